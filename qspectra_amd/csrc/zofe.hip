// Classical RK4 for the ZOFE master equation (gfx950), optionally driven by
// classical fields.  The equation of qspectra/dynamics/zofe.py:121-225 for
// the density matrix rho (N x N) and the auxiliary operators O[p, s]
// (pseudomode p, site s), with L_s the coupling operators (the negated
// system-bath couplings), Osum_s = sum_p O[p, s]:
//     a      = sum_s L_s^+ Osum_s,           b = -i H - a
//     c      = sum_s L_s rho Osum_s^+,       d = b rho + c
//     f      = rho (i H - a^+) + sum_s Osum_s rho L_s^+          (default)
//              rho b^+ + sum_s Osum_s rho L_s^+                   (ham_hermit)
//              rho (i H - a^+) + c^+                             (rho_hermit)
//              d^+                                               (both)
//     rho'   = unit (d + f)
//     O'[p,s]= unit (Gamma[p,s] L_s - w[p,s] O[p,s] + b O[p,s] - O[p,s] b)
// plus, for field terms, sum_i f_i(t) [V_i, X] on rho and on every O[p, s]
// (the ZOFE commutator of qspectra/dynamics/zofe.py:24-34; f_i = -i E_i, E
// conjugated for '+', qspectra/simulate/eom.py:86-93).
//
// One work-group per right-hand side.  The stage vector (rho and all O) and
// the per-site intermediates (Osum_s, L_s rho, Osum_s rho, L_s^+ Osum_s,
// L_s rho Osum_s^+, Osum_s rho L_s^+, b, i H - a^+ and be = unit b +
// sum_i f_i V_i) live in LDS (the operators are read through the cache).
// Per stage, in phases separated by barriers and split into per-site items
// so that no item loops longer than max(N, S, P): (1) Osum; (2) the three
// per-site products; (3) the two per-site triple products, and a summed
// over sites (stored as b, i H - a^+ and be); (4) the derivative of every
// owned element and its RK4 update into the workspace; (5) the next stage
// vector copied into LDS.  The O derivative is unit (Gamma L - w O) +
// be O - O be (the field commutators folded into be).  Thread t owns the
// elements t, t + NT, ...; their state y, RK4 accumulator and next stage
// value sit in a workspace slice of the right-hand side, read and written by
// the owner only (L2 resident), the next element's entries loaded while the
// current one is computed.  The host state layout is the reference's
// (vec(rho) then vec(O) of shape (P, S, N, N), both column-major); in LDS
// rho and each O[p, s] are row-major N x N blocks, O ordered p-major.

#include "qsx_common.h"

#include <algorithm>

namespace qsx {
namespace {

constexpr int kZofeMaxFields = 4;

struct ZofeArgs {
  int N, S, P, size, flags, nfield, K, R, apply;
  double unit;
  const double2* H;       // [B|1][N][N] rotating-frame H (not multiplied by unit)
  int64_t strideH;
  const double2* L;       // [B|1][S][N][N] coupling operators L_s
  int64_t strideL;
  const double2* G;       // [B|1][P][S] Gamma = Omega^2 huang
  const double2* W;       // [B|1][P][S] w = i Omega + gamma
  int64_t strideG;
  const double2* V;       // [B|1][nfield][N][N] dipole operators (fields)
  int64_t strideV;
  const double2* F;       // [B|1][nF][3][nfield] field values at the stage times
  int64_t strideF, nF;
  const double2* proj;    // [B|1][K][N*N] rows on vec(rho) (column-major); null: full state
  int64_t strideP;
};

__constant__ double kZW[4] = {1.0, 2.0, 2.0, 1.0};
__constant__ double kZC[3] = {0.5, 0.5, 1.0};

__device__ inline double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
__device__ inline void cfmad(double2& acc, double2 a, double2 b) {
  acc.x = fma(a.x, b.x, acc.x);
  acc.x = fma(-a.y, b.y, acc.x);
  acc.y = fma(a.x, b.y, acc.y);
  acc.y = fma(a.y, b.x, acc.y);
}

// reference index (column-major vec of rho, then of O[p][s][i][j] with p
// fastest) of internal element e (rho row-major, then O[p*S+s] row-major)
__device__ inline int zofe_ref_index(int e, int N, int S, int P) {
  const int N2 = N * N;
  if (e < N2) return (e / N) + N * (e % N);
  const int r = e - N2, ps = r / N2, ij = r % N2;
  const int i = ij / N, j = ij % N, p = ps / S, s = ps % S;
  return N2 + p + P * (s + S * (i + N * j));
}

// LDS of a stage work-group (row-major N x N blocks)
struct ZofeLds {
  double2* z;    // [size] stage vector: rho, then O[p * S + s]
  double2* Os;   // [S][N2] sum over pseudomodes
  double2* T1;   // [S][N2] L_s rho
  double2* T2;   // [S][N2] Osum_s rho
  double2* U;    // [S][N2] L_s^+ Osum_s
  double2* X1;   // [S][N2] L_s rho Osum_s^+
  double2* X2;   // [S][N2] Osum_s rho L_s^+
  double2* bm;   // [N2]    b = -i H - a
  double2* gm;   // [N2]    i H - a^+
  double2* be;   // [N2]    unit b + sum_i f_i V_i (the O blocks' commutator operator)
  double2* fb;   // [2][3 * kZofeMaxFields] field values
};

__device__ inline ZofeLds zofe_lds(unsigned char* smem, int N, int S, int size) {
  const int N2 = N * N, SN2 = S * N2;
  ZofeLds l;
  l.z = reinterpret_cast<double2*>(smem);
  l.Os = l.z + size;
  l.T1 = l.Os + SN2;
  l.T2 = l.T1 + SN2;
  l.U = l.T2 + SN2;
  l.X1 = l.U + SN2;
  l.X2 = l.X1 + SN2;
  l.bm = l.X2 + SN2;
  l.gm = l.bm + N2;
  l.be = l.gm + N2;
  l.fb = l.be + N2;
  return l;
}

// Phases (1)-(3) of a stage at stage input l.z: Osum; the per-site products
// L rho, Osum rho, L^+ Osum; the triple products, a = sum_s L_s^+ Osum_s and
// b, i H - a^+ and be = unit b + sum_i f_i V_i.  Every sum over sites or pseudomodes is split
// into per-site items, so no item loops longer than max(N, S, P).  Ends
// after a barrier.
template <int NT>
__device__ __forceinline__ void zofe_prepare(const ZofeArgs& a, const ZofeLds& l,
                                             const double2* Hb, const double2* Lb,
                                             const double2* Vb, const double2* fs, int tid) {
  const int N = a.N, S = a.S, P = a.P, N2 = N * N, SN2 = S * N2;
  const double2* rho = l.z;
  for (int it = tid; it < SN2; it += NT) {             // (1) Osum
    const int s = it / N2, ij = it % N2;
    double2 v = make_double2(0.0, 0.0);
    for (int p = 0; p < P; ++p) v = cadd(v, l.z[N2 + (p * S + s) * N2 + ij]);
    l.Os[it] = v;
  }
  __syncthreads();
  for (int it = tid; it < 3 * SN2; it += NT) {         // (2) L rho, Osum rho, L^+ Osum
    const int which = it / SN2, w = it % SN2;
    const int s = w / N2, i = (w % N2) / N, k = w % N;
    const double2* Ls = Lb + s * N2;
    const double2* Oss = l.Os + s * N2;
    double2 v = make_double2(0.0, 0.0);
    if (which == 0) {
      for (int j = 0; j < N; ++j) cfmad(v, Ls[i * N + j], rho[j * N + k]);
      l.T1[w] = v;
    } else if (which == 1) {
      for (int j = 0; j < N; ++j) cfmad(v, Oss[i * N + j], rho[j * N + k]);
      l.T2[w] = v;
    } else {
      for (int j = 0; j < N; ++j) cfmad(v, cconj(Ls[j * N + i]), Oss[j * N + k]);
      l.U[w] = v;
    }
  }
  __syncthreads();
  for (int it = tid; it < 2 * SN2 + N2; it += NT) {    // (3) X1, X2, b, i H - a^+, be
    if (it < 2 * SN2) {
      const int which = it / SN2, w = it % SN2;
      const int s = w / N2, i = (w % N2) / N, j = w % N;
      double2 v = make_double2(0.0, 0.0);
      if (which == 0) {                                   // (L rho)(Osum)^+
        for (int k = 0; k < N; ++k)
          cfmad(v, l.T1[s * N2 + i * N + k], cconj(l.Os[s * N2 + j * N + k]));
        l.X1[w] = v;
      } else {                                            // (Osum rho) L^+
        for (int k = 0; k < N; ++k)
          cfmad(v, l.T2[s * N2 + i * N + k], cconj(Lb[(s * N + j) * N + k]));
        l.X2[w] = v;
      }
    } else {
      const int ik = it - 2 * SN2, i = ik / N, k = ik % N;
      double2 v = make_double2(0.0, 0.0);
      for (int s = 0; s < S; ++s) v = cadd(v, l.U[s * N2 + ik]);     // a_ik
      const double2 hh = Hb[ik], hk = Hb[k * N + i];
      const double2 bik = make_double2(hh.y - v.x, -hh.x - v.y);     // -i H_ik - a_ik
      l.bm[ik] = bik;
      l.gm[k * N + i] = make_double2(-hk.y - v.x, hk.x + v.y);      // i H_ki - conj(a_ik)
      double2 e = make_double2(a.unit * bik.x, a.unit * bik.y);
      for (int fi = 0; fi < a.nfield; ++fi) e = cadd(e, cmul(fs[fi], Vb[fi * N2 + ik]));
      l.be[ik] = e;
    }
  }
  __syncthreads();
}

// d rho_ij / dt (element e = i N + j of the row-major rho), with the field
// terms; needs the intermediates of zofe_prepare.
__device__ __forceinline__ double2 zofe_rho_derivative(const ZofeArgs& a, const ZofeLds& l,
                                                       const double2* Vb, const double2* fs,
                                                       int e) {
  const int N = a.N, S = a.S, N2 = N * N;
  const bool ham_h = a.flags & 1, rho_h = a.flags & 2;
  const double2* rho = l.z;
  const int i = e / N, j = e % N;
  double2 d = make_double2(0.0, 0.0), f = make_double2(0.0, 0.0);
  if (rho_h && ham_h) {                                 // f = d^+
    double2 dt = make_double2(0.0, 0.0);
    for (int k = 0; k < N; ++k) cfmad(dt, l.bm[j * N + k], rho[k * N + i]);
    for (int s = 0; s < S; ++s) dt = cadd(dt, l.X1[s * N2 + j * N + i]);
    f = cconj(dt);
  } else if (ham_h) {                                   // rho b^+
    for (int k = 0; k < N; ++k) cfmad(f, rho[i * N + k], cconj(l.bm[j * N + k]));
  } else {                                              // rho (i H - a^+)
    for (int k = 0; k < N; ++k) cfmad(f, rho[i * N + k], l.gm[k * N + j]);
  }
  if (!rho_h) {                                         // + sum_s Osum rho L^+
    for (int s = 0; s < S; ++s) f = cadd(f, l.X2[s * N2 + e]);
  } else if (!ham_h) {                                  // + c^+_ij = conj(c_ji)
    double2 cc = make_double2(0.0, 0.0);
    for (int s = 0; s < S; ++s) cc = cadd(cc, l.X1[s * N2 + j * N + i]);
    f = cadd(f, cconj(cc));
  }
  for (int k = 0; k < N; ++k) cfmad(d, l.bm[i * N + k], rho[k * N + j]);
  for (int s = 0; s < S; ++s) d = cadd(d, l.X1[s * N2 + e]);
  double2 v = cadd(d, f);
  v = make_double2(a.unit * v.x, a.unit * v.y);
  for (int fi = 0; fi < a.nfield; ++fi) {               // f_i [V_i, rho]
    const double2* Vi = Vb + fi * N2;
    double2 cm = make_double2(0.0, 0.0);
    for (int k = 0; k < N; ++k) {
      cfmad(cm, Vi[i * N + k], rho[k * N + j]);
      const double2 t = cmul(rho[i * N + k], Vi[k * N + j]);
      cm.x -= t.x;
      cm.y -= t.y;
    }
    v = cadd(v, cmul(fs[fi], cm));
  }
  return v;
}

// RK4 bookkeeping of one element: returns the next stage value, updates
// the accumulator an (stages 0-2) or the state yv (stage 3).
__device__ __forceinline__ double2 zofe_rk4(double2 v, double2& yv, double2& an, int st,
                                            double h) {
  const double2 acc = caxpy(kZW[st] * h / 6.0, v, st == 0 ? yv : an);
  if (st < 3) {
    an = acc;
    return caxpy(kZC[st] * h, v, yv);
  }
  yv = acc;
  return acc;
}

// Saves of the state in l.z at save point s: the projections of vec(rho) or
// the whole state (reference layout).
template <int NT>
__device__ __forceinline__ void zofe_save(const ZofeArgs& a, const ZofeLds& l,
                                          const double2* Pb, double2* ob, int s, int tid,
                                          bool& bad) {
  const int N = a.N, N2 = N * N;
  if (Pb) {
    for (int k = tid; k < a.K; k += NT) {
      double2 v = make_double2(0.0, 0.0);
      for (int e = 0; e < N2; ++e) cfmad(v, Pb[(int64_t)k * N2 + (e % N) * N + e / N], l.z[e]);
      ob[(int64_t)s * a.K + k] = v;
      if (!cfinite(v)) bad = true;
    }
  } else {
    for (int e = tid; e < a.size; e += NT) {
      const double2 v = l.z[e];
      ob[(int64_t)s * a.size + zofe_ref_index(e, N, a.S, a.P)] = v;
      if (!cfinite(v)) bad = true;
    }
  }
}

// Per-element kernel (any N): thread t owns the elements t, t + NT, ...;
// their state y, RK4 accumulator and next stage value sit in a workspace
// slice of the right-hand side, read and written by the owner only.
template <int NT>
__global__ __launch_bounds__(NT) void zofe_kernel(ZofeArgs a, const double2* __restrict__ y0,
                                                  const int* __restrict__ nsub,
                                                  const double* __restrict__ hs, int nsave,
                                                  double2* __restrict__ out,
                                                  double2* __restrict__ work,
                                                  int* __restrict__ status) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int N = a.N, S = a.S, P = a.P, N2 = N * N, size = a.size;
  const ZofeLds l = zofe_lds(smem, N, S, size);
  const int tid = threadIdx.x;
  const int r = blockIdx.x, b = blockIdx.y;
  const double2* Hb = a.H + (int64_t)b * a.strideH;
  const double2* Lb = a.L + (int64_t)b * a.strideL;
  const double2* Gb = a.G + (int64_t)b * a.strideG;
  const double2* Wb = a.W + (int64_t)b * a.strideG;
  const double2* Vb = a.V ? a.V + (int64_t)b * a.strideV : nullptr;
  const double2* Fb = a.F ? a.F + (int64_t)b * a.strideF : nullptr;
  const int nfld = a.nfield;
  const bool loader = tid < 3 * nfld;

  const double2* yb0 = y0 + ((int64_t)b * a.R + r) * size;
  double2* yw = work + ((int64_t)b * a.R + r) * 3 * size;   // state y
  double2* aw = yw + size;                                  // RK4 accumulator
  double2* zw = aw + size;                                  // next stage value
  for (int e = tid; e < size; e += NT) {
    const double2 v = yb0[zofe_ref_index(e, N, S, P)];
    yw[e] = v;
    l.z[e] = v;
  }
  if (loader && a.nF > 0) l.fb[tid] = Fb[tid];
  __syncthreads();

  auto stage = [&](const double2* fs, int st, double h) {
    zofe_prepare<NT>(a, l, Hb, Lb, Vb, fs, tid);
    // the workspace entries of the next owned element are loaded while the
    // current one is computed
    double2 y_next = make_double2(0.0, 0.0), a_next = make_double2(0.0, 0.0);
    if (!a.apply && tid < size) {
      y_next = yw[tid];
      a_next = st == 0 ? y_next : aw[tid];
    }
    for (int e = tid; e < size; e += NT) {                 // (4) owned elements
      double2 yv = y_next, an = a_next;
      if (!a.apply && e + NT < size) {
        y_next = yw[e + NT];
        a_next = st == 0 ? y_next : aw[e + NT];
      }
      double2 v;
      if (e < N2) {
        v = zofe_rho_derivative(a, l, Vb, fs, e);
      } else {
        const int rr = e - N2, ps = rr / N2, ij = rr % N2, s = ps % S;
        const int i = ij / N, j = ij % N;
        const double2* X = l.z + N2 + ps * N2;
        const double2 g = cmul(Gb[ps], Lb[s * N2 + ij]), wx = cmul(Wb[ps], X[ij]);
        v = make_double2(a.unit * (g.x - wx.x), a.unit * (g.y - wx.y));
        for (int k = 0; k < N; ++k) {                       // be X - X be
          cfmad(v, l.be[i * N + k], X[k * N + j]);
          const double2 t = cmul(X[i * N + k], l.be[k * N + j]);
          v.x -= t.x;
          v.y -= t.y;
        }
      }
      if (a.apply) {                                        // derivative only
        zw[e] = v;
        continue;
      }
      zw[e] = zofe_rk4(v, yv, an, st, h);
      if (st < 3) aw[e] = an;
      else yw[e] = yv;
    }
    __syncthreads();                                       // all reads of z done
  };

  int64_t g = 0;
  bool bad = false;
  if (a.apply) {                                           // out = F(y0), no fields
    stage(l.fb, 0, 0.0);
    double2* ob = out + ((int64_t)b * a.R + r) * size;
    for (int e = tid; e < size; e += NT) ob[zofe_ref_index(e, N, S, P)] = zw[e];
    return;
  }
  double2* ob = out + ((int64_t)b * a.R + r) * nsave * (a.proj ? a.K : size);
  const double2* Pb = a.proj ? a.proj + (int64_t)b * a.strideP : nullptr;
  const int vz = opaque_zero();
  int n_next = nsub[vz];
  double h_next = hs[vz];
  for (int s = 0; s < nsave; ++s) {
    const int n = max(wave_uniform(n_next), 0);
    const double h = wave_uniform(h_next);
    if (s + 1 < nsave) {
      n_next = nsub[s + 1 + vz];
      h_next = hs[s + 1 + vz];
    }
    for (int step = 0; step < n; ++step, ++g) {
      if (nfld > 0 && g >= a.nF) {
        if (tid == 0) status[0] = 2;
        return;
      }
      double2 fnext = make_double2(0.0, 0.0);
      if (loader) fnext = Fb[(g + 1 < a.nF ? g + 1 : g) * 3 * nfld + tid];
      const double2* fc = l.fb + (g & 1) * 3 * kZofeMaxFields;
      for (int st = 0; st < 4; ++st) {
        const int ti = st == 0 ? 0 : (st == 3 ? 2 : 1);
        stage(fc + ti * nfld, st, h);                      // field values in LDS
        for (int e = tid; e < size; e += NT) l.z[e] = zw[e];
        if (st == 3 && loader) l.fb[((g + 1) & 1) * 3 * kZofeMaxFields + tid] = fnext;
        __syncthreads();
      }
    }
    zofe_save<NT>(a, l, Pb, ob, s, tid, bad);
  }
  if (bad) status[0] = 1;
}

// Column form for diagonal coupling operators (site occupations; kZofeDiagonal)
// and N <= 8.  C neighbouring columns of O[m] (m = p S + s) belong to one
// thread, which keeps their state y and RK4 accumulator in registers through
// the whole launch: a stage moves nothing through the workspace and needs no
// copy back into LDS.  Per stage, three barriers:
//   (1) Osum, and from it in the same phase a = sum_s L_s^+ Osum_s (only the
//       sites that occupy the row), b, i H - a^+ and be;
//   (2) per thread  Gamma L - w X + be X - X be  of its columns: row i of X
//       is read once for all C columns, the entries of be's column k are
//       spread over the 16 lanes of each row and broadcast from there (DPP),
//       so a column costs N^2 / C + 4 N LDS reads of 16 B where the
//       element-wise kernel takes 4 N per element; eight lanes derive each
//       element of rho, one term of its sums per lane, those over sites again
//       only over the sites that couple;
//   (3) the RK4 update written back into LDS.
// Measured (7 sites, 16 modes, one right-hand side): 7.7 us per stage (kernel
// trace: 100 steps 3.09 ms), with the element-wise kernel 16.2 us (its LDS reads,
// phases and workspace round trips).  The 784 FP64 multiply-adds of a thread in
// (2), two wavefronts per SIMD, are 2.6 us of issue at 2.4 GHz; the rest is
// latency: LDS reads and broadcasts between them, (1), (3) and the barriers.
// LDS: a thread's columns are NC apart and the blocks start 16 banks apart
// (4 entries modulo 16), so that the 16 lanes of an access, NC neighbouring
// columns of 16 / NC blocks, meet different banks.
constexpr int kZofeDiagonal = 4;                            // flag bit
constexpr int kColumnThreads = 512;

__host__ __device__ constexpr int zofe_stride(int N) {
  return (N * N + 11) / 16 * 16 + 4;
}

inline size_t zofe_column_lds_bytes(int N, int S, int P) {
  const size_t N2 = (size_t)N * N;
  return ((1 + (size_t)P * S) * zofe_stride(N) + S * N2 + 7 * N2 + (size_t)S * N +
          2 * (size_t)P * S + 2 * 3 * kZofeMaxFields) * sizeof(double2) +
         (size_t)N * (S + 1) * sizeof(int);
}

// d[c][i] += be[i][k] x[c] for i = I .. N - 1, be[i][k] held by lane i
template <int I, int N, int C>
struct ColumnFma {
  static __device__ __forceinline__ void run(double2 (&d)[C][N], double2 bk, const double2 (&x)[C]) {
    const double2 bi = make_double2(row_lane<I>(bk.x), row_lane<I>(bk.y));
#pragma unroll
    for (int c = 0; c < C; ++c) cfmad(d[c][I], bi, x[c]);
    ColumnFma<I + 1, N, C>::run(d, bk, x);
  }
};
template <int N, int C>
struct ColumnFma<N, N, C> {
  static __device__ __forceinline__ void run(double2 (&)[C][N], double2, const double2 (&)[C]) {}
};

// FIELDS: with field terms (their own kernel: what they hold in registers
// would not fit beside the columns).
template <int N, int C, bool FIELDS>
__global__ __launch_bounds__(kColumnThreads) void zofe_column_kernel(
    ZofeArgs a, const double2* __restrict__ y0, const int* __restrict__ nsub,
    const double* __restrict__ hs, int nsave, double2* __restrict__ out,
    int* __restrict__ status) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int N2 = N * N, BS = zofe_stride(N), NC = (N + C - 1) / C;
  const int S = a.S, PS = a.P * a.S, size = a.size, nt = blockDim.x;
  double2* rho = reinterpret_cast<double2*>(smem);          // [BS] density matrix
  double2* O = rho + BS;                                    // [PS][BS] auxiliary operators
  double2* Os = O + PS * BS;                                // [S][N2] sum over pseudomodes
  double2* bm = Os + S * N2;                                // [N2] b = -i H - a
  double2* gm = bm + N2;                                    // [N2] i H - a^+
  double2* be = gm + N2;                                    // [N2] unit b + sum_i f_i V_i
  double2* Hl = be + N2;                                    // [N2] H
  double2* dr = Hl + N2;                                    // [N2] derivative of rho,
  double2* yr = dr + N2;                                    // [N2] its state
  double2* sr = yr + N2;                                    // [N2] and its RK4 sum
  double2* Ld = sr + N2;                                    // [S][N] diagonals of L_s
  double2* gw = Ld + S * N;                                 // [2][PS] unit Gamma, unit w
  double2* fb = gw + 2 * PS;                                // [2][3 * kZofeMaxFields]
  int* sites = reinterpret_cast<int*>(fb + 2 * 3 * kZofeMaxFields);   // [N][1 + S]: how many
                                                            // sites couple to a state, and which
  const int tid = threadIdx.x, lane = tid & 63;
  const int r = blockIdx.x, b = blockIdx.y;
  const double2* Hb = a.H + (int64_t)b * a.strideH;
  const double2* Lb = a.L + (int64_t)b * a.strideL;
  const double2* Vb = a.V ? a.V + (int64_t)b * a.strideV : nullptr;
  const double2* Fb = a.F ? a.F + (int64_t)b * a.strideF : nullptr;
  const int nfld = FIELDS ? a.nfield : 0;
  const bool loader = FIELDS && tid < 3 * nfld;
  const bool ham_h = a.flags & 1, rho_h = a.flags & 2;

  // the thread's columns j0, j0 + NC, ... of O[m].  Lanes and slots without a
  // column repeat the last one, with the same values: every lane takes part
  // in the broadcasts, and the stages have no branch that the registers of
  // all columns would have to live across.
  const int t = min(tid, PS * NC - 1), m = t / NC, j0 = t % NC, s = m % S;
  const double2* X = O + m * BS;
  // element (ri, rj) of rho and of b belongs to eight lanes, each with one
  // term k of its sums (nt >= 8 N^2)
  const int er = min(tid >> 3, N2 - 1), ri = er / N, rj = er % N;
  const int kl = tid & 7, kk = min(kl, N - 1);
  const bool lead = kl == 0 && (tid >> 3) < N2;
  // reference index -> LDS entry
  auto entry = [&](int e) { return e < N2 ? e : BS + (e - N2) / N2 * BS + (e - N2) % N2; };
  const double2* yb0 = y0 + ((int64_t)b * a.R + r) * size;
#pragma unroll 1
  for (int e = tid; e < size; e += nt) rho[entry(e)] = yb0[zofe_ref_index(e, N, S, a.P)];
#pragma unroll 1
  for (int e = tid; e < S * N; e += nt) Ld[e] = Lb[(int64_t)(e / N) * N2 + e % N * (N + 1)];
#pragma unroll 1
  for (int e = tid; e < N2; e += nt) Hl[e] = Hb[e];
  if (loader && a.nF > 0) fb[tid] = Fb[tid];
  __syncthreads();
#pragma unroll 1
  for (int e = tid; e < 2 * PS; e += nt) {
    const double2 v = e < PS ? a.G[(int64_t)b * a.strideG + e]
                             : a.W[(int64_t)b * a.strideG + e - PS];
    gw[e] = make_double2(a.unit * v.x, a.unit * v.y);
  }
  if (tid < N) {
    int cnt = 0;
    for (int q = 0; q < S; ++q) {
      const double2 l = Ld[q * N + tid];
      if (l.x != 0.0 || l.y != 0.0) sites[tid * (1 + S) + ++cnt] = q;
    }
    sites[tid * (1 + S)] = cnt;
  }
  __syncthreads();      // every wavefront reads the lists in the first stage's (1)
  double2 y[C][N], acc[C][N];
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int i = 0; i < N; ++i) y[c][i] = acc[c][i] = X[i * N + min(j0 + c * NC, N - 1)];
  if (tid < N2) yr[tid] = sr[tid] = rho[tid];

  // term k of (sum_s L_s rho Osum_s^+)_ij, (sum_s Osum_s rho L_s^+)_ij, (b rho)_ij
  auto c_term = [&](int i, int j, int k) {
    double2 v = make_double2(0.0, 0.0);
    const int* list = sites + i * (1 + S);
#pragma unroll 1
    for (int n = list[0]; n > 0; --n) {
      const int q = list[n];
      cfmad(v, cmul(Ld[q * N + i], rho[i * N + k]), cconj(Os[q * N2 + j * N + k]));
    }
    return v;
  };
  auto e_term = [&](int i, int j, int k) {
    double2 v = make_double2(0.0, 0.0);
    const int* list = sites + j * (1 + S);
#pragma unroll 1
    for (int n = list[0]; n > 0; --n) {
      const int q = list[n];
      cfmad(v, cmul(cconj(Ld[q * N + j]), Os[q * N2 + i * N + k]), rho[k * N + j]);
    }
    return v;
  };
  auto b_rho = [&](int i, int j, int k) { return cmul(bm[i * N + k], rho[k * N + j]); };
  auto sum8 = [&](double2 v) { return make_double2(seg_sum<8>(v.x), seg_sum<8>(v.y)); };

  int64_t g = 0;
  bool bad = false;
  double2* ob = out + ((int64_t)b * a.R + r) * nsave * (a.proj ? a.K : size);
  const double2* Pb = a.proj ? a.proj + (int64_t)b * a.strideP : nullptr;
  const int vz = opaque_zero();
  int n = 0, step = 0, sv = -1, st = 0;
  double h = 0.0, h6 = 0.0;
  int n_next = nsub[vz];
  double h_next = hs[vz];
  double2 fnext = make_double2(0.0, 0.0);
  // one loop over all stages (nested loops over saves, steps and stages would
  // keep copies of the register arrays for each of their levels)
#pragma unroll 1
  for (;;) {
    while (step == n) {                                     // a save point is reached
      if (sv >= 0) {
        if (Pb) {                                               // save
#pragma unroll 1
          for (int k = tid; k < a.K; k += nt) {
            double2 v = make_double2(0.0, 0.0);
#pragma unroll 1
            for (int e = 0; e < N2; ++e) cfmad(v, Pb[(int64_t)k * N2 + (e % N) * N + e / N], rho[e]);
            ob[(int64_t)sv * a.K + k] = v;
            if (!cfinite(v)) bad = true;
          }
        } else {
#pragma unroll 1
          for (int e = tid; e < size; e += nt) {
            const double2 v = rho[entry(e)];
            ob[(int64_t)sv * size + zofe_ref_index(e, N, S, a.P)] = v;
            if (!cfinite(v)) bad = true;
          }
        }
      }
      if (++sv == nsave) {
        if (bad) status[0] = 1;
        return;
      }
      step = 0;
      n = max(wave_uniform(n_next), 0);
      h = wave_uniform(h_next);
      h6 = h / 6.0;
      if (sv + 1 < nsave) {
        n_next = nsub[sv + 1 + vz];
        h_next = hs[sv + 1 + vz];
      }
    }
    if (st == 0) {
      if (FIELDS && g >= a.nF) {
        if (tid == 0) status[0] = 2;
        return;
      }
      if (loader) fnext = Fb[(g + 1 < a.nF ? g + 1 : g) * 3 * nfld + tid];
    }
    const double2* fc = fb + (g & 1) * 3 * kZofeMaxFields;
    const double2* fs = fc + (st == 0 ? 0 : (st == 3 ? 2 : 1)) * nfld;
    // (1) Osum; b, i H - a^+ and be
#pragma unroll 1
    for (int it = tid; it < S * N2; it += nt) {
      const int q = it / N2, ij = it - q * N2;
      double2 v = make_double2(0.0, 0.0);
#pragma unroll 8
      for (int p = 0; p < a.P; ++p) v = cadd(v, O[(p * S + q) * BS + ij]);
      Os[it] = v;
    }
    {
      const int* list = sites + ri * (1 + S);
      double2 v = make_double2(0.0, 0.0);                   // a_ij, pseudomodes kl, kl + 8, ..
#pragma unroll 1
      for (int n = list[0]; n > 0; --n) {
        const int q = list[n];
        double2 u = make_double2(0.0, 0.0);
#pragma unroll 2
        for (int p = kl; p < a.P; p += 8) u = cadd(u, O[(p * S + q) * BS + er]);
        cfmad(v, cconj(Ld[q * N + ri]), u);
      }
      v = sum8(v);
      if (lead) {
        const double2 hh = Hl[er], hk = Hl[rj * N + ri];
        const double2 bik = make_double2(hh.y - v.x, -hh.x - v.y);       // -i H_ij - a_ij
        bm[er] = bik;
        gm[rj * N + ri] = make_double2(-hk.y - v.x, hk.x + v.y);         // i H_ji - conj(a_ij)
        double2 e = make_double2(a.unit * bik.x, a.unit * bik.y);
#pragma unroll 1
        for (int fi = 0; fi < nfld; ++fi) e = cadd(e, cmul(fs[fi], Vb[fi * N2 + er]));
        be[er] = e;
      }
    }
    __syncthreads();
    // (2) derivatives
    {
      double2 f;
      if (rho_h && ham_h) {                                 // d^+
        f = cconj(cadd(b_rho(rj, ri, kk), c_term(rj, ri, kk)));
      } else {                                              // rho b^+ or rho (i H - a^+)
        f = cmul(rho[ri * N + kk], ham_h ? cconj(bm[rj * N + kk]) : gm[kk * N + rj]);
        f = cadd(f, rho_h ? cconj(c_term(rj, ri, kk)) : e_term(ri, rj, kk));
      }
      const double2 v = cadd(cadd(b_rho(ri, rj, kk), c_term(ri, rj, kk)), f);
      double2 w = make_double2(a.unit * v.x, a.unit * v.y);
#pragma unroll 1
      for (int fi = 0; fi < nfld; ++fi) {                   // f_i [V_i, rho]
        const double2* Vi = Vb + fi * N2;
        const double2 p = cmul(Vi[ri * N + kk], rho[kk * N + rj]);
        const double2 q = cmul(rho[ri * N + kk], Vi[kk * N + rj]);
        w = cadd(w, cmul(fs[fi], make_double2(p.x - q.x, p.y - q.y)));
      }
      w = sum8(kl < N ? w : make_double2(0.0, 0.0));
      if (lead) dr[er] = w;
    }
    double2 d[C][N];
    const double2 gam = gw[m], wm = gw[PS + m];
    int jj = j0;       // opaque: the selects below stay in the stage
    asm volatile("" : "+v"(jj));
#pragma unroll
    for (int c = 0; c < C; ++c) {                           // Gamma L
      const int j = min(jj + c * NC, N - 1);
      const double2 src = cmul(gam, Ld[s * N + j]);
#pragma unroll
      for (int i = 0; i < N; ++i) d[c][i] = i == j ? src : make_double2(0.0, 0.0);
    }
    const int bl = min(lane & 15, N - 1) * N;
#pragma unroll 1
    for (int k = 0; k < N; ++k) {
      double2 x[C], q[C], xr[N];
      const double2 bk = be[bl + k];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int j = min(j0 + c * NC, N - 1);
        x[c] = X[k * N + j];
        q[c] = be[k * N + j];
      }
#pragma unroll
      for (int i = 0; i < N; ++i) xr[i] = X[i * N + k];
      ColumnFma<0, N, C>::run(d, bk, x);              // be X
#pragma unroll
      for (int c = 0; c < C; ++c) {                   // - X (be + w)
        const bool dia = k == min(j0 + c * NC, N - 1);
        q[c] = make_double2(-q[c].x - (dia ? wm.x : 0.0), -q[c].y - (dia ? wm.y : 0.0));
#pragma unroll
        for (int i = 0; i < N; ++i) cfmad(d[c][i], xr[i], q[c]);
      }
    }
    __syncthreads();                                    // all reads of the stage done
    // (3) update: the sum (started from y) and the next stage value; the
    // last stage's sum is the new state.  opaque: one copy of this code
    // for the four stages
    int stage = st;
    asm volatile("" : "+s"(stage));
    const bool last = stage == 3;
    const double wh = stage == 0 || last ? h6 : 2.0 * h6;
    const double ch = last ? 0.0 : (stage == 2 ? h : 0.5 * h);
    auto update = [&](double2 k, double2& yv, double2& sum) {
      sum = caxpy(wh, k, sum);
      yv = make_double2(last ? sum.x : yv.x, last ? sum.y : yv.y);
      return caxpy(ch, k, yv);
    };
    if (tid < N2) rho[tid] = update(dr[tid], yr[tid], sr[tid]);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int i = 0; i < N; ++i)
        O[m * BS + i * N + min(j0 + c * NC, N - 1)] = update(d[c][i], y[c][i], acc[c][i]);
    if (st == 3 && loader) fb[((g + 1) & 1) * 3 * kZofeMaxFields + tid] = fnext;
    __syncthreads();
    st = (st + 1) & 3;
    if (st == 0) {
      ++step;
      ++g;
    }
  }
}

inline size_t zofe_lds_bytes(int N, int S, int size) {
  const size_t N2 = (size_t)N * N;
  return ((size_t)size + 6 * (size_t)S * N2 + 3 * N2 + 2 * 3 * kZofeMaxFields) *
         sizeof(double2);
}

}  // namespace
}  // namespace qsx

static int32_t zofe_launch(int apply,
    int32_t B, int32_t R, int32_t N, int32_t S, int32_t P, const void* H, int64_t strideH,
    const void* L, int64_t strideL, const void* Gamma, const void* w, int64_t strideG,
    int32_t flags, double unit_convert, int32_t nfield, const void* V, int64_t strideV,
    const void* F, int64_t strideF, int64_t nF, const void* y0, const int32_t* nsub,
    const double* h, int32_t nsave, int32_t K, const void* proj, int64_t strideP, void* out,
    void* workspace, int32_t* status, void* stream);


extern "C" int64_t qsx_zofe_workspace_bytes(int32_t B, int32_t R, int32_t N, int32_t S,
                                            int32_t P) {
  if (B < 1 || R < 1 || N < 1 || S < 1 || P < 1) return -1;
  return 3 * (int64_t)B * R * N * N * (1 + (int64_t)P * S) * 16;
}

extern "C" int32_t qsx_zofe_apply(int32_t B, int32_t R, int32_t N, int32_t S, int32_t P,
                                  const void* H, int64_t strideH, const void* L,
                                  int64_t strideL, const void* Gamma, const void* w,
                                  int64_t strideG, int32_t flags, double unit_convert,
                                  const void* y, void* out, void* workspace, void* stream) {
  // the apply launch returns before it reads a schedule or writes a status
  return zofe_launch(1, B, R, N, S, P, H, strideH, L, strideL, Gamma, w, strideG, flags,
                     unit_convert, 0, nullptr, 0, nullptr, 0, 0, y, nullptr, nullptr, 1, 0,
                     nullptr, 0, out, workspace, nullptr, stream);
}

extern "C" int32_t qsx_zofe_propagate(
    int32_t B, int32_t R, int32_t N, int32_t S, int32_t P, const void* H, int64_t strideH,
    const void* L, int64_t strideL, const void* Gamma, const void* w, int64_t strideG,
    int32_t flags, double unit_convert, int32_t nfield, const void* V, int64_t strideV,
    const void* F, int64_t strideF, int64_t nF, const void* y0, const int32_t* nsub,
    const double* h, int32_t nsave, int32_t K, const void* proj, int64_t strideP, void* out,
    void* workspace, int32_t* status, void* stream) {
  return zofe_launch(0, B, R, N, S, P, H, strideH, L, strideL, Gamma, w, strideG, flags,
                     unit_convert, nfield, V, strideV, F, strideF, nF, y0, nsub, h, nsave, K,
                     proj, strideP, out, workspace, status, stream);
}

static int32_t zofe_launch(int apply,
    int32_t B, int32_t R, int32_t N, int32_t S, int32_t P, const void* H, int64_t strideH,
    const void* L, int64_t strideL, const void* Gamma, const void* w, int64_t strideG,
    int32_t flags, double unit_convert, int32_t nfield, const void* V, int64_t strideV,
    const void* F, int64_t strideF, int64_t nF, const void* y0, const int32_t* nsub,
    const double* h, int32_t nsave, int32_t K, const void* proj, int64_t strideP, void* out,
    void* workspace, int32_t* status, void* stream) {
  using namespace qsx;
  QSX_CHECK_ARG(H && L && Gamma && w && y0 && out && workspace &&
                    (apply || (nsub && h && status)),
                "qsx_zofe_propagate: null pointer");
  QSX_CHECK_ARG(B >= 1 && R >= 1 && N >= 1 && S >= 1 && P >= 1 && nsave >= 1 && B <= 65535,
                "qsx_zofe_propagate: bad sizes B=%d R=%d N=%d S=%d P=%d", B, R, N, S, P);
  QSX_CHECK_ARG(nfield >= 0 && nfield <= kZofeMaxFields,
                "qsx_zofe_propagate: %d field terms (0..%d)", nfield, kZofeMaxFields);
  QSX_CHECK_ARG(nfield == 0 || (V && F && nF >= 0 && (strideF == 0 || strideF >= nF * 3 * nfield)),
                "qsx_zofe_propagate: field terms need V and F");
  QSX_CHECK_ARG(K == 0 || (proj && K >= 1), "qsx_zofe_propagate: projection rows need proj");
  const int64_t size64 = (int64_t)N * N * (1 + (int64_t)P * S);
  QSX_CHECK_ARG(size64 <= 8192, "qsx_zofe_propagate: state of %lld elements exceeds 8192",
                (long long)size64);
  const int size = (int)size64;
  const size_t shmem = zofe_lds_bytes(N, S, size);
  QSX_CHECK_ARG(shmem <= 160 * 1024, "qsx_zofe_propagate: %zu bytes of LDS", shmem);
  ZofeArgs a;
  a.N = N;
  a.S = S;
  a.P = P;
  a.size = size;
  a.flags = flags;
  a.nfield = nfield;
  a.K = proj ? K : 0;
  a.R = R;
  a.apply = apply;
  a.unit = unit_convert;
  a.H = (const double2*)H;
  a.strideH = strideH;
  a.L = (const double2*)L;
  a.strideL = strideL;
  a.G = (const double2*)Gamma;
  a.W = (const double2*)w;
  a.strideG = strideG;
  a.V = nfield ? (const double2*)V : nullptr;
  a.strideV = strideV;
  a.F = nfield ? (const double2*)F : nullptr;
  a.strideF = strideF;
  a.nF = nfield ? nF : 0;
  a.proj = (const double2*)proj;
  a.strideP = strideP;
  hipStream_t st = as_stream(stream);
  dim3 grid(R, B);
  // the column form wherever its threads and LDS suffice: 2.1 times as fast
  // as the element-wise kernel at 7 sites and 16 modes (20 steps 615 us for
  // 1300), 1.05 to 3.4 times over 1..8 states and 1..16 modes, one right-hand side
  // or 300.  One column per thread while that takes at most one wavefront per
  // SIMD, two beyond (each row of X then read once for both; one column in 128
  // registers measured 13.2 us per stage, two 7.7).  At 6 and 7 states it
  // holds one work-group per CU (122 and 147 us per 256 right-hand sides and 8
  // steps) where the element-wise kernel with few modes holds up to four: from
  // two to four rounds on that one is taken (8 steps, 1024 right-hand sides, column /
  // element-wise: 6 states, P S = 5, 10, 12, 20: 481 / 290, 487 / 351, 491 / 401,
  // 499 / 467; 7 states, P S = 6: 593 / 451, P S = 12 the column form 1.3 times
  // as fast).
  const int cols = (P * S * N <= 256) ? 1 : 2, need = P * S * ((N + cols - 1) / cols);
  const size_t cshmem = zofe_column_lds_bytes(N, S, P);
  const int64_t groups = (int64_t)R * B;
  const bool crowded = (N == 6 && groups > (P * S <= 5 ? 256 : P * S <= 12 ? 512 : 768) &&
                        P * S <= 20) || (N == 7 && P * S <= 6 && groups > 768);
  if (!apply && (flags & kZofeDiagonal) && N <= 8 && need <= kColumnThreads &&
      cshmem <= 160 * 1024 && !crowded) {
    const int nt = (std::max(need, 8 * N * N) + 63) / 64 * 64;    // <= kColumnThreads
#define QSX_ZOFE_COLUMN(N_, C_)                                                                \
  if (N == N_ && cols == C_) {                                                                 \
    auto kern = nfield ? zofe_column_kernel<N_, C_, true> : zofe_column_kernel<N_, C_, false>; \
    if (cshmem > 64 * 1024)                                                                    \
      QSX_CHECK_HIP(hipFuncSetAttribute((const void*)kern,                                     \
                                        hipFuncAttributeMaxDynamicSharedMemorySize,            \
                                        (int)cshmem));                                         \
    hipLaunchKernelGGL(kern, grid, dim3(nt), cshmem, st, a, (const double2*)y0, nsub, h,       \
                       nsave, (double2*)out, status);                                          \
    QSX_CHECK_HIP(hipGetLastError());                                                          \
    return QSX_OK;                                                                             \
  }
#define QSX_ZOFE_COLUMNS(N_) QSX_ZOFE_COLUMN(N_, 1) QSX_ZOFE_COLUMN(N_, 2)
    QSX_ZOFE_COLUMNS(1) QSX_ZOFE_COLUMNS(2) QSX_ZOFE_COLUMNS(3) QSX_ZOFE_COLUMNS(4)
    QSX_ZOFE_COLUMNS(5) QSX_ZOFE_COLUMNS(6) QSX_ZOFE_COLUMNS(7) QSX_ZOFE_COLUMNS(8)
#undef QSX_ZOFE_COLUMNS
#undef QSX_ZOFE_COLUMN
  }
#define QSX_ZOFE(NT_, LIMIT_)                                                                  \
  if (size <= LIMIT_) {                                                                        \
    auto kern = zofe_kernel<NT_>;                                                              \
    if (shmem > 64 * 1024)                                                                     \
      QSX_CHECK_HIP(hipFuncSetAttribute((const void*)kern,                                     \
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem)); \
    hipLaunchKernelGGL(kern, grid, dim3(NT_), shmem, st, a, (const double2*)y0, nsub, h,       \
                       nsave, (double2*)out, (double2*)workspace, status);                     \
    QSX_CHECK_HIP(hipGetLastError());                                                          \
    return QSX_OK;                                                                             \
  }
  QSX_ZOFE(256, 1024)
  QSX_ZOFE(1024, 8192)
#undef QSX_ZOFE
  set_error("qsx_zofe_propagate: no kernel for %d elements", size);
  return QSX_EINVAL;
}
