// Propagation y_p = P y_{p-1} of small blocks (M <= 16) and its reverse mode,
// parallel in time (gfx950).
//
// A step-by-step recursion of N products leaves the chip waiting on one
// dependent chain per right-hand side.  The N steps are cut into np pieces of
// `len` steps (a power of two); with Q = P^len (squarings)
//   forward   the piece starts y_{j len} = Q^j y_0 (a chain of np products),
//             then every piece steps on its own and writes its save points;
//   reverse   every piece first forms its own contribution mu_j to the
//             cotangent at its start (from the save points inside it), the
//             chain Lam_{j-1} = Q^H Lam_j + mu_j gives the cotangent at the
//             end of every piece, and every piece then recomputes its states
//             (into LDS) and walks back from there, accumulating its part of
//             dLoss/dP; the parts are added in order.
// The chain is np + len products instead of N; the values are those of the
// step-by-step recursion up to the rounding of P^len.
//
// Lanes: a piece per 16-lane row of a wavefront (four per wavefront), lane i
// holding row i of the operator and entry i of the vector, entry j broadcast
// to the row by DPP: a product is 2 M moves and 4 M FMAs for four pieces, with
// no LDS exchange, shuffle or barrier.
//
// Measured (512 right-hand sides of M = 7, 4095 steps, signals, pieces of 64):
// forward 0.12 ms (power, chain, pieces) where the step-by-step stepper takes
// 1.31 ms plus 0.37 ms for the projection; reverse 0.45 ms (contributions
// 0.09, chain 0.03, walk back 0.32) where the checkpointed recursion takes
// 4.98 ms.  The walk back is bound by its latency at the five work-groups per
// CU that the piece states leave in LDS.
//
// Schedule tables (device, int32): pos[s] the step after which save s is
// taken (non-decreasing, the last equal to or below N), first[j] for
// j < np the number of saves with pos <= j len, first[np] = nsave.

#include "qsx_common.h"

#include <algorithm>
#include <type_traits>

namespace qsx {
namespace {

constexpr int kMaxM = 16;
constexpr int kMaxLen = 64;              // states of a piece held in LDS

__device__ inline double2 conj2(double2 a) { return make_double2(a.x, -a.y); }

// acc[j & 3] += row[j] z_j for j = J .. M - 1, z_j held by lane j of the row
template <int J, int M>
struct Dot {
  static __device__ __forceinline__ void run(const double2 (&row)[M], double2 z, double2 (&acc)[4]) {
    const double2 zj = make_double2(row_lane<J>(z.x), row_lane<J>(z.y));
    cfma<double>(acc[J & 3], row[J], zj);
    Dot<J + 1, M>::run(row, z, acc);
  }
};
template <int M>
struct Dot<M, M> {
  static __device__ __forceinline__ void run(const double2 (&)[M], double2, double2 (&)[4]) {}
};
template <int M>
__device__ __forceinline__ double2 row_product(const double2 (&row)[M], double2 z) {
  double2 acc[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) acc[q] = make_double2(0.0, 0.0);
  Dot<0, M>::run(row, z, acc);
  return make_double2((acc[0].x + acc[1].x) + (acc[2].x + acc[3].x),
                      (acc[0].y + acc[1].y) + (acc[2].y + acc[3].y));
}

// Row i of X (CONJ: of X^H) in lane i, zero from lane M on.
template <int M, bool CONJ>
__device__ __forceinline__ void load_row(const double2* __restrict__ X, int i, bool live,
                                         double2 (&row)[M]) {
#pragma unroll
  for (int j = 0; j < M; ++j) {
    double2 v = make_double2(0.0, 0.0);
    if (live && i < M) v = CONJ ? conj2(X[j * M + i]) : X[i * M + j];
    row[j] = v;
  }
}

struct PieceArgs {
  const double2* A;        // [nA][M][M] one-step propagators
  int64_t strideA;         // M*M or 0
  const double2* Q;        // [nA][M][M] A^len
  int R, nrhs;             // right-hand sides per operator, all of them
  int N, len, np, nsave;
  const int* pos;
  const int* first;
  const double2* v;        // [M] signal vector, or null: whole states
};

// Q[b] = A[b]^len: log2(len) squarings, one work-group per operator
__global__ __launch_bounds__(kMaxM * kMaxM) void piece_power_kernel(
    const double2* __restrict__ A, int64_t strideA, int M, int len, double2* __restrict__ Q) {
  __shared__ double2 X[kMaxM][kMaxM + 1];
  const int t = threadIdx.x, i = t / M, j = t % M;
  const bool on = t < M * M;
  const int64_t b = blockIdx.x;
  double2 v = make_double2(0.0, 0.0);
  if (on) v = A[b * strideA + t];
  for (int n = 1; n < len; n *= 2) {
    if (on) X[i][j] = v;
    __syncthreads();
    if (on) {
      v = make_double2(0.0, 0.0);
      for (int k = 0; k < M; ++k) cfma<double>(v, X[i][k], X[k][j]);
    }
    __syncthreads();
  }
  if (on) Q[b * M * M + t] = v;
}

// Injection of save s into lane i's cotangent: gout [nrhs][nsave][M], or
// gout [nrhs][nsave] times conj(v) for a signal.
template <int M, bool SIGNAL>
__device__ __forceinline__ double2 injection(const PieceArgs& a, const double2* __restrict__ gout,
                                             int64_t rhs, int s, int i, double2 vc) {
  if (SIGNAL) return cmul(gout[rhs * a.nsave + s], vc);
  return i < M ? gout[(rhs * a.nsave + s) * M + i] : make_double2(0.0, 0.0);
}

// The chain over pieces: the starts Y[rhs][j] = Q^j y0, or (reverse) the
// cotangents Lam[rhs][j] at the end of piece j from the contributions
// mu[rhs][j], and gy0.
template <int M, bool SIGNAL>
__global__ __launch_bounds__(64) void piece_chain_kernel(
    PieceArgs a, bool reverse, const double2* __restrict__ y0, double2* __restrict__ Y,
    const double2* __restrict__ mu, const double2* __restrict__ gout, double2* __restrict__ Lam,
    double2* __restrict__ gy0) {
  const int g = threadIdx.x >> 4, i = threadIdx.x & 15;
  const int64_t rhs = (int64_t)blockIdx.x * 4 + g;
  const bool live = rhs < a.nrhs, mine = live && i < M;
  const double2* Q = a.Q + (a.strideA ? (live ? rhs / a.R : 0) * M * M : 0);
  const int64_t base = live ? rhs * a.np * M + i : 0;
  double2 row[M];
  if (!reverse) {
    load_row<M, false>(Q, i, live, row);
    double2 y = mine ? y0[rhs * M + i] : make_double2(0.0, 0.0);
    for (int j = 0; j < a.np; ++j) {
      if (mine) Y[base + (int64_t)j * M] = y;
      y = row_product<M>(row, y);
    }
    return;
  }
  load_row<M, true>(Q, i, live, row);
  double2 lam = make_double2(0.0, 0.0);
  double2 next = mine ? mu[base + (int64_t)(a.np - 1) * M] : lam;
  for (int j = a.np - 1; j >= 0; --j) {
    const double2 m = next;
    if (mine && j > 0) next = mu[base + (int64_t)(j - 1) * M];
    if (mine) Lam[base + (int64_t)j * M] = lam;
    lam = cadd(row_product<M>(row, lam), m);
  }
  if (mine) {                                          // saves of y_0 itself
    const double2 vc = SIGNAL ? conj2(a.v[i]) : lam;
    for (int s = 0; s < min(a.first[0], a.nsave); ++s)
      lam = cadd(lam, injection<M, SIGNAL>(a, gout, rhs, s, i, vc));
    if (gy0 != nullptr) gy0[rhs * M + i] = lam;
  }
}

// Forward: the save points of every piece.  SIGNAL: the row after the state's
// rows holds v^T P, so that the signal v . y of a save comes out of the
// product that reaches it (M < 16).
template <int M, bool SIGNAL>
__global__ __launch_bounds__(64) void piece_forward_kernel(PieceArgs a,
                                                           const double2* __restrict__ Y,
                                                           double2* __restrict__ out,
                                                           int* __restrict__ status) {
  const int g = threadIdx.x >> 4, i = threadIdx.x & 15;
  const int64_t id = (int64_t)blockIdx.x * 4 + g;
  const bool live = id < (int64_t)a.nrhs * a.np;
  const int64_t rhs = live ? id / a.np : 0;
  const int j = live ? (int)(id - rhs * a.np) : 0;
  const double2* A = a.A + rhs / a.R * a.strideA;
  double2 row[M];
  load_row<M, false>(A, i, live, row);
  double2 y = live && i < M ? Y[(rhs * a.np + j) * M + i] : make_double2(0.0, 0.0);
  double2 x = y;                                       // SIGNAL: lane M holds v . y
  if (SIGNAL) {
    const double2 vi = i < M ? a.v[i] : make_double2(0.0, 0.0);
    const double2 dot = cmul(vi, y);
    x = make_double2(seg_sum<16>(dot.x), seg_sum<16>(dot.y));
    if (live && i == M) {
#pragma unroll
      for (int c = 0; c < M; ++c) {
        double2 w = make_double2(0.0, 0.0);
        for (int q = 0; q < M; ++q) cfma<double>(w, a.v[q], A[q * M + c]);
        row[c] = w;
      }
    }
  }
  const bool writer = live && (SIGNAL ? i == M : i < M);
  const int64_t width = SIGNAL ? 1 : M;
  double2* o = out + rhs * a.nsave * width + (SIGNAL ? 0 : i);
  // piece 0 also writes the saves of y_0
  int s = j == 0 ? 0 : min(max(a.first[j], 0), a.nsave);
  const int s1 = live ? min(a.first[j + 1], a.nsave) : s;
  const int p0 = j * a.len, p1 = live ? min(p0 + a.len, a.N) : p0;
  int next = s < s1 ? a.pos[s] : INT32_MAX;
  for (int p = p0;; ++p) {
    while (next <= p) {
      if (writer) o[s * width] = SIGNAL ? x : y;
      next = ++s < s1 ? a.pos[s] : INT32_MAX;
    }
    if (p >= p1) break;
    y = row_product<M>(row, y);
    x = y;
  }
  if (live && i <= (SIGNAL ? M : M - 1) && !cfinite(y)) status[0] = 1;
}

// Reverse: the contribution mu of every piece to the cotangent at its start,
// from the saves inside it.
template <int M, bool SIGNAL>
__global__ __launch_bounds__(64) void piece_local_kernel(PieceArgs a,
                                                         const double2* __restrict__ gout,
                                                         double2* __restrict__ mu) {
  const int g = threadIdx.x >> 4, i = threadIdx.x & 15;
  const int64_t id = (int64_t)blockIdx.x * 4 + g;
  const bool live = id < (int64_t)a.nrhs * a.np;
  const int64_t rhs = live ? id / a.np : 0;
  const int j = live ? (int)(id - rhs * a.np) : 0;
  double2 row[M];
  load_row<M, true>(a.A + rhs / a.R * a.strideA, i, live, row);
  const double2 vc = SIGNAL && i < M ? conj2(a.v[i]) : make_double2(0.0, 0.0);
  const int s0 = min(max(a.first[j], 0), a.nsave);
  int s = live ? min(a.first[j + 1], a.nsave) - 1 : s0 - 1;
  const int p0 = j * a.len, p1 = live ? min(p0 + a.len, a.N) : p0;
  double2 lam = make_double2(0.0, 0.0), inj = lam;
  int next = -1;
  if (s >= s0) {
    next = a.pos[s];
    inj = injection<M, SIGNAL>(a, gout, rhs, s, i, vc);
  }
  for (int p = p1; p > p0; --p) {
    while (next >= p) {
      lam = cadd(lam, inj);
      next = -1;
      if (--s >= s0) {
        next = a.pos[s];
        inj = injection<M, SIGNAL>(a, gout, rhs, s, i, vc);
      }
    }
    lam = row_product<M>(row, lam);
  }
  if (live && i < M) mu[(rhs * a.np + j) * M + i] = lam;
}

// Reverse: every piece's part of G = sum_p lambda_p y_{p-1}^H, Gp [nrhs][np][M][M].
template <int M, bool SIGNAL>
__global__ __launch_bounds__(64) void piece_adjoint_kernel(
    PieceArgs a, const double2* __restrict__ Y, const double2* __restrict__ gout,
    const double2* __restrict__ Lam, double2* __restrict__ Gp, int* __restrict__ status) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int g = threadIdx.x >> 4, i = threadIdx.x & 15;
  double2* ys = reinterpret_cast<double2*>(smem) + g * a.len * M;     // [len][M]
  const int64_t id = (int64_t)blockIdx.x * 4 + g;
  const bool live = id < (int64_t)a.nrhs * a.np, mine = live && i < M;
  const int64_t rhs = live ? id / a.np : 0;
  const int j = live ? (int)(id - rhs * a.np) : 0;
  const double2* A = a.A + rhs / a.R * a.strideA;
  const int p0 = j * a.len, p1 = live ? min(p0 + a.len, a.N) : p0;
  double2 row[M];
  load_row<M, false>(A, i, live, row);
  double2 y = mine ? Y[(rhs * a.np + j) * M + i] : make_double2(0.0, 0.0);
  for (int p = p0; p < p1; ++p) {                      // states p0 .. p1 - 1
    if (i < M) ys[(p - p0) * M + i] = y;
    y = row_product<M>(row, y);
  }
  __syncthreads();
  load_row<M, true>(A, i, live, row);
  const double2 vc = SIGNAL && i < M ? conj2(a.v[i]) : make_double2(0.0, 0.0);
  const int s0 = min(max(a.first[j], 0), a.nsave);
  int s = live ? min(a.first[j + 1], a.nsave) - 1 : s0 - 1;
  double2 lam = mine ? Lam[(rhs * a.np + j) * M + i] : make_double2(0.0, 0.0), inj = lam;
  int next = -1;
  if (s >= s0) {
    next = a.pos[s];
    inj = injection<M, SIGNAL>(a, gout, rhs, s, i, vc);
  }
  double2 G[M];
#pragma unroll
  for (int c = 0; c < M; ++c) G[c] = make_double2(0.0, 0.0);
  for (int p = p1; p > p0; --p) {
    while (next >= p) {
      lam = cadd(lam, inj);
      next = -1;
      if (--s >= s0) {
        next = a.pos[s];
        inj = injection<M, SIGNAL>(a, gout, rhs, s, i, vc);
      }
    }
    const double2* yq = ys + (p - 1 - p0) * M;
#pragma unroll
    for (int c = 0; c < M; ++c) cfma<double>(G[c], lam, conj2(yq[c]));
    lam = row_product<M>(row, lam);
  }
  if (mine) {
    double2* o = Gp + ((rhs * a.np + j) * M + i) * M;
    bool bad = !cfinite(lam);
#pragma unroll
    for (int c = 0; c < M; ++c) {
      o[c] = G[c];
      bad |= !cfinite(G[c]);
    }
    if (bad) status[0] = 1;
  }
}

// gA[rhs] = sum over the pieces of Gp
__global__ __launch_bounds__(256) void piece_sum_kernel(const double2* __restrict__ Gp, int mm,
                                                        int np, int64_t total,
                                                        double2* __restrict__ gA) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= total) return;
  const int64_t rhs = e / mm, r = e - rhs * mm;
  const double2* p = Gp + rhs * np * mm + r;
  double2 v = make_double2(0.0, 0.0);
#pragma unroll 8
  for (int j = 0; j < np; ++j) v = cadd(v, p[(int64_t)j * mm]);
  gA[e] = v;
}

int check_pieces(const char* who, const void* A, int64_t strideA, int M, int R, int B,
                 int nsave, int64_t N, int len, const void* pos, const void* first, const void* v,
                 PieceArgs& a) {
  QSX_CHECK_ARG(A && pos && first, "%s: null pointer", who);
  QSX_CHECK_ARG(M >= 1 && M <= kMaxM && R >= 1 && B >= 1 && nsave >= 1 &&
                    (int64_t)R * B <= (1 << 24),
                "%s: bad sizes M=%d R=%d B=%d nsave=%d", who, M, R, B, nsave);
  QSX_CHECK_ARG(N >= 1 && N <= (1 << 24) && len >= 2 && len <= kMaxLen && (len & (len - 1)) == 0,
                "%s: bad schedule N=%lld len=%d", who, (long long)N, len);
  QSX_CHECK_ARG(strideA == 0 || strideA == (int64_t)M * M, "%s: bad strideA", who);
  QSX_CHECK_ARG(v == nullptr || M < kMaxM, "%s: signals need M < %d", who, kMaxM);
  a.A = static_cast<const double2*>(A);
  a.strideA = strideA;
  a.R = R;
  a.nrhs = R * B;
  a.N = (int)N;
  a.len = len;
  a.np = (int)((N + len - 1) / len);
  QSX_CHECK_ARG((int64_t)a.nrhs * a.np < (int64_t)1 << 31, "%s: too many pieces", who);
  a.nsave = nsave;
  a.pos = static_cast<const int*>(pos);
  a.first = static_cast<const int*>(first);
  a.v = static_cast<const double2*>(v);
  return QSX_OK;
}

// fn(std::integral_constant<int, M>()) for 1 <= M <= kMaxM
template <int M = 1, typename F>
void with_m(int m, const F& fn) {
  if (m == M) {
    fn(std::integral_constant<int, M>());
  } else if constexpr (M < kMaxM) {
    with_m<M + 1>(m, fn);
  }
}

template <bool SIGNAL>
void launch_forward(const PieceArgs& a, int M, const double2* y0, double2* Y, double2* out,
                    int* status, hipStream_t s) {
  const dim3 chain((a.nrhs + 3) / 4), pieces((unsigned)(((int64_t)a.nrhs * a.np + 3) / 4));
  with_m(M, [&](auto m) {
    constexpr int kM = decltype(m)::value;
    hipLaunchKernelGGL((piece_chain_kernel<kM, SIGNAL>), chain, dim3(64), 0, s, a, false, y0, Y,
                       nullptr, nullptr, nullptr, nullptr);
    hipLaunchKernelGGL((piece_forward_kernel<kM, SIGNAL>), pieces, dim3(64), 0, s, a, Y, out,
                       status);
  });
}

template <bool SIGNAL>
void launch_reverse(const PieceArgs& a, int M, const double2* Y, const double2* gout,
                    double2* mu, double2* Lam, double2* Gp, double2* gy0, int* status,
                    hipStream_t s) {
  const dim3 chain((a.nrhs + 3) / 4), pieces((unsigned)(((int64_t)a.nrhs * a.np + 3) / 4));
  const size_t lds = (size_t)4 * a.len * M * sizeof(double2);          // <= 64 KB
  with_m(M, [&](auto m) {
    constexpr int kM = decltype(m)::value;
    hipLaunchKernelGGL((piece_local_kernel<kM, SIGNAL>), pieces, dim3(64), 0, s, a, gout, mu);
    hipLaunchKernelGGL((piece_chain_kernel<kM, SIGNAL>), chain, dim3(64), 0, s, a, true, nullptr,
                       nullptr, mu, gout, Lam, gy0);
    hipLaunchKernelGGL((piece_adjoint_kernel<kM, SIGNAL>), pieces, dim3(64), lds, s, a, Y, gout,
                       Lam, Gp, status);
  });
}

}  // namespace
}  // namespace qsx

extern "C" int32_t qsx_propagate_pieces(const void* A, int64_t strideA, int32_t M,
                                        const void* y0, int32_t R, int32_t B, const int32_t* pos,
                                        const int32_t* first, int32_t nsave, int64_t N,
                                        int32_t len, const void* v, void* Q, void* Y, void* out,
                                        int32_t* status, void* stream) {
  using namespace qsx;
  PieceArgs a;
  const int st = check_pieces("qsx_propagate_pieces", A, strideA, M, R, B, nsave, N, len, pos,
                              first, v, a);
  if (st) return st;
  QSX_CHECK_ARG(y0 && Q && Y && out && status, "qsx_propagate_pieces: null pointer");
  hipStream_t s = as_stream(stream);
  a.Q = static_cast<const double2*>(Q);
  hipLaunchKernelGGL(piece_power_kernel, dim3(strideA ? B : 1), dim3(kMaxM * kMaxM), 0, s, a.A,
                     strideA, M, len, static_cast<double2*>(Q));
  if (v != nullptr)
    launch_forward<true>(a, M, static_cast<const double2*>(y0), static_cast<double2*>(Y),
                         static_cast<double2*>(out), status, s);
  else
    launch_forward<false>(a, M, static_cast<const double2*>(y0), static_cast<double2*>(Y),
                          static_cast<double2*>(out), status, s);
  QSX_CHECK_HIP(hipGetLastError());
  return QSX_OK;
}

extern "C" int64_t qsx_propagate_pieces_adjoint_workspace_bytes(int32_t M, int32_t R, int32_t B,
                                                                int64_t N, int32_t len) {
  if (M < 1 || M > qsx::kMaxM || R < 1 || B < 1 || N < 1 || len < 1) return -1;
  const int64_t np = (N + len - 1) / len;
  return (int64_t)R * B * np * M * (2 + M) * (int64_t)sizeof(double2);
}

extern "C" int32_t qsx_propagate_pieces_adjoint(
    const void* A, int64_t strideA, int32_t M, int32_t R, int32_t B, const int32_t* pos,
    const int32_t* first, int32_t nsave, int64_t N, int32_t len, const void* v, const void* Q,
    const void* Y, const void* gout, void* workspace, int64_t workspace_bytes, void* gA,
    void* gy0, int32_t* status, void* stream) {
  using namespace qsx;
  PieceArgs a;
  const int st = check_pieces("qsx_propagate_pieces_adjoint", A, strideA, M, R, B, nsave, N, len,
                              pos, first, v, a);
  if (st) return st;
  QSX_CHECK_ARG(Q && Y && gout && workspace && gA && status,
                "qsx_propagate_pieces_adjoint: null pointer");
  QSX_CHECK_ARG(workspace_bytes >= qsx_propagate_pieces_adjoint_workspace_bytes(M, R, B, N, len),
                "qsx_propagate_pieces_adjoint: workspace too small");
  hipStream_t s = as_stream(stream);
  a.Q = static_cast<const double2*>(Q);
  const int64_t vec = (int64_t)a.nrhs * a.np * M;
  double2* mu = static_cast<double2*>(workspace);
  double2 *Lam = mu + vec, *Gp = Lam + vec;
  if (v != nullptr)
    launch_reverse<true>(a, M, static_cast<const double2*>(Y), static_cast<const double2*>(gout),
                         mu, Lam, Gp, static_cast<double2*>(gy0), status, s);
  else
    launch_reverse<false>(a, M, static_cast<const double2*>(Y), static_cast<const double2*>(gout),
                          mu, Lam, Gp, static_cast<double2*>(gy0), status, s);
  const int64_t total = (int64_t)a.nrhs * M * M;
  hipLaunchKernelGGL(piece_sum_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, Gp,
                     M * M, a.np, total, static_cast<double2*>(gA));
  QSX_CHECK_HIP(hipGetLastError());
  return QSX_OK;
}
