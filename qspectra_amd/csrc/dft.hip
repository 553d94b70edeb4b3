// The Fourier transform of qspectra/simulate/utils.py:128-219 on the GPU, as
// a direct sum (gfx950).
//
// The reference zero-pads a signal of n samples to a grid of N points
// symmetric about t = 0 (the samples at positions lo .. lo+n-1), scales by
// dt, and applies ifftshift, FFT, fftshift (and a reversal for sign = +1).
// Written out, output r is
//
//   X[r] = dt * sum_j x[j] * exp(-2 pi i s_r (lo + j - c) / N),   c = N / 2,
//   s_r  = r - c            (sign = -1)
//   s_r  = N - 1 - c - r    (sign = +1).
//
// Only the n nonzero samples enter, so the direct sum costs N*n complex
// multiply-adds, with no plan and nothing compiled at run time (a library FFT
// of a new length is compiled on first use).  The exponent is reduced exactly
// in integers, m = s_r * (lo + j - c) mod N; every 16th twiddle is read from
// a table exp(-2 pi i m / N) built once per call, the ones in between are
// advanced by one complex multiplication with the step twiddle.  The adjoint (the backward of the
// transform, x -> conj(F)^T X) is the same sum over r with conjugated
// twiddles.
//
// Layout: one thread per pair of outputs with opposite s (conjugate
// twiddles: their four real products per sample are the same, so a pair costs
// one complex multiply-add per sample) and R = 1, 2 or 4 batch rows (the
// twiddles are the rows'): 4 + 4 / R FP64 operations per sample for two
// outputs, where one output of one row took 8.  The rows are staged through
// LDS in tiles (every thread reads the same sample: broadcast), 8 or 16 KB per
// work-group, and a launch has threads for the pairs that have an
// output only, where they fill the chip in work-groups of whole wavefronts:
// short grids (up to 127 points: one wavefront) and the adjoints of short signals
// far from t = 0 keep up to twenty work-groups on a CU.  Four chains of
// twiddles, each advanced by four samples' step, hide their latency.
// Measured (host call): 129 rows of 1000 samples onto 1999 points 63 us, with
// one output of one row per thread 122 us; 20000 rows of 61 samples onto 121
// points 26 us, the adjoint 39 us, with N / 2 + 1 pairs in work-groups of 256
// and 32 KB of samples 64 and 112 us, with one output per thread 76 and 94 us;
// adjoint of 3000 rows from 4000 points to 100 samples at their end 443, 4306
// and 677 us.
//
// Long transforms (both lengths >= kChirpMin) take Bluestein's chirp-z form
// instead, O(N log N) per row.  Both directions are one sum
//
//   out[u] = scale * sum_v in[v] * exp(-2 pi i sigma (u + A)(v + D) / N)
//
// (sigma = +-1), and with pq = (p^2 + q^2 - (q - p)^2) / 2
//
//   out[u] = scale * c(u + A) * sum_v [in[v] c(v + D)] * conj(c(u - v + A - D)),
//   c(k)   = exp(-pi i sigma (k^2 mod 2N) / N)    (exact integer reduction),
//
// a linear convolution.  It is cut into input pieces of P samples and output
// chunks of H points with P + H - 1 <= L = 8192, so that every piece/chunk
// pair is one cyclic convolution of length L: FFT of the chirped piece (in
// LDS), times the FFT of the pair's chirp kernel (a table built once per call,
// it depends on the pair only), inverse FFT by conjugation.  A row of the
// absorption workload (4096 samples onto 8191 points) is one piece and two
// chunks: four FFTs of 8192 points on one row held in LDS, the row read twice
// (the second time from the cache) and its transform written once.  The FFT is a Stockham autosort FFT
// (one radix-2 pass, three radix-16 passes; Govindaraju et al., "High
// performance discrete Fourier transforms on graphics processors", SC 2008)
// on 512 threads, 16 points per thread, the LDS rows padded by one entry in
// 16 against bank conflicts.

#include "qsx_common.h"

#include <algorithm>
#include <type_traits>

namespace qsx {
namespace {

constexpr int kDftThreads = 256;
constexpr int kAnchor = 16;   // samples between exact twiddles (divides a tile)
// samples per row in LDS: 8 KB for four rows, whose launches fill the chip (also
// with work-groups of one wavefront), 8 and 16 KB for one and two
constexpr int dft_tile(int R) { return R == 4 ? 128 : 512; }

__global__ __launch_bounds__(kDftThreads) void dft_twiddle_kernel(int N, double2* __restrict__ T) {
  const int m = blockIdx.x * kDftThreads + threadIdx.x;
  if (m >= N) return;
  double s, c;
  sincospi(2.0 * (double)m / (double)N, &s, &c);
  T[m] = make_double2(c, -s);
}

__device__ inline int64_t mod_n(int64_t a, int64_t N) {
  const int64_t r = a % N;
  return r < 0 ? r + N : r;
}

// out[b, u] = scale * sum_v in[b, v] * T[(a_u * d_v) mod N] (conj if adj),
// a_u = a0 + da * u, d_v = d0 + dd * v.  A thread forms the outputs with
// a_u = q and a_u = -q (mod N), where they exist, of R rows, for its one of the
// nq values q = q0, q0 + 1, .. <= N/2 that have any.  Wavefronts beyond them
// only stage samples.
template <int R>
__global__ __launch_bounds__(kDftThreads) void dft_kernel(
    const double2* __restrict__ in, int64_t batch, int n_in, int n_out, int N, int64_t a0,
    int da, int64_t d0, int dd, int q0, int nq, int adj, double scale,
    const double2* __restrict__ T, double2* __restrict__ out) {
  constexpr int kTile = dft_tile(R), U = 2;
  __shared__ double2 xs[R][kTile];
  const int nt = R == 4 ? blockDim.x : kDftThreads;
  const int64_t q = (int64_t)blockIdx.x * nt + threadIdx.x;
  const bool mine = q < nq, busy = __any(mine);
  const int64_t a = q0 + min(q, (int64_t)(nq - 1));
  const int64_t u0 = mod_n(da * (a - a0), N), u1 = mod_n(da * (-a - a0), N);
  const bool w0 = mine && u0 < n_out, w1 = mine && u1 < n_out && u1 != u0;
  const int step = (int)mod_n(a * dd, N);
  // unsigned: two residues add up to less than 2^32
  const unsigned anchor_step = (unsigned)mod_n((int64_t)step * kAnchor, N);
  const unsigned m0 = (unsigned)mod_n(a * mod_n(d0, N), N);
  const double sg = adj ? -1.0 : 1.0;
  const double2 w = make_double2(T[step].x, sg * T[step].y), w2 = cmul(w, w), w4 = cmul(w2, w2);
  for (int64_t b0 = (int64_t)blockIdx.y * R; b0 < batch; b0 += (int64_t)gridDim.y * R) {
    double rr[R], ii[R], ri[R], ir[R];       // sums of x.x t.x, x.y t.y, x.x t.y, x.y t.x
#pragma unroll
    for (int r = 0; r < R; ++r) rr[r] = ii[r] = ri[r] = ir[r] = 0.0;
    unsigned m = m0;
    for (int v0 = 0; v0 < n_in; v0 += kTile) {
      const int len = min(kTile, n_in - v0);
      __syncthreads();
      if constexpr (R == 2) {         // R U loads in flight (129 rows as above: 63 us for 66)
        for (int k0 = threadIdx.x; k0 < len; k0 += U * nt) {
          double2 x[R][U];
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const double2* row = in + min(b0 + r, batch - 1) * n_in + v0;
#pragma unroll
            for (int u = 0; u < U; ++u) x[r][u] = row[min(k0 + u * nt, len - 1)];
          }
#pragma unroll
          for (int r = 0; r < R; ++r)
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (k0 + u * nt < len) xs[r][k0 + u * nt] = x[r][u];
        }
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const double2* row = in + min(b0 + r, batch - 1) * n_in + v0;
          for (int k = threadIdx.x; k < len; k += nt) xs[r][k] = row[k];
        }
      }
      __syncthreads();
      // exact twiddle from the table every kAnchor samples, in between multiplied
      // by step twiddles: with one rounding error for a table entry and one for
      // a product, w, w2 and w4 carry 1, 3 and 7 of them, t[3] starts with 7, and
      // each of its three products with w4 adds 8: at most 31 (first order)
      auto samples = [&](int k0, int count, auto full) {
        constexpr bool FULL = decltype(full)::value;
        double2 t[4];
        t[0] = make_double2(T[m].x, sg * T[m].y);
        t[1] = cmul(t[0], w);
        t[2] = cmul(t[0], w2);
        t[3] = cmul(t[1], w2);
#pragma unroll
        for (int k = 0; k < kAnchor; ++k) {
          if (FULL || k < count) {
            double2& tk = t[k & 3];
#pragma unroll
            for (int r = 0; r < R; ++r) {
              const double2 x = xs[r][k0 + k];
              rr[r] = fma(x.x, tk.x, rr[r]);
              ii[r] = fma(x.y, tk.y, ii[r]);
              ri[r] = fma(x.x, tk.y, ri[r]);
              ir[r] = fma(x.y, tk.x, ir[r]);
            }
            tk = cmul(tk, w4);
          }
        }
        m += anchor_step;
        if (m >= (unsigned)N) m -= N;
      };
      if (!busy) continue;
      int k0 = 0;
      for (; k0 + kAnchor <= len; k0 += kAnchor) samples(k0, kAnchor, std::true_type());
      if (k0 < len) samples(k0, len - k0, std::false_type());
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (b0 + r >= batch) break;
      double2* o = out + (b0 + r) * n_out;
      if (w0) o[u0] = make_double2(scale * (rr[r] - ii[r]), scale * (ri[r] + ir[r]));
      if (w1) o[u1] = make_double2(scale * (rr[r] + ii[r]), scale * (ir[r] - ri[r]));
    }
  }
}


// ---------------------------------------------------------------------------
// chirp-z transform for long rows

constexpr int kFftL = 8192;                    // cyclic convolution length
constexpr int kFftThreads = 512;
constexpr int kFftPer = kFftL / kFftThreads;   // 16 points per thread
constexpr int kFftPadded = kFftL + kFftL / 16; // one pad entry per 16
constexpr int kTw1 = 128, kTw2 = kFftL / kTw1; // two-level twiddle table
constexpr size_t kFftLds = (size_t)(kFftPadded + kTw1 + kTw2) * sizeof(double2);
constexpr int kChirpMin = 2048;                // shorter transforms: direct sum
constexpr int kChirpMaxTables = 64;

struct ChirpGeom {
  int n_in, n_out;
  int P, H;              // input piece and output chunk lengths, P + H - 1 <= L
  int pieces, chunks;
  int sigma;
  int64_t N, A, D;
};

__device__ __forceinline__ int fpad(int i) { return i + (i >> 4); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) {
  return make_double2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
// a * (-i) and a * (+i)
__device__ __forceinline__ double2 mul_mi(double2 a) { return make_double2(a.y, -a.x); }
__device__ __forceinline__ double2 mul_pi(double2 a) { return make_double2(-a.y, a.x); }

// c(k) = exp(-pi i sigma (k^2 mod 2N) / N), the exponent reduced exactly
// in integers (64-bit divisions: evaluated once per call, into tables)
__device__ __forceinline__ double2 chirp_exact(int64_t k, int64_t N) {
  const int64_t N2 = 2 * N;
  int64_t m = k % N2;
  if (m < 0) m += N2;
  double s, c;
  sincospi((double)((m * m) % N2) / (double)N, &s, &c);
  return make_double2(c, -s);
}

// exp(-2 pi i k / L) = tw1[k mod 128] * tw2[k / 128]
__device__ __forceinline__ void build_fft_twiddles(double2* tw1, double2* tw2) {
  const int t = threadIdx.x;
  double s, c;
  if (t < kTw1) {
    sincospi(2.0 * (double)t / (double)kFftL, &s, &c);
    tw1[t] = make_double2(c, -s);
  } else if (t < kTw1 + kTw2) {
    sincospi(2.0 * (double)((t - kTw1) * kTw1) / (double)kFftL, &s, &c);
    tw2[t - kTw1] = make_double2(c, -s);
  }
}

// 4-point forward DFT in place: y_k = sum_m x_m (-i)^(mk)
__device__ __forceinline__ void dft4(double2& x0, double2& x1, double2& x2, double2& x3) {
  const double2 s02 = cadd(x0, x2), d02 = csub(x0, x2);
  const double2 s13 = cadd(x1, x3), d13 = mul_mi(csub(x1, x3));
  x0 = cadd(s02, s13);
  x2 = csub(s02, s13);
  x1 = cadd(d02, d13);
  x3 = csub(d02, d13);
}

// 16-point forward DFT of v (natural order in and out) as 4 x 4: DFTs over
// the stride-4 subsequences, twiddles exp(-2 pi i q k1 / 16), DFTs over q
__device__ __forceinline__ void dft16(double2 (&v)[16]) {
  constexpr double c1 = 0.92387953251128674;   // cos(pi / 8)
  constexpr double s1 = 0.38268343236508978;   // sin(pi / 8)
  constexpr double h = 0.70710678118654752;    // sqrt(1 / 2)
#pragma unroll
  for (int q = 0; q < 4; ++q) dft4(v[q], v[q + 4], v[q + 8], v[q + 12]);
  // v[q + 4 k1] now holds b[q][k1]; twiddle by w16^(q k1)
  v[5] = cmul(v[5], make_double2(c1, -s1));     // q 1, k1 1: e 1
  v[9] = cmul(v[9], make_double2(h, -h));       // q 1, k1 2: e 2
  v[13] = cmul(v[13], make_double2(s1, -c1));   // q 1, k1 3: e 3
  v[6] = cmul(v[6], make_double2(h, -h));       // q 2, k1 1: e 2
  v[10] = mul_mi(v[10]);                        // q 2, k1 2: e 4
  v[14] = cmul(v[14], make_double2(-h, -h));    // q 2, k1 3: e 6
  v[7] = cmul(v[7], make_double2(s1, -c1));     // q 3, k1 1: e 3
  v[11] = cmul(v[11], make_double2(-h, -h));    // q 3, k1 2: e 6
  v[15] = cmul(v[15], make_double2(-c1, s1));   // q 3, k1 3: e 9
#pragma unroll
  for (int k1 = 0; k1 < 4; ++k1)
    dft4(v[4 * k1], v[4 * k1 + 1], v[4 * k1 + 2], v[4 * k1 + 3]);
  // v[4 k1 + k2] holds X[k1 + 4 k2]: transpose the 4 x 4 index
  double2 t;
  t = v[1]; v[1] = v[4]; v[4] = t;
  t = v[2]; v[2] = v[8]; v[8] = t;
  t = v[3]; v[3] = v[12]; v[12] = t;
  t = v[6]; v[6] = v[9]; v[9] = t;
  t = v[7]; v[7] = v[13]; v[13] = t;
  t = v[11]; v[11] = v[14]; v[14] = t;
}

// The butterflies of one radix-16 Stockham pass over the padded LDS row:
// thread j reads entries j + r L/16 and leaves in v[r] the pass's outputs
// for entries (j - j mod Ns) 16 + j mod Ns + r Ns.
__device__ __forceinline__ void radix16_butterflies(const double2* buf, int Ns,
                                                    const double2* tw1, const double2* tw2,
                                                    double2 (&v)[16]) {
  const int j = threadIdx.x;   // butterfly index, kFftL / 16 of them
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = buf[fpad(j + r * (kFftL / 16))];
  const int jm = j & (Ns - 1);
  const int k1 = jm * (kFftL / (Ns * 16));
  const double2 w1 = cmul(tw1[k1 & (kTw1 - 1)], tw2[k1 / kTw1]);
  double2 w = w1;
#pragma unroll
  for (int r = 1; r < 16; ++r) {
    v[r] = cmul(v[r], w);
    w = cmul(w, w1);
  }
  dft16(v);
}

// One radix-16 Stockham pass, in place: every thread's reads finish before
// the barrier, its writes follow it.
__device__ __forceinline__ void radix16_pass(double2* buf, int Ns, const double2* tw1,
                                             const double2* tw2) {
  double2 v[16];
  radix16_butterflies(buf, Ns, tw1, tw2, v);
  const int j = threadIdx.x, jm = j & (Ns - 1);
  const int idx = (j - jm) * 16 + jm;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; ++r) buf[fpad(idx + r * Ns)] = v[r];
  __syncthreads();
}

// The last three passes of an FFT whose radix-2 pass is in LDS: the final
// pass (Ns = L / 16) leaves entry t + r L/16 of the transform in v[r] of
// thread t, the entries that thread read, so it needs no write-back.
__device__ __forceinline__ void fft_tail_to_registers(double2* buf, const double2* tw1,
                                                      const double2* tw2, double2 (&v)[16]) {
  radix16_pass(buf, 2, tw1, tw2);
  radix16_pass(buf, 32, tw1, tw2);
  radix16_butterflies(buf, kFftL / 16, tw1, tw2, v);
}

// Forward FFT of the L-point row in LDS (natural order in and out).  Expects
// the row's writes to have been made visible by a barrier.
__device__ void fft_row(double2* buf, const double2* tw1, const double2* tw2) {
  const int t = threadIdx.x;
  double2 v[16];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int j = t + q * kFftThreads;
    v[2 * q] = buf[fpad(j)];
    v[2 * q + 1] = buf[fpad(j + kFftL / 2)];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int j = t + q * kFftThreads;
    buf[fpad(2 * j)] = cadd(v[2 * q], v[2 * q + 1]);
    buf[fpad(2 * j + 1)] = csub(v[2 * q], v[2 * q + 1]);
  }
  __syncthreads();
  radix16_pass(buf, 2, tw1, tw2);
  radix16_pass(buf, 32, tw1, tw2);
  radix16_pass(buf, 512, tw1, tw2);
}

// The chirps of the input samples, cin[v] = c(v + D), and of the output
// points, cout[u] = c(u + A) (conjugated for sigma = -1): the same for
// every row.
__global__ __launch_bounds__(256) void chirp_vectors_kernel(ChirpGeom g, double2* __restrict__ cin,
                                                           double2* __restrict__ cout) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (j < g.n_in) {
    const double2 c = chirp_exact(j + g.D, g.N);
    cin[j] = make_double2(c.x, g.sigma > 0 ? c.y : -c.y);
  }
  if (j < g.n_out) {
    const double2 c = chirp_exact(j + g.A, g.N);
    cout[j] = make_double2(c.x, g.sigma > 0 ? c.y : -c.y);
  }
}

// The FFT of each piece/chunk pair's cyclic chirp kernel: G[k] =
// conj(c(delta + k + A - D)) for k < H and conj(c(delta - (L - k) + A - D))
// for k > L - P, delta = j0 - i0.  One work-group per pair.
__global__ __launch_bounds__(kFftThreads) void chirp_tables_kernel(ChirpGeom g,
                                                                  double2* __restrict__ Gt) {
  extern __shared__ double2 lds[];
  double2* buf = lds;
  double2* tw1 = lds + kFftPadded;
  double2* tw2 = tw1 + kTw1;
  build_fft_twiddles(tw1, tw2);
  const int id = blockIdx.x;
  const int j = id / g.pieces, i = id - j * g.pieces;
  const int64_t delta = (int64_t)j * g.H - (int64_t)i * g.P, dl = g.A - g.D;
  for (int r = 0; r < kFftPer; ++r) {
    const int k = threadIdx.x + r * kFftThreads;
    const int64_t e = k < g.H ? delta + k : delta - (kFftL - k);
    const double2 c = chirp_exact(e + dl, g.N);   // conj(c) for sigma = +1
    buf[fpad(k)] = make_double2(c.x, g.sigma > 0 ? -c.y : c.y);
  }
  __syncthreads();
  fft_row(buf, tw1, tw2);
  double2* G = Gt + (size_t)id * kFftL;
#pragma unroll
  for (int r = 0; r < kFftPer; ++r) {
    const int k = threadIdx.x + r * kFftThreads;
    G[k] = buf[fpad(k)];
  }
}

// Piece i of a row, chirped and zero-padded to L points, into LDS.
__device__ __forceinline__ void load_piece(double2* buf, const double2* __restrict__ row,
                                           const ChirpGeom& g, int i,
                                           const double2* __restrict__ cin) {
  const int i0 = i * g.P, pe = min(g.P, g.n_in - i0);
  // four points at a time: their sample and chirp loads issue together
#pragma unroll
  for (int r0 = 0; r0 < kFftPer; r0 += 4) {
    double2 x[4], c[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int v = threadIdx.x + (r0 + q) * kFftThreads;
      x[q] = make_double2(0.0, 0.0);
      c[q] = make_double2(0.0, 0.0);
      if (v < pe) {
        x[q] = row[i0 + v];
        c[q] = cin[i0 + v];
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
      buf[fpad(threadIdx.x + (r0 + q) * kFftThreads)] = cmul(x[q], c[q]);
  }
  __syncthreads();
}

// One work-group per row (grid-stride over the batch): the chirp-z form of
// the transform.  Every piece/chunk pair is two FFTs in LDS with nothing
// held in registers across them (16 points per thread of the in-place passes
// already take most of the 256 registers a thread has here): the chirped
// piece, its product with the pair's kernel spectrum, the inverse FFT.  A
// chunk of several pieces adds their contributions in the output row.
__global__ __launch_bounds__(kFftThreads) void chirp_rows_kernel(
    const double2* __restrict__ in, int64_t batch, ChirpGeom g, const double2* __restrict__ cin,
    const double2* __restrict__ cout, const double2* __restrict__ Gt, double scale,
    double2* __restrict__ out) {
  extern __shared__ double2 lds[];
  double2* buf = lds;
  double2* tw1 = lds + kFftPadded;
  double2* tw2 = tw1 + kTw1;
  build_fft_twiddles(tw1, tw2);
  __syncthreads();
  const int t = threadIdx.x;
  const double oscale = scale / (double)kFftL;   // the inverse FFT's 1 / L
  for (int64_t b = blockIdx.x; b < batch; b += gridDim.x) {
    const double2* row = in + b * g.n_in;
    double2* orow = out + b * g.n_out;
    if (g.pieces == 1) {
      // one piece (P = L/2 samples, zero-padded to L): its spectrum, kept in
      // registers (entry t + r L/16 in S[r] of thread t), serves every
      // chunk.  The radix-2 pass of its FFT only duplicates each sample (the
      // upper half is zero), so the samples go straight to both outputs.
      __syncthreads();                 // the previous row's reads are done
#pragma unroll
      for (int r0 = 0; r0 < kFftPer / 2; r0 += 4) {
        double2 x[4], c[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int v = t + (r0 + q) * kFftThreads;
          x[q] = make_double2(0.0, 0.0);
          c[q] = make_double2(0.0, 0.0);
          if (v < g.n_in) {
            x[q] = row[v];
            c[q] = cin[v];
          }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int v = t + (r0 + q) * kFftThreads;
          const double2 y = cmul(x[q], c[q]);
          buf[fpad(2 * v)] = y;
          buf[fpad(2 * v + 1)] = y;
        }
      }
      __syncthreads();
      double2 S[kFftPer];
      fft_tail_to_registers(buf, tw1, tw2, S);
      for (int j = 0; j < g.chunks; ++j) {
        const int j0 = j * g.H, he = min(g.H, g.n_out - j0);
        const double2* G = Gt + (size_t)j * kFftL;
        // the inverse FFT (conj(FFT(conj(.))) / L) of S times the kernel
        // spectrum, its radix-2 pass from registers: entries t + q L/16 and
        // t + (q + 8) L/16 are this thread's S[q], S[q + 8]
        __syncthreads();               // every thread's reads of buf are done
#pragma unroll
        for (int q = 0; q < kFftPer / 2; ++q) {
          const int jj = t + q * kFftThreads;
          const double2 a = cconj(cmul(S[q], G[jj]));
          const double2 b = cconj(cmul(S[q + kFftPer / 2], G[jj + kFftL / 2]));
          buf[fpad(2 * jj)] = cadd(a, b);
          buf[fpad(2 * jj + 1)] = csub(a, b);
        }
        __syncthreads();
        // the last pass reads and writes only this thread's entries t + r
        // L/16 (no barrier), which the output then reads back
        {
          double2 y[kFftPer];
          fft_tail_to_registers(buf, tw1, tw2, y);
#pragma unroll
          for (int r = 0; r < kFftPer; ++r) buf[fpad(t + r * kFftThreads)] = y[r];
        }
#pragma unroll
        for (int r = 0; r < kFftPer; ++r) {
          const int u = t + r * kFftThreads;
          if (u < he) {
            const double2 z = cmul(cout[j0 + u], cconj(buf[fpad(u)]));
            orow[j0 + u] = make_double2(oscale * z.x, oscale * z.y);
          }
        }
      }
      continue;
    }
    for (int j = 0; j < g.chunks; ++j) {
      const int j0 = j * g.H, he = min(g.H, g.n_out - j0);
      for (int i = 0; i < g.pieces; ++i) {
        load_piece(buf, row, g, i, cin);
        fft_row(buf, tw1, tw2);
        // times the kernel spectrum, conjugated: the inverse FFT is
        // conj(FFT(conj(.))) / L
        const double2* G = Gt + (size_t)(j * g.pieces + i) * kFftL;
#pragma unroll
        for (int r = 0; r < kFftPer; ++r) {
          const int k = t + r * kFftThreads;
          buf[fpad(k)] = cconj(cmul(buf[fpad(k)], G[k]));
        }
        __syncthreads();
        fft_row(buf, tw1, tw2);
#pragma unroll
        for (int r = 0; r < kFftPer; ++r) {
          const int u = t + r * kFftThreads;
          if (u < he) {
            const double2 y = cconj(buf[fpad(u)]);
            double2 z = cmul(cout[j0 + u], y);
            z = make_double2(oscale * z.x, oscale * z.y);
            // the same thread wrote this entry for the previous piece
            orow[j0 + u] = i == 0 ? z : cadd(orow[j0 + u], z);
          }
        }
        __syncthreads();
      }
    }
  }
}

// The real parts of two rows' transforms at once, where the samples start at
// the grid's zero (v + D = v >= 0): Re X[u] is the transform of the row's
// Hermitian extension (x[v] / 2 at v > 0, conj(x[v]) / 2 at -v, Re x[0]), so
// one complex transform of h_a + i h_b has the two real parts as its real and
// imaginary part.  Both halves of the extension are pieces of n samples; a
// chunk's spectrum is the sum of their products, so a pair of rows takes two
// forward FFTs and one inverse FFT per chunk, where two rows alone take two
// forward and two inverse FFTs per chunk, and the output is written as
// doubles.  Row b is scaled by a power of two to row a's magnitude (each
// row's rounding error stays relative to its own); rows that cannot share
// (non-finite, zero, row a beyond 2^+-500 or the rows that far apart) are
// transformed one by one:
// row a in the first launch, which marks row b for the second (ALONE).
// Bound by the FFT passes (LDS and FP64 issue, one work-group per CU).
// Measured (5120 rows of 4096 samples onto 8191 points): 530 + 6 us; row by
// row with complex output 650 us.  The halves' loop stays rolled: unrolled,
// the compiler keeps both FFTs' registers and spills.
constexpr long long kAloneMark = 0x7ff8000000a10e5eLL;   // a NaN

template <bool ALONE>
__global__ __launch_bounds__(kFftThreads) void chirp_pairs_kernel(
    const double2* __restrict__ in, int64_t batch, ChirpGeom g, const double2* __restrict__ cin,
    const double2* __restrict__ cout, const double2* __restrict__ Gt, double scale,
    double* __restrict__ out) {
  extern __shared__ double2 lds[];
  double2* buf = lds;
  double2* tw1 = lds + kFftPadded;
  double2* tw2 = tw1 + kTw1;
  __shared__ double smax[2][kFftThreads / 64];
  const int t = threadIdx.x, n = g.P;
  const double oscale = scale / (double)kFftL;
  const int64_t ra = 2 * (int64_t)blockIdx.x, rb = ra + 1;
  // the rows left alone by the first launch: their first entry holds the mark
  if (ALONE && (rb >= batch || __double_as_longlong(out[rb * g.n_out]) != kAloneMark)) return;
  build_fft_twiddles(tw1, tw2);
  const double2* rowa = in + ra * n;
  const double2* rowb = rb < batch ? in + rb * n : rowa;
  int shift = 0, share = 0;
  if (!ALONE) {
    double ma = 0.0, mb = 0.0;
    bool finite = true;
#pragma unroll
    for (int r = 0; r < kFftPer / 2; ++r) {
      const int v = t + r * kFftThreads;
      if (v < n) {
        const double2 xa = rowa[v], xb = rowb[v];
        finite = finite && isfinite(xa.x) && isfinite(xa.y) && isfinite(xb.x) && isfinite(xb.y);
        ma = fmax(ma, fmax(fabs(xa.x), fabs(xa.y)));
        mb = fmax(mb, fmax(fabs(xb.x), fabs(xb.y)));
      }
    }
    for (int o = 32; o > 0; o >>= 1) {
      ma = fmax(ma, __shfl_xor(ma, o));
      mb = fmax(mb, __shfl_xor(mb, o));
    }
    if ((t & 63) == 0) {
      smax[0][t >> 6] = ma;
      smax[1][t >> 6] = mb;
    }
    const bool all_finite = __syncthreads_and(finite) != 0;
    for (int q = 0; q < kFftThreads / 64; ++q) {
      ma = fmax(ma, smax[0][q]);
      mb = fmax(mb, smax[1][q]);
    }
    shift = __builtin_amdgcn_readfirstlane(ma > 0.0 && mb > 0.0 ? ilogb(ma) - ilogb(mb) : 0);
    // row b takes row a's magnitude: away from both ends of the exponent range,
    // so that it neither overflows nor loses bits where it would not alone
    share = __builtin_amdgcn_readfirstlane(rb < batch && all_finite && ma > 0.0 && mb > 0.0 &&
                                           abs(ilogb(ma)) < 500 && abs(shift) < 500);
  }
  // the power of two of each row (0: not in it)
  const double fa = ALONE ? 0.0 : 0.5, fb = ALONE ? 0.5 : (share ? ldexp(0.5, shift) : 0.0);
  const double oa = oscale, ob = share ? ldexp(oscale, -shift) : oscale;
  double2 S[kFftPer], R[kFftPer];
#pragma unroll 1
  for (int half = 0; half < 2; ++half) {     // samples at v >= 0, then at v < 0
    __syncthreads();
#pragma unroll
    for (int r0 = 0; r0 < kFftPer / 2; r0 += 4) {
      double2 xa[4], xb[4], c[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int v = t + (r0 + q) * kFftThreads;
        const int m = half == 0 ? v : n - v;            // the sample behind entry v
        xa[q] = xb[q] = c[q] = make_double2(0.0, 0.0);
        if (v < n && m < n) {
          if (fa != 0.0) xa[q] = rowa[m];
          if (fb != 0.0) xb[q] = rowb[m];
          c[q] = cin[m];
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int v = t + (r0 + q) * kFftThreads;
        // h_a + i h_b
        const double sg = half == 0 ? 1.0 : -1.0;
        double2 w = make_double2(fa * xa[q].x - sg * (fb * xb[q].y),
                                 sg * (fa * xa[q].y) + fb * xb[q].x);
        if (half == 0 && v == 0) w = make_double2(2.0 * fa * xa[q].x, 2.0 * fb * xb[q].x);
        const double2 y = cmul(w, c[q]);
        buf[fpad(2 * v)] = y;
        buf[fpad(2 * v + 1)] = y;
      }
    }
    __syncthreads();
    fft_tail_to_registers(buf, tw1, tw2, R);
    if (half == 0)
#pragma unroll
      for (int r = 0; r < kFftPer; ++r) S[r] = R[r];
  }
  __syncthreads();                 // every thread's reads of buf are done
  // chunk 0's spectrum through the radix-2 pass of its inverse FFT into
  // LDS, chunk 1's kept in S (tables: chunk, then half v < 0, v >= 0)
#pragma unroll
  for (int q = 0; q < kFftPer / 2; ++q) {
    const int jj = t + q * kFftThreads;
    double2 e[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const double2* G = Gt + jj + u * (kFftL / 2);
      const int x = q + u * (kFftPer / 2);
      e[u] = cconj(cadd(cmul(S[x], G[kFftL]), cmul(R[x], G[0])));
      if (g.chunks == 2)
        S[x] = cconj(cadd(cmul(S[x], G[3 * kFftL]), cmul(R[x], G[2 * kFftL])));
    }
    buf[fpad(2 * jj)] = cadd(e[0], e[1]);
    buf[fpad(2 * jj + 1)] = csub(e[0], e[1]);
  }
  for (int j = 0; j < g.chunks; ++j) {
    const int j0 = j * g.H, he = min(g.H, g.n_out - j0);
    if (j > 0) {
      __syncthreads();
#pragma unroll
      for (int q = 0; q < kFftPer / 2; ++q) {
        const int jj = t + q * kFftThreads;
        buf[fpad(2 * jj)] = cadd(S[q], S[q + kFftPer / 2]);
        buf[fpad(2 * jj + 1)] = csub(S[q], S[q + kFftPer / 2]);
      }
    }
    __syncthreads();
    {
      double2 y[kFftPer];
      fft_tail_to_registers(buf, tw1, tw2, y);
#pragma unroll
      for (int r = 0; r < kFftPer; ++r) buf[fpad(t + r * kFftThreads)] = y[r];
    }
#pragma unroll
    for (int r = 0; r < kFftPer; ++r) {
      const int u = t + r * kFftThreads;
      if (u < he) {
        const double2 z = cmul(cout[j0 + u], cconj(buf[fpad(u)]));
        if (fa != 0.0) out[ra * g.n_out + j0 + u] = oa * z.x;
        if (fb != 0.0) out[rb * g.n_out + j0 + u] = ob * z.y;
      }
    }
  }
  if (!ALONE && !share && rb < batch && t == 0)
    out[rb * g.n_out] = __longlong_as_double(kAloneMark);
}

// Piece/chunk geometry of a transform, or false for the direct sum.
bool chirp_geometry(int n_in, int n_out, int N, int64_t a0, int da, int64_t d0, int dd, int adj,
                    ChirpGeom* g) {
  if (n_in < kChirpMin || n_out < kChirpMin) return false;
  g->n_in = n_in;
  g->n_out = n_out;
  g->P = std::min(n_in, kFftL / 2);
  g->H = kFftL - g->P + 1;
  g->pieces = (n_in + g->P - 1) / g->P;
  g->chunks = (n_out + g->H - 1) / g->H;
  if (g->pieces * g->chunks > kChirpMaxTables) return false;
  // (a0 + da u)(d0 + dd v) = da dd (u + da a0)(v + dd d0), da, dd = +-1
  g->sigma = da * dd * (adj ? -1 : 1);
  g->N = N;
  g->A = da * a0;
  g->D = dd * d0;
  return true;
}

// Whether chirp_pairs_kernel takes n samples at lo of N points: chirp lengths,
// one piece, the first sample at the grid's zero, two chunks at most.
bool chirp_pairs_ok(int n, int N, int lo) {
  return n >= kChirpMin && n <= kFftL / 2 && lo == N / 2 && N <= 2 * (kFftL - n + 1);
}

// Entries (complex) of the chirp tables' workspace beyond the direct sum's
// N-entry twiddle table: the input and output chirps (n_in + n_out <= 2N)
// and the pair spectra (four for the two halves and chunks of paired rows).
int64_t chirp_workspace_entries(int64_t N) {
  if (N < kChirpMin) return 0;
  const int64_t per = (N + kFftL / 2 - 1) / (kFftL / 2);   // pieces or chunks, at most
  return 2 * N + std::min<int64_t>(kChirpMaxTables, std::max<int64_t>(4, per * per)) * kFftL;
}

}  // namespace
}  // namespace qsx

using namespace qsx;

extern "C" int64_t qsx_fourier_workspace_bytes(int32_t N) {
  if (N < 1) return -1;
  return ((int64_t)N + chirp_workspace_entries(N)) * (int64_t)sizeof(double2);
}

extern "C" int32_t qsx_fourier_transform(const void* x, int64_t batch, int32_t n, int32_t N,
                                         int32_t lo, int32_t sign, double dt, int32_t adjoint,
                                         void* workspace, void* out, void* stream) {
  QSX_CHECK_ARG(x && out && workspace, "qsx_fourier_transform: null pointer");
  QSX_CHECK_ARG(n >= 1 && N >= n && lo >= 0 && lo + n <= N && batch >= 1,
                "qsx_fourier_transform: bad sizes n=%d N=%d lo=%d batch=%lld", n, N, lo,
                (long long)batch);
  QSX_CHECK_ARG(sign == 1 || sign == -1, "qsx_fourier_transform: sign must be +1 or -1");
  hipStream_t s = as_stream(stream);
  double2* T = static_cast<double2*>(workspace);
  const int64_t c = N / 2;
  // output index r -> s_r = a0 + da * r; sample index j -> lo + j - c
  const int64_t sa0 = sign == -1 ? -c : (int64_t)N - 1 - c;
  const int sda = sign == -1 ? 1 : -1;
  const int64_t ja0 = (int64_t)lo - c;
  const int n_out = adjoint ? n : N, n_in = adjoint ? N : n;
  const int64_t a0 = adjoint ? ja0 : sa0, d0 = adjoint ? sa0 : ja0;
  const int da = adjoint ? 1 : sda, dd = adjoint ? sda : 1;
  ChirpGeom g;
  if (chirp_geometry(n_in, n_out, N, a0, da, d0, dd, adjoint != 0, &g)) {
    double2* cin = T + N;
    double2* cout = cin + n_in;
    double2* Gt = cin + 2 * (int64_t)N;
    hipLaunchKernelGGL(chirp_vectors_kernel, dim3((unsigned)((std::max(n_in, n_out) + 255) / 256)),
                       dim3(256), 0, s, g, cin, cout);
    QSX_CHECK_HIP(hipFuncSetAttribute((const void*)chirp_tables_kernel,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFftLds));
    QSX_CHECK_HIP(hipFuncSetAttribute((const void*)chirp_rows_kernel,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFftLds));
    hipLaunchKernelGGL(chirp_tables_kernel, dim3(g.pieces * g.chunks), dim3(kFftThreads), kFftLds,
                       s, g, Gt);
    const unsigned gx = (unsigned)std::min<int64_t>(batch, 1 << 20);
    hipLaunchKernelGGL(chirp_rows_kernel, dim3(gx), dim3(kFftThreads), kFftLds, s,
                       static_cast<const double2*>(x), batch, g, (const double2*)cin,
                       (const double2*)cout, (const double2*)Gt, dt, static_cast<double2*>(out));
    QSX_CHECK_HIP(hipGetLastError());
    return QSX_OK;
  }
  hipLaunchKernelGGL(dft_twiddle_kernel, dim3((N + kDftThreads - 1) / kDftThreads), dim3(kDftThreads),
                     0, s, N, T);
  // the pairs q = |a| of the outputs' a = a0 .. a0 + da (n_out - 1), which lie in
  // [-N/2, N/2]: all of 0 .. N/2 forward, the samples' own in the adjoint
  const int64_t a1 = a0 + (int64_t)da * (n_out - 1);
  const int64_t amin = std::min(a0, a1), amax = std::max(a0, a1);
  const int q0 = (int)(amin > 0 ? amin : (amax < 0 ? -amax : 0));
  const int nq = (int)std::max(-amin, amax) - q0 + 1;
  // more rows per thread while that leaves two wavefronts (four rows) or one (two
  // rows) for every SIMD; work-groups of as few wavefronts as the pairs need
  // where they fill the chip, else all 256 threads stage the samples
  const int64_t gx = (nq + kDftThreads - 1) / kDftThreads;
  int waves = (int)(((nq + gx - 1) / gx + 63) / 64);
  const int R = gx * waves * ((batch + 3) / 4) >= 2048 ? 4
              : (gx * waves * ((batch + 1) / 2) >= 1024 ? 2 : 1);
  if (R < 4) waves = kDftThreads / 64;
  const auto kern = R == 4 ? dft_kernel<4> : (R == 2 ? dft_kernel<2> : dft_kernel<1>);
  const unsigned gy = (unsigned)std::min<int64_t>((batch + R - 1) / R, 65535);
  hipLaunchKernelGGL(kern, dim3((unsigned)gx, gy), dim3(64 * waves), 0, s,
                     static_cast<const double2*>(x), batch, n_in, n_out, N, a0, da, d0, dd, q0,
                     nq, (int)(adjoint != 0), dt, T, static_cast<double2*>(out));
  QSX_CHECK_HIP(hipGetLastError());
  return QSX_OK;
}

extern "C" int32_t qsx_fourier_real_pairs(int32_t n, int32_t N, int32_t lo) {
  return n >= 1 && N >= n && lo >= 0 && lo <= N - n && chirp_pairs_ok(n, N, lo) ? 1 : 0;
}

extern "C" int32_t qsx_fourier_transform_real(const void* x, int64_t batch, int32_t n, int32_t N,
                                              int32_t lo, int32_t sign, double dt,
                                              void* workspace, double* out, void* stream) {
  QSX_CHECK_ARG(x && out && workspace, "qsx_fourier_transform_real: null pointer");
  QSX_CHECK_ARG(batch >= 1 && batch < (int64_t)1 << 31 && qsx_fourier_real_pairs(n, N, lo),
                "qsx_fourier_transform_real: bad sizes n=%d N=%d lo=%d batch=%lld", n, N, lo,
                (long long)batch);
  QSX_CHECK_ARG(sign == 1 || sign == -1, "qsx_fourier_transform_real: sign must be +1 or -1");
  hipStream_t s = as_stream(stream);
  double2* cin = static_cast<double2*>(workspace) + N;
  double2* cout = cin + n;
  double2* Gt = cin + 2 * (int64_t)N;
  // output index r -> s_r = a0 + da r as in the complex transform; D = 0
  const int64_t c = N / 2, a0 = sign == -1 ? -c : (int64_t)N - 1 - c;
  const int da = sign == -1 ? 1 : -1;
  ChirpGeom g;
  g.n_in = n;
  g.n_out = N;
  g.P = n;
  g.H = kFftL - n + 1;
  g.pieces = 2;
  g.chunks = (N + g.H - 1) / g.H;
  g.sigma = da;
  g.N = N;
  g.A = da * a0;
  g.D = 0;
  hipLaunchKernelGGL(chirp_vectors_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, g,
                     cin, cout);
  g.D = -n;                          // the tables' pieces: v = -n .. -1, then 0 .. n - 1
  QSX_CHECK_HIP(hipFuncSetAttribute((const void*)chirp_tables_kernel,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFftLds));
  for (const void* k : {(const void*)chirp_pairs_kernel<false>, (const void*)chirp_pairs_kernel<true>})
    QSX_CHECK_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFftLds));
  hipLaunchKernelGGL(chirp_tables_kernel, dim3(2 * g.chunks), dim3(kFftThreads), kFftLds, s, g,
                     Gt);
  for (const auto k : {chirp_pairs_kernel<false>, chirp_pairs_kernel<true>})
    hipLaunchKernelGGL(k, dim3((unsigned)((batch + 1) / 2)), dim3(kFftThreads), kFftLds, s,
                       static_cast<const double2*>(x), batch, g, (const double2*)cin,
                       (const double2*)cout, (const double2*)Gt, dt, out);
  QSX_CHECK_HIP(hipGetLastError());
  return QSX_OK;
}
