// DMRG two-site effective Hamiltonian: operator build, matvec and a Lanczos
// eigensolver whose Krylov recurrence, tridiagonal eigensolve and Ritz vector
// stay on the device (the host waits for the residual at the end of a restart cycle
// and, for large operators, at every second step).
//
// Replaces QuadraticForm.two_site_operator (src/seemps/operators/quadratic.py:
// 187-237) and the scipy eigsh / ARPACK call of _diagonalize_two_site
// (src/seemps/optimization/dmrg.py:15-23).
#include <cmath>

#include "common.h"
#include "gemm_direct.h"
#include "jacobi_inner.h"
#include "wave.h"

namespace seemps {
namespace {

// Hm[(c,k,l), (ko,lo,d)] = sum_e O1[c, ko, k, e] O2[e, lo, l, d]
__global__ void two_site_op_kernel(int c_, int d1, int e_, int d2, int w2,
                                   const double2* __restrict__ O1, const double2* __restrict__ O2,
                                   double2* __restrict__ Hm) {
  const int rows = c_ * d1 * d2, cols = d1 * d2 * w2;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= rows * cols) return;
  const int row = idx / cols, col = idx % cols;
  const int c = row / (d1 * d2), k = (row / d2) % d1, l = row % d2;
  const int ko = col / (d2 * w2), lo = (col / w2) % d2, d = col % w2;
  double2 acc = make_double2(0.0, 0.0);
  for (int e = 0; e < e_; ++e) {
    const double2 a = O1[((c * d1 + ko) * d1 + k) * e_ + e];
    const double2 b = O2[((e * d2 + lo) * d2 + l) * w2 + d];
    acc = cfma(a, b, acc);
  }
  Hm[idx] = acc;
}

struct PermDesc {
  int ndim;
  int64_t out_dims[8];
  int64_t in_strides_perm[8];  // stride in the input of output axis k
};

__global__ void permute_kernel(int64_t total, PermDesc p, const double2* __restrict__ in,
                               double2* __restrict__ out) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    int64_t rem = e, src = 0;
    for (int k = p.ndim - 1; k >= 0; --k) {
      const int64_t i = rem % p.out_dims[k];
      rem /= p.out_dims[k];
      src += i * p.in_strides_perm[k];
    }
    out[e] = in[src];
  }
}


// Scalars of one Lanczos cycle kept on the device.
struct LzScalars {
  double alpha[64];
  double beta[64];
  double y[64];
  double2 h;        // first-pass coefficient of the last basis vector
  int kd;           // effective Krylov dimension of the cycle
  double scl[64];   // running max |alpha| + |beta| after step j (breakdown reference)
  int brk[64];      // breakdown seen up to step j
};

// Bound of the basis size (register arrays of one entry per basis vector).
constexpr int LZ_KREG = 24;
constexpr int LZ_THREADS = 256;

constexpr int LZ_BLOCKS = 256;

// Blocks of the orthogonalisation launches: an element per thread up to one
// block per CU, so that a short vector is spread over as many CUs as it can use.
inline int lz_blocks(int64_t n) {
  int64_t b = ceil_div(n, (int64_t)LZ_THREADS);
  if (b > LZ_BLOCKS) b = LZ_BLOCKS;
  if (b < 1) b = 1;
  return (int)b;
}

// sum_b pn[b], b < nb <= 256, in every lane of a wavefront (fixed order).
__device__ __forceinline__ double lz_wave_sum(int nb, const double* __restrict__ pn) {
  const int lane = threadIdx.x & 63;
  double t[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) t[q] = pn[min(lane + 64 * q, nb - 1)];
  double r = 0.0;
#pragma unroll
  for (int q = 0; q < 4; ++q) r += lane + 64 * q < nb ? t[q] : 0.0;
  return wave::sum(r);
}

// Per-thread partials (k of the KR complex values, one real) to
// part[j * nb + block] and pn[block].
template <int KR>
__device__ __forceinline__ void lz_store_partials(const double2 (&acc)[KR], int k, double nrm,
                                                  double2* __restrict__ part,
                                                  double* __restrict__ pn) {
  __shared__ double red[LZ_THREADS / 64][2 * KR + 1];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, row = lane >> 4;
#pragma unroll
  for (int j = 0; j < KR; j += 2) {
    const double s = wave::row_sum(wave::fold16(wave::fold32(acc[j].x, acc[j].y),
                                                wave::fold32(acc[j + 1].x, acc[j + 1].y)));
    // rows 0, 2: value j; rows 1, 3: value j + 1
    if ((lane & 15) == 0) red[wv][2 * (j + (row & 1)) + (row >> 1)] = s;
  }
  nrm = wave::sum(nrm);
  if (lane == 0) red[wv][2 * KR] = nrm;
  __syncthreads();
  const int t = threadIdx.x;
  if (t < 2 * k || t == 2 * KR) {
    double v = red[0][t];
#pragma unroll
    for (int q = 1; q < LZ_THREADS / 64; ++q) v += red[q][t];
    if (t < 2 * k)
      ((double*)part)[2 * ((t >> 1) * (int64_t)gridDim.x + blockIdx.x) + (t & 1)] = v;
    else
      pn[blockIdx.x] = v;
  }
}

// hs[j] = sum_b part[j * nb + b], j < k: eight lanes per j each add every
// eighth partial, eight loads in flight, then a tree.  Fixed order: every block
// derives the same hs.  Called by every thread; the caller synchronises.
__device__ __forceinline__ void lz_load_coeffs(int k, int nb, const double2* __restrict__ part,
                                               double2* hs) {
  const int j = (int)threadIdx.x >> 3, sub = (int)threadIdx.x & 7;
  const double2* p = part + (int64_t)min(j, k - 1) * nb;
  double2 acc = make_double2(0.0, 0.0);
  for (int b0 = sub; b0 - sub < nb; b0 += 64) {
    double2 v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = p[min(b0 + 8 * q, nb - 1)];
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (b0 + 8 * q < nb) acc = cadd(acc, v[q]);
  }
#define SEEMPS_LZ_STEP(ctrl)            \
  acc.x += wave::dpp<ctrl>(acc.x);      \
  acc.y += wave::dpp<ctrl>(acc.y);
  SEEMPS_LZ_STEP(0xB1)   // quad_perm 1 0 3 2
  SEEMPS_LZ_STEP(0x4E)   // quad_perm 2 3 0 1
  SEEMPS_LZ_STEP(0x141)  // row_half_mirror
#undef SEEMPS_LZ_STEP
  if (j < k && sub == 0) hs[j] = acc;
}

// The k entries V[j][i]; those past k repeat the last.
template <int KR>
__device__ __forceinline__ void lz_column(int64_t n, int k, int64_t i,
                                          const double2* __restrict__ V, double2 (&v)[KR]) {
#pragma unroll
  for (int j = 0; j < KR; ++j) v[j] = V[min(j, k - 1) * n + i];
}

// Classical Gram-Schmidt of w = H v_{k-1} against V[0..k) with the DGKS second
// pass (applied only when the first removed more than half of |w|^2), the norm
// and the scalars, in three launches.  Each is bound by its launch and by one
// round of loads: with n = 36864 the basis is 0.6 MB a vector and lies in the
// last-level cache.  So a thread takes one element and asks for all its basis
// entries at once (KR >= k of them, a multiple of four, in registers; testing
// j < k load by load serialises them), sums go through DPP, and partials lie so
// that blocks read them back coalesced.  A step at n = 36864, averaged over k = 1..20:
// 46.6 us in four launches of four elements a thread and a fifth for the Ritz pair of
// some steps, now 15.7 (passes 3.8, 5.1 and 6.8), and 13.5 with the first pass in the
// last product of H v.
//
// Pass 1: part = block sums of conj(V_j) w; pn0 = block sums of |w|^2.
template <int KR>
__global__ __launch_bounds__(LZ_THREADS) void lz_orth1(int64_t n, int k,
                                                       const double2* __restrict__ V,
                                                       const double2* __restrict__ w,
                                                       double2* __restrict__ part,
                                                       double* __restrict__ pn0) {
  double2 acc[KR];
#pragma unroll
  for (int j = 0; j < KR; ++j) acc[j] = make_double2(0.0, 0.0);
  double nrm = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)LZ_THREADS + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * LZ_THREADS) {
    double2 v[KR];
    lz_column<KR>(n, k, i, V, v);
    const double2 x = w[i];
    nrm += cabs2(x);
#pragma unroll
    for (int j = 0; j < KR; ++j) acc[j] = cfmac(v[j], x, acc[j]);
  }
  lz_store_partials<KR>(acc, k, nrm, part, pn0);
}

// Pass 1 in the last product of H v, out = x2 R^T on 16 x 16 tiles: a thread of the
// finished tile holds one element of w, as in lz_orth1, and a tile stands for a
// block.  Saves the launch and the reading of w: at n = 36864 the product and the
// pass took 5.7 + 3.8 us, together 7.3.
template <int KR>
__global__ __launch_bounds__(LZ_THREADS) void lz_product_dots(
    int64_t M, int64_t N, int64_t K, const double2* __restrict__ x2, const double2* __restrict__ R,
    double2* __restrict__ w, int k, const double2* __restrict__ V, double2* __restrict__ part,
    double* __restrict__ pn0) {
  extern __shared__ double2 lds[];
  const int64_t tiles_n = ceil_div(N, (int64_t)16);
  const int64_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double2 x = make_double2(0.0, 0.0);
  int64_t i = 0;
  direct::tile<SEEMPS_OP_N, SEEMPS_OP_T, 1, 4, true>(
      M, N, K, x2, K, R, K, tile / tiles_n * 16, tile % tiles_n * 16, wv, lds,
      [&](int64_t m, int64_t n, double2 out) {
        i = m * N + n;
        x = out;
        w[i] = x;
      });
  double2 v[KR], acc[KR];
  lz_column<KR>(M * N, k, i, V, v);
#pragma unroll
  for (int j = 0; j < KR; ++j) acc[j] = cmulc(v[j], x);
  lz_store_partials<KR>(acc, k, cabs2(x), part, pn0);
}

// Pass 2: h = sum of the nb_in pass-1 partials (h_{k-1} is kept); w -= V h; then the
// block sums of conj(V_j) w (part_out) and |w|^2 (pn1) of the updated w.
template <int KR>
__global__ __launch_bounds__(LZ_THREADS) void lz_orth2(int64_t n, int k,
                                                       const double2* __restrict__ V,
                                                       double2* __restrict__ w, int nb_in,
                                                       const double2* __restrict__ part_in,
                                                       double2* __restrict__ part_out,
                                                       double* __restrict__ pn1,
                                                       LzScalars* __restrict__ s) {
  __shared__ double2 hs[LZ_KREG];
  const int64_t step = (int64_t)gridDim.x * LZ_THREADS;
  int64_t i = blockIdx.x * (int64_t)LZ_THREADS + threadIdx.x;
  double2 v[KR], x = w[min(i, n - 1)];
  lz_column<KR>(n, k, min(i, n - 1), V, v);
  if (threadIdx.x < LZ_KREG) hs[threadIdx.x] = make_double2(0.0, 0.0);
  __syncthreads();
  lz_load_coeffs(k, nb_in, part_in, hs);
  __syncthreads();
  if (blockIdx.x == 0 && threadIdx.x == 0) s->h = hs[k - 1];
  double2 acc[KR];
#pragma unroll
  for (int j = 0; j < KR; ++j) acc[j] = make_double2(0.0, 0.0);
  double nrm = 0.0;
  for (; i < n;) {
#pragma unroll
    for (int j = 0; j < KR; ++j) {
      const double2 t = cmul(v[j], hs[j]);
      x.x -= t.x;
      x.y -= t.y;
    }
    w[i] = x;
    nrm += cabs2(x);
#pragma unroll
    for (int j = 0; j < KR; ++j) acc[j] = cfmac(v[j], x, acc[j]);
    i += step;
    if (i < n) {
      x = w[i];
      lz_column<KR>(n, k, i, V, v);
    }
  }
  lz_store_partials<KR>(acc, k, nrm, part_out, pn1);
}

// Lowest eigenpair of the symmetric tridiagonal tridiag(beta, alpha, beta) of
// dimension kd < LZ_KREG, by one wavefront; a[] and b[] in LDS (b[kd - 1] may hold
// anything).  64-way multisection on whether T - x has a negative pivot for
// theta: ten rounds narrow the Gershgorin interval by 65^10 (about 1e-18 of its
// width), below the spacing of doubles.  Then inverse iteration for y in every
// lane alike.
//
// Both are chains of kd dependent steps, so what counts is the length of a step.
// The pivots d_i = a_i - x - b_{i-1}^2 / d_{i-1} are taken as ratios of the
// leading minors p_i = (a_i - x) p_{i-1} - b_{i-1}^2 p_{i-2} (one dependent FMA, no
// division; T is scaled by a power of two and the minors rescaled on the way, so
// they stay in range).  The shift of the inverse iteration lies just below the
// interval, where T - x is positive definite: its L D L^T needs no pivoting and
// the iterates no intermediate norm.  All loops run to the constant bound over
// rows that continue T as decoupled ones of a large diagonal.  At kd = 20 29 us as
// a kernel of its own, about 5 at the end of the step's last launch.
__device__ void lz_tridiag(const double* a, const double* b, int kd, double* theta_out,
                           double (&y)[LZ_KREG]) {
  const int lane = threadIdx.x & 63;
  const double al = lane < kd ? a[lane] : 0.0;
  const double bl = lane < kd - 1 ? fabs(b[lane]) : 0.0;
  const double bp = lane > 0 && lane < kd ? fabs(b[lane - 1]) : 0.0;
  double lo = lane < kd ? al - bl - bp : HUGE_VAL, hi = lane < kd ? al + bl + bp : -HUGE_VAL;
  for (int off = 32; off > 0; off >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, off, 64));
    hi = fmax(hi, __shfl_xor(hi, off, 64));
  }
  const double top = fmax(fabs(lo), fabs(hi));
  const double pad = 1e-12 * top + 1e-300;
  lo -= pad;
  hi += pad;
  const int ex = top > 0.0 && top < HUGE_VAL ? ilogb(top) + 1 : 0;  // |T| <= 1 scaled
  lo = ldexp(lo, -ex);
  hi = ldexp(hi, -ex);
  double A[LZ_KREG], B2[LZ_KREG];
#pragma unroll
  for (int i = 0; i < LZ_KREG; ++i) {
    A[i] = i < kd ? ldexp(a[i], -ex) : 4.0;
    const double t = i < kd - 1 ? ldexp(b[i], -ex) : 0.0;
    B2[i] = t * t;
  }
  for (int round = 0; round < 10; ++round) {
    const double x = lo + (hi - lo) * (double)(lane + 1) / 65.0;
    double p = A[0] - x, q = 1.0;
    bool neg = p < 0.0;
#pragma unroll
    for (int i = 1; i < LZ_KREG; ++i) {
      const double r = fma(A[i] - x, p, -B2[i - 1] * q);
      q = p;
      p = r;
      neg = neg || p < 0.0;
      if (i % 4 == 0) {
        const int e = p != 0.0 ? __builtin_amdgcn_frexp_exp(p) : 0;
        p = ldexp(p, -e);
        q = ldexp(q, -e);
      }
    }
    // smallest lane whose point has at least one eigenvalue below it
    const unsigned long long mask = __ballot(neg);
    const int l = mask ? __ffsll((long long)mask) - 1 : 64;
    const double nlo = l == 0 ? lo : lo + (hi - lo) * (double)l / 65.0;
    hi = l == 64 ? hi : lo + (hi - lo) * (double)(l + 1) / 65.0;
    lo = nlo;
  }
  *theta_out = ldexp(0.5 * (lo + hi), ex);
  // T - x = L D L^T, x below every eigenvalue by a rounding or two
  const double x = lo - 4.440892098500626e-16;
  double rd[LZ_KREG], l[LZ_KREG];
  double d = A[0] - x;
#pragma unroll
  for (int i = 0; i < LZ_KREG; ++i) {
    rd[i] = jac::rcp_nr(fmax(d, 2.220446049250313e-16));
    const double t = i < kd - 1 ? ldexp(b[i], -ex) : 0.0;
    l[i] = t * rd[i];
    if (i + 1 < LZ_KREG) d = fma(-t, l[i], A[i + 1] - x);
  }
#pragma unroll
  for (int i = 0; i < LZ_KREG; ++i) y[i] = i < kd ? 1.0 : 0.0;
  for (int it = 0; it < 4; ++it) {
#pragma unroll
    for (int i = 1; i < LZ_KREG; ++i) y[i] = fma(-l[i - 1], y[i - 1], y[i]);
#pragma unroll
    for (int i = 0; i < LZ_KREG; ++i) y[i] *= rd[i];
#pragma unroll
    for (int i = LZ_KREG - 2; i >= 0; --i) y[i] = fma(-l[i], y[i + 1], y[i]);
  }
  // unit norm, largest component positive
  double big = 0.0;
#pragma unroll
  for (int i = 0; i < LZ_KREG; ++i)
    if (fabs(y[i]) > fabs(big)) big = y[i];
  const double inv = 1.0 / big;
  double nn = 0.0;
#pragma unroll
  for (int i = 0; i < LZ_KREG; ++i) {
    y[i] *= inv;
    nn = fma(y[i], y[i], nn);
  }
  const double sc = 1.0 / sqrt(nn);
#pragma unroll
  for (int i = 0; i < LZ_KREG; ++i) y[i] *= sc;
}

// Pass 3 and the end of step j = k - 1.  DGKS: if |w|^2 after pass 1 is at least
// half of |w|^2 before it, the first pass was accurate and w is kept (h2 = 0);
// otherwise w -= V h2 with h2 = the pass-2 coefficients, and |w|^2 falls by
// |h2|^2 (V is orthonormal and h2 the projections on it; where that cancels, w is
// the rounding of H v and far below the breakdown bound either way).  Then
// beta_j = |w|, alpha_j = Re(h_j + h2_j), the breakdown test and
// v_{j+1} = w / beta_j (0 after a breakdown).  Block 0 records the scalars and,
// with `ritz`, the lowest Ritz pair of the k vectors: y for the combination,
// theta and the residual beta_j |y_j| to the host's `out`,
// published as ticket `ritz`.
template <int KR>
__global__ __launch_bounds__(LZ_THREADS) void lz_orth3(int64_t n, int k,
                                                       const double2* __restrict__ V,
                                                       double2* __restrict__ w,
                                                       const double2* __restrict__ part_in,
                                                       int nb0, const double* __restrict__ pn0,
                                                       const double* __restrict__ pn1,
                                                       LzScalars* __restrict__ s, uint64_t ritz,
                                                       double* __restrict__ out) {
  __shared__ double2 hs[LZ_KREG];
  __shared__ double as[LZ_KREG], bs[LZ_KREG];
  const int nb = gridDim.x, j = k - 1;
  const int64_t step = (int64_t)gridDim.x * LZ_THREADS;
  int64_t i = blockIdx.x * (int64_t)LZ_THREADS + threadIdx.x;
  double2 v[KR], x = w[min(i, n - 1)];
  lz_column<KR>(n, k, min(i, n - 1), V, v);
  const double h = s->h.x;
  const double prev = j > 0 ? s->beta[j - 1] : 0.0, scale_prev = j > 0 ? s->scl[j - 1] : 0.0;
  const int brk_prev = j > 0 ? s->brk[j - 1] : 0;
  const int kd_prev = s->kd;
  const double n0 = lz_wave_sum(nb0, pn0), n1 = lz_wave_sum(nb, pn1);
  if (threadIdx.x < LZ_KREG) hs[threadIdx.x] = make_double2(0.0, 0.0);
  __syncthreads();
  const bool second = !(n1 >= 0.5 * n0);
  if (second) lz_load_coeffs(k, nb, part_in, hs);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const double h2 = wave::sum(lane < k ? cabs2(hs[lane]) : 0.0);
  const double a = h + hs[j].x;
  const double beta = sqrt(fmax(n1 - h2, 0.0));
  const double ref = fmax(scale_prev, fabs(a) + prev);
  const int brk = brk_prev || (beta <= 1e-12 * ref);
  const double inv = brk ? 0.0 : 1.0 / beta;
  for (; i < n;) {
    if (second) {
#pragma unroll
      for (int q = 0; q < KR; ++q) {
        const double2 t = cmul(v[q], hs[q]);
        x.x -= t.x;
        x.y -= t.y;
      }
    }
    w[i] = make_double2(x.x * inv, x.y * inv);
    i += step;
    if (i < n) {
      x = w[i];
      if (second) lz_column<KR>(n, k, i, V, v);
    }
  }
  if (blockIdx.x != 0 || threadIdx.x >= 64) return;
  const int kd_new = brk && !brk_prev ? k : kd_prev;
  if (lane == 0) {
    s->alpha[j] = a;
    s->beta[j] = brk ? 0.0 : beta;
    s->scl[j] = ref;
    s->brk[j] = brk;
    s->kd = kd_new;
  }
  if (!ritz) return;
  if (lane < k) {
    as[lane] = lane == j ? a : s->alpha[lane];
    bs[lane] = lane == j ? (brk ? 0.0 : beta) : s->beta[lane];
  }
  __builtin_amdgcn_wave_barrier();
  const int kd = brk ? kd_new : k;
  double theta, y[LZ_KREG];
  lz_tridiag(as, bs, kd, &theta, y);
  if (lane == 0) {
    double last = 0.0;
#pragma unroll
    for (int q = 0; q < LZ_KREG; ++q) {
      s->y[q] = y[q];
      if (q == kd - 1) last = y[q];
    }
    out[0] = theta;
    out[1] = brk ? 0.0 : fabs(beta * last);
    host_publish(host_flag(out), ritz);
  }
}

// x = sum_{j<k} y_j V_j over V_0 (k > 0), or x unchanged (k == 0), with the
// block sums of |x|^2 in pn.
__global__ __launch_bounds__(LZ_THREADS) void lz_combine(int64_t n, int k, double2* __restrict__ x,
                                                         const double* __restrict__ y,
                                                         double* __restrict__ pn) {
  __shared__ double red[LZ_THREADS / 64];
  double nrm = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)LZ_THREADS + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * LZ_THREADS) {
    double2 acc;
    if (k == 0) {
      acc = x[i];
    } else {
      acc = make_double2(0.0, 0.0);
      for (int j0 = 0; j0 < k; j0 += 8) {
        double2 v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = x[min(j0 + q, k - 1) * n + i];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const double t = j0 + q < k ? y[j0 + q] : 0.0;
          acc.x = fma(v[q].x, t, acc.x);
          acc.y = fma(v[q].y, t, acc.y);
        }
      }
      x[i] = acc;
    }
    nrm += cabs2(acc);
  }
  nrm = wave::sum(nrm);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = nrm;
  __syncthreads();
  if (threadIdx.x == 0) pn[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// v = x / |x| from the block sums pn of |x|^2 (0 if x is), to `copy` as well if
// given; the scalars are reset for the cycle that starts from v.
__global__ __launch_bounds__(LZ_THREADS) void lz_unit(int64_t n, int nb,
                                                      const double* __restrict__ pn,
                                                      const double2* x, double2* v, double2* copy,
                                                      LzScalars* __restrict__ s) {
  const double nn = sqrt(fmax(lz_wave_sum(nb, pn), 0.0));
  const double inv = (nn > 0.0) ? 1.0 / nn : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) s->kd = 0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double2 t = x[i], u = make_double2(t.x * inv, t.y * inv);
    v[i] = u;
    if (copy) copy[i] = u;
  }
}

struct EigWork {
  double2* V;      // (m + 1) x n
  double2* x1;     // a*c*d1*d2*f
  double2* x2;     // a*d1*d2*w2*f
  double2* part;   // reduction partials (LZ_KREG x blocks)
  double2* part2;  // second-pass partials (LZ_KREG x blocks)
  double* pnorm;   // partial squared norms (2 x blocks: before pass 1, after it)
  double2* ks;     // split-K partials of the matvec GEMMs
  LzScalars* sc;
};

inline int64_t al256(int64_t x) { return (x + 255) & ~int64_t(255); }

// Split-K scratch (elements) of the two matvec GEMMs.
int64_t matvec_ks_elems(int64_t a, int64_t c, int64_t b, int64_t d1, int64_t d2, int64_t w2,
                        int64_t f, int64_t g) {
  const int64_t k1 = splitk_workspace(a * c, d1 * d2 * f, b);
  const int64_t k2 = splitk_workspace(a * d1 * d2, g, w2 * f);
  return k1 > k2 ? k1 : k2;
}

int64_t eig_bytes_full(int64_t chiL, int64_t c, int64_t d1, int64_t d2, int64_t w2, int64_t chiR,
                       int64_t m) {
  const int64_t n = chiL * d1 * d2 * chiR;
  int64_t b = 0;
  b += al256((m + 1) * n * 16);
  b += al256(chiL * c * d1 * d2 * chiR * 16);
  b += al256(chiL * d1 * d2 * w2 * chiR * 16);
  b += al256(LZ_KREG * LZ_BLOCKS * 16);
  b += al256(LZ_KREG * LZ_BLOCKS * 16);
  b += al256(2 * LZ_BLOCKS * 8);
  b += al256(matvec_ks_elems(chiL, c, chiL, d1, d2, w2, chiR, chiR) * 16);
  b += al256(sizeof(LzScalars));
  return b;
}

EigWork eig_carve(void* work, int64_t chiL, int64_t c, int64_t d1, int64_t d2, int64_t w2,
                  int64_t chiR, int64_t m) {
  const int64_t n = chiL * d1 * d2 * chiR;
  char* p = (char*)work;
  EigWork w;
  w.V = (double2*)p;
  p += al256((m + 1) * n * 16);
  w.x1 = (double2*)p;
  p += al256(chiL * c * d1 * d2 * chiR * 16);
  w.x2 = (double2*)p;
  p += al256(chiL * d1 * d2 * w2 * chiR * 16);
  w.part = (double2*)p;
  p += al256(LZ_KREG * LZ_BLOCKS * 16);
  w.part2 = (double2*)p;
  p += al256(LZ_KREG * LZ_BLOCKS * 16);
  w.pnorm = (double*)p;
  p += al256(2 * LZ_BLOCKS * 8);
  w.ks = (double2*)p;
  p += al256(matvec_ks_elems(chiL, c, chiL, d1, d2, w2, chiR, chiR) * 16);
  w.sc = (LzScalars*)p;
  return w;
}

unsigned grid_for(int64_t n) {
  int64_t b = ceil_div(n, 256);
  if (b > 2048) b = 2048;
  if (b < 1) b = 1;
  return (unsigned)b;
}

}  // namespace

// x2[a, ko, lo, d, f] = sum L[a,c,b] Hm[(c,k,l),(ko,lo,d)] v[b,k,l,f]
static int two_site_half(int64_t a, int64_t c, int64_t b, int64_t d1, int64_t d2, int64_t w2,
                         int64_t f, const double2* L, const double2* Hm, const double2* v,
                         double2* x1, double2* x2, double2* ks, int64_t ks_elems,
                         hipStream_t stream, int prec) {
  int st;
  // x1[(a,c), (k,l,f)] = L[(a,c), b] v[b, (k,l,f)]
  if ((st = zgemm_ws(SEEMPS_OP_N, SEEMPS_OP_N, a * c, d1 * d2 * f, b, make_double2(1.0, 0.0), L, b,
                     v, d1 * d2 * f, make_double2(0.0, 0.0), x1, d1 * d2 * f, ks, ks_elems, stream,
                     prec)))
    return st;
  // x2[a, (ko,lo,d), f] = sum_{(c,k,l)} x1[a, (c,k,l), f] Hm[(c,k,l), (ko,lo,d)]
  return zlocal_impl(a, c * d1 * d2, f, d1 * d2 * w2, 1, x1, Hm, x2, 0, stream);
}

// out[a, ko, lo, g] = sum L[a,c,b] Hm[(c,k,l),(ko,lo,d)] v[b,k,l,f] R[g,d,f]
int two_site_matvec_impl(int64_t a, int64_t c, int64_t b, int64_t d1, int64_t d2, int64_t w2,
                         int64_t f, int64_t g, const double2* L, const double2* Hm,
                         const double2* R, const double2* v, double2* out, double2* x1,
                         double2* x2, double2* ks, int64_t ks_elems, hipStream_t stream,
                         int prec) {
  int st;
  const double2 one = make_double2(1.0, 0.0), zero = make_double2(0.0, 0.0);
  if ((st = two_site_half(a, c, b, d1, d2, w2, f, L, Hm, v, x1, x2, ks, ks_elems, stream, prec)))
    return st;
  // out[(a,ko,lo), g] = x2[(a,ko,lo), (d,f)] R[g, (d,f)]^T
  return zgemm_ws(SEEMPS_OP_N, SEEMPS_OP_T, a * d1 * d2, g, w2 * f, one, x2, w2 * f, R, w2 * f,
                  zero, out, g, ks, ks_elems, stream, prec);
}

}  // namespace seemps

using namespace seemps;

extern "C" int seemps_two_site_operator(int64_t c, int64_t d1, int64_t e, int64_t d2, int64_t w2,
                                        const void* O1, const void* O2, void* Hm, void* stream) {
  SEEMPS_CHECK_ARG(c >= 1 && d1 >= 1 && e >= 1 && d2 >= 1 && w2 >= 1,
                   "two_site_operator: bad dimensions");
  const int64_t total = c * d1 * d2 * d1 * d2 * w2;
  hipLaunchKernelGGL(two_site_op_kernel, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0,
                     (hipStream_t)stream, (int)c, (int)d1, (int)e, (int)d2, (int)w2,
                     (const double2*)O1, (const double2*)O2, (double2*)Hm);
  return check_launch("two_site_operator");
}

extern "C" int seemps_zpermute(int ndim, const int64_t* dims, const int* perm, const void* in,
                               void* out, void* stream) {
  SEEMPS_CHECK_ARG(ndim >= 1 && ndim <= 8, "permute: 1 <= ndim <= 8");
  PermDesc p;
  p.ndim = ndim;
  int64_t strides[8];
  int64_t acc = 1;
  for (int k = ndim - 1; k >= 0; --k) {
    strides[k] = acc;
    acc *= dims[k];
  }
  int seen[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int k = 0; k < ndim; ++k) {
    SEEMPS_CHECK_ARG(perm[k] >= 0 && perm[k] < ndim && !seen[perm[k]], "permute: invalid perm");
    seen[perm[k]] = 1;
    p.out_dims[k] = dims[perm[k]];
    p.in_strides_perm[k] = strides[perm[k]];
  }
  const int64_t total = acc;
  if (total == 0) return SEEMPS_OK;
  hipLaunchKernelGGL(permute_kernel, dim3(grid_for(total)), dim3(256), 0, (hipStream_t)stream,
                     total, p, (const double2*)in, (double2*)out);
  return check_launch("permute");
}

extern "C" int64_t seemps_two_site_matvec_workspace(int64_t a, int64_t c, int64_t b, int64_t d1,
                                                    int64_t d2, int64_t w2, int64_t f) {
  return al256(a * c * d1 * d2 * f * 16) + al256(a * d1 * d2 * w2 * f * 16) +
         al256(matvec_ks_elems(a, c, b, d1, d2, w2, f, a) * 16);
}

extern "C" int seemps_two_site_matvec(int64_t a, int64_t c, int64_t b, int64_t d1, int64_t d2,
                                      int64_t w2, int64_t f, int64_t g, const void* L,
                                      const void* Hm, const void* R, const void* v, void* out,
                                      void* work, int64_t work_bytes, void* stream) {
  SEEMPS_CHECK_ARG(work_bytes >= seemps_two_site_matvec_workspace(a, c, b, d1, d2, w2, f),
                   "two_site_matvec: workspace too small");
  double2* x1 = (double2*)work;
  double2* x2 = (double2*)((char*)work + al256(a * c * d1 * d2 * f * 16));
  double2* ks = (double2*)((char*)x2 + al256(a * d1 * d2 * w2 * f * 16));
  // the split-K size depends on g too; the workspace query assumed g = a
  const int64_t ks_avail = (work_bytes - ((char*)ks - (char*)work)) / 16;
  return two_site_matvec_impl(a, c, b, d1, d2, w2, f, g, (const double2*)L, (const double2*)Hm,
                              (const double2*)R, (const double2*)v, (double2*)out, x1, x2, ks,
                              ks_avail, (hipStream_t)stream, SEEMPS_PREC_FP64);
}

extern "C" int64_t seemps_eigensolve_workspace(int64_t chiL, int64_t c, int64_t d1, int64_t d2,
                                               int64_t w2, int64_t chiR, int64_t ncv) {
  const int64_t n = chiL * d1 * d2 * chiR;
  const int64_t m = ncv < n ? ncv : n;
  return eig_bytes_full(chiL, c, d1, d2, w2, chiR, m);
}

namespace {

// The last product of wv = H V[k-1] (x2 in w.x2), its orthogonalisation against
// V[0..k), norm and scalars.
struct LzProduct {
  int64_t M, N, K;
  const double2* R;
  int prec;
  int64_t ks_elems;
};

template <int KR>
int lz_step_kr(const LzProduct& pr, int k, int nb, const EigWork& w, double2* wv, double* pn0,
               double* pn1, uint64_t ritz, double* out, hipStream_t s) {
  const int64_t n = pr.M * pr.N, tiles = ceil_div(pr.M, (int64_t)16) * ceil_div(pr.N, (int64_t)16);
  const double orth = 8.0 * n * k;
  int nb_in = nb;
  if (pr.prec == SEEMPS_PREC_FP64 && tiles <= LZ_BLOCKS &&
      gemm_on_small_tiles(SEEMPS_OP_N, SEEMPS_OP_T, pr.M, pr.N, pr.K)) {
    nb_in = (int)tiles;
    TimedLaunch timed("lz_product_dots", s, 8.0 * n * pr.K + orth);
    hipLaunchKernelGGL(lz_product_dots<KR>, dim3(nb_in), dim3(LZ_THREADS), 4 * 4 * 64 * 16, s,
                       pr.M, pr.N, pr.K, w.x2, pr.R, wv, k, w.V, w.part, pn0);
  } else {
    const int st = zgemm_ws(SEEMPS_OP_N, SEEMPS_OP_T, pr.M, pr.N, pr.K, make_double2(1.0, 0.0),
                            w.x2, pr.K, pr.R, pr.K, make_double2(0.0, 0.0), wv, pr.N, w.ks,
                            pr.ks_elems, s, pr.prec);
    if (st) return st;
    TimedLaunch timed("lz_orth1", s, orth);
    hipLaunchKernelGGL(lz_orth1<KR>, dim3(nb), dim3(LZ_THREADS), 0, s, n, k, w.V, wv, w.part,
                       pn0);
  }
  {
    TimedLaunch timed("lz_orth2", s, 2.0 * orth);
    hipLaunchKernelGGL(lz_orth2<KR>, dim3(nb), dim3(LZ_THREADS), 0, s, n, k, w.V, wv, nb_in,
                       w.part, w.part2, pn1, w.sc);
  }
  TimedLaunch timed("lz_orth3", s, orth);
  hipLaunchKernelGGL(lz_orth3<KR>, dim3(nb), dim3(LZ_THREADS), 0, s, n, k, w.V, wv, w.part2, nb_in,
                     pn0, pn1, w.sc, ritz, out);
  return check_launch("lanczos step");
}

int lz_step(const LzProduct& pr, int k, int nb, const EigWork& w, double2* wv, double* pn0,
            double* pn1, uint64_t ritz, double* out, hipStream_t s) {
  switch ((k + 3) / 4) {
    case 1: return lz_step_kr<4>(pr, k, nb, w, wv, pn0, pn1, ritz, out, s);
    case 2: return lz_step_kr<8>(pr, k, nb, w, wv, pn0, pn1, ritz, out, s);
    case 3: return lz_step_kr<12>(pr, k, nb, w, wv, pn0, pn1, ritz, out, s);
    case 4: return lz_step_kr<16>(pr, k, nb, w, wv, pn0, pn1, ritz, out, s);
    case 5: return lz_step_kr<20>(pr, k, nb, w, wv, pn0, pn1, ritz, out, s);
    default: return lz_step_kr<24>(pr, k, nb, w, wv, pn0, pn1, ritz, out, s);
  }
}

int eigensolve_impl(int prec, int64_t chiL, int64_t c, int64_t d1, int64_t d2, int64_t w2,
                    int64_t chiR, const void* L, const void* Hm, const void* R, const void* v0,
                    void* evec, int64_t ncv, double tol, int64_t maxiter, double* stats,
                    int nstats, void* work, int64_t work_bytes, hipStream_t st_) {
  SEEMPS_CHECK_ARG(prec == SEEMPS_PREC_FP64 || prec == SEEMPS_PREC_FP32 ||
                       prec == SEEMPS_PREC_MIXED,
                   "eigensolve: invalid precision");
  SEEMPS_CHECK_ARG(chiL >= 1 && chiR >= 1 && c >= 1 && w2 >= 1 && d1 >= 1 && d2 >= 1,
                   "eigensolve: bad dimensions");
  SEEMPS_CHECK_ARG(ncv >= 2 && ncv < LZ_KREG, "eigensolve: ncv must be in [2, %d]",
                   LZ_KREG - 1);
  SEEMPS_CHECK_ARG(maxiter >= 1, "eigensolve: maxiter must be positive");
  const int64_t n = chiL * d1 * d2 * chiR;
  const int64_t m = ncv < n ? ncv : n;
  SEEMPS_CHECK_ARG(work_bytes >= eig_bytes_full(chiL, c, d1, d2, w2, chiR, m),
                   "eigensolve: workspace too small");
  if (tol <= 0.0) tol = 2.220446049250313e-16;
  const double eps23 = pow(2.220446049250313e-16, 2.0 / 3.0);
  EigWork w = eig_carve(work, chiL, c, d1, d2, w2, chiR, m);
  const double2* L_ = (const double2*)L;
  const double2* H_ = (const double2*)Hm;
  const double2* R_ = (const double2*)R;
  const int nbk = lz_blocks(n);
  const int64_t ks_elems = matvec_ks_elems(chiL, c, chiL, d1, d2, w2, chiR, chiR);
  int st;
  double* pn0 = w.pnorm;
  double* pn1 = w.pnorm + LZ_BLOCKS;
  // V[0] = v0 / ||v0||
  hipLaunchKernelGGL(lz_combine, dim3(nbk), dim3(LZ_THREADS), 0, st_, n, 0, (double2*)v0,
                     w.sc->y, pn0);
  hipLaunchKernelGGL(lz_unit, dim3(nbk), dim3(LZ_THREADS), 0, st_, n, nbk, pn0,
                     (const double2*)v0, w.V, (double2*)nullptr, w.sc);
  if ((st = check_launch("lz_unit"))) return st;
  double theta = 0.0, resid = 0.0;
  double* hp = (double*)pinned_stage(PINNED_BYTES);  // host reads of the scalars
  SEEMPS_CHECK_ARG(hp != nullptr, "pinned host staging could not be allocated");
  void* dev = nullptr;
  SEEMPS_HIP(hipHostGetDevicePointer(&dev, hp, 0));
  double* hp_dev = (double*)dev;
  uint64_t ticket = 0;
  *host_flag(hp) = 0;
  int64_t matvecs = 0, matvecs32 = 0, cycle = 0;
  bool converged = false;
  // FP32 phase: the operator is applied with FP32 products, whose rounding
  // (~1e-7 relative) floors the residual near 1e-7 |theta|.  MIXED enters it
  // only when the start vector's residual (the first step's beta, from an FP64
  // product) exceeds 1e-4 |alpha|, and leaves it at 1e-5 |theta| or when a
  // restart gains less than a factor 4.  A good start vector (a converged
  // DMRG sweep) thus stays in FP64, where one short cycle suffices.
  int mv_prec = prec == SEEMPS_PREC_FP32 ? SEEMPS_PREC_FP32 : SEEMPS_PREC_FP64;
  const double fp32_floor = 1e-5, fp32_start = 1e-4;
  double last_resid = HUGE_VAL;
  // In FP64 cycles the Ritz residual is also tested after steps 4, 6, 8, ...
  // (a tridiagonal solve at the end of the step's last launch and a wait for its
  // flag each), so that a warm start stops well before ncv products; only for
  // operators large enough that a product outweighs the check.
  const bool early = n >= 8192;
  const int64_t first_check = 4, check_every = 2;
  for (cycle = 0; cycle < maxiter; ++cycle) {
    int64_t kd_eff = m;
    for (int64_t j = 0; j < m; ++j) {
      double2* vj = w.V + j * n;
      double2* wv = w.V + (j + 1) * n;
      if ((st = two_site_half(chiL, c, chiL, d1, d2, w2, chiR, L_, H_, vj, w.x1, w.x2, w.ks,
                              ks_elems, st_, mv_prec)))
        return st;
      ++matvecs;
      if (mv_prec == SEEMPS_PREC_FP32) ++matvecs32;
      // the Ritz pair after the last step and after each one that is checked
      const int64_t kd = j + 1;
      const bool check = early && mv_prec == SEEMPS_PREC_FP64 && kd < m && kd >= first_check &&
                         (kd - first_check) % check_every == 0;
      if (check || kd == m) ticket = next_ticket();
      const LzProduct last{chiL * d1 * d2, chiR, w2 * chiR, R_, mv_prec, ks_elems};
      if ((st = lz_step(last, (int)kd, nbk, w, wv, pn0, pn1, check || kd == m ? ticket : 0, hp_dev,
                        st_)))
        return st;
      if (prec == SEEMPS_PREC_MIXED && cycle == 0 && j == 0) {
        double* ab = hp + 2;
        SEEMPS_HIP(hipMemcpyAsync(&ab[0], &w.sc->alpha[0], 8, hipMemcpyDeviceToHost, st_));
        SEEMPS_HIP(hipMemcpyAsync(&ab[1], &w.sc->beta[0], 8, hipMemcpyDeviceToHost, st_));
        SEEMPS_HIP(hipStreamSynchronize(st_));
        if (ab[1] > fp32_start * fmax(eps23, fabs(ab[0]))) mv_prec = SEEMPS_PREC_FP32;
      }
      if (check) {
        if ((st = wait_host_flag(host_flag(hp), ticket, st_))) return st;
        if (hp[1] <= tol * fmax(eps23, fabs(hp[0]))) {
          kd_eff = kd;
          break;
        }
      }
    }
    // Ritz vector over V[0], normalised: the result, or the next cycle's start
    hipLaunchKernelGGL(lz_combine, dim3(nbk), dim3(LZ_THREADS), 0, st_, n, (int)kd_eff, w.V,
                       w.sc->y, pn0);
    hipLaunchKernelGGL(lz_unit, dim3(nbk), dim3(LZ_THREADS), 0, st_, n, nbk, pn0, w.V, w.V,
                       (double2*)evec, w.sc);
    if ((st = check_launch("lz_unit"))) return st;
    if ((st = wait_host_flag(host_flag(hp), ticket, st_))) return st;
    theta = hp[0];
    resid = hp[1];
    const double scale = fmax(eps23, fabs(theta));
    if (mv_prec == SEEMPS_PREC_FP32 && prec == SEEMPS_PREC_MIXED) {
      // An FP32 residual meets the test only for tolerances FP32 can resolve.
      if (tol >= fp32_floor && resid <= tol * scale) {
        converged = true;
        ++cycle;
        break;
      }
      if (resid <= fp32_floor * scale || resid > 0.25 * last_resid) mv_prec = SEEMPS_PREC_FP64;
      last_resid = resid;
      continue;
    }
    if (resid <= tol * scale) {
      converged = true;
      ++cycle;
      break;
    }
  }
  SEEMPS_HIP(hipStreamSynchronize(st_));
  if (stats) {
    stats[0] = theta;
    stats[1] = resid;
    stats[2] = (double)matvecs;
    stats[3] = (double)cycle;
    if (nstats > 4) stats[4] = (double)matvecs32;
  }
  if (!converged) {
    set_error("eigensolve: no convergence after %lld restarts (residual %g)", (long long)cycle,
              resid);
    return SEEMPS_ERR_NOCONVERGE;
  }
  return SEEMPS_OK;
}

}  // namespace

extern "C" int seemps_two_site_eigensolve(int64_t chiL, int64_t c, int64_t d1, int64_t d2,
                                          int64_t w2, int64_t chiR, const void* L, const void* Hm,
                                          const void* R, const void* v0, void* evec, int64_t ncv,
                                          double tol, int64_t maxiter, double* stats, void* work,
                                          int64_t work_bytes, void* stream) {
  return eigensolve_impl(SEEMPS_PREC_FP64, chiL, c, d1, d2, w2, chiR, L, Hm, R, v0, evec, ncv,
                         tol, maxiter, stats, 4, work, work_bytes, (hipStream_t)stream);
}

extern "C" int seemps_two_site_eigensolve_prec(int precision, int64_t chiL, int64_t c,
                                               int64_t d1, int64_t d2, int64_t w2, int64_t chiR,
                                               const void* L, const void* Hm, const void* R,
                                               const void* v0, void* evec, int64_t ncv,
                                               double tol, int64_t maxiter, double* stats5,
                                               void* work, int64_t work_bytes, void* stream) {
  return eigensolve_impl(precision, chiL, c, d1, d2, w2, chiR, L, Hm, R, v0, evec, ncv, tol,
                         maxiter, stats5, 5, work, work_bytes, (hipStream_t)stream);
}
