// Householder QR of a column-major working matrix (FP64 complex), used to
// precondition the one-sided Jacobi SVD (Jacobi on R^H converges in a few
// sweeps even for strongly graded spectra, where Jacobi on A needs tens) and
// to orthonormalise sketches.
//
// Storage: A_cm holds ncol columns of length len (len >= ncol), column c at
// A_cm + c * len.  qr_factor leaves R[0..c, c] in rows 0..c of column c (the
// rows below are scratch), tau, and the reflectors explicitly: row c of Vall
// (length len) is v_c, zeros above row c included.
//
// Up to 1024 rows both kernels keep columns in registers, one column's rows spread
// over the 64 lanes of a wavefront, so a dot product is a few FMAs per lane and one
// wavefront reduction (wave.h).  A panel is one workgroup of eight wavefronts
// with one barrier per column; the trailing columns then take the panel's
// reflectors one after the other in one launch, every column by itself (no
// compact-WY factor, no GEMMs).  Longer columns stay in memory.
//
// Reflector convention: H = I - tau v v^H with H^H [alpha; x] = [beta; 0], beta
// real of the sign opposite to Re alpha, v = [alpha - beta; x] (not scaled to a
// leading 1: that needs a division per column and nothing reads it) and
// tau = -1 / (beta conj(alpha - beta)).
#include <cmath>

#include "jacobi_inner.h"
#include "wave.h"

namespace seemps {
namespace {

__device__ __forceinline__ double2 rscale(double f, double2 x) {
  return make_double2(f * x.x, f * x.y);
}

struct Reflector {
  double beta;
  double2 d, tau;  // (alpha - beta) up, tau
  double up;       // v = up [alpha - beta; x]
  bool any;        // false: H = I
};

// None for a column of squared norm below 1e-300 (tau, about 1 / |v|^2, nears the
// largest number there); NaN gets one, and spreads.
__device__ __forceinline__ Reflector make_reflector(double2 alpha, double xnorm2) {
  Reflector h;
  h.beta = alpha.x;
  h.d = h.tau = make_double2(0.0, 0.0);
  h.up = 1.0;
  const double s = cabs2(alpha) + xnorm2;
  h.any = !(xnorm2 == 0.0 && alpha.y == 0.0) && !(s < 1e-300);
  if (h.any) {
    const double r = jac::rsqrt_nr(s), sg = (alpha.x >= 0.0) ? -1.0 : 1.0;
    h.beta = sg * (s * r);
    h.d = make_double2(alpha.x - h.beta, alpha.y);
    const double q = jac::rcp_nr(cabs2(h.d)), ib = -sg * r;  // 1 / |d|^2, -1 / beta
    h.tau = make_double2((h.d.x * ib) * q, (h.d.y * ib) * q);
  }
  return h;
}

// The reflector of such a column, v scaled up by a power of two.  Asked for where
// make_reflector gave none, so that the other columns do not pay for it (a test of the
// norm and a scale in that chain made the panels 5 % slower).
__device__ __forceinline__ Reflector tiny_reflector(double2 alpha, double xnorm2) {
  Reflector h = make_reflector(rscale(0x1p500, alpha), (xnorm2 * 0x1p500) * 0x1p500);
  h.beta *= 0x1p-500;
  h.up = 0x1p500;
  return h;
}

// Panel of nb <= NW CPW columns from j0 on, L = len - j0 <= 64 RPT rows.
// Wavefront w holds columns w, w + NW, ... (CPW of them), lane l rows l,
// l + 64, ... (RPT).  Step j: the unscaled column j is in LDS (published by its
// owner at the end of the step before); every wavefront forms its norm below
// the diagonal and its dot products with the wavefront's own later columns,
// derives the reflector (redundantly, the same arithmetic everywhere) and
// updates those columns in registers; the owner of column j + 1 publishes it.
// One barrier per column.
//
// Bound by instruction issue on one CU, half of it the reductions (14
// instructions a column against 8 FMAs a row and column).  64 columns of 64
// rows take 80 us, 16 of 512 rows 23 us; with the panel in LDS instead (every
// update a read and a write there) 16 columns took 54 and 64 us.  Eight
// wavefronts: each derives the reflector by itself, and 16 of them spent 125 us
// on the 64 x 64 panel.
template <int NW, int RPT, int CPW>
__global__ __launch_bounds__(64 * NW) void qr_panel(double2* __restrict__ A, int64_t len,
                                                             int64_t j0, int nb,
                                                             double2* __restrict__ tau,
                                                             double2* __restrict__ Vall) {
  __shared__ double2 xs[2][64 * RPT];
  __shared__ double2 s_tau[NW * CPW];
  __shared__ double s_beta[NW * CPW];
  const int L = (int)(len - j0);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  double2 a[CPW][RPT];
#pragma unroll
  for (int i = 0; i < CPW; ++i) {
    const int c = wv + NW * i;
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int row = lane + 64 * r;
      a[i][r] = (c < nb && row < L) ? A[(j0 + c) * len + j0 + row] : make_double2(0.0, 0.0);
    }
  }
  if (wv == 0) {
#pragma unroll
    for (int r = 0; r < RPT; ++r) xs[0][lane + 64 * r] = a[0][r];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < CPW; ++i) {
    for (int w = 0; w < NW; ++w) {
      const int j = NW * i + w;
      if (j >= nb) break;
      const double2* xb = xs[j & 1];
      double2 x[RPT];
      double nn = 0.0;
#pragma unroll
      for (int r = 0; r < RPT; ++r) {
        x[r] = (lane + 64 * r > j) ? xb[lane + 64 * r] : make_double2(0.0, 0.0);
        nn += cabs2(x[r]);
      }
      const double2 alpha = xb[j];
      double2 d[CPW];
#pragma unroll
      for (int k = 0; k < CPW; ++k) {
        d[k] = make_double2(0.0, 0.0);
        if (k < i) continue;
#pragma unroll
        for (int r = 0; r < RPT; ++r) d[k] = cfmac(x[r], a[k][r], d[k]);
      }
      nn = wave::sum(nn);
#pragma unroll
      for (int k = i; k < CPW; k += 2) {
        if (k + 1 < CPW)
          wave::sum4(d[k], d[k + 1]);
        else
          d[k] = wave::sum2(d[k]);
      }
      Reflector h = make_reflector(alpha, nn);
      if (!h.any) {
        h = tiny_reflector(alpha, nn);
#pragma unroll
        for (int r = 0; r < RPT; ++r) x[r] = rscale(h.up, x[r]);
#pragma unroll
        for (int k = 0; k < CPW; ++k) d[k] = rscale(h.up, d[k]);
      }
#pragma unroll
      for (int r = 0; r < RPT; ++r)
        if (lane + 64 * r == j) x[r] = h.d;  // x is v from here on
      if (h.any) {
        // c <- c - conj(tau) (v^H c) v,  v^H c = x^H c + conj(d) c[j]
        const double2 ct = make_double2(h.tau.x, -h.tau.y);
#pragma unroll
        for (int k = i; k < CPW; ++k) {
          if (k == i && wv <= w) continue;  // column j itself or an earlier one
          const double2 cj = make_double2(wave::bcast(a[k][(NW * i) / 64].x, j & 63),
                                          wave::bcast(a[k][(NW * i) / 64].y, j & 63));
          const double2 f = cmul(ct, cfmac(h.d, cj, d[k]));
          const double2 g = make_double2(-f.x, -f.y);
#pragma unroll
          for (int r = 0; r < RPT; ++r) a[k][r] = cfma(g, x[r], a[k][r]);
        }
      }
      if (wv == w) {
        // column j is done: R above the diagonal, the reflector from it on
#pragma unroll
        for (int r = 0; r < RPT; ++r)
          if (lane + 64 * r >= j) a[i][r] = x[r];
        if (lane == 0) {
          s_beta[j] = h.beta;
          s_tau[j] = h.tau;
        }
      }
      // the next column's owner publishes it
      const int wn = (w + 1) % NW;
      if (wv == wn) {
        double2* nx = xs[(j + 1) & 1];
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
          if (w + 1 < NW)
            nx[lane + 64 * r] = a[i][r];
          else if (i + 1 < CPW)
            nx[lane + 64 * r] = a[i + 1 < CPW ? i + 1 : i][r];
        }
      }
      __syncthreads();
    }
  }
#pragma unroll
  for (int i = 0; i < CPW; ++i) {
    const int c = wv + NW * i;
    if (c >= nb) continue;
    double2* v = Vall + (j0 + c) * len;
    for (int64_t row = lane; row < j0; row += 64) v[row] = make_double2(0.0, 0.0);
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int row = lane + 64 * r;
      if (row < L) v[j0 + row] = (row < c) ? make_double2(0.0, 0.0) : a[i][r];
      if (row < L && row <= c)
        A[(j0 + c) * len + j0 + row] = (row < c) ? a[i][r] : make_double2(s_beta[c], 0.0);
    }
    if (lane == 0) tau[j0 + c] = s_tau[c];
  }
}

// Row q of a matrix with L double2 a row, as a buffer resource: reads past the
// row's end give zero, so the lanes need no bounds tests (a test would put each
// load behind a branch, and the loads ahead would wait for one another).
__device__ __forceinline__ double2 row_load(__amdgpu_buffer_rsrc_t row, int elem) {
  const auto w = __builtin_amdgcn_raw_buffer_load_b128(row, elem * 16, 0, 0);
  return make_double2(__hiloint2double((int)w[1], (int)w[0]), __hiloint2double((int)w[3], (int)w[2]));
}

// Reflectors j1 - 1 .. j0 (FORWARD: j0 .. j1 - 1, adjoint) on the columns of Y
// (ny of length len), rows r0 .. len - 1 (L <= 64 RPT; the reflectors are zero
// above r0).  One wavefront per CW columns, its rows in registers; the next
// reflectors are loaded while one is applied.  Bound by the chain of the dot
// product, its reduction and the update: 0.31 us a reflector at 512 rows (8 us
// for a panel's 16 on the trailing columns, 160 us for Q of 512 reflectors on
// 512 columns; as compact-WY GEMMs three launches took 20 us a panel).
template <int RPT, int CW, bool FORWARD>
__global__ __launch_bounds__(64) void qr_reflect(double2* __restrict__ Y, int64_t len, int64_t ny,
                                                 int64_t r0, int64_t j0, int64_t j1,
                                                 const double2* __restrict__ tau,
                                                 const double2* __restrict__ Vall) {
  const int lane = threadIdx.x;
  const int L = (int)(len - r0);
  const int64_t c0 = (int64_t)blockIdx.x * CW;
  // reflectors loaded ahead of the one applied (the registers hold no more of
  // them at 1024 rows)
  constexpr int AHEAD = RPT <= 8 ? 2 : 1;
  double2 y[CW][RPT], v[AHEAD][RPT];
  const int nq = (int)(j1 - j0);
  const double2* vrow = Vall + (FORWARD ? j0 : j1 - 1) * len + r0;
  const double2* trow = tau + (FORWARD ? j0 : j1 - 1);
  auto load_v = [&](int q, double2* vq) {
    const int64_t qq = q < nq ? q : nq - 1;
    const auto row = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(vrow + (FORWARD ? qq : -qq) * len), 0, L * 16, 0x00027000);
#pragma unroll
    for (int r = 0; r < RPT; ++r) vq[r] = row_load(row, lane + 64 * r);
  };
#pragma unroll
  for (int p = 0; p < AHEAD; ++p) load_v(p, v[p]);
#pragma unroll
  for (int k = 0; k < CW; ++k)
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int row = lane + 64 * r;
      y[k][r] = (c0 + k < ny && row < L) ? Y[(c0 + k) * len + r0 + row] : make_double2(0.0, 0.0);
    }
  for (int qb = 0; qb < nq; qb += 64) {
    // 64 tau in the lanes, one readlane each
    const int ql = min(qb + lane, nq - 1);
    double2 tl = trow[FORWARD ? ql : -ql];
    if (FORWARD) tl.y = -tl.y;
    // past the last reflector tau = 0 (H = I), so that no step is conditional
    if (qb + lane >= nq) tl = make_double2(0.0, 0.0);
    const int qe = min(64, nq - qb);
    for (int q0 = 0; q0 < qe; q0 += AHEAD) {
#pragma unroll
      for (int p = 0; p < AHEAD; ++p) {
        double2 u[RPT], d[CW];
#pragma unroll
        for (int r = 0; r < RPT; ++r) u[r] = v[p][r];
        load_v(qb + q0 + p + AHEAD, v[p]);
#pragma unroll
        for (int k = 0; k < CW; ++k) {
          d[k] = make_double2(0.0, 0.0);
#pragma unroll
          for (int r = 0; r < RPT; ++r) d[k] = cfmac(u[r], y[k][r], d[k]);
        }
        if (CW == 2)
          wave::sum4(d[0], d[CW - 1]);
        else
          d[0] = wave::sum2(d[0]);
        const double2 t = make_double2(wave::bcast(tl.x, q0 + p), wave::bcast(tl.y, q0 + p));
#pragma unroll
        for (int k = 0; k < CW; ++k) {
          const double2 f = cmul(t, d[k]), g = make_double2(-f.x, -f.y);
#pragma unroll
          for (int r = 0; r < RPT; ++r) y[k][r] = cfma(g, u[r], y[k][r]);
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < CW; ++k)
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int row = lane + 64 * r;
      if (c0 + k < ny && row < L) Y[(c0 + k) * len + r0 + row] = y[k][r];
    }
}

// ---- columns longer than the registers hold (more than 64 REG_RPT rows) ------

constexpr int REG_RPT = 16;
constexpr int LONG_NB = 8;

__device__ double2 block_sum(double2 v, double2* red) {
  v = wave::sum2(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double2 s = make_double2(0.0, 0.0);
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s = cadd(s, red[w]);
  return s;
}

// y <- y - f (v^H y) v over rows [lo, len) by one workgroup, v and y in memory.
// A thread keeps the same rows (its index modulo the workgroup's size) whatever
// lo is: what it reads of y it has written itself, with no barrier between
// calls.
__device__ void long_reflect(double2* __restrict__ y, const double2* __restrict__ v, int64_t lo,
                             int64_t len, double2 f, double2* red) {
  const int64_t step = blockDim.x, tid = threadIdx.x;
  const int64_t first = tid + (lo > tid ? ceil_div(lo - tid, step) * step : 0);
  double2 d = make_double2(0.0, 0.0);
  for (int64_t r = first; r < len; r += step) d = cfmac(v[r], y[r], d);
  d = cmul(f, block_sum(d, red));
  for (int64_t r = first; r < len; r += step) {
    const double2 p = cmul(d, v[r]);
    y[r] = make_double2(y[r].x - p.x, y[r].y - p.y);
  }
}

// Panel of nb <= NB columns from j0 on, columns in memory, one workgroup.  A thread
// keeps the same rows throughout.  Step j: one pass applies reflector j to the later
// columns and forms, from the values in hand, the norm of column j + 1 below its
// diagonal and its dot products with the columns after it; a wavefront then derives
// reflector j + 1 and the factors of the next pass.  Two barriers a column.  Bound by
// what one CU moves, so panels are narrow: 16 columns of 4096 rows take 134 us in two
// of eight (and 50 on the reflectors in between), 205 in one of sixteen, and took 501
// with a pass for every dot product and every update.
constexpr int LONG_THREADS = 512;

template <int NB>
struct LongLds {
  double2 red[LONG_THREADS / 64][NB];  // wavefronts' sums: |x|^2 of the next column, x^H a_k
  double2 row[NB];                     // the next column's diagonal row
  double2 f[NB];                       // -conj(tau) v^H a_k
  Reflector h;
};

// Steps J, J + 1, .. of the panel (P, V: its columns of A and of Vall); J = -1 only
// forms the sums of column 0.
template <int NB, int J>
__device__ __forceinline__ void long_steps(double2* __restrict__ P, double2* __restrict__ V,
                                           int64_t len, int64_t j0, int nb,
                                           double2* __restrict__ tau, LongLds<NB>& L) {
  constexpr int NW = LONG_THREADS / 64, T = NB - 1 - J;  // columns after column J
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t c = j0 + J;
  const bool any = J >= 0 && L.h.any;
  double2 acc[T];
#pragma unroll
  for (int k = 0; k < T; ++k) acc[k] = make_double2(0.0, 0.0);
  for (int64_t r = j0 + threadIdx.x; r < len; r += LONG_THREADS) {
    double2 v = make_double2(0.0, 0.0);
    if (J >= 0) {
      double2* x = P + J * len + r;
      if (r >= c) v = r == c ? L.h.d : rscale(L.h.up, *x);
      V[J * len + r] = v;
      if (r == c) *x = make_double2(L.h.beta, 0.0);
      if (r < c) continue;
    }
    double2 a[T];
    double2* const p = P + (J + 1) * len + r;
#pragma unroll
    for (int k = 0; k < T; ++k) a[k] = p[min(k, nb - 2 - J) * len];
    if (any) {
#pragma unroll
      for (int k = 0; k < T; ++k) a[k] = cfma(L.f[J + 1 + k], v, a[k]);
#pragma unroll
      for (int k = 0; k < T; ++k)
        if (k < nb - 1 - J) p[k * len] = a[k];
    }
    if (r == c + 1) {
#pragma unroll
      for (int k = 0; k < T; ++k) L.row[J + 1 + k] = a[k];
    } else if (r > c + 1) {
      acc[0].x += cabs2(a[0]);
#pragma unroll
      for (int k = 1; k < T; ++k) acc[k] = cfmac(a[0], a[k], acc[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < T; k += 2) {
    if (k + 1 < T)
      wave::sum4(acc[k], acc[k + 1 < T ? k + 1 : k]);
    else
      acc[k] = wave::sum2(acc[k]);
    if (lane == 0) {
      L.red[wv][J + 1 + k] = acc[k];
      if (k + 1 < T) L.red[wv][J + 2 + k] = acc[k + 1 < T ? k + 1 : k];
    }
  }
  __syncthreads();
  if (wv == 0) {
    const int k = min(max(lane, J + 1), NB - 1);
    double2 t = make_double2(0.0, 0.0);
    for (int q = 0; q < NW; ++q) t = cadd(t, L.red[q][k]);
    const double2 alpha = L.row[J + 1];
    const double nn = wave::bcast(t.x, J + 1);
    Reflector h = make_reflector(alpha, nn);
    if (!h.any) h = tiny_reflector(alpha, nn);
    // v^H a_k = conj(d) a_k[c + 1] + up x^H a_k
    if (lane > J + 1 && lane < NB)
      L.f[k] = cmul(make_double2(-h.tau.x, h.tau.y), cfmac(h.d, L.row[k], rscale(h.up, t)));
    if (lane == 0) {
      L.h = h;
      tau[c + 1] = h.tau;
    }
  }
  __syncthreads();
  if constexpr (J + 2 < NB) {
    if (J + 2 < nb) long_steps<NB, J + 1>(P, V, len, j0, nb, tau, L);
  }
}

template <int NB>
__global__ __launch_bounds__(LONG_THREADS) void qr_panel_long(double2* __restrict__ A, int64_t len,
                                                              int64_t j0, int nb,
                                                              double2* __restrict__ tau,
                                                              double2* __restrict__ Vall) {
  __shared__ LongLds<NB> L;
  long_steps<NB, -1>(A + j0 * len, Vall + j0 * len, len, j0, nb, tau, L);
  // the last column: its reflector
  const int64_t c = j0 + nb - 1;
  for (int64_t r = j0 + threadIdx.x; r < len; r += LONG_THREADS) {
    double2* x = A + c * len + r;
    Vall[c * len + r] = r < c    ? make_double2(0.0, 0.0)
                        : r == c ? L.h.d
                                 : rscale(L.h.up, *x);
    if (r == c) *x = make_double2(L.h.beta, 0.0);
  }
}

// Reflectors j0 .. j1 - 1 (adjoint, ascending) or j1 - 1 .. j0 on one column
// of Y per workgroup, in memory.  16 reflectors on 16 columns of 20000 rows: 587 us
// with 256 threads, 259 with 1024; up to 4096 rows the barriers of 256 are the shorter.
__global__ __launch_bounds__(1024) void qr_reflect_long(double2* __restrict__ Y, int64_t len,
                                                        int64_t j0, int64_t j1, int forward,
                                                        const double2* __restrict__ tau,
                                                        const double2* __restrict__ Vall) {
  __shared__ double2 red[16];
  double2* y = Y + (int64_t)blockIdx.x * len;
  for (int64_t q = 0; q < j1 - j0; ++q) {
    const int64_t j = forward ? j0 + q : j1 - 1 - q;
    double2 t = tau[j];
    if (forward) t.y = -t.y;
    long_reflect(y, Vall + j * len, j, len, t, red);
  }
}

// Rows per lane of the smallest instantiation that holds L rows (0: none).
inline int rows_per_lane(int64_t L) {
  for (int r = 1; r <= REG_RPT; r <<= 1)
    if (L <= 64 * r) return r;
  return 0;
}

// Panel width of a register panel with r rows per lane: 64 columns up to 128
// rows, 32 up to 256, 16 up to 512, 8 beyond (eight, four, two, one columns on
// each of eight wavefronts: what the registers hold).
inline int panel_width(int r) { return r <= 2 ? 64 : r <= 4 ? 32 : r <= 8 ? 16 : 8; }

int panel(int r, double2* A, int64_t len, int64_t j0, int nb, double2* tau, double2* Vall,
          hipStream_t stream) {
  TimedLaunch timed("qr_panel", stream, 0.0);
#define SEEMPS_PANEL(W, R, C)                                                             \
  hipLaunchKernelGGL((qr_panel<W, R, C>), dim3(1), dim3(64 * W), 0, stream, A, len, j0, nb, tau, \
                     Vall)
  if (r == 1)
    SEEMPS_PANEL(8, 1, 8);
  else if (r == 2)
    SEEMPS_PANEL(8, 2, 8);
  else if (r == 4)
    SEEMPS_PANEL(8, 4, 4);
  else if (r == 8)
    SEEMPS_PANEL(8, 8, 2);
  else if (r == 16)
    SEEMPS_PANEL(8, 16, 1);
  else
    hipLaunchKernelGGL(nb <= 4 ? qr_panel_long<4> : qr_panel_long<LONG_NB>,
                       dim3(1), dim3(LONG_THREADS), 0, stream, A, len, j0, nb, tau, Vall);
#undef SEEMPS_PANEL
  return check_launch("qr_panel");
}

// Reflectors [j0, j1) on the ny columns of Y, rows r0 .. len - 1.
template <bool FORWARD>
int reflect(double2* Y, int64_t len, int64_t ny, int64_t r0, int64_t j0, int64_t j1,
            const double2* tau, const double2* Vall, hipStream_t stream) {
  if (ny <= 0 || j1 <= j0) return SEEMPS_OK;
  TimedLaunch timed("qr_reflect", stream, 16.0 * (double)(len - r0) * ny * (j1 - j0));
  // two columns per wavefront share each load of a reflector once one column
  // each would put more than a wavefront on every SIMD
  const bool two = ny > 1024;
  const dim3 grid((unsigned)(two ? ceil_div(ny, 2) : ny)), wg(64);
#define SEEMPS_REFLECT(R)                                                                       \
  if (two)                                                                                      \
    hipLaunchKernelGGL((qr_reflect<R, 2, FORWARD>), grid, wg, 0, stream, Y, len, ny, r0, j0, j1, \
                       tau, Vall);                                                              \
  else                                                                                          \
    hipLaunchKernelGGL((qr_reflect<R, 1, FORWARD>), grid, wg, 0, stream, Y, len, ny, r0, j0, j1, \
                       tau, Vall)
  switch (rows_per_lane(len - r0)) {
    case 1: SEEMPS_REFLECT(1); break;
    case 2: SEEMPS_REFLECT(2); break;
    case 4: SEEMPS_REFLECT(4); break;
    case 8: SEEMPS_REFLECT(8); break;
    case 16: SEEMPS_REFLECT(16); break;
    default:
      hipLaunchKernelGGL(qr_reflect_long, dim3((unsigned)ny), dim3(len > 4096 ? 1024 : 256), 0,
                         stream, Y, len, j0, j1, (int)FORWARD, tau, Vall);
  }
#undef SEEMPS_REFLECT
  return check_launch("qr_reflect");
}

}  // namespace

// In-place QR of A_cm (ncol columns of length len, len >= ncol).
// Work: Vall (ncol * len complex), tau (ncol).
int qr_factor(double2* A, int64_t len, int64_t ncol, double2* Vall, double2* tau,
              hipStream_t stream) {
  int st;
  for (int64_t j0 = 0; j0 < ncol;) {
    const int r = rows_per_lane(len - j0);
    const int64_t wide = r ? panel_width(r) : LONG_NB;
    const int nb = (int)(ncol - j0 < wide ? ncol - j0 : wide);
    if ((st = panel(r, A, len, j0, nb, tau, Vall, stream))) return st;
    if ((st = reflect<true>(A + (j0 + nb) * len, len, ncol - j0 - nb, j0, j0, j0 + nb, tau, Vall,
                            stream)))
      return st;
    j0 += nb;
  }
  return SEEMPS_OK;
}

// Y <- Q Y for Y column-major (ny columns of length len), Q from qr_factor with
// ncol columns.
int qr_apply_q(double2* Y, int64_t len, int64_t ny, int64_t ncol, const double2* Vall,
               const double2* tau, hipStream_t stream) {
  return reflect<false>(Y, len, ny, 0, 0, ncol, tau, Vall, stream);
}

}  // namespace seemps
