// Memory-bound kernels of the hot path: the small-index "local operator"
// contraction shared by MPO application, MPO environments, the DMRG matvec and
// two-site gates; elementwise scalings; deterministic two-pass reductions.
#include "common.h"

namespace seemps {
namespace {

constexpr int LIC = 64;  // rows of the operator staged in LDS at a time

// out[p, j1, q, j2] (+)= sum_i in[p, i, q] Mop[i, j1, j2]; outputs j = j1 J2 + j2.
// A thread takes one (p, q), numbered through so that no width of q leaves lanes
// idle, and JT consecutive outputs in registers.  It reads its inputs straight from
// memory, eight ahead of the eight in use, and the operator's entries, the same
// for all lanes, from LDS: one LDS read for four FMAs and one load for 4 JT.  What
// bounds a short call is its launch and the loads of i in turn, a long one the
// memory.  The J / JT groups of one (p, q) run lie next to each other on one XCD
// and share the inputs in its L2.  P = Q = 96, I = J = 20: staging inputs in LDS
// with a thread per five outputs, two LDS reads for four FMAs, took 9.6 us, this 5.6;
// P = Q = 256 16.1 -> 13.9.
template <int JT>
__global__ __launch_bounds__(256) void zlocal_kernel(int64_t PQ, int I, int64_t Q, int J1, int J2,
                                                     int groups, const double2* __restrict__ in,
                                                     const double2* __restrict__ Mop,
                                                     double2* __restrict__ out, int accumulate) {
  constexpr int U = 8;
  __shared__ double2 ms[LIC * JT];
  const int J = J1 * J2;
  const int64_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const int j0 = (int)(tile % groups) * JT;
  const int64_t e = tile / groups * 256 + threadIdx.x;
  const int64_t ec = min(e, PQ - 1);  // lanes past the end read the last, store nothing
  const int64_t p = PQ <= 0x7fffffff ? (int64_t)((uint32_t)ec / (uint32_t)Q) : ec / Q;
  const int64_t q = ec - p * Q;
  const double2* x = in + p * I * Q + q;
  double2 acc[JT];
#pragma unroll
  for (int j = 0; j < JT; ++j) acc[j] = make_double2(0.0, 0.0);
  double2 v[2][U];
  auto load = [&](int i, double2 (&r)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) r[u] = x[min(i + u, I - 1) * Q];
  };
  load(0, v[0]);
  if (I > U) load(U, v[1]);
  for (int i0 = 0; i0 < I; i0 += LIC) {
    const int n = min(LIC, I - i0);
    if (i0) __syncthreads();
    for (int t = threadIdx.x; t < n * JT; t += 256)
      ms[t] = Mop[(int64_t)(i0 + t / JT) * J + min(j0 + t % JT, J - 1)];
    __syncthreads();
    for (int b = 0; b < n; b += 2 * U) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int i = b + h * U;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (i + u < n) {
#pragma unroll
            for (int j = 0; j < JT; ++j) acc[j] = cfma(v[h][u], ms[(i + u) * JT + j], acc[j]);
          }
        }
        if (i0 + i + 2 * U < I) load(i0 + i + 2 * U, v[h]);
      }
    }
  }
  if (e >= PQ) return;
#pragma unroll
  for (int j = 0; j < JT; ++j) {
    if (j0 + j >= J) break;
    const int j1 = (j0 + j) / J2, j2 = (j0 + j) % J2;
    const int64_t o = ((p * J1 + j1) * Q + q) * J2 + j2;
    if (accumulate) acc[j] = cadd(acc[j], out[o]);
    out[o] = acc[j];
  }
}

__global__ void zaxpby_kernel(int64_t n, double2 a, const double2* __restrict__ x, int conj_x,
                              double2 b, double2* __restrict__ y, int use_b) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * blockDim.x) {
    double2 v = make_double2(0.0, 0.0);
    if (x) {
      double2 xv = x[k];
      if (conj_x) xv.y = -xv.y;
      v = cmul(a, xv);
    }
    if (use_b) v = cfma(b, y[k], v);
    y[k] = v;
  }
}

// Site-wise product of two MPS tensors (the MPS Hadamard product):
// out[(x, y), k, (u, v)] = A[x, k, u] * B[y, k, v], A (a, d, b), B (c, d, e).
__global__ void zsite_product_kernel(int64_t a, int64_t d, int64_t b, int64_t c, int64_t e,
                                     const double2* __restrict__ A, const double2* __restrict__ B,
                                     double2* __restrict__ out) {
  const int64_t be = b * e, total = a * c * d * be;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t col = i % be, row = i / be;  // row = (x * c + y) * d + k
    const int64_t k = row % d, xy = row / d;
    const int64_t x = xy / c, y = xy % c, u = col / e, v = col % e;
    out[i] = cmul(A[(x * d + k) * b + u], B[(y * d + k) * e + v]);
  }
}

__global__ void zscale2d_kernel(int64_t rows, int64_t cols, const double* __restrict__ sr,
                                const double* __restrict__ sc, const double2* __restrict__ src,
                                int64_t ld_src, double2* __restrict__ dst, int64_t ld_dst) {
  const int64_t total = rows * cols;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = e / cols, c = e % cols;
    double f = 1.0;
    if (sr) f *= sr[r];
    if (sc) f *= sc[c];
    const double2 v = src[r * ld_src + c];
    dst[r * ld_dst + c] = make_double2(f * v.x, f * v.y);
  }
}

// Block-wide sum of one complex value per thread (256 threads).
__device__ double2 block_sum(double2 v, double2* red) {
  for (int off = 32; off > 0; off >>= 1) {
    v.x += __shfl_down(v.x, off, 64);
    v.y += __shfl_down(v.y, off, 64);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double2 s = make_double2(0.0, 0.0);
  if (threadIdx.x == 0)
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s = cadd(s, red[w]);
  __syncthreads();
  return s;  // valid in thread 0
}

// Pass 1: partial[blk * nv + j] = sum over this block's chunk of conj(V_j) w.
__global__ __launch_bounds__(256) void zmdotc_partial(int64_t n, int nv,
                                                      const double2* __restrict__ V, int64_t ldv,
                                                      const double2* __restrict__ w,
                                                      double2* __restrict__ partial) {
  __shared__ double2 red[4];
  const int64_t chunk = (n + gridDim.x - 1) / gridDim.x;
  const int64_t lo = blockIdx.x * chunk;
  const int64_t hi = min(n, lo + chunk);
  for (int j = 0; j < nv; ++j) {
    double2 acc = make_double2(0.0, 0.0);
    for (int64_t k = lo + threadIdx.x; k < hi; k += blockDim.x)
      acc = cfmac(V[j * ldv + k], w[k], acc);
    const double2 s = block_sum(acc, red);
    if (threadIdx.x == 0) partial[blockIdx.x * nv + j] = s;
  }
}

// Pass 2: result[j] = sum_blk partial[blk * nv + j], fixed order.
// result[j] = sum_b partial[b * nv + j]: block j, thread t adds the partials
// b = t, t + 256, ..., then a shuffle and LDS tree (a fixed order).  256 threads.
__global__ __launch_bounds__(256) void zmdotc_final(int nblk, int nv,
                                                    const double2* __restrict__ partial,
                                                    double2* __restrict__ result) {
  __shared__ double2 red[4];
  const int j = blockIdx.x;
  double2 s = make_double2(0.0, 0.0);
  for (int b = threadIdx.x; b < nblk; b += blockDim.x) s = cadd(s, partial[b * nv + j]);
  for (int off = 32; off > 0; off >>= 1) {
    s.x += __shfl_down(s.x, off, 64);
    s.y += __shfl_down(s.y, off, 64);
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) result[j] = cadd(cadd(red[0], red[1]), cadd(red[2], red[3]));
}

}  // namespace

int64_t reduce_blocks(int64_t n) {
  int64_t b = ceil_div(n, 4096);
  if (b < 1) b = 1;
  if (b > 512) b = 512;
  return b;
}

int zlocal_impl(int64_t P, int64_t I, int64_t Q, int64_t J1, int64_t J2, const double2* in,
                const double2* Mop, double2* out, int accumulate, hipStream_t stream) {
  SEEMPS_CHECK_ARG(P >= 0 && I >= 1 && Q >= 0 && J1 >= 1 && J2 >= 1, "zlocal: bad dimensions");
  SEEMPS_CHECK_ARG(I <= 0x7fffffff && J1 * J2 <= 0x7fffffff, "zlocal: dimensions too large");
  if (P == 0 || Q == 0) return SEEMPS_OK;
  const int64_t J = J1 * J2, PQ = P * Q;
  // Ten outputs a thread where that still leaves eight wavefronts a CU or more,
  // four for more wavefronts otherwise.
  const int64_t runs = ceil_div(PQ, 256);
  const bool wide = runs * ceil_div(J, 10) >= 512 && J > 4;
  const int64_t groups = ceil_div(J, wide ? 10 : 4);
  SEEMPS_CHECK_ARG(runs * groups <= 0x7fffffff, "zlocal: grid too large");
  TimedLaunch timed("zlocal_kernel", stream, 8.0 * P * I * Q * J);
  hipLaunchKernelGGL(wide ? zlocal_kernel<10> : zlocal_kernel<4>, dim3((unsigned)(runs * groups)),
                     dim3(256), 0, stream, PQ, (int)I, Q, (int)J1, (int)J2, (int)groups, in, Mop,
                     out, accumulate);
  return check_launch("zlocal");
}

int zaxpby_impl(int64_t n, double2 a, const double2* x, int conj_x, double2 b, double2* y,
                hipStream_t stream) {
  if (n <= 0) return SEEMPS_OK;
  const int use_b = (b.x != 0.0 || b.y != 0.0);
  int64_t blocks = ceil_div(n, 256);
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(zaxpby_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, n, a, x, conj_x,
                     b, y, use_b);
  return check_launch("zaxpby");
}

int zscale2d_impl(int64_t rows, int64_t cols, const double* sr, const double* sc,
                  const double2* src, int64_t ld_src, double2* dst, int64_t ld_dst,
                  hipStream_t stream) {
  if (rows <= 0 || cols <= 0) return SEEMPS_OK;
  int64_t blocks = ceil_div(rows * cols, 256);
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(zscale2d_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, rows, cols,
                     sr, sc, src, ld_src, dst, ld_dst);
  return check_launch("zscale2d");
}

int zmdotc_impl(int64_t n, int64_t nv, const double2* V, int64_t ldv, const double2* w,
                double2* result, double2* work, hipStream_t stream) {
  SEEMPS_CHECK_ARG(nv >= 1 && nv <= 64, "zmdotc: number of vectors out of range");
  const int64_t nblk = reduce_blocks(n);
  hipLaunchKernelGGL(zmdotc_partial, dim3((unsigned)nblk), dim3(256), 0, stream, n, (int)nv, V,
                     ldv, w, work);
  int st = check_launch("zmdotc_partial");
  if (st) return st;
  hipLaunchKernelGGL(zmdotc_final, dim3((unsigned)nv), dim3(256), 0, stream, (int)nblk, (int)nv,
                     work, result);
  return check_launch("zmdotc_final");
}

}  // namespace seemps

extern "C" int seemps_zlocal(int64_t P, int64_t I, int64_t Q, int64_t J1, int64_t J2,
                             const void* in, const void* Mop, void* out, int accumulate,
                             void* stream) {
  return seemps::zlocal_impl(P, I, Q, J1, J2, (const double2*)in, (const double2*)Mop,
                             (double2*)out, accumulate, (hipStream_t)stream);
}

extern "C" int seemps_zaxpby(int64_t n, double a_re, double a_im, const void* x, int conj_x,
                             double b_re, double b_im, void* y, void* stream) {
  return seemps::zaxpby_impl(n, make_double2(a_re, a_im), (const double2*)x, conj_x,
                             make_double2(b_re, b_im), (double2*)y, (hipStream_t)stream);
}

extern "C" int seemps_zscale2d(int64_t rows, int64_t cols, const double* sr, const double* sc,
                               const void* src, int64_t ld_src, void* dst, int64_t ld_dst,
                               void* stream) {
  return seemps::zscale2d_impl(rows, cols, sr, sc, (const double2*)src, ld_src, (double2*)dst,
                               ld_dst, (hipStream_t)stream);
}

extern "C" int64_t seemps_reduce_workspace(int64_t n) {
  return seemps::reduce_blocks(n) * (int64_t)sizeof(double2);
}

extern "C" int seemps_zdotc(int64_t n, const void* x, const void* y, void* result, void* work,
                            int64_t work_bytes, void* stream) {
  SEEMPS_CHECK_ARG(n >= 0, "zdotc: negative length");
  SEEMPS_CHECK_ARG(work_bytes >= seemps_reduce_workspace(n), "zdotc: workspace too small");
  if (n == 0) {
    return seemps::zaxpby_impl(1, make_double2(0.0, 0.0), nullptr, 0, make_double2(0.0, 0.0),
                               (double2*)result, (hipStream_t)stream);
  }
  return seemps::zmdotc_impl(n, 1, (const double2*)x, n, (const double2*)y, (double2*)result,
                             (double2*)work, (hipStream_t)stream);
}

extern "C" int seemps_zsite_product(int64_t a, int64_t d, int64_t b, int64_t c, int64_t e,
                                    const void* A, const void* B, void* out, void* stream) {
  using namespace seemps;
  SEEMPS_CHECK_ARG(a >= 1 && d >= 1 && b >= 1 && c >= 1 && e >= 1,
                   "site_product: bad dimensions");
  const int64_t total = a * c * d * b * e;
  int64_t blocks = ceil_div(total, 256);
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(zsite_product_kernel, dim3((unsigned)blocks), dim3(256), 0,
                     (hipStream_t)stream, a, d, b, c, e, (const double2*)A, (const double2*)B,
                     (double2*)out);
  return check_launch("site_product");
}
