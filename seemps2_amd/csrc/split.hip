// Truncated split of a matrix, A ~ U_D (S VH)_D (mode 0) or (U S)_D VH_D (mode 1),
// by the QR-preconditioned Jacobi of svd.hip.
//
// With B = A (m >= n) or A^H of ncol = min(m, n) columns and P its columns by
// decreasing norm: B P = Q R, X = R^H, X V = W = U_X Sigma.  The right singular
// vectors of B are P U_X, the left ones Q V.  The host waits once, for D and the
// error, which a kernel writes to pinned memory with the Jacobi's status; Q is
// applied to the D kept columns of V only, and the two factors are written in
// one launch.  Replaces svd.pxi:17-83 with schmidt.pxi:123-174 of the reference.
#include <cmath>

#include "svd_work.h"
#include "wave.h"

namespace seemps {
namespace {

struct SplitWork {
  SvdWork w;           // Y unused
  double* S;           // ncol, descending
  int64_t* D;
};

SvdShape split_shape(int64_t m, int64_t n, int num_cu) {
  SvdShape s;
  s.m = m;
  s.n = n;
  s.transposed = m < n;  // B = A^H
  s.ncol = m < n ? m : n;
  s.lenA = m < n ? n : m;
  s.use_qr = 1;
  s.len = s.ncol;
  jacobi_shape(&s, num_cu);
  return s;
}

// base == nullptr only sizes the layout.
int64_t split_carve(const SvdShape& s, void* base, SplitWork* out) {
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    void* q = base ? (void*)((char*)base + off) : nullptr;
    off += align256(bytes);
    return q;
  };
  SplitWork x;
  x.w.Y = nullptr;
  x.w.Acm = (double2*)take(s.ncol * s.lenA * 16);
  x.w.Vall = (double2*)take(s.ncol * s.lenA * 16);
  x.w.tau = (double2*)take(s.ncol * 16);
  x.w.W = (double2*)take(s.ncolp * s.len * 16);
  x.w.V = (double2*)take(s.ncolp * s.ncolp * 16);
  x.w.part = (double2*)take(2 * s.P * RMAX * PW * PW * 16);
  x.w.sync = (unsigned int*)take(sync_words(s) * 4);
  x.w.colnrm = (double*)take(s.ncol * 8);
  x.w.colperm = (int*)take(s.ncol * 4);
  x.w.sigma = (double*)take(s.ncolp * 8);
  x.w.perm = (int*)take(s.ncolp * 4);
  x.w.ctrl = (Ctrl*)take(sizeof(Ctrl));
  x.S = (double*)take(s.ncol * 8);
  x.D = (int64_t*)take(8);
  if (out) *out = x;
  return off;
}

// What the host reads after the Jacobi, in pinned memory.
struct SplitResult {
  int64_t D;
  double err;
  int tiny;                 // a kept singular value is negligible
  int status[3];            // of the Jacobi: sweeps, converged, aborted
};

// Squared norms of the columns of B: of A's rows (adj, a wavefront each) ...
__global__ __launch_bounds__(256) void row_norms(int64_t rows, int64_t cols,
                                                 const double2* __restrict__ A,
                                                 double* __restrict__ nrm) {
  const int64_t r = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  double acc = 0.0;
  for (int64_t c = threadIdx.x & 63; c < cols; c += 64) acc += cabs2(A[r * cols + c]);
  acc = wave::sum(acc);
  if ((threadIdx.x & 63) == 0) nrm[r] = acc;
}
// ... or of A's columns (cw = 16, 32 or 64 to a workgroup; the rows over
// its wavefronts and their 64 / cw groups of lanes).
__global__ __launch_bounds__(1024) void column_norms(int64_t rows, int64_t cols, int cw,
                                                     const double2* __restrict__ A,
                                                     double* __restrict__ nrm) {
  __shared__ double red[1024];
  const int64_t c = (int64_t)blockIdx.x * cw + (threadIdx.x & (cw - 1));
  double acc = 0.0;
  if (c < cols) {
#pragma unroll 4
    for (int64_t r = threadIdx.x / cw; r < rows; r += 1024 / cw) acc += cabs2(A[r * cols + c]);
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  if ((int)threadIdx.x < cw && c < cols) {
    for (int q = cw; q < 1024; q += cw) acc += red[q + threadIdx.x];
    nrm[c] = acc;
  }
}

// Block sums over 256 threads, in every thread.
__device__ double block_sum256(double x, double* red) {
  x = wave::sum(x);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// Workgroup c puts column c of B at its place among the columns by decreasing
// norm (ties by index; NaN last, so the places form a permutation), and the
// grid resets the control block (tiny2 from the norms' sum) and the counters.
__global__ __launch_bounds__(256) void load_sorted(SvdShape s, const double2* __restrict__ A,
                                                   SvdWork w) {
  __shared__ double red[4];
  const int64_t c = blockIdx.x;
  auto key = [&](int64_t d) {
    const double x = w.colnrm[d];
    return isnan(x) ? -1.0 : x;
  };
  const double kc = key(c);
  double before = 0.0, total = 0.0;
  for (int64_t d = threadIdx.x; d < s.ncol; d += 256) {
    const double kd = key(d);
    before += (kd > kc || (kd == kc && d < c)) ? 1.0 : 0.0;
    total += w.colnrm[d];
  }
  const int64_t pos = (int64_t)block_sum256(before, red);
  if (threadIdx.x == 0) w.colperm[pos] = (int)c;
  double2* dst = w.Acm + pos * s.lenA;
  for (int64_t r = threadIdx.x; r < s.lenA; r += 256) {
    double2 v = s.transposed ? A[c * s.n + r] : A[r * s.n + c];
    if (s.transposed) v.y = -v.y;
    dst[r] = v;
  }
  for (int64_t e = c * 256 + threadIdx.x; e < sync_words(s); e += (int64_t)gridDim.x * 256)
    w.sync[e] = 0u;
  if (c == 0) {
    total = block_sum256(total, red);
    if (threadIdx.x == 0) {
      Ctrl* k = w.ctrl;
      k->barrier = k->abort = 0;
      for (int i = 0; i < 3; ++i) k->off[i] = 0;
      for (int i = 0; i < 4; ++i) k->info[i] = 0;
      for (int i = 0; i < 8; ++i) k->prof[i] = 0;
      k->frob2 = total;
      k->tiny2 = negligible2(s.len, total);
    }
  }
}

// The columns of X = R^H, W[c][k] = conj(R[c][k]) for k >= c (zero elsewhere and
// in the padding; column k of R at Acm + k lenA), and V = identity.
__global__ void load_adjoint(SvdShape s, SvdWork w) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < s.ncolp * s.ncolp;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = e / s.ncolp, k = e % s.ncolp;
    w.V[e] = make_double2((c == k && c < s.ncol) ? 1.0 : 0.0, 0.0);
    if (k >= s.len) continue;
    double2 v = make_double2(0.0, 0.0);
    if (c < s.ncol && k >= c) {
      v = w.Acm[k * s.lenA + c];
      v.y = -v.y;
    }
    w.W[c * s.len + k] = v;
  }
}

// sigma_c = ||w_c||, a wavefront a column.
__global__ __launch_bounds__(256) void column_sigma(SvdShape s, SvdWork w) {
  const int64_t c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= s.ncolp) return;
  double acc = 0.0;
  for (int64_t r = threadIdx.x & 63; r < s.len; r += 64) acc += cabs2(w.W[c * s.len + r]);
  acc = wave::sum(acc);
  if ((threadIdx.x & 63) == 0) w.sigma[c] = sqrt(acc);
}

// Order of the singular values (descending, ties by index, NaN last), the
// truncation rule on them and the host's result.  One workgroup; 8 lanes count
// the predecessors of a value.  keys: 2 ncolp doubles (LDS, or memory for
// spectra too long for it).
constexpr int64_t SORT_LDS = 4096;
template <bool STAGED>
__global__ __launch_bounds__(1024) void sort_truncate(SvdShape s, SvdWork w, double* S,
                                                      int64_t* D_dev, int method, double tol,
                                                      int64_t max_bond, double* spill,
                                                      SplitResult* host, uint64_t* flag,
                                                      uint64_t ticket) {
  extern __shared__ double lds[];
  __shared__ int64_t sD;
  __shared__ int s_tiny;
  const int tid = threadIdx.x, sub = tid & 7;
  double* const key = STAGED ? lds : spill;
  double* const ss = key + s.ncolp;
  if (tid == 0) s_tiny = 0;
  for (int64_t d = tid; d < s.ncolp; d += 1024) {
    const double x = w.sigma[d];
    key[d] = isnan(x) ? -1.0 : x;
  }
  __syncthreads();
  const int nc = (int)s.ncolp;
  for (int c = tid >> 3; c < ((nc + 127) & ~127); c += 128) {
    const double kc = c < nc ? key[c] : 0.0;
    int rank = 0;
#pragma unroll 4
    for (int d = sub; d < nc; d += 8) {
      const double kd = key[d];
      rank += (int)(kd > kc) + (int)(kd == kc && d < c);
    }
    for (int o = 1; o < 8; o <<= 1) rank += __shfl_xor(rank, o, 64);
    if (c < nc && sub == 0) {
      w.perm[rank] = c;
      ss[rank] = w.sigma[c];
    }
  }
  __syncthreads();
  if (tid == 0) {
    double err = 0.0;
    truncation_rule(s.ncol, ss, method, tol, max_bond, &sD, &err);
    *D_dev = sD;
    host->D = sD;
    host->err = err;
  }
  for (int64_t k = tid; k < s.ncol; k += 1024) S[k] = ss[k];
  __syncthreads();
  const double tiny2 = w.ctrl->tiny2;
  for (int64_t k = tid; k < sD; k += 1024)
    if (!(ss[k] > 0.0 && ss[k] * ss[k] > tiny2)) atomicOr(&s_tiny, 1);
  __syncthreads();
  if (tid == 0) {
    host->tiny = s_tiny;
    host->status[0] = w.ctrl->info[0];
    host->status[1] = w.ctrl->info[1];
    host->status[2] = (int)w.ctrl->abort;
    host_publish(flag, ticket);
  }
}

// Y[k][x] = V[perm[k]][x], x < ncol, zero below: the kept columns, before Q.
__global__ void gather_v(SvdShape s, SvdWork w, int64_t D, double2* __restrict__ Y) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < D * s.lenA;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t k = e / s.lenA, x = e % s.lenA;
    Y[e] = x < s.ncol ? w.V[(int64_t)w.perm[k] * s.ncolp + x] : make_double2(0.0, 0.0);
  }
}

// Z[k][x] = W[perm[k]][x] / S[k], zero where S[k] is negligible.
__global__ void gather_w(SvdShape s, SvdWork w, const double* __restrict__ S, int64_t D,
                         double2* __restrict__ Z) {
  const double tiny2 = w.ctrl->tiny2;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < D * s.len;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t k = e / s.len, x = e % s.len;
    const double sg = S[k];
    double2 v = make_double2(0.0, 0.0);
    if (sg > 0.0 && sg * sg > tiny2) {
      v = w.W[(int64_t)w.perm[k] * s.len + x];
      v = make_double2(v.x / sg, v.y / sg);
    }
    Z[e] = v;
  }
}

// Both factors, D columns of U (m x D) and D rows of VH.  Y: the left vectors of
// B; the right ones are W's columns, normalised (wnorm) unless they carry the
// singular values, or Z when given; the left ones times S when those do not.
// B = A: U from Y, VH from W; B = A^H: the other way round.
__global__ void store_factors(SvdShape s, SvdWork w, const double* __restrict__ S, int64_t D,
                              const double2* __restrict__ Y, const double2* __restrict__ Z,
                              int wnorm, double2* __restrict__ U, double2* __restrict__ VH) {
  const int64_t ny = D * s.lenA, nw = D * s.len;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < ny + nw;
       e += (int64_t)gridDim.x * blockDim.x) {
    const bool left = e < ny;
    const int64_t f = left ? e : e - ny, len = left ? s.lenA : s.len;
    const bool to_u = left != (s.transposed != 0);
    // consecutive threads write consecutive elements
    const int64_t k = to_u ? f % D : f / len, x = to_u ? f / D : f % len;
    double2 v;
    int64_t xo = x;
    if (left) {
      v = Y[k * s.lenA + x];
      if (wnorm) v = make_double2(v.x * S[k], v.y * S[k]);
    } else {
      xo = w.colperm[x];
      if (Z) {
        v = Z[k * s.len + x];
      } else {
        v = w.W[(int64_t)w.perm[k] * s.len + x];
        if (wnorm) v = make_double2(v.x / S[k], v.y / S[k]);
      }
    }
    if (to_u)
      U[xo * D + k] = v;
    else
      VH[k * s.n + xo] = make_double2(v.x, -v.y);
  }
}

unsigned blocks_for(int64_t n) {
  int64_t b = ceil_div(n, 256);
  if (b > 2048) b = 2048;
  if (b < 1) b = 1;
  return (unsigned)b;
}

}  // namespace

int64_t svd_split_bytes(int64_t m, int64_t n) {
  // sized for the largest row split, independent of the device
  return split_carve(split_shape(m, n, 1 << 20), nullptr, nullptr);
}

int svd_split_impl(int64_t m, int64_t n, const double2* A, int mode, int method, double tolerance,
                   int64_t max_bond, double2* outA, double2* outB, double* s_out,
                   int64_t* D_host, double* err_host, void* work, int64_t work_bytes,
                   int32_t* info, hipStream_t st_) {
  SEEMPS_CHECK_ARG(m >= 1 && n >= 1, "svd_split: empty matrix");
  SEEMPS_CHECK_ARG(mode == 0 || mode == 1, "svd_split: invalid mode");
  SEEMPS_CHECK_ARG(work_bytes >= svd_split_bytes(m, n), "svd_split: workspace too small");
  SEEMPS_CHECK_ARG(method >= 0 && method <= 3, "truncate: invalid method %d", method);
  SEEMPS_CHECK_ARG(max_bond >= 1, "truncate: invalid max bond dimension");
  DeviceInfo di;
  int st = device_info(&di);
  if (st) return st;
  char* hp = (char*)pinned_stage(PINNED_BYTES);
  SEEMPS_CHECK_ARG(hp != nullptr, "pinned host staging could not be allocated");
  SplitResult* res = (SplitResult*)hp;
  void* res_dev = nullptr;
  SEEMPS_HIP(hipHostGetDevicePointer(&res_dev, res, 0));
  const uint64_t ticket = next_ticket();
  *host_flag(hp) = 0;
  const SvdShape s = split_shape(m, n, di.num_cu);
  SplitWork x;
  split_carve(s, work, &x);
  const SvdWork& w = x.w;
  if (s.transposed)
    hipLaunchKernelGGL(row_norms, dim3((unsigned)ceil_div(m, 4)), dim3(256), 0, st_, m, n, A,
                       w.colnrm);
  else {
    int cw = 64;
    while (cw > 16 && cw / 2 >= n) cw /= 2;
    hipLaunchKernelGGL(column_norms, dim3((unsigned)ceil_div(n, cw)), dim3(1024), 0, st_, m, n, cw,
                       A, w.colnrm);
  }
  if ((st = check_launch("split norms"))) return st;
  hipLaunchKernelGGL(load_sorted, dim3((unsigned)s.ncol), dim3(256), 0, st_, s, A, w);
  if ((st = check_launch("load_sorted"))) return st;
  if ((st = qr_factor(w.Acm, s.lenA, s.ncol, w.Vall, w.tau, st_))) return st;
  hipLaunchKernelGGL(load_adjoint, dim3(blocks_for(s.ncolp * s.ncolp)), dim3(256), 0, st_, s, w);
  if ((st = check_launch("load_adjoint"))) return st;
  if ((st = jacobi_enqueue(s, w, st_))) return st;
  hipLaunchKernelGGL(column_sigma, dim3((unsigned)ceil_div(s.ncolp, 4)), dim3(256), 0, st_, s, w);
  if ((st = check_launch("column_sigma"))) return st;
  if (s.ncolp <= SORT_LDS)
    hipLaunchKernelGGL(sort_truncate<true>, dim3(1), dim3(1024), 2 * s.ncolp * sizeof(double), st_,
                       s, w, x.S, x.D, method, tolerance, max_bond, (double*)nullptr,
                       (SplitResult*)res_dev, host_flag(res_dev), ticket);
  else
    hipLaunchKernelGGL(sort_truncate<false>, dim3(1), dim3(1024), 0, st_, s, w, x.S, x.D, method,
                       tolerance, max_bond, (double*)w.part, (SplitResult*)res_dev,
                       host_flag(res_dev), ticket);
  if ((st = check_launch("sort_truncate"))) return st;
  if ((st = wait_host_flag(host_flag(hp), ticket, st_))) return st;
  const SplitResult got = *res;
  if (got.status[2] || !got.status[1] || getenv("SEEMPS_SVD_PROFILE")) {
    if ((st = svd_read_ctrl(work, (int)((char*)w.ctrl - (char*)work), info, st_))) return st;
  } else if (info) {
    info[0] = got.status[0];
    info[1] = got.status[1];
  }
  const int64_t D = got.D;
  // W's side holds the right vectors of B: it is normalised where it is the isometry
  const int wnorm = (mode == 0) == (s.transposed != 0);
  double2* Y = w.Acm;  // free by now
  hipLaunchKernelGGL(gather_v, dim3(blocks_for(D * s.lenA)), dim3(256), 0, st_, s, w, D, Y);
  if ((st = check_launch("gather_v"))) return st;
  if ((st = qr_apply_q(Y, s.lenA, D, s.ncol, w.Vall, w.tau, st_))) return st;
  double2* Z = nullptr;
  if (wnorm && got.tiny) {
    Z = w.Vall;  // free once Q is applied
    hipLaunchKernelGGL(gather_w, dim3(blocks_for(D * s.len)), dim3(256), 0, st_, s, w, x.S, D, Z);
    if ((st = check_launch("gather_w"))) return st;
    if ((st = complete_enqueue(w, Z, s.len, 1, 0, s.ncol, s.len, x.D, st_))) return st;
  }
  hipLaunchKernelGGL(store_factors, dim3(blocks_for(D * (s.lenA + s.len))), dim3(256), 0, st_, s, w,
                     x.S, D, Y, Z, wnorm, outA, outB);
  if ((st = check_launch("store_factors"))) return st;
  if (s_out)
    SEEMPS_HIP(hipMemcpyAsync(s_out, x.S, s.ncol * 8, hipMemcpyDeviceToDevice, st_));
  *D_host = D;
  *err_host = got.err;
  return SEEMPS_OK;
}

}  // namespace seemps

extern "C" int64_t seemps_svd_split_workspace(int64_t m, int64_t n) {
  return seemps::svd_split_bytes(m, n);
}

extern "C" int seemps_svd_split(int64_t m, int64_t n, const void* A, int mode, int method,
                                double tolerance, int64_t max_bond, void* outA, void* outB,
                                double* s_out, int64_t* D_host, double* err_host, void* work,
                                int64_t work_bytes, int32_t* info, void* stream) {
  return seemps::svd_split_impl(m, n, (const double2*)A, mode, method, tolerance, max_bond,
                                (double2*)outA, (double2*)outB, s_out, D_host, err_host, work,
                                work_bytes, info, (hipStream_t)stream);
}
