// FP64 complex SVD (QR-preconditioned one-sided block Jacobi) and the Strategy
// truncation rule.
//
// Pipeline for an m x n matrix A (B = A if m >= n, else B = A^H; B is
// len x ncol with len >= ncol):
//   1. B is copied column-major (column c contiguous).
//   2. If ncol > 16: blocked Householder QR, B = Q R (qr.hip).  The Jacobi then
//      works on X = R^H (ncol x ncol); Jacobi on R^H converges in a handful of
//      sweeps even for graded spectra (Drmac-Veselic preconditioning).
//      Otherwise the Jacobi works on B directly.
//   3. One-sided block Jacobi on the working matrix W (columns of X or B):
//      column blocks of width BW, every pair of blocks visited once per sweep
//      in a round-robin (circle) schedule; per pair the 2BW x 2BW Gram matrix is
//      formed (partial sums over row chunks in different workgroups), and the
//      rotations of an inner Hermitian Jacobi sweep on it are applied to the
//      pair's columns of W and V as they come.
//      Stops when every normalised off-diagonal |G_ij| / sqrt(G_ii G_jj) seen in
//      a sweep is below 32 sqrt(len) eps (relative orthogonality), when it was
//      already below 1e-9 (quadratic convergence: that sweep's rotations leave
//      ~1e-18), or when it stalls within 16x of the target.
//   4. sigma_k = ||w_k||, sorted descending; the W side gives the normalised
//      singular vectors of the working matrix, V (times Q in the QR path) the
//      other side.  Exactly-zero singular values get an orthonormal completion.
//
// The Jacobi runs as one cooperative persistent kernel.  With one work item
// per workgroup, steps are ordered by per-pair and per-row-chunk counters and
// one bounded grid barrier per sweep reduces the convergence measure;
// otherwise two bounded grid barriers per block step.  A workgroup that waits
// too long raises an abort flag that every waiter observes, so every wave
// always exits.
//
// Replaces _destructive_svd (src/seemps/cython/svd.pxi:17-83) and the
// truncation rules of src/seemps/cython/truncation.pxi:222-334.
#include <cmath>
#include <cstdlib>

#include "svd_work.h"
#include "wave.h"

namespace seemps {

namespace {

// Relative off-diagonal measure from which one more sweep is known to suffice
// (quadratic convergence: the sweep leaves ~1e-18 against a target ~1e-13).
constexpr double QUAD_STOP = 1e-9;
constexpr int QR_MIN_COLS = 17; // use the QR preconditioner from this many columns
constexpr int MAX_SWEEPS = 60;
constexpr unsigned long long SPIN_LIMIT = 4000000ull;

SvdShape svd_shape(int64_t m, int64_t n, int num_cu, bool precondition = true) {
  SvdShape s;
  s.m = m;
  s.n = n;
  s.transposed = (m < n);
  s.lenA = s.transposed ? n : m;
  s.ncol = s.transposed ? m : n;
  s.use_qr = precondition && (s.ncol >= QR_MIN_COLS);
  s.len = s.use_qr ? s.ncol : s.lenA;
  jacobi_shape(&s, num_cu);
  return s;
}

// Inner sweeps per step: a single pair (two blocks) has nothing to wait for, but
// tiles that replay the rotations find only the last sweep's.
__host__ __device__ inline int inner_sweeps_of(const SvdShape& s) {
  return s.nb == 2 && ceil_div(s.len, s.R) <= RT && ceil_div(s.ncolp, s.R) <= RT ? 3 : 1;
}
// First level of a full inner sweep: of 32 indices, unless a single pair holds
// fewer columns (the padding is zero and takes no rotation).
__host__ __device__ inline int inner_top_of(const SvdShape& s) {
  int top = 16;
  while (s.nb == 2 && top > 1 && s.ncol <= top) top >>= 1;
  return top;
}

#define SEEMPS_SVD_REGIONS(X)                                         \
  X(Acm, s.use_qr ? s.ncol * s.lenA : 0, double2)                     \
  X(Vall, s.use_qr ? s.ncol * s.lenA : 0, double2)                    \
  X(tau, s.use_qr ? s.ncol : 0, double2)                              \
  X(Y, s.use_qr ? s.ncol * s.lenA : 0, double2)                       \
  X(W, s.ncolp * s.len, double2)                                      \
  X(V, s.ncolp * s.ncolp, double2)                                    \
  X(part, 2 * s.P * RMAX * PW * PW, double2)                          \
  X(sync, sync_words(s), unsigned int)                                \
  X(colnrm, s.use_qr ? s.ncol : 0, double)                            \
  X(colperm, s.use_qr ? s.ncol : 0, int)                              \
  X(sigma, s.ncolp, double)                                           \
  X(perm, s.ncolp, int)                                               \
  X(ctrl, 1, Ctrl)

int64_t svd_bytes(const SvdShape& s) {
  int64_t b = 0;
#define X(name, count, type) b += align256((int64_t)(count) * (int64_t)sizeof(type));
  SEEMPS_SVD_REGIONS(X)
#undef X
  return b;
}

SvdWork svd_carve(const SvdShape& s, void* work) {
  char* p = (char*)work;
  SvdWork w;
#define X(name, count, type)                                   \
  w.name = (type*)p;                                           \
  p += align256((int64_t)(count) * (int64_t)sizeof(type));
  SEEMPS_SVD_REGIONS(X)
#undef X
  return w;
}

// B column-major: dst[c * lenA + r] = A[r][c] (m >= n) or conj(A[c][r]) (m < n),
// zero for padded columns c >= ncol (dst has ncols_dst columns).
__global__ void load_colmajor(SvdShape s, const double2* __restrict__ A, int64_t lda,
                              double2* __restrict__ dst, int64_t ncols_dst,
                              const int* __restrict__ perm) {
  const int64_t total = ncols_dst * s.lenA;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = e / s.lenA, r = e % s.lenA;
    double2 v = make_double2(0.0, 0.0);
    if (c < s.ncol) {
      const int64_t cs = perm ? perm[c] : c;  // column of B stored at position c
      if (!s.transposed) {
        v = A[r * lda + cs];
      } else {
        v = A[cs * lda + r];
        v.y = -v.y;
      }
    }
    dst[e] = v;
  }
}

// Squared norms of the ncol columns of B (B = A, or A^H when transposed).
__global__ void col_norms(SvdShape s, const double2* __restrict__ A, int64_t lda,
                          double* __restrict__ nrm) {
  for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < s.ncol;
       c += (int64_t)gridDim.x * blockDim.x) {
    double acc = 0.0;
    if (!s.transposed) {
      for (int64_t r = 0; r < s.lenA; ++r) acc += cabs2(A[r * lda + c]);
    } else {
      for (int64_t r = 0; r < s.lenA; ++r) acc += cabs2(A[c * lda + r]);
    }
    nrm[c] = acc;
  }
}

// perm[rank] = c with decreasing norm, ties by index (the QR then sees the
// heaviest columns first, which leaves R^H graded the way one-sided Jacobi
// converges fast on).
__global__ void col_rank(SvdShape s, const double* __restrict__ nrm, int* __restrict__ perm) {
  for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < s.ncol;
       c += (int64_t)gridDim.x * blockDim.x) {
    // NaN keys sort last, so the ranks always form a permutation
    const double nc = isnan(nrm[c]) ? -1.0 : nrm[c];
    int rank = 0;
    for (int64_t d = 0; d < s.ncol; ++d) {
      const double nd = isnan(nrm[d]) ? -1.0 : nrm[d];
      rank += (nd > nc || (nd == nc && d < c)) ? 1 : 0;
    }
    perm[rank] = (int)c;
  }
}

// W[c][k] = conj(R[c][k]) = conj(Acm[k][c]) for k >= c (columns of X = R^H).
__global__ void load_w_from_r(SvdShape s, const double2* __restrict__ Acm,
                              double2* __restrict__ W) {
  const int64_t total = s.ncolp * s.len;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = e / s.len, k = e % s.len;
    double2 v = make_double2(0.0, 0.0);
    if (c < s.ncol && k >= c) {
      v = Acm[k * s.lenA + c];
      v.y = -v.y;
    }
    W[e] = v;
  }
}

// V = identity on the real columns; control block reset.
__global__ void init_v_ctrl(SvdShape s, SvdWork w) {
  const int64_t totalV = s.ncolp * s.ncolp;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < totalV;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = e / s.ncolp, r = e % s.ncolp;
    w.V[e] = make_double2((c == r && c < s.ncol) ? 1.0 : 0.0, 0.0);
  }
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < sync_words(s);
       e += (int64_t)gridDim.x * blockDim.x)
    w.sync[e] = 0u;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    w.ctrl->barrier = 0;
    w.ctrl->abort = 0;
    w.ctrl->off[0] = 0;
    w.ctrl->off[1] = 0;
    w.ctrl->off[2] = 0;
    for (int i = 0; i < 4; ++i) w.ctrl->info[i] = 0;
    for (int i = 0; i < 8; ++i) w.ctrl->prof[i] = 0;
  }
}

// ctrl->frob2 = ||W||_F^2 (fixed summation order), ctrl->tiny2 = (len eps)^2 frob2.
// One workgroup of 1024 threads.
__global__ __launch_bounds__(1024) void svd_frob(SvdShape s, SvdWork w) {
  __shared__ double red[16];
  const int64_t total = s.ncolp * s.len;
  double acc = 0.0;
  for (int64_t e = threadIdx.x; e < total; e += blockDim.x) acc += cabs2(w.W[e]);
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int q = 0; q < (int)(blockDim.x >> 6); ++q) t += red[q];
    const double le = (double)s.len * 2.220446049250313e-16;
    w.ctrl->frob2 = t;
    w.ctrl->tiny2 = le * le * t;
  }
}

// Y[c][r] = V[c][r] for r < ncol, 0 below (input of Q V).
__global__ void load_y(SvdShape s, SvdWork w) {
  const int64_t total = s.ncol * s.lenA;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t c = e / s.lenA, r = e % s.lenA;
    w.Y[e] = (r < s.ncol) ? w.V[c * s.ncolp + r] : make_double2(0.0, 0.0);
  }
}

// ---- data that workgroups hand to one another --------------------------------
//
// W, V and the partial Gram matrices are read and written past the caches that
// are not coherent between the XCDs (sc1: agent scope), so a reader needs no
// cache invalidation, which would also drop what the other workgroups of its
// XCD hold.  A writer waits for its stores in every wavefront (vmcnt), then
// releases and sets the counter.  128 workgroups handing 64 KB (8 KB) to one
// another: 6.7 (3.3) us, against 11.1 (6.7) with plain accesses and an acquire.
constexpr int SC1 = 16;  // cache policy bit of the raw buffer operations

__device__ __forceinline__ __amdgpu_buffer_rsrc_t shared_rsrc(const double2* base, int elems) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, elems * 16, 0x00027000);
}
// Element e of the resource (zero past its end).
__device__ __forceinline__ double2 shared_load(__amdgpu_buffer_rsrc_t r, int e) {
  const auto w = __builtin_amdgcn_raw_buffer_load_b128(r, e * 16, 0, SC1);
  return make_double2(__hiloint2double((int)w[1], (int)w[0]), __hiloint2double((int)w[3], (int)w[2]));
}
// (dropped past its end)
__device__ __forceinline__ void shared_store(__amdgpu_buffer_rsrc_t r, int e, double2 v) {
  typedef unsigned int u4 __attribute__((ext_vector_type(4)));
  const u4 w = {(unsigned)__double2loint(v.x), (unsigned)__double2hiint(v.x),
                (unsigned)__double2loint(v.y), (unsigned)__double2hiint(v.y)};
  __builtin_amdgcn_raw_buffer_store_b128(w, r, e * 16, 0, SC1);
}
// This workgroup's stores are done and released: called by every thread, then
// thread 0 may set a counter.
__device__ __forceinline__ void publish() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
}

// Bounded wait (thread 0 polls, the block follows) until every counter has
// reached target.  Returns false if the wait was aborted.
__device__ bool wait_counters(Ctrl* ctrl, const unsigned int* c0, const unsigned int* c1,
                              unsigned int target, int* s_flag) {
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long spins = 0;
    int ok = 1;
    while (__hip_atomic_load(c0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target ||
           (c1 && __hip_atomic_load(c1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target)) {
      if (__hip_atomic_load(&ctrl->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        ok = 0;
        break;
      }
      if (++spins > SPIN_LIMIT) {
        atomicExch(&ctrl->abort, 1u);
        ok = 0;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    *s_flag = ok;
  }
  // the loads that follow must stay behind the counter's
  asm volatile("" ::: "memory");
  __syncthreads();
  return *s_flag != 0;
}

// Bounded wait of a step: counters c[i0] and c[i1] at `target`, and the n < 62
// counters from c[guard] on at `guard_target`; a lane of the first wavefront each.
__device__ bool wait_step(Ctrl* ctrl, const unsigned int* c, int64_t i0, int64_t i1,
                          unsigned int target, int64_t guard, int64_t n,
                          unsigned int guard_target, int* s_flag) {
  __syncthreads();
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    const unsigned int* mine = &c[lane == 0 ? i0 : lane == 1 ? i1 : lane < n + 2 ? guard + lane - 2 : i0];
    const unsigned int want = lane >= 2 && lane < n + 2 ? guard_target : target;
    unsigned long long spins = 0;
    int ok = 1;
    while (!__all(__hip_atomic_load(mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= want)) {
      if (__hip_atomic_load(&ctrl->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        ok = 0;
        break;
      }
      if (++spins > SPIN_LIMIT) {
        if (lane == 0) atomicExch(&ctrl->abort, 1u);
        ok = 0;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    if (lane == 0) *s_flag = ok;
  }
  asm volatile("" ::: "memory");
  __syncthreads();
  return *s_flag != 0;
}

// Bounded grid barrier.  Returns false if the barrier was aborted.
__device__ bool grid_barrier(Ctrl* ctrl, unsigned int target, int* s_flag) {
  publish();
  if (threadIdx.x == 0) atomicAdd(&ctrl->barrier, 1u);
  return wait_counters(ctrl, &ctrl->barrier, nullptr, target, s_flag);
}

__device__ void signal_add(unsigned int* c) {
  publish();
  if (threadIdx.x == 0) atomicAdd(c, 1u);
}
__device__ void signal_set(unsigned int* c, unsigned int v) {
  publish();
  if (threadIdx.x == 0) __hip_atomic_store(c, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Block indices of pair p in round k of the circle schedule over nb blocks.
__device__ __forceinline__ void pair_blocks(int64_t nb, int64_t k, int64_t p, int64_t* bi,
                                            int64_t* bj) {
  auto idx = [&](int64_t x) { return 1 + (x + k) % (nb - 1); };
  if (p == 0) {
    *bi = 0;
    *bj = idx(0);
  } else {
    *bi = idx(p);
    *bj = idx(nb - 1 - p);
  }
}

// Column index (in W / V) of local column t (0 <= t < PW) of the pair.
__device__ __forceinline__ int64_t pair_col(int64_t bi, int64_t bj, int t) {
  return (t < BW) ? bi * BW + t : bj * BW + (t - BW);
}

__device__ __forceinline__ long long now_ticks() { return (long long)wall_clock64(); }

// Pair owning block x in round k of the circle schedule (inverse of pair_blocks).
__device__ __forceinline__ int64_t block_owner(int64_t nb, int64_t k, int64_t x) {
  if (x == 0) return 0;
  const int64_t y = ((x - 1 - k) % (nb - 1) + (nb - 1)) % (nb - 1);  // idx(y) == x
  if (y == 0) return 0;
  return (y < nb / 2) ? y : nb - 1 - y;
}

// ---- one block pair on one workgroup --------------------------------------
//
// 768 threads.  A tile of RT rows of the pair's PW columns of W sits in LDS
// (column-major, padded), and one of V; the Gram matrix is taken from the former
// on the matrix cores, then the inner Jacobi rotates G and both tiles in
// registers.
//
// A level H of the inner Jacobi pairs index base + t with base + H + (t + k) mod H
// in round k (base = 0, 2H, ..): H rounds of 16 disjoint rotations that visit
// every pair across the two halves of each group of 2H indices once.  Level 16
// visits the pairs across the two blocks; levels 16, 8, 4, 2, 1 together every
// pair of the 32.  The first index of a pair stays where it is and the second
// moves one place a round, so wavefronts 0-3 keep G in registers, a 2 x 2 block
// a thread, and pass entries to the neighbouring thread: along a row of threads
// by DPP, between rows through LDS.  Wavefronts 4-7 hold W's tile, a row a lane,
// four pairs of columns a wavefront, and pass one column a round; 8-11 hold V's.  One barrier
// a round: the thread that holds pair p's own block derives its rotation from
// what it has (the second index's diagonal entry comes with that pair's
// rotation), everyone applies it after the barrier.
//
// A round takes 0.51 us, two thirds of it instruction issue (48 FP64
// operations a thread in either role, the rotation's chain of 45); with G and
// the tile in LDS it took 1.07 us, LDS traffic (100 KB a round).  G's rounds are
// not unrolled: in fours the 64 x 64 split took 634 us for 625 (more spills).
constexpr int JT = 768;            // threads
constexpr int TP = RT + 1;         // padded tile column (complex)
constexpr int NP = PW / 2;         // pairs a round
constexpr int ROUNDS = PW - 1;     // rounds of all levels

// Rotation of a pair, [x_a, x_b] <- [cs x_a - conj(s) x_b, s x_a + cs x_b], and
// the diagonal entry that it gives index b.
struct Rot {
  double cs, gbb;
  double2 s;
};

// Indices of pair p in round k of level H.
__device__ __forceinline__ void slot_cols(int H, int p, int k, int* a, int* b) {
  const int t = p & (H - 1), base = (p - t) * 2;
  *a = base + t;
  *b = base + H + ((t + k) & (H - 1));
}
// The pair whose second index pair p takes over in the next round.
__device__ __forceinline__ int slot_next(int H, int p) {
  return (p & ~(H - 1)) | ((p + 1) & (H - 1));
}
// x of the thread of pair slot_next(q) (q: the thread's place in its row of 16).
template <int H>
__device__ __forceinline__ double lane_next(double x) {
  if (H == 16) return wave::dpp<0x12F>(x);  // row_ror:15
  if (H == 8) {
    const double u = wave::dpp<0x12F>(x), v = wave::dpp<0x127>(x);  // row_ror:15, :7
    return (threadIdx.x & 7) == 7 ? v : u;
  }
  if (H == 4) return wave::dpp<0x39>(x);  // quad_perm 1, 2, 3, 0
  if (H == 2) return wave::dpp<0xB1>(x);  // quad_perm 1, 0, 3, 2
  return x;
}

struct PairLds {
  double2 tile[2][PW * TP];   // of W, of V
  double2 G[PW * GP];
  union {
    double2 G2[PW * GP];          // second half's Gram matrix
    double2 sh[2][2][NP * NP];    // second rows of the 2 x 2 blocks, by round parity
  };
  double2 xch[2][2][4][RT];   // the tiles' columns on their way, by round parity
  Rot rec[ROUNDS * NP];       // rotations of a sweep's rounds
  double off[JT / 64];
  int flag;
};

// 1/sqrt(x) and 1/x to a few ulp by one step of third order on the hardware's
// estimate (about 5e-8): two dependent operations shorter than jac::rsqrt_nr and
// rcp_nr, but an ulp low at x = 1, where those are exact.
__device__ __forceinline__ double rsqrt_short(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double rcp_short(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, y, 1.0);
  return fma(y, fma(e, e, e), y);
}

// Rotation that annihilates c = G_ab; identity when the pair is orthogonal to
// tol or either column negligible.  With d = G_bb - G_aa the tangent is
// t = w |c|, w = 2 sign(d) / (|d| + sqrt(d^2 + 4 |c|^2)) (the smaller root of
// t^2 + d t / |c| - 1 = 0), so |c| itself is not needed; all to a few ulp.
// cs = 1/sqrt(1 + t^2) must be unbiased where it is close to one (jac::rsqrt_nr is):
// an ulp lost in each of the hundreds of small rotations of a column adds up
// (1.4e-14 against 8.9e-15 on 64 columns).
__device__ __forceinline__ Rot pair_rotation(double gaa, double gbb, double2 c, double tol2,
                                             double tiny2) {
  Rot q;
  q.cs = 1.0;
  q.gbb = gbb;
  q.s = make_double2(0.0, 0.0);
  const double s2 = cabs2(c), d = gbb - gaa;
  const bool any = s2 > 0.0 && gaa > tiny2 && gbb > tiny2 && s2 > (tol2 * gaa) * gbb;
  const double h = fma(d, d, 4.0 * s2);
  const double w = copysign(2.0 * rcp_short(fma(h, rsqrt_short(h), fabs(d))), d);
  const double tc = w * s2;  // t |c|
  const double cs = jac::rsqrt_nr(fma(w, tc, 1.0)), sn = w * cs;
  if (any) {
    q.cs = cs;
    q.gbb = gbb + tc;
    q.s = make_double2(c.x * sn, c.y * sn);
  }
  return q;
}

__device__ __forceinline__ double2 rscale(double f, double2 x) {
  return make_double2(f * x.x, f * x.y);
}

// One row of a pair's columns, rotated by the Rot at doubles N .. N + 3 of rd.
template <int N>
__device__ __forceinline__ void rotate_columns(double2& x, double2& y, double rd) {
  const double cs = wave::row_bcast<N>(rd);
  const double2 sp = make_double2(wave::row_bcast<N + 2>(rd), wave::row_bcast<N + 3>(rd));
  const double2 x0 = x;
  x = cfma(make_double2(-sp.x, sp.y), y, rscale(cs, x0));
  y = cfma(sp, x0, rscale(cs, y));
}

// Level H on L.G and the tiles (ONE: the first only), on every wavefront of
// the workgroup; rec receives its H x NP rotations.  Ends with a barrier.
template <int H, bool ONE>
__device__ __forceinline__ void inner_level(PairLds& L, Rot* rec, double tol2, double tiny2) {
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (wv < 4) {
    const int p = tid >> 4, q = tid & 15, pn = slot_next(H, p);
    int a, b, c, d;
    slot_cols(H, p, 0, &a, &b);
    slot_cols(H, q, 0, &c, &d);
    double2 ac = L.G[a * GP + c], ad = L.G[a * GP + d];
    double2 bc = L.G[b * GP + c], bd = L.G[b * GP + d];
    double gbb = bd.x;
#pragma unroll 1
    for (int k = 0; k < H; ++k) {
      Rot* rot = rec + k * NP;
      const Rot own = pair_rotation(ac.x, gbb, ad, tol2, tiny2);
      if (p == q) rot[p] = own;
      __syncthreads();
      const Rot rp = rot[p], rq = rot[q];
      gbb = rot[pn].gbb;
      if (k > 0) {
        bc = L.sh[k & 1][0][pn * NP + q];
        bd = L.sh[k & 1][1][pn * NP + q];
      }
      // Z = J_p^H X J_q on the block (rows of pair p, columns of pair q)
      const double2 mq = make_double2(-rq.s.x, rq.s.y), mp = make_double2(-rp.s.x, -rp.s.y);
      const double2 cp = make_double2(rp.s.x, -rp.s.y);
      const double2 yac = cfma(mq, ad, rscale(rq.cs, ac)), yad = cfma(rq.s, ac, rscale(rq.cs, ad));
      const double2 ybc = cfma(mq, bd, rscale(rq.cs, bc)), ybd = cfma(rq.s, bc, rscale(rq.cs, bd));
      ac = cfma(mp, ybc, rscale(rp.cs, yac));
      ad = cfma(mp, ybd, rscale(rp.cs, yad));
      bc = cfma(cp, yac, rscale(rp.cs, ybc));
      bd = cfma(cp, yad, rscale(rp.cs, ybd));
      if (k + 1 < H) {
        ad = make_double2(lane_next<H>(ad.x), lane_next<H>(ad.y));
        bd = make_double2(lane_next<H>(bd.x), lane_next<H>(bd.y));
        L.sh[(k + 1) & 1][0][tid] = bc;
        L.sh[(k + 1) & 1][1][tid] = bd;
      }
    }
    slot_cols(H, p, H - 1, &a, &b);
    slot_cols(H, q, H - 1, &c, &d);
    L.G[a * GP + c] = ac;
    L.G[a * GP + d] = ad;
    L.G[b * GP + c] = bc;
    L.G[b * GP + d] = bd;
  } else if (ONE && wv >= 8) {
    for (int k = 0; k < H; ++k) __syncthreads();
  } else {
    const int w = wv & 3, which = wv >= 8;
    double2* tile = L.tile[which];
    const int wn = H == 16 ? (w + 1) & 3 : H == 8 ? w ^ 1 : w;  // owner of the column to come
    double2 xa[4], xb[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int a, b;
      slot_cols(H, 4 * w + i, 0, &a, &b);
      xa[i] = tile[a * TP + lane];
      xb[i] = tile[b * TP + lane];
    }
#pragma unroll 4
    for (int k = 0; k < H; ++k) {
      __syncthreads();
      // the four rotations (16 doubles) in the lanes of each row, broadcast from there
      const double rd = ((const double*)(rec + k * NP + 4 * w))[lane & 15];
      if (H >= 8 && k > 0) xb[3] = L.xch[k & 1][which][wn][lane];
      rotate_columns<0>(xa[0], xb[0], rd);
      rotate_columns<4>(xa[1], xb[1], rd);
      rotate_columns<8>(xa[2], xb[2], rd);
      rotate_columns<12>(xa[3], xb[3], rd);
      if (k + 1 < H) {
        const double2 x = xb[0];
        if (H == 2) {
          xb[0] = xb[1];
          xb[1] = x;
          const double2 y = xb[2];
          xb[2] = xb[3];
          xb[3] = y;
        } else {
          if (H >= 8) L.xch[(k + 1) & 1][which][w][lane] = x;
          xb[0] = xb[1];
          xb[1] = xb[2];
          xb[2] = xb[3];
          if (H == 4) xb[3] = x;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int a, b;
      slot_cols(H, 4 * w + i, H - 1, &a, &b);
      tile[a * TP + lane] = xa[i];
      tile[b * TP + lane] = xb[i];
    }
  }
  __syncthreads();
}

// Inner sweeps: level 16 (cross) or the levels from top down to 1.  Returns the
// number of rounds of the last one, whose rotations L.rec holds.
template <bool ONE>
__device__ int inner_rounds(PairLds& L, double tol, double tiny2, int sweeps, bool cross, int top) {
  const double tol2 = tol * tol;
  Rot* rec = L.rec;
  int n = 0;
  for (int sw = 0; sw < sweeps; ++sw) {
    n = 0;
    if (top == 16) {
      inner_level<16, ONE>(L, rec + n * NP, tol2, tiny2);
      n += 16;
      if (cross) continue;
    }
    if (top >= 8) {
      inner_level<8, ONE>(L, rec + n * NP, tol2, tiny2);
      n += 8;
    }
    if (top >= 4) {
      inner_level<4, ONE>(L, rec + n * NP, tol2, tiny2);
      n += 4;
    }
    if (top >= 2) {
      inner_level<2, ONE>(L, rec + n * NP, tol2, tiny2);
      n += 2;
    }
    inner_level<1, ONE>(L, rec + n * NP, tol2, tiny2);
    n += 1;
  }
  return n;
}

// Rows [rb, rb + nr) of the pair's columns of M into the tile (zeros below), a
// column a wavefront.
__device__ __forceinline__ void load_tile(const double2* __restrict__ M, int64_t ld, int64_t bi,
                                          int64_t bj, int64_t rb, int nr, double2* tile) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int t = wv; t < PW; t += JT / 64)
    tile[t * TP + lane] = shared_load(shared_rsrc(M + pair_col(bi, bj, t) * ld + rb, nr), lane);
}
__device__ __forceinline__ void store_tile(double2* __restrict__ M, int64_t ld, int64_t bi,
                                           int64_t bj, int64_t rb, int nr, const double2* tile) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int t = wv; t < PW; t += JT / 64)
    shared_store(shared_rsrc(M + pair_col(bi, bj, t) * ld + rb, nr), lane, tile[t * TP + lane]);
}

// A wavefront's share of the Gram matrix's upper 16 x 16 tiles: tile
// (00, 11 or 01), real or imaginary part, first or second half of the rows.
struct GramShare {
  int ti, tj, im, half;
};
__device__ __forceinline__ GramShare gram_share(int q) {
  const int tl = q % 3;
  return GramShare{tl == 1 ? 1 : 0, tl == 0 ? 0 : 1, (q / 3) & 1, q / 6};
}

typedef double d4 __attribute__((ext_vector_type(4)));

// acc += this share of the tile's Gram matrix (nr valid rows).
__device__ __forceinline__ void gram_accumulate(const double2* tile, int nr, GramShare q, d4* acc) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int steps = (nr + 3) >> 2, mid = (steps + 1) >> 1;
  const double2* ca = tile + (q.ti * 16 + li) * TP + lk;
  const double2* cb = tile + (q.tj * 16 + li) * TP + lk;
  for (int k = q.half ? mid : 0; k < (q.half ? steps : mid); ++k) {
    const double2 x = ca[4 * k], y = cb[4 * k];
    // conj(x) y: re = xr yr + xi yi, im = xr yi - xi yr
    *acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, q.im ? y.y : y.x, *acc, 0, 0, 0);
    *acc = __builtin_amdgcn_mfma_f64_16x16x4f64(q.im ? -x.y : x.y, q.im ? y.x : y.y, *acc, 0, 0, 0);
  }
}

// The share into its half's buffer (upper tiles of the PW x PW matrix).
__device__ __forceinline__ void gram_store(double2* dst, GramShare q, d4 acc) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  double* d = (double*)dst + q.im;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    d[2 * ((q.ti * 16 + lk + 4 * r) * GP + q.tj * 16 + li)] = acc[r];
}

// Rows of V that chunk r of W rotates; one tile of them rotates along with W's.
template <bool VSEP>
__device__ __forceinline__ bool v_rows(const SvdShape& s, const SvdWork& w, int64_t r, int64_t* v0,
                                       int64_t* v1) {
  *v0 = *v1 = 0;
  if (VSEP) return false;  // V has workgroups of its own
  const int64_t rcv = ceil_div(s.ncolp, s.R);
  *v0 = r * rcv;
  *v1 = min(s.ncolp, *v0 + rcv);
  return w.V && rcv <= RT && *v0 < *v1;
}

// Phase A for item (p, r): the Gram matrix of rows [r0, r1) of the pair's
// columns; the last tile of the rows stays in LDS, with V's.  R > 1: into dst
// (PW x PW, i <= j only), to be summed over the chunks or read by V's workgroups;
// with R = 1 the two halves are left in L.G and L.G2 as well.
template <bool VSEP>
__device__ void partial_gram(const SvdShape& s, const SvdWork& w, int64_t bi, int64_t bj, int64_t r,
                             int64_t r0, int64_t r1, double2* __restrict__ dst, PairLds& L) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const GramShare q = gram_share(wv);
  d4 c = {0.0, 0.0, 0.0, 0.0};
  int64_t v0, v1;
  const bool v_live = v_rows<VSEP>(s, w, r, &v0, &v1);
  constexpr int PER = (PW + JT / 64 - 1) / (JT / 64);  // columns of a tile per wavefront
  double2 vt[PER];
  for (int64_t rb = r0; rb == r0 || rb < r1; rb += RT) {
    const int nr = (int)max((int64_t)0, min((int64_t)RT, r1 - rb));
    __syncthreads();
    load_tile(w.W, s.len, bi, bj, rb, nr, L.tile[0]);
    if (rb == r0 && v_live) {
      // V's tile is on its way while the Gram matrix is formed
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int t = min(wv + i * (JT / 64), PW - 1);
        vt[i] = shared_load(
            shared_rsrc(w.V + pair_col(bi, bj, t) * s.ncolp + v0, (int)(v1 - v0)), lane);
      }
    }
    __syncthreads();
    gram_accumulate(L.tile[0], nr, q, &c);
  }
  if (v_live) {
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (wv + i * (JT / 64) < PW) L.tile[1][(wv + i * (JT / 64)) * TP + lane] = vt[i];
  }
  gram_store(q.half ? L.G2 : L.G, q, c);
  __syncthreads();
  if (s.R == 1 && !VSEP) return;
  const auto out = shared_rsrc(dst, PW * PW);
  for (int e = threadIdx.x; e < PW * PW; e += JT) {
    const int i = e / PW, j = e % PW;
    if (i <= j) shared_store(out, e, cadd(L.G[i * GP + j], L.G2[i * GP + j]));
  }
}

// The recorded rotations of n rounds on rows [lo, hi) of the pair's columns of
// M, a tile at a time in LDS.
__device__ void replay(double2* __restrict__ M, int64_t ld, int64_t bi, int64_t bj, int64_t lo,
                       int64_t hi, int n, bool cross, int top, PairLds& L) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int64_t rb = lo; rb < hi; rb += RT) {
    const int nr = (int)min((int64_t)RT, hi - rb);
    __syncthreads();
    double2* tile = L.tile[0];
    load_tile(M, ld, bi, bj, rb, nr, tile);
    __syncthreads();
    int H = top, k = 0;
    for (int m = 0; m < n; ++m) {
      for (int t = wave; t < NP; t += JT / 64) {
        int a, b;
        slot_cols(H, t, k, &a, &b);
        const Rot q = L.rec[m * NP + t];
        const double2 x = tile[a * TP + lane], y = tile[b * TP + lane];
        tile[a * TP + lane] = cfma(make_double2(-q.s.x, q.s.y), y, rscale(q.cs, x));
        tile[b * TP + lane] = cfma(q.s, x, rscale(q.cs, y));
      }
      __syncthreads();
      if (++k == H) {  // the next level; the first again after the last (or, cross, at once)
        k = 0;
        H = cross || H == 1 ? top : H >> 1;
      }
    }
    store_tile(M, ld, bi, bj, rb, nr, tile);
  }
}

// LDS of item (p, r) as partial_gram left it, in a workgroup that has held
// other items since.
__device__ void reload(const SvdShape& s, const SvdWork& w, int64_t bi, int64_t bj, int64_t r,
                       int64_t r0, int64_t r1, PairLds& L) {
  if (s.R == 1) {
    partial_gram<false>(s, w, bi, bj, r, r0, r1, nullptr, L);
    return;
  }
  __syncthreads();
  if (r0 < r1) {
    const int64_t last = r0 + (r1 - r0 - 1) / RT * RT;
    load_tile(w.W, s.len, bi, bj, last, (int)(r1 - last), L.tile[0]);
  }
  int64_t v0, v1;
  if (v_rows<false>(s, w, r, &v0, &v1)) load_tile(w.V, s.ncolp, bi, bj, v0, (int)(v1 - v0), L.tile[1]);
}

// Phases B + C for item (p, r): G = sum of the R partials at src (R > 1), the
// pair's off-diagonal measure (r == 0) into *off_slot, inner Jacobi, rotation of
// this chunk's rows of W and V (r >= R: chunk r - R of V's, its tile in LDS).  prof/pt/t0: phase timing of workgroup 0.
template <bool VSEP>
__device__ void pair_update(const SvdShape& s, const SvdWork& w, int64_t bi, int64_t bj,
                            int64_t r, const double2* __restrict__ src,
                            unsigned long long* off_slot, double tol, double tiny2,
                            int inner_sweeps, bool cross, PairLds& L, bool prof, long long* pt,
                            long long* t0) {
  const int tid = threadIdx.x;
  const int64_t rc = ceil_div(s.len, s.R);
  const auto parts = shared_rsrc(src, RMAX * PW * PW);
  // Upper triangle; the lower one mirrors it, so G is exactly Hermitian.
  for (int e = tid; e < PW * PW; e += JT) {
    const int i = e / PW, j = e % PW;
    if (i > j) continue;
    double2 g;
    if (s.R == 1 && (!VSEP || r == 0)) {
      g = cadd(L.G[i * GP + j], L.G2[i * GP + j]);
    } else {
      g = make_double2(0.0, 0.0);
      for (int q0 = 0; q0 < s.R; q0 += 4) {
        double2 gq[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          gq[q] = (q0 + q < s.R) ? shared_load(parts, (q0 + q) * PW * PW + e)
                                 : make_double2(0.0, 0.0);
#pragma unroll
        for (int q = 0; q < 4; ++q) g = cadd(g, gq[q]);
      }
    }
    if (i == j) g.y = 0.0;
    L.G[i * GP + j] = g;
    L.G[j * GP + i] = make_double2(g.x, -g.y);
  }
  __syncthreads();
  // max normalised off-diagonal over non-negligible column pairs (every
  // workgroup of the pair derives the same value from the same G)
  double mx = 0.0;
  for (int e = tid; e < PW * PW; e += JT) {
    const int i = e / PW, j = e % PW;
    if (i < j) {
      const double gi = L.G[i * GP + i].x, gj = L.G[j * GP + j].x;
      if (gi > tiny2 && gj > tiny2) mx = fmax(mx, cabs2(L.G[i * GP + j]) / gi / gj);
    }
  }
  for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_down(mx, off, 64));
  if ((tid & 63) == 0) L.off[tid >> 6] = mx;
  __syncthreads();
  double pair_off = 0.0;
  for (int q = 0; q < JT / 64; ++q) pair_off = fmax(pair_off, L.off[q]);
  pair_off = sqrt(pair_off);
  if (r == 0 && tid == 0) atomicMax(off_slot, (unsigned long long)__double_as_longlong(pair_off));
  if (prof) {
    const long long t1 = now_ticks();
    pt[2] += t1 - *t0;
    *t0 = t1;
  }
  // already orthogonal to tolerance: no rotation is applied to this pair
  if (pair_off <= tol) return;
  int64_t v0, v1;
  const bool v_live = v_rows<VSEP>(s, w, r, &v0, &v1);
  const int n = inner_rounds<VSEP>(L, tol, tiny2, inner_sweeps, cross, inner_top_of(s));
  if (prof) {
    const long long t1 = now_ticks();
    pt[3] += t1 - *t0;
    *t0 = t1;
  }
  if (VSEP && r >= s.R) {
    const int64_t v0 = (r - s.R) * RT;
    store_tile(w.V, s.ncolp, bi, bj, v0, (int)min((int64_t)RT, s.ncolp - v0), L.tile[0]);
    return;
  }
  // the tile in LDS is the chunk's last one
  const int64_t r0 = r * rc, r1 = min(s.len, r0 + rc);
  if (r0 < r1) {
    const int64_t last = r0 + (r1 - r0 - 1) / RT * RT;
    store_tile(w.W, s.len, bi, bj, last, (int)(r1 - last), L.tile[0]);
    replay(w.W, s.len, bi, bj, r0, last, n, cross, inner_top_of(s), L);
  }
  if (v_live)
    store_tile(w.V, s.ncolp, bi, bj, v0, (int)(v1 - v0), L.tile[1]);
  else if (w.V && !VSEP)
    replay(w.V, s.ncolp, bi, bj, v0, v1, n, cross, inner_top_of(s), L);
  if (prof) {
    const long long t1 = now_ticks();
    pt[4] += t1 - *t0;
    *t0 = t1;
  }
}

// Work item (pair p, row chunk r) of workgroup b when every item has its own
// workgroup.  Workgroups are dispatched round-robin over the XCDs (b mod 8), so
// the items are laid out XCD by XCD: each XCD takes whole pairs first (their
// partial Grams then meet in that XCD's L2 instead of crossing XCDs through
// memory), and the pairs left over fill the remaining slots.  A bijection of
// [0, G) onto the items for every G = P R.
constexpr int64_t NXCD = 8;
__device__ inline void local_item(int64_t b, int64_t G, int64_t R, int64_t* p, int64_t* r) {
  if (G % NXCD) {
    *p = b / R;
    *r = b % R;
    return;
  }
  const int64_t per = G / NXCD, x = b % NXCD, j = b / NXCD;
  const int64_t f = per / R;  // whole pairs per XCD
  if (j < f * R) {
    *p = x * f + j / R;
    *r = j % R;
    return;
  }
  const int64_t q = x * (per - f * R) + (j - f * R);
  *p = NXCD * f + q / R;
  *r = q % R;
}

// One-sided block Jacobi sweeps.  Work item (p, r) = row chunk r of pair p.
// LOCAL: one item per workgroup (gridDim.x == P R); the steps are ordered by
// local counters only -- the R workgroups of a pair meet after their partial
// Grams (pair counter), and a workgroup starts a step once the two pairs that
// held its blocks in the previous step have rotated its row chunk (chunk step
// counters).  One grid barrier per sweep reduces the convergence measure.
// VSEP (LOCAL, VS > 0): the rows of V are rotated by VS more workgroups per pair, which
// take the Gram matrix from W's and solve it like them.  An inner round is bound by
// the instructions of three wavefronts a SIMD (G, a tile of W, one of V), so V on
// other CUs shortens it; V's workgroups follow W's by a step or so and hold them up
// only if they fall two behind (the partial Grams alternate between two buffers) or
// at the end.  They read the convergence measure but are not counted in the barrier.
// An inner round 0.52 -> 0.44 us (64 columns).
// !LOCAL: items are strided over the grid, with two grid barriers per step.
template <bool LOCAL, bool VSEP>
__global__ __launch_bounds__(JT) void svd_jacobi(SvdShape s, SvdWork w, double tol,
                                                 int max_sweeps) {
  __shared__ PairLds L;

  const int tid = threadIdx.x;
  const bool prof = (blockIdx.x == 0 && tid == 0);
  long long pt[6] = {0, 0, 0, 0, 0, 0};
  long long t0 = 0;
  const int64_t items = s.P * s.R;
  const int64_t rc = ceil_div(s.len, s.R);  // rows of W per chunk
  const int64_t steps = s.nb - 1;
  const int inner_sweeps = inner_sweeps_of(s);
  const double tiny2 = w.ctrl->tiny2;
  const int64_t RA = s.R + (VSEP ? s.VS : 0);  // workgroups of a pair
  const size_t part_stride = (size_t)s.P * RMAX * PW * PW;
  unsigned int* pair_ctr = w.sync;
  unsigned int* chunk_ctr = w.sync + s.P;
  unsigned int barrier_no = 0;
  const unsigned int G_ = LOCAL ? (unsigned int)items : gridDim.x;  // arrivals at the barrier
  bool v_side = false;
  int sweep = 0;
  int converged = 0;
  double off_prev = 1.0e300;
  for (; sweep < max_sweeps; ++sweep) {
    // Slot (sweep + 1) % 3 was last read after the grid barrier ending sweep
    // sweep - 2; every workgroup has passed the barrier ending sweep - 1 since.
    if (blockIdx.x == 0 && tid == 0)
      __hip_atomic_store(&w.ctrl->off[(sweep + 1) % 3], 0ull, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    unsigned long long* off_slot = &w.ctrl->off[sweep % 3];
    for (int64_t k = 0; k < steps; ++k) {
      const int64_t g = (int64_t)sweep * steps + k;
      const bool cross = s.cross_inner && k != 0 && (s.cross_inner == 1 || sweep > 0);
      double2* part = w.part + (g & 1) * part_stride;
      if (prof) t0 = now_ticks();
      if (LOCAL) {
        int64_t p, r;
        local_item(blockIdx.x, gridDim.x, RA, &p, &r);
        v_side = VSEP && r >= s.R;
        int64_t bi, bj;
        pair_blocks(s.nb, k, p, &bi, &bj);
        if (g > 0) {
          const int64_t kp = (k == 0) ? steps - 1 : k - 1;
          const int64_t oi = block_owner(s.nb, kp, bi), oj = block_owner(s.nb, kp, bj);
          // (VSEP) and V's chunks have read the partial Grams of step g - 2
          const bool ok =
              VSEP ? wait_step(w.ctrl, chunk_ctr, oi * RA + r, oj * RA + r, (unsigned int)g,
                               p * RA + s.R, v_side ? 0 : s.VS, (unsigned int)(g - 1), &L.flag)
                   : wait_counters(w.ctrl, &chunk_ctr[oi * RA + r], &chunk_ctr[oj * RA + r],
                                   (unsigned int)g, &L.flag);
          if (!ok) return;
        }
        if (prof) {
          const long long t1 = now_ticks();
          pt[5] += t1 - t0;
          t0 = t1;
        }
        if (v_side) {
          const int64_t v0 = (r - s.R) * RT;
          load_tile(w.V, s.ncolp, bi, bj, v0, (int)min((int64_t)RT, s.ncolp - v0), L.tile[0]);
        } else {
          partial_gram<VSEP>(s, w, bi, bj, r, r * rc, min(s.len, r * rc + rc),
                             part + (p * RMAX + r) * PW * PW, L);
        }
        if (prof) {
          const long long t1 = now_ticks();
          pt[0] += t1 - t0;
          t0 = t1;
        }
        if (s.R > 1) {
          if (!v_side) signal_add(&pair_ctr[p]);
          if (!wait_counters(w.ctrl, &pair_ctr[p], nullptr, (unsigned int)((g + 1) * s.R),
                             &L.flag))
            return;
        } else if (VSEP && v_side) {  // the only chunk of W does not stop to publish its Gram matrix
          if (!wait_counters(w.ctrl, &chunk_ctr[p * RA], nullptr, (unsigned int)(g + 1), &L.flag))
            return;
        }
        if (prof) {
          const long long t1 = now_ticks();
          pt[1] += t1 - t0;
          t0 = t1;
        }
        pair_update<VSEP>(s, w, bi, bj, r, part + p * RMAX * PW * PW, off_slot, tol, tiny2,
                          inner_sweeps, cross, L, prof, pt, &t0);
        signal_set(&chunk_ctr[p * RA + r], (unsigned int)(g + 1));
      } else {
        for (int64_t it = blockIdx.x; it < items && s.R > 1; it += G_) {
          const int64_t p = it / s.R, r = it % s.R;
          int64_t bi, bj;
          pair_blocks(s.nb, k, p, &bi, &bj);
          partial_gram<false>(s, w, bi, bj, r, r * rc, min(s.len, r * rc + rc),
                              part + (p * RMAX + r) * PW * PW, L);
        }
        if (prof) {
          const long long t1 = now_ticks();
          pt[0] += t1 - t0;
          t0 = t1;
        }
        if (!grid_barrier(w.ctrl, (++barrier_no) * G_, &L.flag)) return;
        if (prof) {
          const long long t1 = now_ticks();
          pt[1] += t1 - t0;
          t0 = t1;
        }
        for (int64_t it = blockIdx.x; it < items; it += G_) {
          const int64_t p = it / s.R, r = it % s.R;
          int64_t bi, bj;
          pair_blocks(s.nb, k, p, &bi, &bj);
          // the chunk's last tile (and, R = 1, its Gram matrix) again: L has
          // held other items since
          reload(s, w, bi, bj, r, r * rc, min(s.len, r * rc + rc), L);
          pair_update<false>(s, w, bi, bj, r, part + p * RMAX * PW * PW, off_slot, tol, tiny2,
                             inner_sweeps, cross, L, prof, pt, &t0);
        }
        if (!grid_barrier(w.ctrl, (++barrier_no) * G_, &L.flag)) return;
        if (prof) pt[5] += now_ticks() - t0;
      }
    }
    if (LOCAL) {
      // all pairs' measures of this sweep are in *off_slot after the barrier.  Slot
      // (sweep + 1) % 3 is not reset before V's workgroups have read sweep - 2's: at the
      // end of sweep - 1 they had all finished its first step (steps >= 3).
      ++barrier_no;
      if (v_side) {
        if (!wait_counters(w.ctrl, &w.ctrl->barrier, nullptr, barrier_no * G_, &L.flag)) return;
      } else if (!grid_barrier(w.ctrl, barrier_no * G_, &L.flag)) {
        return;
      }
    }
    {
      const unsigned long long bits =
          __hip_atomic_load(off_slot, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
      const double off_sweep = __longlong_as_double((long long)bits);
      if (blockIdx.x == 0 && tid == 0 && sweep < 64) w.ctrl->offhist[sweep] = off_sweep;
      // Converged at the target, or stalled within 16x of it: near convergence
      // Jacobi reduces the measure quadratically, so a sweep that gains less than
      // 4x there is sitting on the rounding floor.  A sweep whose measure (taken
      // before each pair's rotation) was already below QUAD_STOP leaves an
      // off-diagonal of order QUAD_STOP^2, far below tol: the sweep that would
      // only confirm it is skipped.
      if (off_sweep <= tol || off_sweep <= QUAD_STOP ||
          (off_sweep <= 16.0 * tol && off_sweep > 0.25 * off_prev)) {
        converged = 1;
        ++sweep;
        break;
      }
      off_prev = off_sweep;
    }
  }
  if (prof) {
    w.ctrl->info[0] = sweep;
    w.ctrl->info[1] = converged;
    for (int i = 0; i < 6; ++i) w.ctrl->prof[i] = pt[i];
  }
}

// sigma_c = ||w_c||.
__global__ void svd_sigma(SvdShape s, SvdWork w) {
  __shared__ double red[256];
  for (int64_t c = blockIdx.x; c < s.ncolp; c += gridDim.x) {
    double acc = 0.0;
    for (int64_t r = threadIdx.x; r < s.len; r += blockDim.x) acc += cabs2(w.W[c * s.len + r]);
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
      if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
      __syncthreads();
    }
    if (threadIdx.x == 0) w.sigma[c] = sqrt(red[0]);
    __syncthreads();
  }
}

// perm[rank] = c with descending sigma, ties by index.  The keys are staged in
// LDS (dynamic, ncolp doubles) when the launch provides it, else read from
// memory.
__global__ void svd_rank(SvdShape s, SvdWork w, int staged) {
  extern __shared__ double keys[];
  // NaN keys sort last, so the ranks always form a permutation
  auto key = [&](int64_t d) -> double {
    const double x = staged ? keys[d] : w.sigma[d];
    return isnan(x) ? -1.0 : x;
  };
  if (staged) {
    for (int64_t d = threadIdx.x; d < s.ncolp; d += blockDim.x) keys[d] = w.sigma[d];
    __syncthreads();
  }
  for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < s.ncolp;
       c += (int64_t)gridDim.x * blockDim.x) {
    const double sc = key(c);
    int rank = 0;
    for (int64_t d = 0; d < s.ncolp; ++d) {
      const double sd = key(d);
      rank += (sd > sc || (sd == sc && d < c)) ? 1 : 0;
    }
    w.perm[rank] = (int)c;
  }
}

// Output.  W side: normalised columns of the working matrix (length len);
// V side: V (no QR; stride ncolp, length ncol) or Y = Q V (QR; stride lenA,
// length lenA).  wside_u: the W side is U (columns) rather than VH (conj rows).
__global__ void svd_output(SvdShape s, SvdWork w, double2* __restrict__ U, double* __restrict__ S,
                           double2* __restrict__ VH) {
  const int64_t r = s.ncol;
  const int wside_u = (s.use_qr == s.transposed);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  for (int64_t k = t0; k < r; k += stride) S[k] = w.sigma[w.perm[k]];
  const double tiny2 = w.ctrl->tiny2;
  for (int64_t e = t0; e < r * s.len; e += stride) {
    const int64_t k = e / s.len, x = e % s.len;
    const int64_t c = w.perm[k];
    const double sg = w.sigma[c];
    double2 v = w.W[c * s.len + x];
    // negligible columns get an orthonormal completion afterwards
    v = (sg > 0.0 && sg * sg > tiny2) ? make_double2(v.x / sg, v.y / sg) : make_double2(0.0, 0.0);
    // with QR, coordinate x of the W side is B's column colperm[x]
    const int64_t xo = s.use_qr ? (int64_t)w.colperm[x] : x;
    if (wside_u)
      U[xo * r + k] = v;
    else
      VH[k * s.n + xo] = make_double2(v.x, -v.y);
  }
  const double2* src = s.use_qr ? w.Y : w.V;
  const int64_t ld = s.use_qr ? s.lenA : s.ncolp;
  const int64_t vlen = s.use_qr ? s.lenA : s.ncol;
  for (int64_t e = t0; e < r * vlen; e += stride) {
    const int64_t k = e / vlen, x = e % vlen;
    const double2 v = src[(int64_t)w.perm[k] * ld + x];
    if (wside_u)
      VH[k * s.n + x] = make_double2(v.x, -v.y);
    else
      U[x * r + k] = v;
  }
}

// Complete the W-side singular vectors of negligible singular values
// (sigma^2 <= tiny2: at the rounding level of the factorisation, where the
// directions are not determined) to an orthonormal set.  The singular values
// themselves are kept.  For slot k the candidate is the unit vector e_x whose
// coordinate x has the smallest leverage sum_{j<k} |u_j[x]|^2 among the
// vectors already fixed; its residual after projection then has squared norm
// 1 - leverage >= 1 - k/len > 0, so the completion cannot fail.  Projection is
// classical Gram-Schmidt applied twice, one wavefront per dot product.  Only
// slots k < *kmax are completed when kmax is given (the caller keeps no more).
// One workgroup of 1024 threads; w.part holds at least r complex values.
__global__ __launch_bounds__(1024) void svd_complete(SvdWork w, double2* __restrict__ base,
                                                     int64_t sk, int64_t sx, int conj, int64_t r,
                                                     int64_t len, const int64_t* __restrict__ kmax) {
  const double cy = conj ? -1.0 : 1.0;
  // component x of vector k, as a plain (unconjugated) one
  auto load = [&](int64_t k, int64_t x) -> double2 {
    const double2 v = base[k * sk + x * sx];
    return make_double2(v.x, cy * v.y);
  };
  auto store = [&](int64_t k, int64_t x, double2 v) {
    base[k * sk + x * sx] = make_double2(v.x, cy * v.y);
  };
  __shared__ double s_val[16];
  __shared__ int64_t s_idx[16];
  __shared__ int64_t s_best;
  __shared__ double s_nrm;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nwaves = (int)(blockDim.x >> 6);
  double2* coef = w.part;
  const double tiny2 = w.ctrl->tiny2;
  int64_t kend = r;
  if (kmax && *kmax < kend) kend = *kmax;
  // Usually no kept column is negligible: find out in parallel first, and
  // leave without the sequential scan when none is.
  __shared__ int s_any;
  if (tid == 0) s_any = 0;
  __syncthreads();
  for (int64_t k = tid; k < kend; k += blockDim.x) {
    const double sg = w.sigma[w.perm[k]];
    if (!(sg > 0.0 && sg * sg > tiny2)) atomicOr(&s_any, 1);
  }
  __syncthreads();
  if (!s_any) return;
  for (int64_t k = 0; k < kend; ++k) {
    const double sg = w.sigma[w.perm[k]];
    if (sg > 0.0 && sg * sg > tiny2) continue;
    // Candidate coordinate: smallest leverage, ties to the smallest index.
    double best = 1.0e300;
    int64_t bx = len;
    for (int64_t x = tid; x < len; x += blockDim.x) {
      double lev = 0.0;
      for (int64_t j = 0; j < k; ++j) lev += cabs2(load(j, x));
      if (lev < best) {
        best = lev;
        bx = x;
      }
    }
    for (int off = 32; off > 0; off >>= 1) {
      const double ov = __shfl_down(best, off, 64);
      const int64_t ox = __shfl_down(bx, off, 64);
      if (ov < best || (ov == best && ox < bx)) {
        best = ov;
        bx = ox;
      }
    }
    if (lane == 0) {
      s_val[wave] = best;
      s_idx[wave] = bx;
    }
    __syncthreads();
    if (tid == 0) {
      double bv = s_val[0];
      int64_t bi = s_idx[0];
      for (int q = 1; q < nwaves; ++q)
        if (s_val[q] < bv || (s_val[q] == bv && s_idx[q] < bi)) {
          bv = s_val[q];
          bi = s_idx[q];
        }
      s_best = bi;
    }
    __syncthreads();
    const int64_t xb = s_best;
    for (int64_t x = tid; x < len; x += blockDim.x)
      store(k, x, make_double2(x == xb ? 1.0 : 0.0, 0.0));
    __syncthreads();
    for (int pass = 0; pass < 2; ++pass) {
      for (int64_t j = wave; j < k; j += nwaves) {
        double2 acc = make_double2(0.0, 0.0);
        for (int64_t x = lane; x < len; x += 64) acc = cfmac(load(j, x), load(k, x), acc);
        for (int off = 32; off > 0; off >>= 1) {
          acc.x += __shfl_down(acc.x, off, 64);
          acc.y += __shfl_down(acc.y, off, 64);
        }
        if (lane == 0) coef[j] = acc;
      }
      __syncthreads();
      for (int64_t x = tid; x < len; x += blockDim.x) {
        double2 b = load(k, x);
        for (int64_t j = 0; j < k; ++j) {
          const double2 pa = cmul(coef[j], load(j, x));
          b = make_double2(b.x - pa.x, b.y - pa.y);
        }
        store(k, x, b);
      }
      __syncthreads();
    }
    double acc = 0.0;
    for (int64_t x = tid; x < len; x += blockDim.x) acc += cabs2(load(k, x));
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
    if (lane == 0) s_val[wave] = acc;
    __syncthreads();
    if (tid == 0) {
      double t = 0.0;
      for (int q = 0; q < nwaves; ++q) t += s_val[q];
      s_nrm = sqrt(t);
    }
    __syncthreads();
    const double nrm = s_nrm;
    for (int64_t x = tid; x < len; x += blockDim.x) {
      const double2 b = load(k, x);
      store(k, x, make_double2(b.x / nrm, b.y / nrm));
    }
    __syncthreads();
  }
}

// Truncation rule: one lane runs it over an LDS copy of s
// (STAGED, spectra of up to TRUNC_STAGE values) or over s itself.
constexpr int64_t TRUNC_STAGE = 4096;
template <bool STAGED>
__global__ void truncate_kernel(int64_t N, const double* __restrict__ s, int method, double tol,
                                int64_t max_bond, int64_t* D_out, double* err_out) {
  extern __shared__ double stage[];
  if (STAGED) {
    for (int64_t i = threadIdx.x; i < N; i += blockDim.x) stage[i] = s[i];
    __syncthreads();
  }
  const double* ss = STAGED ? stage : s;
  if (threadIdx.x != 0) return;
  truncation_rule(N, ss, method, tol, max_bond, D_out, err_out);
}

// Kernel of each variant, and the workgroups of it that can be resident at once.
const void* jacobi_kernel(int variant) {
  return variant == JACOBI_V_APART ? (const void*)svd_jacobi<true, true>
         : variant == JACOBI_LOCAL ? (const void*)svd_jacobi<true, false>
                                   : (const void*)svd_jacobi<false, false>;
}
int resident_workgroups(int64_t* lim) {
  DeviceInfo di;
  int st = device_info(&di);
  if (st) return st;
  static thread_local int occ_dev = -1, occ[3];
  if (occ_dev != di.device) {
    for (int v = 0; v < 3; ++v) {
      occ[v] = 0;
      SEEMPS_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ[v], jacobi_kernel(v), JT, 0));
    }
    occ_dev = di.device;
  }
  for (int v = 0; v < 3; ++v) lim[v] = (int64_t)occ[v] * di.num_cu;
  return SEEMPS_OK;
}

unsigned blocks_for(int64_t n) {
  int64_t b = ceil_div(n, 256);
  if (b > 2048) b = 2048;
  if (b < 1) b = 1;
  return (unsigned)b;
}

}  // namespace

void jacobi_shape(SvdShape* s, int num_cu) {
  int64_t nb = ceil_div(s->ncol, BW);
  if (nb < 2) nb = 2;
  nb += (nb & 1);
  s->nb = nb;
  s->ncolp = nb * BW;
  s->P = nb / 2;
  // Row chunks per pair: a tile each, as far as one workgroup per CU allows.
  // The chunk's rotations then hide behind the inner rounds; a longer chunk
  // replays them tile by tile.
  int64_t R = num_cu / s->P;
  // tuning knob: cap on the row chunks per pair (SEEMPS_SVD_ROW_CHUNKS)
  static const int64_t r_cap = [] {
    const char* e = getenv("SEEMPS_SVD_ROW_CHUNKS");
    const long v = e ? atol(e) : 0;
    return (int64_t)(v > 0 ? v : RMAX);
  }();
  if (R > r_cap) R = r_cap;
  const int64_t rmax_len = ceil_div(s->len, RT);
  if (R > rmax_len) R = rmax_len;
  if (R > RMAX) R = RMAX;
  if (R < 1) R = 1;
  s->R = R;
  // V's rows to workgroups of their own as long as all of them take a quarter of the
  // CUs (256 columns); with more, the waits between them cost what the shorter rounds
  // give.  A square matrix, us, V apart / along with W: 64 columns 653 / 680, 128
  // 1549 / 1707, 256 3640 / 3842, 320 5674 / 5667, 416 8378 / 8158, 512 9976 / 9237.
  const int64_t vs = ceil_div(s->ncolp, RT);
  s->VS = nb > 2 && 4 * s->P * (R + vs) <= num_cu ? vs : 0;
  // Inner solves: every block's own pairs are visited at the first step of a
  // sweep (each block meets one partner there); with cross_inner the later
  // steps rotate only the pairs across the two blocks (16 rounds instead of
  // 31).  Measured over whole chi=256 DMRG sweeps this is faster in both the
  // QR-preconditioned and the basis-sketched splits (more sweeps at times,
  // each about half as long); the convergence test is the same either way.
  // SEEMPS_SVD_INNER=full restores the full inner sweep at every step, and
  // SEEMPS_SVD_INNER=hybrid keeps it for the first sweep only (tuning: hybrid
  // converges the sketch matrices in fewer sweeps, but lost over DMRG sweeps).
  static const int inner_mode = [] {
    const char* e = getenv("SEEMPS_SVD_INNER");
    if (e && strcmp(e, "full") == 0) return 0;
    if (e && strcmp(e, "hybrid") == 0) return 2;  // full inner sweeps in sweep 0
    return 1;
  }();
  s->cross_inner = s->nb > 2 ? inner_mode : 0;
}

bool jacobi_plan(int64_t P, int64_t R, int64_t VS, const int64_t* lim, int* variant, int* grid) {
  // an item a workgroup where they all fit: local step ordering
  const int64_t apart = P * (R + VS), local = P * R;
  if (VS > 0 && apart <= lim[JACOBI_V_APART]) {
    *variant = JACOBI_V_APART;
    *grid = (int)apart;
  } else if (local <= lim[JACOBI_LOCAL]) {
    *variant = JACOBI_LOCAL;
    *grid = (int)local;
  } else {
    *variant = JACOBI_STRIDED;
    *grid = (int)(local < lim[JACOBI_STRIDED] ? local : lim[JACOBI_STRIDED]);
  }
  return *grid >= 1;
}

int jacobi_enqueue(const SvdShape& shape, const SvdWork& w, hipStream_t stream) {
  SvdShape s = shape;
  if (!w.V) s.VS = 0;
  int64_t lim[3];
  int st, variant, grid;
  if ((st = resident_workgroups(lim))) return st;
  if (!jacobi_plan(s.P, s.R, s.VS, lim, &variant, &grid)) {
    set_error("svd: kernel cannot be resident on this device");
    return SEEMPS_ERR_RUNTIME;
  }
  if (variant != JACOBI_V_APART) s.VS = 0;
  // Relative orthogonality target: a few times above the rounding floor of the
  // measured Gram entries (~sqrt(len) eps), so that rounding alone cannot keep
  // the measure above it.
  double tol = 32.0 * sqrt((double)s.len) * 2.220446049250313e-16;
  int max_sweeps = MAX_SWEEPS;
  void* args[] = {(void*)&s, (void*)&w, (void*)&tol, (void*)&max_sweeps};
  // nominal SVD flops (complex): 4 * (6 M N^2 + 16 N^3), M >= N
  const double M_ = (double)s.lenA, N_ = (double)s.ncol;
  TimedLaunch timed("svd_jacobi", stream, 4.0 * (6.0 * M_ * N_ * N_ + 16.0 * N_ * N_ * N_));
  const void* fn = jacobi_kernel(variant);
  if (grid == 1) {  // nothing to be resident with
    SEEMPS_HIP(hipLaunchKernel(fn, dim3(1), dim3(JT), args, 0, stream));
    return SEEMPS_OK;
  }
  SEEMPS_HIP(hipLaunchCooperativeKernel(fn, dim3(grid), dim3(JT), args, 0, stream));
  return SEEMPS_OK;
}

int complete_enqueue(const SvdWork& w, double2* base, int64_t sk, int64_t sx, int conj, int64_t r,
                     int64_t len, const int64_t* kmax, hipStream_t stream) {
  TimedLaunch timed("svd_complete", stream, 0.0);
  hipLaunchKernelGGL(svd_complete, dim3(1), dim3(1024), 0, stream, w, base, sk, sx, conj, r, len,
                     kmax);
  return check_launch("svd_complete");
}

namespace {
// The W side's vectors among the outputs: columns of U, or conjugated rows of VH.
int complete_sides(const SvdShape& s, const SvdWork& w, double2* U, double2* VH,
                   const int64_t* kmax, hipStream_t stream) {
  if (s.use_qr == s.transposed)
    return complete_enqueue(w, U, 1, s.ncol, 0, s.ncol, s.len, kmax, stream);
  return complete_enqueue(w, VH, s.n, 1, 1, s.ncol, s.len, kmax, stream);
}
}  // namespace

// Enqueue the SVD.  With kmax_dev == nullptr every slot is completed; otherwise
// svd_complete_enqueue must follow, limited to the slots the caller keeps.
int svd_enqueue(int64_t m, int64_t n, const double2* A, int64_t lda, double2* U, double* S,
                double2* VH, void* work, int64_t work_bytes, hipStream_t stream,
                int* info_dev_off, bool complete, bool precondition) {
  DeviceInfo di;
  int st = device_info(&di);
  if (st) return st;
  const SvdShape s = svd_shape(m, n, di.num_cu, precondition);
  SEEMPS_CHECK_ARG(work_bytes >= svd_bytes(s), "svd: workspace too small (%lld < %lld)",
                   (long long)work_bytes, (long long)svd_bytes(s));
  SvdWork w = svd_carve(s, work);
  if (s.use_qr) {
    hipLaunchKernelGGL(col_norms, dim3(blocks_for(s.ncol)), dim3(256), 0, stream, s, A, lda,
                       w.colnrm);
    if ((st = check_launch("col_norms"))) return st;
    hipLaunchKernelGGL(col_rank, dim3(blocks_for(s.ncol)), dim3(256), 0, stream, s, w.colnrm,
                       w.colperm);
    if ((st = check_launch("col_rank"))) return st;
    hipLaunchKernelGGL(load_colmajor, dim3(blocks_for(s.ncol * s.lenA)), dim3(256), 0, stream, s,
                       A, lda, w.Acm, s.ncol, (const int*)w.colperm);
    if ((st = check_launch("load_colmajor"))) return st;
    if ((st = qr_factor(w.Acm, s.lenA, s.ncol, w.Vall, w.tau, stream))) return st;
    hipLaunchKernelGGL(load_w_from_r, dim3(blocks_for(s.ncolp * s.len)), dim3(256), 0, stream, s,
                       w.Acm, w.W);
    if ((st = check_launch("load_w_from_r"))) return st;
  } else {
    hipLaunchKernelGGL(load_colmajor, dim3(blocks_for(s.ncolp * s.lenA)), dim3(256), 0, stream,
                       s, A, lda, w.W, s.ncolp, (const int*)nullptr);
    if ((st = check_launch("load_colmajor"))) return st;
  }
  hipLaunchKernelGGL(init_v_ctrl, dim3(blocks_for(s.ncolp * s.ncolp)), dim3(256), 0, stream, s, w);
  if ((st = check_launch("init_v_ctrl"))) return st;
  hipLaunchKernelGGL(svd_frob, dim3(1), dim3(1024), 0, stream, s, w);
  if ((st = check_launch("svd_frob"))) return st;
  if ((st = jacobi_enqueue(s, w, stream))) return st;
  hipLaunchKernelGGL(svd_sigma, dim3((unsigned)(s.ncolp < 1024 ? s.ncolp : 1024)), dim3(256), 0,
                     stream, s, w);
  if ((st = check_launch("svd_sigma"))) return st;
  {
    const int staged = s.ncolp <= 8192;  // up to 64 KB of keys per workgroup
    const size_t shmem = staged ? (size_t)s.ncolp * sizeof(double) : 0;
    hipLaunchKernelGGL(svd_rank, dim3(blocks_for(s.ncolp)), dim3(256), shmem, stream, s, w,
                       staged);
  }
  if ((st = check_launch("svd_rank"))) return st;
  if (s.use_qr) {
    hipLaunchKernelGGL(load_y, dim3(blocks_for(s.ncol * s.lenA)), dim3(256), 0, stream, s, w);
    if ((st = check_launch("load_y"))) return st;
    if ((st = qr_apply_q(w.Y, s.lenA, s.ncol, s.ncol, w.Vall, w.tau, stream))) return st;
  }
  const int64_t big = s.ncol * (s.len > s.lenA ? s.len : s.lenA);
  hipLaunchKernelGGL(svd_output, dim3(blocks_for(big)), dim3(256), 0, stream, s, w, U, S, VH);
  if ((st = check_launch("svd_output"))) return st;
  if (complete && (st = complete_sides(s, w, U, VH, nullptr, stream))) return st;
  if (info_dev_off) *info_dev_off = (int)((char*)w.ctrl - (char*)work);
  return SEEMPS_OK;
}

// Orthonormal completion of the slots k < *kmax_dev (see svd_complete).
int svd_complete_enqueue(int64_t m, int64_t n, double2* U, double2* VH, void* work,
                         const int64_t* kmax_dev, hipStream_t stream, bool precondition) {
  DeviceInfo di;
  int st = device_info(&di);
  if (st) return st;
  const SvdShape s = svd_shape(m, n, di.num_cu, precondition);
  SvdWork w = svd_carve(s, work);
  return complete_sides(s, w, U, VH, kmax_dev, stream);
}

int64_t svd_workspace_bytes(int64_t m, int64_t n, bool precondition) {
  // Sized for the largest row split so the size does not depend on the device.
  SvdShape s = svd_shape(m, n, 1 << 20, precondition);
  return svd_bytes(s);
}

int truncate_enqueue(int64_t N, const double* s, int method, double tol, int64_t max_bond,
                     int64_t* D_out, double* err_out, hipStream_t stream) {
  SEEMPS_CHECK_ARG(N >= 1, "truncate: empty spectrum");
  SEEMPS_CHECK_ARG(method >= 0 && method <= 3, "truncate: invalid method %d", method);
  SEEMPS_CHECK_ARG(max_bond >= 1, "truncate: invalid max bond dimension");
  if (N <= TRUNC_STAGE)
    hipLaunchKernelGGL(truncate_kernel<true>, dim3(1), dim3(256), (size_t)N * sizeof(double),
                       stream, N, s, method, tol, max_bond, D_out, err_out);
  else
    hipLaunchKernelGGL(truncate_kernel<false>, dim3(1), dim3(64), 0, stream, N, s, method, tol,
                       max_bond, D_out, err_out);
  return check_launch("truncate");
}

// Read the control block after the stream has been synchronised by the caller's copy.
int svd_read_ctrl(void* work, int off, int32_t* info, hipStream_t stream) {
  static_assert(sizeof(Ctrl) <= PINNED_BYTES - PINNED_CTRL_OFF, "control block too large");
  char* hp = (char*)pinned_stage(PINNED_BYTES);
  SEEMPS_CHECK_ARG(hp != nullptr, "pinned host staging could not be allocated");
  hp += PINNED_CTRL_OFF;
  SEEMPS_HIP(hipMemcpyAsync(hp, (char*)work + off, sizeof(Ctrl), hipMemcpyDeviceToHost, stream));
  SEEMPS_HIP(hipStreamSynchronize(stream));
  Ctrl h;
  memcpy(&h, hp, sizeof(h));
  return ctrl_status(h, info);
}

int ctrl_status(const Ctrl& h, int32_t* info) {
  if (info) {
    info[0] = h.info[0];
    info[1] = h.info[1];
  }
  if (getenv("SEEMPS_SVD_PROFILE")) {
    int dev = 0, rate = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&rate, hipDeviceAttributeWallClockRate, dev);  // kHz
    const double us = rate > 0 ? 1e3 / rate : 0.0;
    fprintf(stderr,
            "[svd] sweeps=%d converged=%d  us: gramA=%.1f bar1=%.1f reduce=%.1f inner=%.1f "
            "rotate=%.1f bar2=%.1f\n",
            h.info[0], h.info[1], h.prof[0] * us, h.prof[1] * us, h.prof[2] * us, h.prof[3] * us,
            h.prof[4] * us, h.prof[5] * us);
    fprintf(stderr, "[svd] off by sweep:");
    for (int i = 0; i < h.info[0] && i < 16; ++i) fprintf(stderr, " %.1e", h.offhist[i]);
    fprintf(stderr, "\n");
  }
  if (h.abort) {
    set_error("svd: grid barrier timed out (cooperative residency lost)");
    return SEEMPS_ERR_RUNTIME;
  }
  if (!h.info[1]) {
    const int ns = h.info[0] < 64 ? h.info[0] : 64;
    set_error("SVD did not converge in %d sweeps (off-diagonal measure by sweep: %.2e %.2e %.2e "
              "... %.2e %.2e; negligible column norm^2 %.2e)",
              h.info[0], ns > 0 ? h.offhist[0] : 0.0, ns > 1 ? h.offhist[1] : 0.0,
              ns > 2 ? h.offhist[2] : 0.0, ns > 1 ? h.offhist[ns - 2] : 0.0,
              ns > 0 ? h.offhist[ns - 1] : 0.0, h.tiny2);
    return SEEMPS_ERR_NOCONVERGE;
  }
  return SEEMPS_OK;
}

}  // namespace seemps

extern "C" int64_t seemps_svd_workspace(int64_t m, int64_t n) {
  return seemps::svd_workspace_bytes(m, n);
}

extern "C" int seemps_zgesvd(int64_t m, int64_t n, const void* A, int64_t lda, void* U, double* S,
                             void* VH, void* work, int64_t work_bytes, int32_t* info,
                             void* stream) {
  SEEMPS_CHECK_ARG(m >= 1 && n >= 1, "svd: empty matrix");
  SEEMPS_CHECK_ARG(lda >= n, "svd: lda < n");
  int off = 0;
  int st = seemps::svd_enqueue(m, n, (const double2*)A, lda, (double2*)U, S, (double2*)VH, work,
                               work_bytes, (hipStream_t)stream, &off);
  if (st) return st;
  return seemps::svd_read_ctrl(work, off, info, (hipStream_t)stream);
}

extern "C" int seemps_truncate(int64_t N, const double* s, int method, double tolerance,
                               int64_t max_bond, int64_t* D_out, double* err_out, void* stream) {
  return seemps::truncate_enqueue(N, s, method, tolerance, max_bond, D_out, err_out,
                                  (hipStream_t)stream);
}
