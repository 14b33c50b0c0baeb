// Shapes, workspaces and steps that the SVD (svd.hip) and the truncated split
// (split.hip) share.
#pragma once

#include "jacobi_inner.h"

namespace seemps {

using jac::GP;
using jac::PW;

constexpr int BW = PW / 2;      // block width (columns); PW, GP from jacobi_inner.h
constexpr int RT = 64;          // rows per LDS tile: a row a lane
constexpr int RMAX = 16;        // max row chunks per pair

struct Ctrl {
  unsigned int barrier;       // grid barrier arrivals
  unsigned int abort;         // set by any workgroup whose wait timed out
  unsigned long long off[3];  // per-sweep max normalised off-diagonal (as bits), slot sweep % 3
  int info[4];                // sweeps, converged (written by workgroup 0), unused
  long long prof[8];          // wall-clock ticks of workgroup 0 per phase
  double frob2;               // ||W||_F^2 (invariant under the rotations)
  double tiny2;               // squared norm below which a column is negligible
  double offhist[64];         // off-diagonal measure of each sweep (diagnostics)
};

struct SvdShape {
  int64_t m, n;         // input shape
  int64_t lenA, ncol;   // working matrix B: ncol columns of length lenA
  int64_t len;          // Jacobi column length (ncol with QR, lenA without)
  int64_t nb, ncolp;    // blocks (even), padded column count
  int64_t P, R;         // pairs per step, row chunks of W
  int64_t VS;           // row chunks of V with workgroups of their own (0: W's rotate V too)
  int transposed;       // 1 if B = A^H
  int use_qr;
  int cross_inner;      // inner solves after a sweep's first step: cross-block pairs only
};

struct SvdWork {
  double2* Acm;   // ncol x lenA (QR in place)
  double2* Vall;  // ncol x lenA (QR vectors)
  double2* tau;   // ncol
  double2* Y;     // ncol x lenA (Q V)
  double2* W;     // ncolp x len
  double2* V;     // ncolp x ncolp
  double2* part;  // 2 x P x RMAX x PW x PW (partial Grams, by step parity)
  unsigned int* sync;  // P pair arrival counters, then P x (R + VS) chunk step counters
  double* colnrm;  // ncol squared column norms of B (QR path)
  int* colperm;    // ncol: B's columns by decreasing norm (QR path)
  double* sigma;  // ncolp
  int* perm;      // ncolp
  Ctrl* ctrl;
};

__host__ __device__ inline int64_t sync_words(const SvdShape& s) { return s.P + s.P * (s.R + s.VS); }
inline int64_t align256(int64_t x) { return (x + 255) & ~int64_t(255); }

// Blocks, pairs and row chunks of a Jacobi on s.ncol columns of length s.len
// (set by the caller, as s.use_qr), at most one workgroup per CU.
void jacobi_shape(SvdShape* s, int num_cu);
// Forms of the Jacobi kernel: V's rows on workgroups of their own, one work item a
// workgroup, items strided over the grid.
enum JacobiVariant { JACOBI_V_APART = 0, JACOBI_LOCAL = 1, JACOBI_STRIDED = 2 };
// The form and its grid for P pairs of R row chunks (and VS of V's), when lim[v]
// workgroups of form v can be resident at once; false if no grid can.
bool jacobi_plan(int64_t P, int64_t R, int64_t VS, const int64_t* lim, int* variant, int* grid);
// Sweeps on w.W (and w.V unless it is null) until converged; w.ctrl reset and
// its tiny2 set beforehand, w.sync zero.
int jacobi_enqueue(const SvdShape& s, const SvdWork& w, hipStream_t stream);
// Squared norm below which a column of length len is negligible in a matrix of
// squared Frobenius norm frob2.
__host__ __device__ inline double negligible2(int64_t len, double frob2) {
  const double le = (double)len * 2.220446049250313e-16;
  return le * le * frob2;
}
// Completes the vectors of negligible singular values among the first *kmax (or
// r: kmax null) to an orthonormal set: vector k has components base[k sk + x sx]
// (conjugated if conj), x < len; w.sigma, w.perm and w.ctrl->tiny2 say which.
int complete_enqueue(const SvdWork& w, double2* base, int64_t sk, int64_t sx, int conj, int64_t r,
                     int64_t len, const int64_t* kmax, hipStream_t stream);
// Status and message of a finished Jacobi from a host copy of its control block.
// `abort` decides over `info`: V's own workgroups are not counted in the last
// barrier, so a wait of theirs may run out after workgroup 0 left as converged.
int ctrl_status(const Ctrl& h, int32_t* info);

// Truncation rule on the descending spectrum ss by one thread: the reference's
// sequential loops (summation order identical to truncation.pxi:251-327,
// products and sums rounded separately as in the reference's compiled loops).
__device__ inline void truncation_rule(int64_t N, const double* ss, int method, double tol,
                                       int64_t max_bond, int64_t* D_out, double* err_out) {
#pragma clang fp contract(off)
  int64_t D = N;
  double err = 0.0;
  if (method == SEEMPS_TRUNC_NONE) {
    D = N;
    err = 0.0;
  } else if (method == SEEMPS_TRUNC_REL_NORM2) {
    // errors[i] = sum of the i smallest s^2, accumulated from the smallest.
    // The loads of eight values are issued together: one add after another would
    // otherwise wait for a load each.
    double total = 0.0, x[8];
    for (int64_t i = 0; i < N; i += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = i + u < N ? ss[N - 1 - i - u] : 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u) total += x[u] * x[u];
    }
    const double max_error = total * tol;
    double acc = 0.0;
    int64_t i_stop = N - 1;
    for (int64_t i = 0; i < N && i_stop == N - 1; i += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = i + u < N ? ss[N - 1 - i - u] : 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (i + u < N && i_stop == N - 1 && acc > max_error) i_stop = i + u - 1;
        acc += x[u] * x[u];
      }
    }
    D = N - i_stop;
    if (D > max_bond) D = max_bond;
    double e = 0.0;  // errors[N - D]
    for (int64_t i = 0; i < N - D; i += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = i + u < N - D ? ss[N - 1 - i - u] : 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u) e += x[u] * x[u];
    }
    err = e;
  } else {
    const double thr = (method == SEEMPS_TRUNC_REL_SV) ? tol * ss[0] : tol;
    D = (N < max_bond) ? N : max_bond;
    for (int64_t i = 1; i < D; ++i) {
      if (ss[i] <= thr) {
        D = i;
        break;
      }
    }
    double e = 0.0;
    for (int64_t i = D; i < N; ++i) e += ss[i] * ss[i];
    err = e;
  }
  *D_out = D;
  *err_out = err;
}

}  // namespace seemps
