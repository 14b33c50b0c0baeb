// One output tile of a complex128 GEMM with the operands loaded straight into the
// layout of v_mfma_f64_16x16x4f64 (A[i][k] from lane i + 16k, B[k][j] from lane
// j + 16k, result item r of lane l is D[l/16 + 4r][l%16]): no LDS staging and no
// barrier in the loop.  FP64 MFMA asks little of the memory path (a 32 x 32 step of
// four k is 768 to 1024 cycles of the matrix core for 4 KB), so a wavefront loads
// its own operands, four steps ahead of the four in use.
#pragma once

#include "common.h"

namespace seemps {
namespace direct {

typedef double d4 __attribute__((ext_vector_type(4)));

// The tile of 16 F x 16 F at (m0, n0), K cut in KS runs over the workgroup's
// wavefronts (wv), whose partial tiles are summed in LDS (`part`, KS x 4 F F x 64,
// unused for KS = 1) in the order of the runs; store(m, n, value) for every entry
// inside M x N.  G3: three real products for a complex one, else four.
template <int OPA, int OPB, int F, int KS, bool G3, class Store>
__device__ __forceinline__ void tile(int64_t M, int64_t N, int64_t K,
                                     const double2* __restrict__ A, int64_t lda,
                                     const double2* __restrict__ B, int64_t ldb, int64_t m0,
                                     int64_t n0, int wv, double2* part, Store store) {
  constexpr int U = 4;  // steps of four k in a block; one block is loaded ahead
  constexpr bool AT = OPA == SEEMPS_OP_T || OPA == SEEMPS_OP_H;
  constexpr bool BT = OPB == SEEMPS_OP_T || OPB == SEEMPS_OP_H;
  constexpr double SGA = (OPA == SEEMPS_OP_C || OPA == SEEMPS_OP_H) ? -1.0 : 1.0;
  constexpr double SGB = (OPB == SEEMPS_OP_C || OPB == SEEMPS_OP_H) ? -1.0 : 1.0;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  // rows and columns past the edge are read from the last one and not stored
  const double2 *pa[F], *pb[F];
#pragma unroll
  for (int f = 0; f < F; ++f) {
    const int64_t m = min(m0 + 16 * f + li, M - 1), n = min(n0 + 16 * f + li, N - 1);
    pa[f] = AT ? A + m : A + m * lda;
    pb[f] = BT ? B + n * ldb : B + n;
  }
  const int64_t stepA = AT ? lda : 1, stepB = BT ? 1 : ldb;
  // G3: sums of ar br, ai bi and (ar + ai)(br + bi); else of the real and imaginary parts
  d4 t1[F][F], t2[F][F], t3[F][F];
#pragma unroll
  for (int a = 0; a < F; ++a)
#pragma unroll
    for (int b = 0; b < F; ++b) t1[a][b] = t2[a][b] = t3[a][b] = d4{0.0, 0.0, 0.0, 0.0};
  auto load = [&](int64_t k, double2 (&x)[F], double2 (&y)[F]) {
#pragma unroll
    for (int f = 0; f < F; ++f) {
      x[f] = pa[f][k * stepA];
      y[f] = pb[f][k * stepB];
    }
  };
  auto mac = [&](const double2 (&x)[F], const double2 (&y)[F]) {
#pragma unroll
    for (int a = 0; a < F; ++a)
#pragma unroll
      for (int b = 0; b < F; ++b) {
        if (G3) {
          t1[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[a].x, y[b].x, t1[a][b], 0, 0, 0);
          t2[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[a].y, y[b].y, t2[a][b], 0, 0, 0);
          t3[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(
              x[a].x + SGA * x[a].y, y[b].x + SGB * y[b].y, t3[a][b], 0, 0, 0);
        } else {
          t1[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[a].x, y[b].x, t1[a][b], 0, 0, 0);
          t1[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(-SGA * SGB * x[a].y, y[b].y, t1[a][b],
                                                          0, 0, 0);
          t2[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[a].x, SGB * y[b].y, t2[a][b], 0, 0,
                                                          0);
          t2[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(SGA * x[a].y, y[b].x, t2[a][b], 0, 0,
                                                          0);
        }
      }
  };
  const int64_t steps = ceil_div(K, (int64_t)4), per = ceil_div(steps, (int64_t)KS);
  const int64_t s0 = min(wv * per, steps), s1 = min(s0 + per, steps);
  const int64_t full = min(s1, K / 4);  // steps [s0, full) need no bounds test
  const int64_t nb = full > s0 ? (full - s0) / U : 0;
  double2 x[2][U][F], y[2][U][F];
  auto load_block = [&](int64_t b, double2 (&xx)[U][F], double2 (&yy)[U][F]) {
#pragma unroll
    for (int u = 0; u < U; ++u) load((s0 + b * U + u) * 4 + lk, xx[u], yy[u]);
  };
  if (nb > 0) load_block(0, x[0], y[0]);
  for (int64_t b = 0; b < nb; b += 2) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (b + i < nb) {
        // a test keeps small tiles from a load too many, large ones hide it
        if (F > 1)
          load_block(min(b + i + 1, nb - 1), x[(i + 1) % 2], y[(i + 1) % 2]);
        else if (b + i + 1 < nb)
          load_block(b + i + 1, x[(i + 1) % 2], y[(i + 1) % 2]);
#pragma unroll
        for (int u = 0; u < U; ++u) mac(x[i][u], y[i][u]);
      }
    }
  }
  // the last steps together: past the run or past K they are read in bounds
  // and count as zero
  if (s0 + nb * U < s1) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t s = s0 + nb * U + u;
      load(min(s * 4 + lk, K - 1), x[0][u], y[0][u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t s = s0 + nb * U + u;
      if (s >= s1) break;
      if (s * 4 + lk >= K) {
#pragma unroll
        for (int f = 0; f < F; ++f) x[0][u][f] = y[0][u][f] = make_double2(0.0, 0.0);
      }
      mac(x[0][u], y[0][u]);
    }
  }
  auto put = [&](int a, int b, int r, double2 acc) {
    const int64_t m = m0 + 16 * a + lk + 4 * r, n = n0 + 16 * b + li;
    if (m < M && n < N) store(m, n, acc);
  };
#pragma unroll
  for (int a = 0; a < F; ++a)
#pragma unroll
    for (int b = 0; b < F; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double u = t1[a][b][r], v = t2[a][b][r];
        const double2 acc = G3 ? make_double2(u - SGA * SGB * v, (t3[a][b][r] - u) - SGA * SGB * v)
                               : make_double2(u, v);
        if (KS == 1)
          put(a, b, r, acc);
        else
          part[(wv * (4 * F * F) + (a * F + b) * 4 + r) * 64 + lane] = acc;
      }
  if (KS == 1) return;
  __syncthreads();
#pragma unroll
  for (int a = 0; a < F; ++a)
#pragma unroll
    for (int b = 0; b < F; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int item = (a * F + b) * 4 + r;
        if (item % KS != wv) continue;
        double2 acc = part[item * 64 + lane];
#pragma unroll
        for (int q = 1; q < KS; ++q) acc = cadd(acc, part[(q * (4 * F * F) + item) * 64 + lane]);
        put(a, b, r, acc);
      }
}

}  // namespace direct
}  // namespace seemps
