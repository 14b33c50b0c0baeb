// Grouped complex GEMM: many independent products C_p = op(A_p) op(B_p) of
// uneven shapes in one launch.  The host lists every output tile of every
// problem once (tile_prob[t] = problem of tile t, tiles of a problem in
// row-major order).  Tile shapes are 64 x 64 and 32 x 32.  Used by the
// batched overlap engine (many MPS of uneven length and bond dimension), where the
// tile shape is chosen by measurement.
#include "common.h"
#include "gemm_direct.h"

namespace seemps {
namespace {

// device-side view of SeempsGemmDesc (same layout, typed pointers)
struct GemmDesc {
  int64_t M, N, K;
  const double2* A;
  int64_t lda;
  const double2* B;
  int64_t ldb;
  double2* C;
  int64_t ldc;
  int64_t tiles_n;
  int64_t tile0;
};
static_assert(sizeof(GemmDesc) == sizeof(SeempsGemmDesc), "descriptor layout");

// Workgroups of four wavefronts, operands loaded straight into registers
// (gemm_direct.h, four real products for a complex one).  S = 64: the tile, a 32 x 32
// quarter for each wavefront.  S = 32: the tile, K cut in four runs.  S = 16: a
// quarter of a 32 x 32 tile, K cut in four runs.  Staging the operands in LDS cost a
// chain of loads and barriers every 16 of K and left the matrix cores idle most of
// the time: 64 overlaps of up to 40 sites, chi up to 128, 4.14 -> 1.86 ms.
template <int OPA, int OPB, int S>
__global__ __launch_bounds__(256) void grouped_zgemm_kernel(const GemmDesc* __restrict__ desc,
                                                            const int32_t* __restrict__ tile_prob) {
  extern __shared__ double2 part[];
  constexpr int QUARTERS = S == 16 ? 4 : 1, T = S == 16 ? 32 : S;
  const int64_t unit = xcd_tile(blockIdx.x, gridDim.x), tile = unit / QUARTERS;
  const GemmDesc d = desc[tile_prob[tile]];
  const int64_t local = tile - d.tile0;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int64_t m0 = (local / d.tiles_n) * T, n0 = (local % d.tiles_n) * T;
  if (S != 32) {
    const int quarter = S == 64 ? wv : (int)(unit % 4);
    m0 += T / 2 * (quarter >> 1);
    n0 += T / 2 * (quarter & 1);
    if (m0 >= d.M || n0 >= d.N) return;
  }
  direct::tile<OPA, OPB, S == 16 ? 1 : 2, S == 64 ? 1 : 4, false>(
      d.M, d.N, d.K, d.A, d.lda, d.B, d.ldb, m0, n0, S == 64 ? 0 : wv, part,
      [&](int64_t m, int64_t n, double2 acc) { d.C[m * d.ldc + n] = acc; });
}

template <int OPA, int OPB>
int launch_grouped(int tile_cfg, const GemmDesc* desc, const int32_t* tile_prob, int64_t ntiles,
                   hipStream_t s) {
  DeviceInfo info;
  const int ist = device_info(&info);
  if (ist) return ist;
  const dim3 block(256);
  if (tile_cfg == SEEMPS_TILE_64x64)
    hipLaunchKernelGGL((grouped_zgemm_kernel<OPA, OPB, 64>), dim3((unsigned)ntiles), block, 0, s,
                       desc, tile_prob);
  else if (ntiles >= 2 * (info.num_cu > 0 ? info.num_cu : 256))
    hipLaunchKernelGGL((grouped_zgemm_kernel<OPA, OPB, 32>), dim3((unsigned)ntiles), block,
                       4 * 16 * 64 * 16, s, desc, tile_prob);
  else  // quarters, for four times the wavefronts where two tiles a CU do not come together
    hipLaunchKernelGGL((grouped_zgemm_kernel<OPA, OPB, 16>), dim3((unsigned)(4 * ntiles)), block,
                       4 * 4 * 64 * 16, s, desc, tile_prob);
  return check_launch("grouped_zgemm");
}

}  // namespace
}  // namespace seemps

extern "C" int64_t seemps_grouped_tiles(int tile_cfg, int64_t M, int64_t N) {
  const int64_t t = tile_cfg == SEEMPS_TILE_64x64 ? 64 : 32;
  return seemps::ceil_div(M, t) * seemps::ceil_div(N, t);
}

extern "C" int seemps_zgemm_grouped(int opA, int opB, int tile_cfg, int64_t nprob,
                                    const void* desc, const int32_t* tile_prob, int64_t ntiles,
                                    void* stream) {
  using namespace seemps;
  SEEMPS_CHECK_ARG(tile_cfg == SEEMPS_TILE_64x64 || tile_cfg == SEEMPS_TILE_32x32,
                   "zgemm_grouped: invalid tile configuration");
  SEEMPS_CHECK_ARG(nprob >= 0 && ntiles >= 0 && ntiles < (1ll << 31),
                   "zgemm_grouped: invalid problem or tile count");
  if (ntiles == 0) return SEEMPS_OK;
  const GemmDesc* d = (const GemmDesc*)desc;
  hipStream_t s = (hipStream_t)stream;
  TimedLaunch timed("grouped_zgemm", s, 0.0);
#define SEEMPS_GROUPED_CASE(x, y) \
  if (opA == x && opB == y) return launch_grouped<x, y>(tile_cfg, d, tile_prob, ntiles, s);
  SEEMPS_GROUPED_CASE(SEEMPS_OP_N, SEEMPS_OP_N)
  SEEMPS_GROUPED_CASE(SEEMPS_OP_H, SEEMPS_OP_N)
  SEEMPS_GROUPED_CASE(SEEMPS_OP_N, SEEMPS_OP_T)
  SEEMPS_GROUPED_CASE(SEEMPS_OP_T, SEEMPS_OP_N)
  SEEMPS_GROUPED_CASE(SEEMPS_OP_C, SEEMPS_OP_N)
  SEEMPS_GROUPED_CASE(SEEMPS_OP_N, SEEMPS_OP_H)
#undef SEEMPS_GROUPED_CASE
  set_error("zgemm_grouped: op pair (%d, %d) not instantiated", opA, opB);
  return SEEMPS_ERR_INVALID;
}
