// Tiles for Q4 weights whose waves stream K on their own (tile_wavek_q4.h).
#include "launch.h"
#include "sk_persistent.h"
#include "tile_wavek_q4.h"
#include "wavek_launch.h"

namespace sk {

template <class P, bool FIXUP>
__global__ __launch_bounds__(P::NT, P::WAVES_PER_EU) void sk_tile_wavek_q4_kernel(typename P::Args a, DevPlan plan, Workspace ws,
                                                                                  const void *bias) {
  __shared__ __attribute__((aligned(1024))) char smem[P::LDS_BYTES];
  run_persistent<P, FIXUP, true>(a, plan, ws, smem, bias);
}

// (what the loop needs leads the arguments, as many as are preloaded -- hence the tiles, at most eight, and the zero point in one; the
// others are read later)
template <class P>
__global__ __launch_bounds__(P::NT, P::WAVES_PER_EU) void sk_tile_wavek_q4_flat_kernel(const half_t *A, const half_t *B, const half_t *scales,
                                                                                       const half_t *zeros, int M, int N, int K, int lda,
                                                                                       int tiles_zero, uint32_t start_scale, half_t *C, int ldc,
                                                                                       const void *bias) {
  __shared__ __attribute__((aligned(1024))) char smem[P::LDS_BYTES];
  WaveKQ4Args a;
  a.A = A; a.B = B; a.C = C;
  a.M = M; a.N = N; a.K = K;
  a.lda = lda; a.ldb = K / 2; a.ldc = ldc;
  a.alpha = 1.f; a.scales = scales; a.zero = tiles_zero >> 8; a.groups = K / 128;
  a.start_scale = start_scale;
  a.zeros = zeros;
  flat_run<P>(a, tiles_zero & 255, bias, smem);
}

int wavek_q4_kernel_infos(KernelInfo *out, int max) {
  int n = 0;
#define INFO(id, DT, TYPE, TILED, NAME, FM, FN)                                                                                   \
  if (n < max) {                                                                                                                  \
    typedef TileWaveKQ4<TYPE, FM, FN, TILED> P;                                                                                   \
    out[n++] = KernelInfo{id, FAMILY_TILE, DT, 0, 10, P::BM, P::BN, P::BK, P::NT, P::LDS_TOTAL, P::CTAS_PER_CU, P::TILE_ELEMS, 0, \
                          0, 128, NAME "_" #FM "x" #FN};                                                                          \
  }
#define X(id, FM, FN)                                    \
  INFO(id, 2, WK_Q4, false, "wavek_q4", FM, FN)          \
  INFO(id + 20, 7, WK_Q4ZP, false, "wavek_q4zp", FM, FN) \
  INFO(id + 40, 4, WK_Q4, true, "wavek_q4t", FM, FN)     \
  INFO(id + 60, 9, WK_Q4ZP, true, "wavek_q4zpt", FM, FN)
  SK_TILE_WAVEK_Q4_KERNELS(X)
#undef X
#undef INFO
  return n;
}

template <class P>
static int launch(const WaveKQ4Args &a, const DevPlan &p, const Workspace &ws, hipStream_t s, const void *bias) {
  if (flat_plan(a, p, P::BK) && a.ldb == a.K / 2 && a.groups == a.K / 128)
    hipLaunchKernelGGL((sk_tile_wavek_q4_flat_kernel<P>), dim3(p.grid), dim3(P::NT), 0, s, a.A, a.B, a.scales, a.zeros, a.M, a.N, a.K,
                       (int)a.lda, p.tiles_m | a.zero << 8, a.start_scale, a.C, (int)a.ldc, bias);
  else if (p.sk_tiles == 0)
    hipLaunchKernelGGL((sk_tile_wavek_q4_kernel<P, false>), dim3(p.grid), dim3(P::NT), 0, s, a, p, ws, bias);
  else
    hipLaunchKernelGGL((sk_tile_wavek_q4_kernel<P, true>), dim3(p.grid), dim3(P::NT), 0, s, a, p, ws, bias);
  return (int)hipGetLastError();
}

int launch_wavek_q4(int id, const GemmArgs &g, const void *zeros, const DevPlan &p, const Workspace &ws, hipStream_t s, const void *bias) {
  WaveKQ4Args a;
  static_cast<GemmArgs &>(a) = g;
  a.start_scale = start_scale(p);
  a.zeros = static_cast<const half_t *>(zeros);
  switch (id) {
#define X(id_, FM, FN)                                                               \
  case id_: return launch<TileWaveKQ4<WK_Q4, FM, FN>>(a, p, ws, s, bias);            \
  case id_ + 20: return launch<TileWaveKQ4<WK_Q4ZP, FM, FN>>(a, p, ws, s, bias);     \
  case id_ + 40: return launch<TileWaveKQ4<WK_Q4, FM, FN, true>>(a, p, ws, s, bias); \
  case id_ + 60: return launch<TileWaveKQ4<WK_Q4ZP, FM, FN, true>>(a, p, ws, s, bias);
    SK_TILE_WAVEK_Q4_KERNELS(X)
#undef X
  }
  return (int)hipErrorInvalidValue;
}

int occupancy_wavek_q4(int id) {
  int occ = 0;
  switch (id) {
#define OCC(id_, TYPE, TILED, FM, FN)                                                                                              \
  case id_: {                                                                                                                      \
    typedef TileWaveKQ4<TYPE, FM, FN, TILED> P;                                                                                    \
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, sk_tile_wavek_q4_kernel<P, true>, P::NT, 0) == hipSuccess ? occ : -1; \
  }
#define X(id_, FM, FN)                   \
  OCC(id_, WK_Q4, false, FM, FN)         \
  OCC(id_ + 20, WK_Q4ZP, false, FM, FN)  \
  OCC(id_ + 40, WK_Q4, true, FM, FN)     \
  OCC(id_ + 60, WK_Q4ZP, true, FM, FN)
    SK_TILE_WAVEK_Q4_KERNELS(X)
#undef X
#undef OCC
  }
  return -1;
}

}  // namespace sk
