// fp32 Stream-K kernels (gfx950): fp32 MFMA tiles, B as [K,N] or [N,K].
#include "launch.h"
#include "sk_persistent.h"
#include "tile_f32.h"

namespace sk {

template <class P, bool FIXUP>
__global__ __launch_bounds__(P::NT, P::WAVES_PER_EU) void sk_f32_kernel(typename P::Args a, DevPlan plan, Workspace ws) {
  __shared__ __attribute__((aligned(1024))) char smem[P::LDS_BYTES];
  run_persistent<P, FIXUP>(a, plan, ws, smem);
}

// X(id, B is [K,N], BM, BN, BK, WM, WN, stages, CTAs per CU); the reference's own fp32 run is 16 x 16384 x 8192
// (streamk_fp32.py:10-12 with the values of :24-28).  A tile without its K-iteration, or a schedule or grid without a tile,
// names the first four: 16 K-values, two CTAs per CU.  The [N,K] tiles of 128 x 128 and 32 x 256 also exist with 32, which
// the planner takes when everything is left to it (weights from HBM, 16 / 32 K-values, in us: 32 x 8192 x 8192 71.6 / 67.4,
// 32 x 28672 x 4096 112 / 106, 32 x 11008 x 4096 53.5 / 52.7, 16 x 16384 x 8192 103 / 104).
#define SK_F32_KERNELS(X)                    \
  X(200, true, 128, 128, 16, 2, 2, 4, 2)     \
  X(201, false, 128, 128, 16, 2, 2, 4, 2)    \
  X(202, true, 32, 256, 16, 1, 4, 4, 2)      \
  X(203, false, 32, 256, 16, 1, 4, 4, 2)     \
  X(204, true, 64, 64, 32, 2, 2, 5, 2)       \
  X(205, false, 64, 64, 32, 2, 2, 5, 2)      \
  X(206, true, 64, 128, 32, 2, 2, 3, 2)      \
  X(207, false, 64, 128, 32, 2, 2, 3, 2)     \
  X(208, true, 32, 64, 32, 1, 4, 6, 2)       \
  X(209, false, 32, 64, 64, 1, 4, 6, 1)      \
  X(212, false, 128, 128, 32, 2, 2, 2, 2)    \
  X(213, false, 32, 256, 32, 1, 4, 4, 1)

int f32_kernel_infos(KernelInfo *out, int max) {
  int n = 0;
#define X(id, KN, TBM, TBN, TBK, TWM, TWN, ST, CT)                                                                        \
  if (n < max) {                                                                                                          \
    typedef TileF32<KN, TBM, TBN, TBK, TWM, TWN, ST, CT> P;                                                               \
    out[n++] = KernelInfo{id, FAMILY_TILE, 1, (KN) ? 1 : 0, 0, TBM, TBN, TBK, P::NT, P::LDS_TOTAL,                        \
                          P::CTAS_PER_CU, P::TILE_ELEMS, 0, 0, 4,                                                         \
                          (KN) ? "tile_f32_nn_" #TBM "x" #TBN "x" #TBK : "tile_f32_nt_" #TBM "x" #TBN "x" #TBK};          \
  }
  SK_F32_KERNELS(X)
#undef X
  return n;
}

int launch_f32(int id, const GemmArgsF32 &a, const DevPlan &p, const Workspace &ws, hipStream_t s) {
  switch (id) {
#define X(id_, KN, TBM, TBN, TBK, TWM, TWN, ST, CT)                                                                      \
  case id_:                                                                                                             \
    if (p.sk_tiles > 0)                                                                                                 \
      hipLaunchKernelGGL((sk_f32_kernel<TileF32<KN, TBM, TBN, TBK, TWM, TWN, ST, CT>, true>), dim3(p.grid), dim3(256), 0, s, a, p, ws); \
    else                                                                                                                \
      hipLaunchKernelGGL((sk_f32_kernel<TileF32<KN, TBM, TBN, TBK, TWM, TWN, ST, CT>, false>), dim3(p.grid), dim3(256), 0, s, a, p, ws); \
    return (int)hipGetLastError();
    SK_F32_KERNELS(X)
#undef X
  }
  return (int)hipErrorInvalidValue;
}

int occupancy_f32(int id) {
  int occ = 0;
  switch (id) {
#define X(id_, KN, TBM, TBN, TBK, TWM, TWN, ST, CT)                                                                       \
  case id_:                                                                                                               \
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(                                                                  \
               &occ, sk_f32_kernel<TileF32<KN, TBM, TBN, TBK, TWM, TWN, ST, CT>, true>, 256, 0) == hipSuccess             \
               ? occ                                                                                                      \
               : -1;
    SK_F32_KERNELS(X)
#undef X
  }
  return -1;
}

}  // namespace sk
