// fp16 / bfloat16 tile kernels for 65 to 128 rows, operands through rings of different depths (tile_ring16.h).
#include "launch.h"
#include "sk_persistent.h"
#include "tile_ring16.h"

namespace sk {

template <class P, bool FIXUP>
__global__ __launch_bounds__(P::NT, P::WAVES_PER_EU) void sk_tile_ring_kernel(typename P::Args a, DevPlan plan, Workspace ws,
                                                                              const void *bias) {
  __shared__ __attribute__((aligned(1024))) char smem[P::LDS_BYTES];
  run_persistent<P, FIXUP, true>(a, plan, ws, smem, bias);
}

int tile_ring_kernel_infos(KernelInfo *out, int max) {
  int n = 0;
#define X(id, BM, BN, BK, WM, WN, KH, WD, AD, BF)                                                                              \
  if (n < max) {                                                                                                           \
    typedef TileRing16<BM, BN, BK, WM, WN, KH, WD, AD, BF> P;                                                                  \
    out[n++] = KernelInfo{id, FAMILY_TILE, (BF) ? 3 : 0, 0, 9, BM, BN, BK, P::NT, P::LDS_TOTAL, P::CTAS_PER_CU,            \
                          P::TILE_ELEMS, 0, 0, 8, (BF) ? "tile_bf16_ring_" #BM "x" #BN "x" #BK : "tile_f16_ring_" #BM "x" #BN "x" #BK}; \
  }
  SK_TILE_RING_KERNELS(X)
#undef X
  return n;
}

int launch_tile_ring(int id, const GemmArgs &a, const DevPlan &p, const Workspace &ws, hipStream_t s, const void *bias) {
  switch (id) {
#define X(id_, BM, BN, BK, WM, WN, KH, WD, AD, BF)                                                                 \
  case id_: {                                                                                                  \
    typedef TileRing16<BM, BN, BK, WM, WN, KH, WD, AD, BF> P;                                                      \
    if (p.sk_tiles == 0)                                                                                       \
      hipLaunchKernelGGL((sk_tile_ring_kernel<P, false>), dim3(p.grid), dim3(P::NT), 0, s, a, p, ws, bias);    \
    else                                                                                                       \
      hipLaunchKernelGGL((sk_tile_ring_kernel<P, true>), dim3(p.grid), dim3(P::NT), 0, s, a, p, ws, bias);     \
    return (int)hipGetLastError();                                                                             \
  }
    SK_TILE_RING_KERNELS(X)
#undef X
  }
  return launch_tile_wavek(id, a, p, ws, s, bias);
}

int occupancy_tile_ring(int id) {
  int occ = 0;
  switch (id) {
#define X(id_, BM, BN, BK, WM, WN, KH, WD, AD, BF)                                                                              \
  case id_: {                                                                                                               \
    typedef TileRing16<BM, BN, BK, WM, WN, KH, WD, AD, BF> P;                                                                   \
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, sk_tile_ring_kernel<P, true>, P::NT, 0) == hipSuccess ? occ : -1; \
  }
    SK_TILE_RING_KERNELS(X)
#undef X
  }
  return occupancy_tile_wavek(id);
}

}  // namespace sk
