// Kernel entry, table entries and launcher of the tiles whose waves stream K on their own, shared by the units that compile them
// for one type each (WAVEK_NAME: what the kernels are called, WAVEK_NN: whether the weights are [K, N]).
#pragma once
#include "launch.h"
#include "sk_persistent.h"
#include "tile_wavek.h"

namespace sk {

template <class P, bool FIXUP>
__global__ __launch_bounds__(P::NT, P::WAVES_PER_EU) void sk_tile_wavek_kernel(typename P::Args a, DevPlan plan, Workspace ws,
                                                                               const void *bias) {
  __shared__ __attribute__((aligned(1024))) char smem[P::LDS_BYTES];
  run_persistent<P, FIXUP, true>(a, plan, ws, smem, bias);
}

// ids of a type
constexpr int wavek_base(int type, bool nn = false) { return (nn ? 600 : 400) + 20 * type; }

#define SK_WAVEK_UNIT(TYPE, SK_DTYPE, NN, LIST)                                                                                \
  template <>                                                                                                                  \
  int wavek_kernel_infos<TYPE, NN>(KernelInfo * out, int max) {                                                                    \
    int n = 0;                                                                                                                 \
    LIST(SK_WAVEK_INFO, TYPE, wavek_base(TYPE, NN))                                                               \
    for (int i = 0; i < n; ++i) out[i].dtype = SK_DTYPE, out[i].layout = NN;                                                                       \
    return n;                                                                                                                  \
  }                                                                                                                            \
  template <>                                                                                                                  \
  int wavek_launch<TYPE, NN>(int id, const GemmArgs &a, const DevPlan &p, const Workspace &ws, hipStream_t s, const void *bias) {  \
    switch (id) { LIST(SK_WAVEK_LAUNCH, TYPE, wavek_base(TYPE, NN)) }                                             \
    return (int)hipErrorInvalidValue;                                                                                          \
  }                                                                                                                            \
  template <>                                                                                                                  \
  int wavek_occupancy<TYPE, NN>(int id) {                                                                                          \
    int occ = 0;                                                                                                               \
    switch (id) { LIST(SK_WAVEK_OCC, TYPE, wavek_base(TYPE, NN)) }                                                \
    return -1;                                                                                                                 \
  }
#define SK_WAVEK_INFO(TYPE, ID, FM, FN)                                                                                          \
  if (n < max) {                                                                                                                 \
    typedef TileWaveK<TYPE, FM, FN, WAVEK_NN> P;                                                                                           \
    constexpr bool one_byte = TYPE >= WK_F8E4M3;                                                                                 \
    out[n++] = KernelInfo{ID, FAMILY_TILE, 0, 0, 10, P::BM, P::BN, one_byte ? 2 * P::BK : P::BK, P::NT, P::LDS_TOTAL,            \
                          P::CTAS_PER_CU, P::TILE_ELEMS, 0, 0, one_byte ? 16 : 8, WAVEK_NAME "_" #FM "x" #FN};                   \
  }
#define SK_WAVEK_LAUNCH(TYPE, ID, FM, FN)                                                                    \
  case ID: {                                                                                                 \
    typedef TileWaveK<TYPE, FM, FN, WAVEK_NN> P;                                                                       \
    if (p.sk_tiles == 0)                                                                                     \
      hipLaunchKernelGGL((sk_tile_wavek_kernel<P, false>), dim3(p.grid), dim3(P::NT), 0, s, a, p, ws, bias); \
    else                                                                                                     \
      hipLaunchKernelGGL((sk_tile_wavek_kernel<P, true>), dim3(p.grid), dim3(P::NT), 0, s, a, p, ws, bias);  \
    return (int)hipGetLastError();                                                                           \
  }
#define SK_WAVEK_OCC(TYPE, ID, FM, FN)                                                                                          \
  case ID: {                                                                                                                    \
    typedef TileWaveK<TYPE, FM, FN, WAVEK_NN> P;                                                                                          \
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, sk_tile_wavek_kernel<P, true>, P::NT, 0) == hipSuccess ? occ : -1; \
  }

}  // namespace sk
