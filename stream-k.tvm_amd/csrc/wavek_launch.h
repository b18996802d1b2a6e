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

// One round of whole tiles, with scalar arguments that the command processor preloads into scalar registers (see
// sk_skinny_flat_kernel; the units are compiled with a preload count of 14): the first loads go out about a microsecond
// earlier than behind the argument structure and the plan.  Tiles are walked down their columns, as a raster of eight rows walks
// up to eight of them; XCD x takes a contiguous range of them.
struct FlatTile {
  int pm, pn;
};
static __device__ __forceinline__ FlatTile flat_tile(int tiles_m, int tiles_n) {
  const int b = blockIdx.x, grid = tiles_m * tiles_n, x = b & 7, id = x * (grid >> 3) + min(x, grid & 7) + (b >> 3);
  const int pn = (int)((uint32_t)id / (uint32_t)tiles_m);
  return FlatTile{id - pn * tiles_m, pn};
}
template <class P>
static __device__ __forceinline__ void flat_run(const typename P::Args &a, int tiles_m, const void *bias, char *smem) {
  const FlatTile t = flat_tile(tiles_m, (a.N + P::BN - 1) / P::BN);   // (gridDim would be a load from memory)
  typename P::Acc acc;
  if (bias != nullptr) P::prefetch_bias(a, acc, t.pn, bias);
  P::mac(a, acc, t.pm, t.pn, 0, (a.K + P::BK - 1) / P::BK, smem);
  P::store_c(a, acc, t.pm, t.pn, smem, bias);
}
template <class P>
__global__ __launch_bounds__(P::NT, P::WAVES_PER_EU) void sk_tile_wavek_flat_kernel(const half_t *A, const half_t *B, half_t *C, int M, int N,
                                                                                    int K, int lda, int ldb, int ldc, int tiles_m,
                                                                                    uint32_t start_scale, const void *bias, float alpha) {
  __shared__ __attribute__((aligned(1024))) char smem[P::LDS_BYTES];
  WaveKArgs a;
  a.A = A; a.B = B; a.C = C;
  a.M = M; a.N = N; a.K = K;
  a.lda = lda; a.ldb = ldb; a.ldc = ldc;
  a.alpha = alpha; a.scales = nullptr; a.zero = 0; a.groups = 0;
  a.start_scale = start_scale;
  flat_run<P>(a, tiles_m, bias, smem);
}
// the plans it runs
static inline bool flat_plan(const GemmArgs &a, const DevPlan &p, int bk) {
  return p.sk_tiles == 0 && p.grid == p.total_tiles && p.tiles_m <= 8 && (p.tiles_m == 1 || p.raster == 8) && p.xcd_remap == 1 &&
         p.ipt == (a.K + bk - 1) / bk && a.lda <= 0x7fffffff && a.ldb <= 0x7fffffff && a.ldc <= 0x7fffffff;
}

static inline uint32_t start_scale(const DevPlan &p) {
  const uint64_t round = (uint64_t)(p.grid < p.total_tiles ? p.grid : p.total_tiles);
  const uint64_t group = (uint64_t)(p.raster <= 0 ? 1 : (p.raster < p.tiles_m ? p.raster : p.tiles_m));
  return (uint32_t)(((group << 32) + round - 1) / round);
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
    typedef TileWaveK<TYPE, FM, FN, WAVEK_NN> P;                                                             \
    WaveKArgs w;                                                                                             \
    static_cast<GemmArgs &>(w) = a;                                                                          \
    w.start_scale = start_scale(p);                                                                          \
    if (flat_plan(a, p, P::BK))                                                                              \
      hipLaunchKernelGGL((sk_tile_wavek_flat_kernel<P>), dim3(p.grid), dim3(P::NT), 0, s, a.A, a.B, a.C, a.M, a.N, a.K, (int)a.lda, \
                         (int)a.ldb, (int)a.ldc, p.tiles_m, w.start_scale, bias, a.alpha);                    \
    else if (p.sk_tiles == 0)                                                                                \
      hipLaunchKernelGGL((sk_tile_wavek_kernel<P, false>), dim3(p.grid), dim3(P::NT), 0, s, w, p, ws, bias); \
    else                                                                                                     \
      hipLaunchKernelGGL((sk_tile_wavek_kernel<P, true>), dim3(p.grid), dim3(P::NT), 0, s, w, p, ws, bias);  \
    return (int)hipGetLastError();                                                                           \
  }
#define SK_WAVEK_OCC(TYPE, ID, FM, FN)                                                                                          \
  case ID: {                                                                                                                    \
    typedef TileWaveK<TYPE, FM, FN, WAVEK_NN> P;                                                                                          \
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, sk_tile_wavek_kernel<P, true>, P::NT, 0) == hipSuccess ? occ : -1; \
  }

}  // namespace sk
