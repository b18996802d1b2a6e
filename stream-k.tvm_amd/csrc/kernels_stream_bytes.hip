// Up to 64 rows of A against fp8 / int8 weights that stream through LDS in contiguous loads (tile_stream_pairs.h).
#include "skinny_launch.h"

namespace sk {

#define SK_STREAM_BYTES_POLICY(MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH, FMT) \
  TileStreamPairs<MB, WM, WN, RK, DEPTH, false, NB, AD, PAD, KH, FMT>

int stream_bytes_kernel_infos(KernelInfo *out, int max) {
  int n = 0;
#define INFO(id, DT, FMT, NAME, MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH)                                                    \
  if (n < max) {                                                                                                          \
    typedef SK_STREAM_BYTES_POLICY(MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH, FMT) P;                                        \
    out[n++] = KernelInfo{id, FAMILY_SKINNY, DT, 0, 8, P::BM, P::BN, 2 * P::BKC, P::NT, P::LDS_BYTES, P::CTAS_PER_CU,     \
                          P::TILE_ELEMS, 0, P::MAX_M, 16, NAME "_mb" #MB "_nb" #NB "_wm" #WM "_wn" #WN "_rk" #RK};        \
  }
#define X(id, MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH)                                   \
  INFO(id, 5, 1, "stream_f8e4m3", MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH)               \
  INFO(id + 10, 8, 2, "stream_f8e5m2", MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH)          \
  INFO(id + 20, 6, 3, "stream_i8", MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH)
  SK_STREAM_BYTES_KERNELS(X)
#undef X
#undef INFO
  return n;
}

int launch_stream_bytes(int id, const SkinnyArgs &a, const DevPlan &p, const Workspace &ws, hipStream_t s, const void *bias) {
  switch (id) {
#define X(id_, MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH)                                                                       \
  case id_:                                                                                                                  \
    return launch_policy<SK_STREAM_BYTES_POLICY(MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH, 1)>(a, p, ws, s, bias);              \
  case id_ + 10:                                                                                                             \
    return launch_policy<SK_STREAM_BYTES_POLICY(MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH, 2)>(a, p, ws, s, bias);              \
  case id_ + 20:                                                                                                             \
    return launch_policy<SK_STREAM_BYTES_POLICY(MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH, 3)>(a, p, ws, s, nullptr);
    SK_STREAM_BYTES_KERNELS(X)
#undef X
  }
  return (int)hipErrorInvalidValue;
}

int occupancy_stream_bytes(int id) {
  int occ = 0;
  switch (id) {
#define OCC(id_, FMT, MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH)                                                              \
  case id_: {                                                                                                              \
    typedef SK_STREAM_BYTES_POLICY(MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH, FMT) P;                                         \
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, sk_skinny_kernel<P>, P::NT, 0) == hipSuccess ? occ : -1;     \
  }
#define X(id_, MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH)               \
  OCC(id_, 1, MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH)                \
  OCC(id_ + 10, 2, MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH)           \
  OCC(id_ + 20, 3, MB, WM, WN, RK, DEPTH, NB, AD, PAD, KH)
    SK_STREAM_BYTES_KERNELS(X)
#undef X
#undef OCC
  }
  return -1;
}

}  // namespace sk
