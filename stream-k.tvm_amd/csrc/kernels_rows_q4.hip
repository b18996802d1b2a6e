// Q4 weights with up to 16 rows of A, every wave streaming K on its own (tile_rows_q4.h).
#include "skinny_launch.h"
#include "tile_rows_q4.h"

namespace sk {

int rows_q4_kernel_infos(KernelInfo *out, int max) {
  int n = 0;
#define X(id, MR, NB, S, ZP, GM, TD)                                                                                       \
  if (n < max) {                                                                                                       \
    typedef TileRowsQ4<MR, NB, S, ZP, GM, TD> P;                                                                           \
    out[n++] = KernelInfo{id, FAMILY_SKINNY, (TD) ? 9 /* SK_Q4_ZP_TILED */ : ((ZP) ? 7 /* SK_Q4_ZP */ : 2 /* SK_Q4 */), 0, 5, P::BM, P::BN, P::BKC, P::NT, \
                          P::LDS_BYTES, P::CTAS_PER_CU, P::TILE_ELEMS, P::MAX_ITERS, P::MAX_M, 128,                    \
                          (TD) ? "rows_q4zpt_m" #MR "_nb" #NB "_s" #S : (ZP) ? "rows_q4zp_m" #MR "_nb" #NB "_s" #S : "rows_q4_m" #MR "_nb" #NB "_s" #S};             \
  }
  SK_ROWS_Q4_KERNELS(X)
#undef X
  return n;
}

int launch_rows_q4(int id, const SkinnyArgs &a, const DevPlan &p, const Workspace &ws, hipStream_t s, const void *bias) {
  switch (id) {
#define X(id_, MR, NB, S, ZP, GM, TD)                                                  \
  case id_:                                                                        \
    return launch_policy<TileRowsQ4<MR, NB, S, ZP, GM, TD>>(a, p, ws, s, bias);
    SK_ROWS_Q4_KERNELS(X)
#undef X
  }
  return launch_stream_bytes(id, a, p, ws, s, bias);
}

int occupancy_rows_q4(int id) {
  int occ = 0;
  switch (id) {
#define X(id_, MR, NB, S, ZP, GM, TD)                                                                                      \
  case id_: {                                                                                                          \
    typedef TileRowsQ4<MR, NB, S, ZP, GM, TD> P;                                                                           \
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, sk_skinny_kernel<P>, P::NT, 0) == hipSuccess ? occ : -1; \
  }
    SK_ROWS_Q4_KERNELS(X)
#undef X
  }
  return occupancy_stream_bytes(id);
}

}  // namespace sk
