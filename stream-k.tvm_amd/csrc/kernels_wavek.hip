// The tiles whose waves stream K on their own: from a kernel's id to the unit of its type.
#include "launch.h"
#include "tile_wavek.h"

namespace sk {

#define FOR_WAVEK_TYPES(F) F(WK_F16) F(WK_BF16) F(WK_F8E4M3) F(WK_F8E5M2) F(WK_I8)

int tile_wavek_kernel_infos(KernelInfo *out, int max) {
  int n = 0;
#define X(TYPE) n += wavek_kernel_infos<TYPE>(out + n, max - n);
  FOR_WAVEK_TYPES(X)
#undef X
  n += wavek_q4_kernel_infos(out + n, max - n);
  return n;
}

int launch_tile_wavek(int id, const GemmArgs &a, const DevPlan &p, const Workspace &ws, hipStream_t s, const void *bias) {
  switch (id >= 400 ? (id - 400) / 20 : -1) {
#define X(TYPE) case TYPE: return wavek_launch<TYPE>(id, a, p, ws, s, bias);
    FOR_WAVEK_TYPES(X)
#undef X
  }
  return launch_tile_q4(id, a, p, ws, s, bias);
}

int occupancy_tile_wavek(int id) {
  switch (id >= 400 ? (id - 400) / 20 : -1) {
#define X(TYPE) case TYPE: return wavek_occupancy<TYPE>(id);
    FOR_WAVEK_TYPES(X)
#undef X
  }
  if (id >= 520) return occupancy_wavek_q4(id);
  return occupancy_tile_q4(id);
}

}  // namespace sk
