// The tiles whose waves stream K on their own: from a kernel's id to the unit of its type.
#include "launch.h"
#include "tile_wavek.h"

namespace sk {

// F(type, [K, N] weights, first id)
#define FOR_WAVEK_UNITS(F)   \
  F(WK_F16, false, 400)      \
  F(WK_BF16, false, 420)     \
  F(WK_F8E4M3, false, 440)   \
  F(WK_F8E5M2, false, 460)   \
  F(WK_I8, false, 480)       \
  F(WK_F16, true, 600)       \
  F(WK_BF16, true, 620)

int tile_wavek_kernel_infos(KernelInfo *out, int max) {
  int n = 0;
#define X(TYPE, NN, BASE) n += wavek_kernel_infos<TYPE, NN>(out + n, max - n);
  FOR_WAVEK_UNITS(X)
#undef X
  n += wavek_q4_kernel_infos(out + n, max - n);
  return n;
}

int launch_tile_wavek(int id, const GemmArgs &a, const DevPlan &p, const Workspace &ws, hipStream_t s, const void *bias) {
  switch (id / 20) {   // (every unit has twenty ids)
#define X(TYPE, NN, BASE) case BASE / 20: return wavek_launch<TYPE, NN>(id, a, p, ws, s, bias);
    FOR_WAVEK_UNITS(X)
#undef X
  }
  return launch_tile_q4(id, a, p, ws, s, bias);
}

int occupancy_tile_wavek(int id) {
  switch (id / 20) {
#define X(TYPE, NN, BASE) case BASE / 20: return wavek_occupancy<TYPE, NN>(id);
    FOR_WAVEK_UNITS(X)
#undef X
  }
  if (id >= 520 && id < 600) return occupancy_wavek_q4(id);
  return occupancy_tile_q4(id);
}

}  // namespace sk
