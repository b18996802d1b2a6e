// The tiles whose waves stream K on their own (tile_wavek.h) for one type of operands.
#define WAVEK_NAME "wavek_f8e4m3"
#define WAVEK_NN false
#include "wavek_launch.h"

namespace sk {
SK_WAVEK_UNIT(WK_F8E4M3, 5, WAVEK_NN, SK_TILE_WAVEK_KERNELS)
}  // namespace sk
