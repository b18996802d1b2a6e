// The tiles whose waves stream K on their own (tile_wavek.h) for one type of operands.
#define WAVEK_NAME "wavek_i8"
#define WAVEK_NN false
#include "wavek_launch.h"

namespace sk {
SK_WAVEK_UNIT(WK_I8, 6, WAVEK_NN, SK_TILE_WAVEK_KERNELS)
}  // namespace sk
