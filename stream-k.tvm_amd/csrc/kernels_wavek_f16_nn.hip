// The tiles whose waves stream K on their own (tile_wavek.h) for [K, N] weights of one type.
#define WAVEK_NAME "wavek_f16_nn"
#define WAVEK_NN true
#include "wavek_launch.h"

namespace sk {
SK_WAVEK_UNIT(WK_F16, 0, WAVEK_NN, SK_TILE_WAVEK_NN_KERNELS)
}  // namespace sk
