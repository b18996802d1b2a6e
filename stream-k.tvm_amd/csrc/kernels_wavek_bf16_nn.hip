// The tiles whose waves stream K on their own (tile_wavek.h) for [K, N] weights of one type.
#define WAVEK_NAME "wavek_bf16_nn"
#define WAVEK_NN true
#include "wavek_launch.h"

namespace sk {
SK_WAVEK_UNIT(WK_BF16, 3, WAVEK_NN, SK_TILE_WAVEK_NN_KERNELS)
}  // namespace sk
