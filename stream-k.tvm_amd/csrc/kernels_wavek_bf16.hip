// The tiles whose waves stream K on their own (tile_wavek.h) for one type of operands.
#define WAVEK_NAME "wavek_bf16"
#include "wavek_launch.h"

namespace sk {
SK_WAVEK_UNIT(WK_BF16, 3, WAVEK_NAME)
}  // namespace sk
