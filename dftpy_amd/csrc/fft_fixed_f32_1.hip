// Size-specialised FFT passes in float, length group 1.
#include "fft_fixed.h"

namespace ofdft {
OFDFT_SIZES_1(OFDFT_SIZE_INST, float)
}  // namespace ofdft
