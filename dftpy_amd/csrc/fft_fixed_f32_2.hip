// Size-specialised FFT passes in float, length group 2.
#include "fft_fixed.h"

namespace ofdft {
OFDFT_SIZES_2(OFDFT_SIZE_INST, float)
}  // namespace ofdft
