// Size-specialised FFT passes in float, length group 0.
#include "fft_fixed.h"

namespace ofdft {
OFDFT_SIZES_0(OFDFT_SIZE_INST, float)
}  // namespace ofdft
