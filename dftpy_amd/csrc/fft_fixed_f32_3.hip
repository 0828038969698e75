// Size-specialised FFT passes in float, length group 3.
#include "fft_fixed.h"

namespace ofdft {
OFDFT_SIZES_3(OFDFT_SIZE_INST, float)
}  // namespace ofdft
