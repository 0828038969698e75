// Size table of the size-specialised FFT passes.
#include "fft_fixed.h"

namespace ofdft {

#define DECLARE(T, N) template <> const SizeOps<T> *size_ops<T, N>();
OFDFT_SIZES(DECLARE, float)
OFDFT_SIZES(DECLARE, double)
#undef DECLARE

#define CASE(T, N) \
    case N: return size_ops<T, N>();

template <> const SizeOps<float> *find_ops<float>(int n) {
    switch (n) {
        OFDFT_SIZES(CASE, float)
        default: return nullptr;
    }
}
template <> const SizeOps<double> *find_ops<double>(int n) {
    switch (n) {
        OFDFT_SIZES(CASE, double)
        default: return nullptr;
    }
}
#undef CASE

bool fixed_size(int n) { return find_ops<float>(n) != nullptr; }

}  // namespace ofdft
