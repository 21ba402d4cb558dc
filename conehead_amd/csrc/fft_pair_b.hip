// fft_pair_b.hip -- instances of the two-stage FFT passes (fft_pair.h).
#include "fft_pair_kernels.h"

namespace ch {

CH_PAIR(96, 12, 8)
CH_PAIR(128, 16, 8)
CH_PAIR(162, 18, 9)
CH_PAIR(240, 16, 15)
CH_PAIR(270, 18, 15)
CH_PAIR(384, 24, 16)

}  // namespace ch
