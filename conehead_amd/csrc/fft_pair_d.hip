// fft_pair_d.hip -- instances of the two-stage FFT passes (fft_pair.h).
#include "fft_pair_kernels.h"

namespace ch {

CH_PAIR(72, 8, 9)
CH_PAIR(90, 10, 9)
CH_PAIR(150, 10, 15)
CH_PAIR(160, 16, 10)
CH_PAIR(256, 16, 16)
CH_PAIR(320, 20, 16)
CH_PAIR(324, 18, 18)

}  // namespace ch
