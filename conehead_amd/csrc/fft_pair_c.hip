// fft_pair_c.hip -- instances of the two-stage FFT passes (fft_pair.h).
#include "fft_pair_kernels.h"

namespace ch {

CH_PAIR(80, 10, 8)
CH_PAIR(108, 12, 9)
CH_PAIR(120, 12, 10)
CH_PAIR(192, 16, 12)
CH_PAIR(216, 18, 12)
CH_PAIR(300, 20, 15)
CH_PAIR(360, 20, 18)

}  // namespace ch
