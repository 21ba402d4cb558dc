// fft_pair_a.hip -- instances of the two-stage FFT passes (fft_pair.h).
#include "fft_pair_kernels.h"

namespace ch {

CH_PAIR(100, 10, 10)
CH_PAIR(144, 12, 12)
CH_PAIR(180, 12, 15)
CH_PAIR(200, 20, 10)
CH_PAIR(288, 18, 16)
CH_PAIR(400, 20, 20)

}  // namespace ch
