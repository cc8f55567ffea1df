// FFT launches in double.
#include "fft_launch.h"

namespace fans {
FANS_FFT_INSTANCES(double)
}
