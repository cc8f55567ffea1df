// FFT launches in float.
#include "fft_launch.h"

namespace fans {
FANS_FFT_INSTANCES(float)
}
