// Assembly launches in float, k_assemble.
#include "assemble_launch.h"

namespace fans {
template void launch_general<float, ASM_CGLIN>(fans_gpu_ctx *, const AsmArgs<float> &, dim3);
}
