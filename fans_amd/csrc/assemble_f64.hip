// Assembly launches in double, k_assemble.
#include "assemble_launch.h"

namespace fans {
template void launch_general<double, ASM_CGLIN>(fans_gpu_ctx *, const AsmArgs<double> &, dim3);
template void launch_general<double, ASM_RESID>(fans_gpu_ctx *, const AsmArgs<double> &, dim3);
}
