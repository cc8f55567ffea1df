// Assembly launches in float.
#include "assemble_launch.h"

namespace fans {
template void launch_modal<float, 1, 8, ASM_CGLIN>(fans_gpu_ctx *, const AsmArgs<float> &, dim3);
template void launch_modal<float, 1, 1, ASM_CGLIN>(fans_gpu_ctx *, const AsmArgs<float> &, dim3);
template void launch_modal<float, 3, 8, ASM_CGLIN>(fans_gpu_ctx *, const AsmArgs<float> &, dim3);
template void launch_modal<float, 3, 1, ASM_CGLIN>(fans_gpu_ctx *, const AsmArgs<float> &, dim3);
}
