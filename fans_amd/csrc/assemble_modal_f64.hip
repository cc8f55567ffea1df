// Assembly launches in FP64, k_assemble_modal.
#include "assemble_launch.h"

namespace fans {
template void launch_modal<double, 1, 8, ASM_CGLIN>(fans_gpu_ctx *, const AsmArgs<double> &, dim3);
template void launch_modal<double, 1, 1, ASM_CGLIN>(fans_gpu_ctx *, const AsmArgs<double> &, dim3);
template void launch_modal<double, 3, 8, ASM_CGLIN>(fans_gpu_ctx *, const AsmArgs<double> &, dim3);
template void launch_modal<double, 3, 1, ASM_CGLIN>(fans_gpu_ctx *, const AsmArgs<double> &, dim3);
template void launch_modal<double, 1, 8, ASM_RESID>(fans_gpu_ctx *, const AsmArgs<double> &, dim3);
template void launch_modal<double, 1, 1, ASM_RESID>(fans_gpu_ctx *, const AsmArgs<double> &, dim3);
template void launch_modal<double, 3, 8, ASM_RESID>(fans_gpu_ctx *, const AsmArgs<double> &, dim3);
template void launch_modal<double, 3, 1, ASM_RESID>(fans_gpu_ctx *, const AsmArgs<double> &, dim3);
}
