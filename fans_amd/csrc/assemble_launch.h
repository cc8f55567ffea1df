// Definitions of the assembly launches declared in context.h.
#pragma once
#include "context.h"

namespace fans {

// k_assemble_modal for the context's materials.  Byte ids find their phase in
// the workgroup's staged table; tensors are staged while they leave room for two
// workgroups per CU (the registers' limit): 64 KiB, about 120 phases in FP64.
template <typename T, int H, int NGP, int MODE>
void launch_modal(fans_gpu_ctx *c, const AsmArgs<T> &a, dim3 g)
{
#define MODAL(VAR, MAT, LDS) \
    hipLaunchKernelGGL((k_assemble_modal<T, H, NGP, MODE, VAR, MAT>), g, dim3(kThreads), LDS, c->stream, a)
    if (!c->all_iso) {
        const size_t lds = sizeof(T) * kTensorLen<T, H>() * std::min(c->nphases, kStagedPhases);
        if (!c->ms16 && lds + modal_static_lds<T, H>() <= 64 * 1024)
            MODAL(ASM_ANISO, MAT_STAGED, lds);
        else
            MODAL(ASM_ANISO, MAT_TABLE, 0);
    } else if (c->cubic) {
        if (c->voxel_moduli)
            MODAL(ASM_ISO_CUBIC, MAT_VOXEL, 0);
        else if (c->ms16)
            MODAL(ASM_ISO_CUBIC, MAT_TABLE, 0);
        else
            MODAL(ASM_ISO_CUBIC, MAT_STAGED, 0);
    } else {
        if (c->voxel_moduli)
            MODAL(ASM_ISO, MAT_VOXEL, 0);
        else if (c->ms16)
            MODAL(ASM_ISO, MAT_TABLE, 0);
        else
            MODAL(ASM_ISO, MAT_STAGED, 0);
    }
#undef MODAL
}

// the residual of nonlinear materials (thermal models are all linear)
template <typename T>
void launch_general(fans_gpu_ctx *c, const AsmArgs<T> &a, dim3 g)
{
#define ASM(VAR)                                                                                \
    do {                                                                                        \
        if (c->ngp == 8)                                                                        \
            hipLaunchKernelGGL((k_assemble<T, 3, 8, VAR>), g, dim3(kThreads), 0, c->stream, a); \
        else                                                                                    \
            hipLaunchKernelGGL((k_assemble<T, 3, 1, VAR>), g, dim3(kThreads), 0, c->stream, a); \
    } while (0)
    if (c->nstr == 9)
        ASM(ASM_LARGE);
    else if (c->has_visco)
        ASM(ASM_GENERAL_VISCO);
    else if (c->has_pnl)
        ASM(ASM_GENERAL_PNL);
    else
        ASM(ASM_GENERAL);
#undef ASM
}

}  // namespace fans
