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

// k_assemble: nonlinear materials (residual only; thermal models are all linear),
// linear ones in the mixed form
template <typename T, int MODE, int H, int NGP>
void launch_general_hn(fans_gpu_ctx *c, const AsmArgs<T> &a, dim3 g)
{
#define ASM(VAR) hipLaunchKernelGGL((k_assemble<T, H, NGP, MODE, VAR>), g, dim3(kThreads), 0, c->stream, a)
    if constexpr (MODE == ASM_RESID && H == 3) {
        if (c->nstr == 9) {
            ASM(ASM_LARGE);
            return;
        }
        if (c->has_visco) {
            ASM(ASM_GENERAL_VISCO);
            return;
        }
        if (c->has_pnl) {
            ASM(ASM_GENERAL_PNL);
            return;
        }
    }
    if constexpr (MODE == ASM_CGLIN && sizeof(T) == 4)
        if (a.cx != a.grp) {  // a batch's deeper workgroups
#define ASMG(VAR) hipLaunchKernelGGL((k_assemble<T, H, NGP, MODE, VAR, true>), g, dim3(kThreads), 0, c->stream, a)
            if (c->all_iso && c->cubic)
                ASMG(ASM_ISO_CUBIC);
            else if (c->all_iso)
                ASMG(ASM_ISO);
            else
                ASMG(ASM_GENERAL);
#undef ASMG
            return;
        }
    if (c->all_iso && c->cubic)
        ASM(ASM_ISO_CUBIC);
    else if (c->all_iso)
        ASM(ASM_ISO);
    else
        ASM(ASM_GENERAL);
#undef ASM
}
template <typename T, int MODE>
void launch_general(fans_gpu_ctx *c, const AsmArgs<T> &a, dim3 g)
{
    if (c->h == 1)
        c->ngp == 8 ? launch_general_hn<T, MODE, 1, 8>(c, a, g) : launch_general_hn<T, MODE, 1, 1>(c, a, g);
    else
        c->ngp == 8 ? launch_general_hn<T, MODE, 3, 8>(c, a, g) : launch_general_hn<T, MODE, 3, 1>(c, a, g);
}

}  // namespace fans
