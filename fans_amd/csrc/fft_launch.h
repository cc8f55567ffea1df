// Definitions of the FFT launches declared in context.h.
#pragma once
#include "context.h"
#include "fft_reg_kernels.h"

namespace fans {

// ---------------------------------------------------------------------------
// register four-step kernels: power-of-two lengths 16..256 and, along y, 48, 80 and
// 96 (256^3 FP64 y 157 us against 189 with the staged kernel, 48^3 5.2 against 6.8)
// ---------------------------------------------------------------------------
inline bool reg_len(int n) { return n == 16 || n == 32 || n == 64 || n == 128 || n == 256; }
inline bool reg_len_y(int n) { return reg_len(n) || n == 96 || n == 80 || n == 48; }
// the x+Green pass: the powers of two; FP32 also 48, 80 and 96, whose FP64 forms
// would spill (one wave)
template <typename T>
bool x_green_reg(int n)
{
    return sizeof(T) == 8 ? reg_len(n) : reg_len_y(n);
}

// columns per block: a power of two (>= 4) within ~72 KiB of LDS (two
// workgroups per CU) and at most MAXT threads; at 256^3 FP64 this gives 16
// columns (256-byte row segments) for the y pass and 4 frequencies for the x
// pass.  The FP32 y pass takes 512 threads (32 columns, 256-byte segments:
// 0.095 -> 0.085 ms at 256^3); the FP32 x pass stays at 256 (wider was slower).
constexpr int kRegLdsKiB = 72;
template <typename T, int N1, int N2, int MAXT = 256>
constexpr int reg_cols()
{
    constexpr int n   = N1 * N2;
    constexpr int lim = (int) (kRegLdsKiB * 1024 / (n * sizeof(cplx<T>)));
    int           c   = 4;
    while (c * 2 <= lim && c * 2 * N2 <= MAXT)
        c *= 2;
    return c;
}
template <typename T>
constexpr int strided_max_threads()
{
    return sizeof(T) == 4 ? 512 : 256;
}

template <typename T, bool INV, int N1, int N2>
void launch_strided_reg(fans_gpu_ctx *c, cplx<T> *spec, const cplx<T> *tw, int64_t sn, int c0, int c1,
                        int64_t ostride, int nouter, const int *done)
{
    constexpr int C   = reg_cols<T, N1, N2, strided_max_threads<T>()>();
    const int     nbx = (c1 - c0 + C - 1) / C;
    hipLaunchKernelGGL((k_fft_strided_reg<T, N1, N2, C, INV>), dim3(nbx * nouter, 1, c->gz), dim3(C * N2), 0,
                       c->stream, spec, tw, sn, c0, c1, ostride, nbx, launch_slots(c, done != nullptr));
}

template <typename T, bool INV>
void launch_strided(fans_gpu_ctx *c, const FftLen &L, const cplx<T> *tw, int bc, size_t smem, cplx<T> *spec,
                    int64_t sn, int c0, int c1, int64_t ostride, int nouter, const int *done)
{
    switch (reg_len_y(L.n) || L.n == 1 ? L.n : 0) {
    case 96: launch_strided_reg<T, INV, 24, 4>(c, spec, tw, sn, c0, c1, ostride, nouter, done); break;
    case 80: launch_strided_reg<T, INV, 20, 4>(c, spec, tw, sn, c0, c1, ostride, nouter, done); break;
    case 48: launch_strided_reg<T, INV, 12, 4>(c, spec, tw, sn, c0, c1, ostride, nouter, done); break;
    case 256: launch_strided_reg<T, INV, 16, 16>(c, spec, tw, sn, c0, c1, ostride, nouter, done); break;
    case 128: launch_strided_reg<T, INV, 16, 8>(c, spec, tw, sn, c0, c1, ostride, nouter, done); break;
    case 64: launch_strided_reg<T, INV, 8, 8>(c, spec, tw, sn, c0, c1, ostride, nouter, done); break;
    case 32: launch_strided_reg<T, INV, 8, 4>(c, spec, tw, sn, c0, c1, ostride, nouter, done); break;
    case 16: launch_strided_reg<T, INV, 4, 4>(c, spec, tw, sn, c0, c1, ostride, nouter, done); break;
    case 1: break;
    default: {
        const int nbx = (c1 - c0 + bc - 1) / bc;
        if constexpr (sizeof(T) == 4)
            hipLaunchKernelGGL((k_fft_strided_stockham<T, INV>), dim3(nbx, nouter, c->gz), dim3(kThreads), smem, c->stream,
                               spec, L, tw, sn, c0, c1, ostride, bc, launch_slots(c, done != nullptr));
        else
            hipLaunchKernelGGL((k_fft_strided<T, INV>), dim3(nbx * nouter, 1, c->gz), dim3(kThreads), smem, c->stream,
                               spec, L, tw, sn, c0, c1, ostride, bc, nbx, launch_slots(c, done != nullptr));
    }
    }
}

// Split transposes (fourstep_split) for the x+Green pass: measured at 256^3
// FP64 they took the pass from 0.29 to 0.50 ms (twice the barriers outweigh the
// doubled residency), so the complex tile stays
constexpr bool kXGreenSplit = false;

template <typename T, int H, int N1, int N2>
int launch_x_green_reg(fans_gpu_ctx *c, cplx<T> *spec, const cplx<T> *tw, const GreenView<T> &gv, int kz_lo,
                       int kz_hi, double *partial, const int *done)
{
    constexpr int C   = reg_cols<T, N1, N2>();
    constexpr int KB  = H == 3 ? (C == 16 ? 5 : C / 4) : C;
    const int     nbk = (kz_hi - kz_lo + KB - 1) / KB;
    // the complex transpose tile of the 256-point FP64 pass (70 KB) allows two
    // workgroups per CU; the split tile (35 KB) four
    constexpr bool SPLIT = kXGreenSplit && (int64_t) N1 * N2 * (C + 1) * sizeof(cplx<T>) > 48 * 1024;
    hipLaunchKernelGGL((k_fft_x_green_reg<T, H, N1, N2, KB, C, SPLIT>), dim3(nbk * c->ny, 1, c->gz), dim3(C * N2),
                       0, c->stream, spec, tw, gv, kz_lo, kz_hi, nbk, partial, launch_slots(c, done != nullptr));
    return nbk * c->ny;
}

template <typename T, int H>
int launch_x_green(fans_gpu_ctx *c, Fft3D<T> &P, cplx<T> *spec, const T *G, int kz_lo, int kz_hi, double *partial,
                   const int *done)
{
    const GreenView<T> gv{G, c->nx, c->ny, c->gxq, c->gyq, P.Mc};
    if constexpr (sizeof(T) == 4) {
        switch (P.Lx.n) {
        case 96: return launch_x_green_reg<T, H, 24, 4>(c, spec, P.twx, gv, kz_lo, kz_hi, partial, done);
        case 80: return launch_x_green_reg<T, H, 20, 4>(c, spec, P.twx, gv, kz_lo, kz_hi, partial, done);
        case 48: return launch_x_green_reg<T, H, 12, 4>(c, spec, P.twx, gv, kz_lo, kz_hi, partial, done);
        default: break;
        }
    }
    switch (P.Lx.n) {
    case 256: return launch_x_green_reg<T, H, 16, 16>(c, spec, P.twx, gv, kz_lo, kz_hi, partial, done);
    case 128: return launch_x_green_reg<T, H, 16, 8>(c, spec, P.twx, gv, kz_lo, kz_hi, partial, done);
    case 64: return launch_x_green_reg<T, H, 8, 8>(c, spec, P.twx, gv, kz_lo, kz_hi, partial, done);
    case 32: return launch_x_green_reg<T, H, 8, 4>(c, spec, P.twx, gv, kz_lo, kz_hi, partial, done);
    case 16: return launch_x_green_reg<T, H, 4, 4>(c, spec, P.twx, gv, kz_lo, kz_hi, partial, done);
    default: {
        const int nbk = (kz_hi - kz_lo + P.bk - 1) / P.bk;
        if constexpr (sizeof(T) == 4)
            hipLaunchKernelGGL((k_fft_x_green_stockham<T, H>), dim3(nbk, c->ny, c->gz), dim3(kThreads), P.smx, c->stream,
                               spec, P.Lx, P.twx, gv, kz_lo, kz_hi, P.bk, partial, launch_slots(c, done != nullptr));
        else
            hipLaunchKernelGGL((k_fft_x_green<T, H>), dim3(nbk * c->ny, 1, c->gz), dim3(kThreads), P.smx, c->stream, spec,
                               P.Lx, P.twx, gv, kz_lo, kz_hi, P.bk, nbk, partial, launch_slots(c, done != nullptr));
        return nbk * c->ny;
    }
    }
}

template <typename T>
int64_t x_green_blocks(const Fft3D<T> &P, int h, int ny)
{
    int kb = 0;
    switch (x_green_reg<T>(P.Lx.n) ? P.Lx.n : 0) {
    case 96: kb = reg_cols<T, 24, 4>(); break;
    case 80: kb = reg_cols<T, 20, 4>(); break;
    case 48: kb = reg_cols<T, 12, 4>(); break;
    case 256: kb = reg_cols<T, 16, 16>(); break;
    case 128: kb = reg_cols<T, 16, 8>(); break;
    case 64: kb = reg_cols<T, 8, 8>(); break;
    case 32: kb = reg_cols<T, 8, 4>(); break;
    case 16: kb = reg_cols<T, 4, 4>(); break;
    default: return (int64_t) ((P.Mc + P.bk - 1) / P.bk) * ny;
    }
    if (h == 3)
        kb = kb == 16 ? 5 : kb / 4;
    return (int64_t) ((P.Mc + kb - 1) / kb) * ny;
}

// z passes: compile-time kernels where M = nz/2 is in {16, 24, 32, 40, 48, 64,
// 128} and the line count divides evenly, else the generic ones
template <typename T, int H, int PRO>
void launch_z_r2c(fans_gpu_ctx *c, Fft3D<T> &P, T *rin, cplx<T> *spec, const ProArgs<T> &pa, const int *done)
{
    const int64_t nlines = (int64_t) c->nx * c->ny;
    const Slots   sl     = launch_slots(c, done != nullptr);
#define ZF(MM)                                                                                                  \
    hipLaunchKernelGGL((k_fft_z_r2c_ct<T, H, MM, PRO>), dim3((unsigned) (nlines / zct_lpb<H, MM>()), 1, c->gz),  \
                       dim3(zct_threads<H, MM>()), 0, c->stream, rin, spec, P.twz, pa, sl)
    switch (P.zct ? P.M : 0) {
    case 128: ZF(128); break;
    case 64: ZF(64); break;
    case 48: ZF(48); break;
    case 40: ZF(40); break;
    case 32: ZF(32); break;
    case 24: ZF(24); break;
    case 16: ZF(16); break;
    default:
        hipLaunchKernelGGL((k_fft_z_r2c<T, H, PRO>), dim3(P.nblk_z, 1, c->gz), dim3(kThreads), P.smz, c->stream, rin,
                           spec, P.Lz, P.twz, c->nz, nlines, P.lpb, pa, sl);
    }
#undef ZF
}

template <typename T, int H, int EPI>
void launch_z_c2r(fans_gpu_ctx *c, Fft3D<T> &P, const cplx<T> *spec, const EpiArgs<T> &ep, const int *done)
{
    const int64_t nlines = (int64_t) c->nx * c->ny;
    const Slots   sl     = launch_slots(c, done != nullptr);
#define ZI(MM)                                                                                                  \
    hipLaunchKernelGGL((k_fft_z_c2r_ct<T, H, MM, EPI>), dim3((unsigned) (nlines / zct_lpb<H, MM>()), 1, c->gz),  \
                       dim3(zct_threads<H, MM>()), 0, c->stream, spec, P.twz, ep, sl)
    switch (P.zct ? P.M : 0) {
    case 128: ZI(128); break;
    case 64: ZI(64); break;
    case 48: ZI(48); break;
    case 40: ZI(40); break;
    case 32: ZI(32); break;
    case 24: ZI(24); break;
    case 16: ZI(16); break;
    default:
        hipLaunchKernelGGL((k_fft_z_c2r<T, H, EPI>), dim3(P.nblk_z, 1, c->gz), dim3(kThreads), P.smz, c->stream, spec,
                           P.Lz, P.twz, c->nz, nlines, P.lpb, ep, sl);
    }
#undef ZI
}

#define FANS_FFT_INSTANCES(T)                                                                                     \
    template void launch_strided<T, false>(fans_gpu_ctx *, const FftLen &, const cplx<T> *, int, size_t, cplx<T> *, \
                                           int64_t, int, int, int64_t, int, const int *);                         \
    template void launch_strided<T, true>(fans_gpu_ctx *, const FftLen &, const cplx<T> *, int, size_t, cplx<T> *, \
                                          int64_t, int, int, int64_t, int, const int *);                          \
    template int64_t x_green_blocks<T>(const Fft3D<T> &, int, int);                                               \
    FANS_FFT_INSTANCES_H(T, 1)                                                                                    \
    FANS_FFT_INSTANCES_H(T, 3)
#define FANS_FFT_INSTANCES_H(T, H)                                                                                \
    template int  launch_x_green<T, H>(fans_gpu_ctx *, Fft3D<T> &, cplx<T> *, const T *, int, int, double *,       \
                                      const int *);                                                               \
    template void launch_z_r2c<T, H, PRO_NONE>(fans_gpu_ctx *, Fft3D<T> &, T *, cplx<T> *, const ProArgs<T> &,     \
                                               const int *);                                                      \
    template void launch_z_r2c<T, H, PRO_CG>(fans_gpu_ctx *, Fft3D<T> &, T *, cplx<T> *, const ProArgs<T> &,       \
                                             const int *);                                                        \
    template void launch_z_r2c<T, H, PRO_CGF>(fans_gpu_ctx *, Fft3D<T> &, T *, cplx<T> *, const ProArgs<T> &,      \
                                              const int *);                                                       \
    FANS_FFT_INSTANCES_C2R(T, H, EPI_STORE)                                                                       \
    FANS_FFT_INSTANCES_C2R(T, H, EPI_CG)                                                                          \
    FANS_FFT_INSTANCES_C2R(T, H, EPI_FP)                                                                          \
    FANS_FFT_INSTANCES_C2R(T, H, EPI_CGD)                                                                         \
    FANS_FFT_INSTANCES_C2R(T, H, EPI_CGDF)
#define FANS_FFT_INSTANCES_C2R(T, H, EPI)                                                                         \
    template void launch_z_c2r<T, H, EPI>(fans_gpu_ctx *, Fft3D<T> &, const cplx<T> *, const EpiArgs<T> &, const int *);

}  // namespace fans
