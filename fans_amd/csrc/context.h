// A context of the C ABI (one load case, or a batch of RVEs of one shape) and
// the kernel launches it is built on.  The launches are templates defined in
// fft_launch.h and assemble_launch.h and instantiated per precision in the
// fft_f*.hip and assemble_f*.hip units, so that the kernels compile in parallel.
#pragma once
#include "fans_gpu.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <functional>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "assemble_kernels.h"
#include "cg_scalars.h"
#include "common.h"
#include "element_kernels.h"
#include "fft_kernels.h"

namespace fans {

struct HostScalars;  // vec_kernels.h
struct MixedCtl;

constexpr int kThreads = 256;

// kernel families for the timing report
enum {
    KF_FFT_Z_FWD = 0,
    KF_FFT_Y_FWD,
    KF_FFT_X_GREEN,
    KF_FFT_Y_INV,
    KF_FFT_Z_INV,
    KF_ASSEMBLE_LIN,
    KF_ASSEMBLE_RES,
    KF_CG_UPDATE,
    KF_REDUCE,
    KF_VECTOR,
    KF_ELEMENT,
    KF_CG_FFT_Z_FWD,  // CG update fused into the forward z pass
    KF_COUNT
};

// ---- host twiddles (long double, then rounded) ------------------------------
template <typename T>
std::vector<cplx<T>> twiddles(int n)
{
    std::vector<cplx<T>> w(n);
    const long double    pi = 3.14159265358979323846264338327950288L;
    for (int k = 0; k < n; ++k) {
        long double th = -2.0L * pi * (long double) k / (long double) n;
        w[k]           = cplx<T>{(T) cosl(th), (T) sinl(th)};
    }
    return w;
}

// n as a product of the fewest stage radices (two at least, unless n is 2, 3 or
// 5), the largest as small as it can be, in descending order; false if n is no
// product of 2, 3 and 5
inline bool make_len(int n, int tws, FftLen &L, int max_radix = 16)
{
    static const int kRadices[] = {16, 15, 12, 10, 9, 8, 6, 5, 4, 3, 2};
    L                           = FftLen{};
    L.n                         = n;
    L.tws                       = tws;
    if (n == 1)
        return true;
    int  cur[kMaxStages], best_max = 0;
    bool found = false;
    for (int nst = n == 2 || n == 3 || n == 5 ? 1 : 2; nst <= kMaxStages && !found; ++nst) {
        // radices non-increasing, depth-first
        std::function<void(int, int, int)> go = [&](int depth, int rest, int from) {
            if (depth == nst) {
                if (rest == 1 && (!found || cur[0] < best_max)) {
                    found    = true;
                    best_max = cur[0];
                    L.nst    = nst;
                    std::copy(cur, cur + nst, L.rad);
                }
                return;
            }
            for (int k = from; k < 11; ++k)
                if (kRadices[k] <= max_radix && rest % kRadices[k] == 0) {
                    cur[depth] = kRadices[k];
                    go(depth + 1, rest / kRadices[k], k);
                }
        };
        go(0, n, 0);
    }
    return found;
}

// the FP32 stages (lds_stockham)
inline bool make_len_stockham(int n, int tws, FftLen &L)
{
    L.n   = n;
    L.tws = tws;
    L.nst = 0;
    int m = n;
    for (int r : {5, 3, 8, 4, 2})
        while (m % r == 0) {
            if (L.nst >= kMaxStages)
                return false;
            L.rad[L.nst++] = r;
            m /= r;
        }
    return m == 1;
}

// lines per block of the compile-time z kernels (0: generic kernels)
inline int zct_lines(int h, int M)
{
    switch (M) {
    case 128: return h == 1 ? zct_lpb<1, 128>() : zct_lpb<3, 128>();
    case 64: return h == 1 ? zct_lpb<1, 64>() : zct_lpb<3, 64>();
    case 48: return h == 1 ? zct_lpb<1, 48>() : zct_lpb<3, 48>();
    case 40: return h == 1 ? zct_lpb<1, 40>() : zct_lpb<3, 40>();
    case 32: return h == 1 ? zct_lpb<1, 32>() : zct_lpb<3, 32>();
    case 24: return h == 1 ? zct_lpb<1, 24>() : zct_lpb<3, 24>();
    case 16: return h == 1 ? zct_lpb<1, 16>() : zct_lpb<3, 16>();
    default: return 0;
    }
}

// threads of the z kernels
inline int zct_nt(int h, int M) { return M / (M >= 32 ? 8 : 4) * zct_lines(h, M) * h; }

template <typename T>
struct Fft3D {
    int           nx = 0, ny = 0, nz = 0, h = 0, M = 0, Mc = 0;
    FftLen        Lz{}, Ly{}, Lx{};
    cplx<T>      *twz = nullptr, *twy = nullptr, *twx = nullptr;
    int           lpb = 1, bc = 8, bk = 2, bcx = 8;
    size_t        smz = 0, smy = 0, smx = 0, smx_plain = 0;
    // LDS budget of one workgroup of the generic (LDS-tiled) passes; it sets
    // their lines / columns per workgroup (FANS_OPT_FFT_LDS_KIB)
    int           lds_kib = 40;
    bool          lds_set = false;

    // largest power of two <= min(limit, cap), at least 1
    static int pow2_cols(int limit, int cap)
    {
        int v = 1;
        while (v * 2 <= limit && v * 2 <= cap)
            v *= 2;
        return v;
    }
    int64_t       nblk_z = 0;
    bool          zct    = false;  // compile-time z kernels in use
    bool          ready  = false;

    hipError_t init(int nx_, int ny_, int nz_, int h_)
    {
        hipError_t e = plan(nx_, ny_, nz_, h_);
        if (e != hipSuccess)
            return e;
        ready   = false;
        auto up = [](cplx<T> *&dst, const std::vector<cplx<T>> &v) {
            hipError_t e = hipMalloc(&dst, sizeof(cplx<T>) * v.size());
            if (e != hipSuccess)
                return e;
            return hipMemcpy(dst, v.data(), sizeof(cplx<T>) * v.size(), hipMemcpyHostToDevice);
        };
        if ((e = up(twz, twiddles<T>(nz))) != hipSuccess)
            return e;
        if ((e = up(twy, twiddles<T>(ny))) != hipSuccess)
            return e;
        if ((e = up(twx, twiddles<T>(nx))) != hipSuccess)
            return e;
        ready = true;
        return hipSuccess;
    }
    // launch shapes and length factorisations only (host arithmetic, no device
    // memory): the twiddle tables twz / twy / twx are the caller's to provide
    hipError_t plan(int nx_, int ny_, int nz_, int h_)
    {
        nx = nx_, ny = ny_, nz = nz_, h = h_;
        M  = nz / 2;
        Mc = M + 1;
        const size_t cb = sizeof(cplx<T>);
        const int    Kc = Mc * h;
        if ((int64_t) M * h > FFT_MAX_ELEMS || ny > FFT_MAX_ELEMS || (int64_t) nx * h > FFT_MAX_ELEMS)
            return hipErrorInvalidValue;
        const int64_t lim = (int64_t) lds_kib * 1024 / (int64_t) cb;
        if constexpr (sizeof(T) == 4) {
            // one padded LDS tile per workgroup, n * columns <= FFT_MAX_ELEMS so the
            // in-place stages keep every butterfly input in registers
            if (!make_len_stockham(M, 2, Lz) || !make_len_stockham(ny, 1, Ly) || !make_len_stockham(nx, 1, Lx))
                return hipErrorInvalidValue;
            const int le = (int) std::min<int64_t>(FFT_MAX_ELEMS, lim);
            lpb          = std::max(1, std::min(16, le / (M * h)));
            smz          = cb * M * (lpb * h + 1);
            bc           = pow2_cols(le / ny, std::min(Kc, 16));
            smy          = cb * ny * (bc + 1);
            bk           = std::max(1, std::min(Mc, le / (nx * h)));
            smx          = cb * nx * (bk * h + 1);
            bcx          = pow2_cols(le / nx, 16);
            smx_plain    = cb * nx * (bcx + 1);
        } else {
            if (!make_len(M, 2, Lz) || !make_len(ny, 1, Ly) ||
                !make_len(nx, 1, Lx, h == 3 ? kXGreenMaxRadix<3>() : kXGreenMaxRadix<1>()))
                return hipErrorInvalidValue;
            // one LDS tile per workgroup, by default 40 KiB (four workgroups per CU).
            // The strided passes go to 64 KiB where that gives rows of 16 columns (192
            // points, 200 x 192 x 160 conduction: 25.5 us against 27.7 with 8
            // columns); the z passes stay within 32 (125 x 120 x 150 52.5 and 50.0 us
            // against 56.8 and 52.0)
            const int64_t wide = lds_set ? lim : 64 * 1024 / (int64_t) cb;
            const int64_t zlim = lds_set ? lim : (int64_t) 32 * 1024 / (int64_t) cb;
            lpb                = (int) std::max<int64_t>(1, std::min<int64_t>(16, zlim / (M * h)));
            smz                = cb * M * (lpb * h + 1) + sizeof(unsigned short) * M;
            bc                 = pow2_cols((int) (wide / ny), std::min(Kc, 16));
            smy                = cb * ny * bc;
            // frequencies per x+Green workgroup: the budget, less where that leaves
            // fewer than 256 workgroups
            const int64_t nbk = std::max<int64_t>({1, (Mc * (int64_t) nx * h + lim - 1) / lim, lds_set ? 1 : 256 / ny});
            bk                = (int) std::max<int64_t>(1, std::min<int64_t>(lim / (nx * h), (Mc + nbk - 1) / nbk));
            smx               = cb * nx * bk * h;
            bcx               = pow2_cols((int) (wide / nx), 16);
            smx_plain         = cb * nx * bcx;
        }
        nblk_z       = ((int64_t) nx * ny + lpb - 1) / lpb;
        const int lct = zct_lines(h, M);
        zct           = lct > 0 && ((int64_t) nx * ny) % lct == 0;
        if (zct)
            nblk_z = (int64_t) nx * ny / lct;
        ready = true;
        return hipSuccess;
    }
    void release()
    {
        (void) hipFree(twz);
        (void) hipFree(twy);
        (void) hipFree(twx);
        twz = twy = twx = nullptr;
        ready           = false;
    }
};

// RVE slots of one batched context at most
constexpr int kMaxSlots = 4096;

// per-RVE device buffers of a context and the stride kind of each (Slots);
// g0 holds 9 entries per slot, the device scalars SC_COUNT / IS_COUNT
#define FANS_SLOT_BUFFERS(X)                                                                                   \
    X(double, u, field) X(double, u_prev, field) X(double, r, field) X(double, s, field) X(double, dA, field)   \
    X(double, dB, field) X(double, rnew, field) X(cplx<double>, spec64, spec) X(double, G64, green)            \
    X(float, G32, green) X(uint8_t, ms, ms) X(Phase<double>, dph64, ph) X(Phase<float>, dph32, ph)            \
    X(double, g0d, g0) X(float, g0f, g0) X(double, partial, part) X(double, partial_e, part) X(double, sc, sc) \
    X(int, is, is) X(double, hist, hist) X(float, r32, field) X(float, s32, field) X(float, dA32, field)       \
    X(float, dB32, field) X(float, rnew32, field) X(float, x32, field) X(cplx<float>, spec32, spec)
enum SlotKind { SK_field, SK_spec, SK_green, SK_ms, SK_ph, SK_g0, SK_part, SK_sc, SK_is, SK_hist };

// slot 0's address of every per-RVE buffer of a batched context
struct SlotBase {
#define X(T, name, kind) T *name = nullptr;
    FANS_SLOT_BUFFERS(X)
#undef X
    double *ring64[kDirRing]{};
    float  *ring32[kDirRing]{};
};

// host state of one RVE of a batched context while another slot is selected
#define FANS_SLOT_HOST(X)                                                                                      \
    X(have_ms) X(have_mat) X(ms16) X(ms_max) X(nphases) X(phase_kind) X(all_linear) X(has_j2) X(all_iso)        \
    X(has_pnl) X(has_visco) X(user_ref) X(voxel_moduli) X(ph64) X(ph32) X(gxq) X(gyq) X(iter) X(inner_iters)    \
    X(outer_iters) X(err_hist) X(solve_ms) X(kref) X(keref) X(g0) X(gvec) X(gvec_prev)
struct SlotHost {
    bool                       have_ms = false, have_mat = false, ms16 = false;
    int                        ms_max = -1, nphases = 0;
    std::vector<int>           phase_kind;
    bool                       all_linear = true, has_j2 = false, all_iso = false, has_pnl = false;
    bool                       has_visco = false, user_ref = false, voxel_moduli = false;
    std::vector<Phase<double>> ph64;
    std::vector<Phase<float>>  ph32;
    int                        gxq = 0, gyq = 0, iter = 0, inner_iters = 0, outer_iters = 0;
    std::vector<double>        err_hist;
    double                     solve_ms = 0;
    double                     kref[81]{}, keref[576]{}, g0[9]{}, gvec[9]{}, gvec_prev[9]{};
};

// what the launches of a captured CG iteration depend on beside the context's
// settings (drop_graphs): the first direction buffer (with it the precision), the
// slots per launch (gz) and whether the z passes fold the scalars
using GraphKey = std::tuple<const void *, int, bool>;

}  // namespace fans

using namespace fans;  // the context is the C ABI's type, at global scope

struct fans_gpu_ctx {
    fans_gpu_desc d{};
    std::string   err;
    int           nx = 0, ny = 0, nz = 0, h = 0, nstr = 0, ngp = 0;
    int64_t       N = 0, Nh = 0, Nf = 0;
    hipStream_t   stream = nullptr;
    int           tol_type = 0;  // current error type (tangent switches it, solver.h:749)
    double        tol      = 0;

    // materials
    bool                        have_ms = false, have_mat = false;
    int                         ms_max  = -1;  // largest phase id of the microstructure
    int                         nphases = 0;
    std::vector<int>            phase_kind;
    bool                        all_linear = true, has_j2 = false, all_iso = false;
    bool                        has_pnl = false;  // a PseudoPlasticNonLinearHardening phase
    bool                        has_visco = false;  // a J2ViscoPlastic phase
    bool                        cubic = false;  // hx == hy == hz
    double                      kref[81]{};
    double                      keref[576]{};
    std::vector<Phase<double>>  ph64;
    std::vector<Phase<float>>   ph32;

    // device buffers
    uint8_t       *ms = nullptr;  // phase ids: bytes, or 16-bit ids when ms16
    bool           ms16 = false;
    int64_t        ms_bytes = 0;  // allocated bytes of ms
    int            nph_cap  = 0;  // allocated entries of dph64 / dph32
    Phase<double> *dph64 = nullptr;
    Phase<float>  *dph32 = nullptr;
    double        *u = nullptr, *u_prev = nullptr, *r = nullptr, *s = nullptr, *dA = nullptr, *dB = nullptr,
           *rnew = nullptr;
    cplx<double> *spec64 = nullptr;
    double       *G64 = nullptr, *keref_d = nullptr;
    float        *G32 = nullptr;
    int           gxq = 0, gyq = 0;  // stored kx / ky counts of the Green operator
    // per-voxel isotropic moduli (K, G; thermal: k in vk), replacing the phase table
    bool          voxel_moduli = false, user_ref = false;
    double       *vk64 = nullptr, *vg64 = nullptr;
    float        *vk32 = nullptr, *vg32 = nullptr;
    double       *ub_d = nullptr, *sens_d = nullptr;
    double       *js = nullptr;
    double       *g0d = nullptr;
    float        *g0f = nullptr;
    double       *partial = nullptr;
    int64_t       partial_len = 0;
    double       *partial_e   = nullptr;  // [nblk_z] of the linear CG's inverse z pass
    int64_t       partial_e_len = 0;
    // nonlinear CG: scalars in pinned host memory, mixed-control state
    HostScalars  *nl_host     = nullptr;
    MixedCtl     *nl_ctl      = nullptr;
    double       *sc = nullptr;
    int          *is = nullptr;
    double       *hist = nullptr;
    // FP32 inner solve (mixed form)
    float        *r32 = nullptr, *s32 = nullptr, *dA32 = nullptr, *dB32 = nullptr, *rnew32 = nullptr, *x32 = nullptr;
    cplx<float>  *spec32 = nullptr;
    // linear CG direction rings: slots 0 and 1 are dA / dB (dA32 / dB32), the
    // others are allocated by the first linear CG solve
    double *ring64[kDirRing]{};
    float  *ring32[kDirRing]{};
    Fft3D<double> fft64;
    Fft3D<float>  fft32;

    // RVE slots (fans_gpu_create_batch): nb same-shape RVEs whose per-RVE
    // device buffers lie nb times at the strides of `strides`.  The buffer
    // fields above address the selected slot `cur`, `base` keeps slot 0's
    // addresses and `parked` the host state of the slots not selected.  A
    // batched solve points the fields at slot 0 and launches gz slots per
    // kernel (grid z) through the device map `slot_map`.
    int                   nb = 1, cur = 0, gz = 1;
    bool                  use_map  = false;
    int                  *slot_map = nullptr;
    int                   map_cap  = 0;
    std::vector<int>      map_h, map_slots;  // uploaded map and the slots it holds
    Slots                 strides{};
    SlotBase              base{};
    std::vector<SlotHost> parked;
    std::array<int, 7>    batch_sig{};

    // launch geometry
    int     cx = 1, nty = 0, ntz = 0, nblk_asm = 0, nblk_vec = 0, nblk_el = 0;
    bool    cx_set = false;  // the caller chose cx (FANS_OPT_ASM_PLANES)
    int64_t nslot = 0;      // J2 state slots per component and Gauss point
    int     js_comps = 0;   // components of the allocated J2 state
    int     nblk_slot = 0;  // workgroups of the state commit (one thread per slot)
    double  g0[9]{};
    Geom    geom{};

    // mixed BC (mixedBCs.h)
    bool                mixed_active = false;
    std::vector<int>    idxE, idxF;
    std::vector<double> FE, PF, M;
    int                 nsteps = 0, step = 0;
    double              gvec[9]{}, gvec_prev[9]{};
    double              alpha_warm = 0.1;

    // results
    int                 iter = 0, inner_iters = 0, outer_iters = 0;
    std::vector<double> err_hist;
    double              solve_ms = 0;

    // timing
    bool                                                timing = false;
    int                                                 fft_chunks = 1;
    // the single-operator entry points run the mixed form's FP32 kernels
    bool                                                op_fp32 = false;
    // single-RVE mixed form with restarted inner solves (as batched contexts)
    bool                                                mixed_restart = false;
    // captured CG iterations (hipGraph)
    bool                                                use_graphs = true;
    std::vector<std::pair<GraphKey, hipGraphExec_t>>    graphs;
    std::array<int, 7>                                  graph_sig{};
    std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> ev_used;
    std::vector<hipEvent_t>                             ev_pool;
    double                                              fam_ms[KF_COUNT]{};
    int                                                 fam_n[KF_COUNT]{};
};

namespace fans {

// slots of a launch: the selected slot alone (its buffers are the fields), or
// during a batched solve the slots of the device map; `gated`: finished slots
// return at entry
inline Slots launch_slots(const fans_gpu_ctx *c, bool gated)
{
    Slots s = c->strides;
    s.map   = c->use_map ? c->slot_map : nullptr;
    s.is    = gated ? c->is : nullptr;
    return s;
}

// partials of one kernel up to which the z passes fold the CG scalars themselves:
// with 2176 (128^3 elastic FP64) the solve went from 9.26 to 9.12 ms, with 2304
// (144^3 mixed) 10.61 to 10.43; with 2400 (200 x 192 x 160 conduction) from 4.77 to
// 4.80 and, mixed, 4.01 to 4.17: every workgroup reads all of them
constexpr int kFoldMax = 2304;
// and, in a batch, the partials that all workgroups of the two z passes read in one
// iteration with every slot running: the reduction launches are shared by the slots
// there.  Folded, 32 RVEs of 64^3 conduction (3 million) solve in 7.5 ms against 7.8,
// 11 of 96^3 (4 million) in 7.1 against 7.2, but 40 of 48^3 elasticity (12 million)
// in 13.0 against 12.7 and 11 of 96^3 (24 million and more) in 18.8 against 17.8.
// Decided per phase instead, from the slots still running, a mixed solve takes the
// same time (40 of 48^3 12.8 ms either way, 32 of 64^3 16.9).
constexpr int64_t kFoldBatch = 8'000'000;

// ---- launches ----------------------------------------------------------------
// z passes, strided (y or x) pass, x+Green pass; x+Green returns its block count
// (one partial of the spectral <r, s> per block when `partial` is set)
template <typename T, int H, int PRO>
void launch_z_r2c(fans_gpu_ctx *c, Fft3D<T> &P, T *rin, cplx<T> *spec, const ProArgs<T> &pa, const int *done);
template <typename T, int H, int EPI>
void launch_z_c2r(fans_gpu_ctx *c, Fft3D<T> &P, const cplx<T> *spec, const EpiArgs<T> &ep, const int *done);
template <typename T, bool INV>
void launch_strided(fans_gpu_ctx *c, const FftLen &L, const cplx<T> *tw, int bc, size_t smem, cplx<T> *spec,
                    int64_t sn, int c0, int c1, int64_t ostride, int nouter, const int *done);
template <typename T, int H>
int launch_x_green(fans_gpu_ctx *c, Fft3D<T> &P, cplx<T> *spec, const T *G, int kz_lo, int kz_hi, double *partial,
                   const int *done);
// blocks of one x+Green launch over all kz (the size of its partial array)
template <typename T>
int64_t x_green_blocks(const Fft3D<T> &P, int h, int ny);
// linear and nonlinear assembly
template <typename T, int H, int NGP, int MODE>
void launch_modal(fans_gpu_ctx *c, const AsmArgs<T> &a, dim3 g);
template <typename T, int MODE>
void launch_general(fans_gpu_ctx *c, const AsmArgs<T> &a, dim3 g);

}  // namespace fans
