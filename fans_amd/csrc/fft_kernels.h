// LDS-staged FFT kernels for 3-D r2c / c2r of nodal fields.
//
// Layouts (all row-major, components fastest):
//   real field      [x][y][z][h]            (T)
//   spectrum        [x][y][kz][h], kz<=nz/2 (cplx<T>)
// The r2c/c2r along z use the half-length complex transform (pairs of reals
// packed into one complex number) and a post/pre-processing twiddle.  The y
// and x passes are batched strided transforms: one workgroup owns a tile of
// contiguous (kz,h) columns for every y (or x) and transforms it in LDS.  The x
// pass carries the Green operator multiply between the forward and inverse
// transforms, so the spectrum is read and written once for that stage.
//
// An FP64 transform of n = r1 r2 ... rs runs as s in-place stages: forward by
// decimation in frequency (natural order in, digit-reversed order out), inverse
// as its exact reversal.  A butterfly reads and writes the same places, so a
// stage holds no data across a barrier, and one barrier separates two stages.  The
// strided passes take their first stage from global memory and give their last
// one to it; the x pass applies the Green operator to the registers of the last
// forward stage and starts the inverse from them.  FP32: see lds_stockham.
#pragma once
#include "cg_scalars.h"
#include "common.h"
#include <type_traits>
#include "fft_butterflies.h"

namespace fans {

constexpr int kMaxStages = 8;
struct FftLen {
    int n;                // transform length
    int nst;              // number of radix stages (0 for n = 1)
    int tws;              // stride into the twiddle table (table length n * tws)
    int rad[kMaxStages];  // radices in forward order
};

// Green operator storage, G[(kxq * gyq + kyq) * Mc + kz][H(H+1)/2] packed
// (00 01 02 11 12 22), 1/N folded in.  Full storage: gxq = nx, gyq = ny.
// Quarter storage (the reference element stiffness is symmetric under the x
// and y mirrors and n_x, n_y are even): only kx <= nx/2 and ky <= ny/2 are
// stored, and G(-kx) = Rx G(kx) Rx with Rx = diag(-1, 1, 1) flips the xy and
// xz entries (G(-ky): the xy and yz entries).
template <typename T>
struct GreenView {
    const T *G;
    int      nx, ny, gxq, gyq, Mc;
};

// Transform lengths (times the components, along z and x) are at most this.
constexpr int FFT_MAX_ELEMS = 3840;

// quotient of 0 <= a < 2^20 by a divisor fixed per launch
struct FastDiv {
    int   d;
    float inv;
    __device__ __forceinline__ explicit FastDiv(int n) : d(n), inv(1.0f / (float) n) {}
    __device__ __forceinline__ int operator()(int a, int &rem) const
    {
        int q = (int) (((float) a + 0.5f) * inv);
        rem   = a - q * d;
        return q;
    }
};

// f(integral_constant<R>) for the stage radix R <= MAXR
template <int MAXR = 16, typename F>
__device__ __forceinline__ void with_radix(int R, F &&f)
{
    if constexpr (MAXR < 16) {
        static_assert(MAXR == 12, "largest radix");
        switch (R) {
        case 2: f(std::integral_constant<int, 2>{}); break;
        case 3: f(std::integral_constant<int, 3>{}); break;
        case 4: f(std::integral_constant<int, 4>{}); break;
        case 5: f(std::integral_constant<int, 5>{}); break;
        case 6: f(std::integral_constant<int, 6>{}); break;
        case 8: f(std::integral_constant<int, 8>{}); break;
        case 9: f(std::integral_constant<int, 9>{}); break;
        case 10: f(std::integral_constant<int, 10>{}); break;
        default: f(std::integral_constant<int, 12>{}); break;
        }
        return;
    }
    switch (R) {
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 9: f(std::integral_constant<int, 9>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    case 12: f(std::integral_constant<int, 12>{}); break;
    case 15: f(std::integral_constant<int, 15>{}); break;
    default: f(std::integral_constant<int, 16>{}); break;
    }
}

// the same for a transform of a single stage (n = 2, 3 or 5)
template <typename F>
__device__ __forceinline__ void with_prime(int R, F &&f)
{
    switch (R) {
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    default: f(std::integral_constant<int, 5>{}); break;
    }
}

// v[k] *= W_m^(+-i k) with tw the table of W_n and step = (n / m) tws
template <typename T, int R, bool CONJ>
__device__ __forceinline__ void stage_twiddle(cplx<T> (&v)[R], const cplx<T> *__restrict__ tw, int i_step)
{
#pragma unroll
    for (int k = 1; k < R; ++k) {
        const cplx<T> w = tw[k * i_step];
        v[k]            = CONJ ? cmulc(v[k], w) : cmul(v[k], w);
    }
}

// Decimation-in-frequency stage of radix R on sub-transforms of length m (of a
// transform of length n): element i + t s, s = m / R, of a sub-transform comes
// from load(place, column) and output k goes to store(place of k, column, k).
// `place` counts the n elements, ncols columns each; INV conjugates.
template <typename T, int R, bool INV, typename Load, typename Store>
__device__ __forceinline__ void dif_stage(int n, int m, const FastDiv &ncols, const cplx<T> *__restrict__ tw, int tws,
                                          Load load, Store store)
{
    const int     s = m / R, total = (n / R) * ncols.d, step = (n / m) * tws;
    const FastDiv ds(s);
    for (int w = threadIdx.x; w < total; w += blockDim.x) {
        int       col, i;
        const int bi = ncols(w, col), q = ds(bi, i), p0 = q * m + i;
        cplx<T>   v[R];
#pragma unroll
        for (int t = 0; t < R; ++t)
            v[t] = load(p0 + t * s, col);
        dft_reg<T, R, INV>(v);
        if (s > 1)
            stage_twiddle<T, R, INV>(v, tw, i * step);
#pragma unroll
        for (int k = 0; k < R; ++k)
            store(p0 + k * s, col, v[k]);
    }
}

// The reversal of the forward dif_stage (decimation in time, inverse transform)
template <typename T, int R, typename Load, typename Store>
__device__ __forceinline__ void dit_stage(int n, int m, const FastDiv &ncols, const cplx<T> *__restrict__ tw, int tws,
                                          Load load, Store store)
{
    const int     s = m / R, total = (n / R) * ncols.d, step = (n / m) * tws;
    const FastDiv ds(s);
    for (int w = threadIdx.x; w < total; w += blockDim.x) {
        int       col, i;
        const int bi = ncols(w, col), q = ds(bi, i), p0 = q * m + i;
        cplx<T>   v[R];
#pragma unroll
        for (int k = 0; k < R; ++k)
            v[k] = load(p0 + k * s, col);
        if (s > 1)
            stage_twiddle<T, R, true>(v, tw, i * step);
        dft_reg<T, R, true>(v);
#pragma unroll
        for (int t = 0; t < R; ++t)
            store(p0 + t * s, col, v[t]);
    }
}

// frequency of the first output of block q of the last forward stage (the
// others follow at a distance of n / r_last)
__device__ __forceinline__ int block_frequency(const FftLen &L, int q)
{
    int f = 0;
    for (int s = L.nst - 2; s > 0; --s) {
        const int p = q / L.rad[s];
        f           = q - p * L.rad[s] + L.rad[s] * f;
        q           = p;
    }
    return q + (L.nst > 1 ? L.rad[0] : 1) * f;
}

// place of frequency k after the forward stages
__device__ __forceinline__ int frequency_place(const FftLen &L, int k)
{
    int p = 0;
    for (int s = 0; s < L.nst; ++s) {
        const int q = k / L.rad[s];
        p           = p * L.rad[s] + (k - q * L.rad[s]);
        k           = q;
    }
    return p;
}

// all stages in place in LDS, element (place, column) at buf[place * ld + column]
// (ends synchronised)
template <typename T, bool INV>
__device__ __forceinline__ void lds_fft(cplx<T> *buf, const FftLen &L, const cplx<T> *__restrict__ tw, int ncols,
                                        int ld)
{
    const FastDiv nc(ncols);
    auto          load  = [&](int p, int c) { return buf[p * ld + c]; };
    auto          store = [&](int p, int c, const cplx<T> &x) { buf[p * ld + c] = x; };
    int           m     = INV ? 1 : L.n;
    for (int j = 0; j < L.nst; ++j) {
        const int R = L.rad[INV ? L.nst - 1 - j : j];
        if (INV)
            m *= R;
        with_radix(R, [&](auto r) {
            constexpr int RR = decltype(r)::value;
            if constexpr (INV)
                dit_stage<T, RR>(L.n, m, nc, tw, L.tws, load, store);
            else
                dif_stage<T, RR, false>(L.n, m, nc, tw, L.tws, load, store);
        });
        if (!INV)
            m /= R;
        __syncthreads();
    }
}

// ---- FP32 stages ----------------------------------------------------------------
// The FP32 transforms (the inner solve of the mixed form) are Stockham stages of
// radices 5, 3, 8, 4 and 2, in this order of operations: a mixed displacement is
// FP32 rounding below about 1e-8 of its size (several outer rounds of FP32
// directions), so that another order moves it by up to 5e-9, more than the form's
// results are compared to.  (The larger radices of the FP64 stages took the 128^3
// mixed solve from 11.6 to 11.0 ms.)
// Register budget of the in-place stages: a thread holds at most FFT_MAXV
// complex values; callers keep n * ncols <= FFT_MAXV * 240 so every radix
// (including 3 and 5, where MAXV/R rounds down) fits.
constexpr int FFT_MAXV = 16;

// ---- one in-place Stockham radix-R stage over `ncols` independent columns --
// element (i, col) lives at buf[i * ld + col]
template <typename T, int R, bool INV>
__device__ __forceinline__ void stockham_stage(cplx<T> *__restrict__ buf, int n, int ncols, int ld, int Ns,
                                               const cplx<T> *__restrict__ tw, int tws)
{
    constexpr int MB    = FFT_MAXV / R;
    const int     nb    = n / R;
    const int     total = nb * ncols;
    const int     tstep = (n / (Ns * R)) * tws;
    cplx<T>       v[MB][R];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const int w = threadIdx.x + b * blockDim.x;
        if (w < total) {
            const int col = w % ncols, j = w / ncols;
#pragma unroll
            for (int t = 0; t < R; ++t)
                v[b][t] = buf[(j + t * nb) * ld + col];
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const int w = threadIdx.x + b * blockDim.x;
        if (w < total) {
            const int col = w % ncols, j = w / ncols, k = j % Ns;
            if (Ns > 1) {
#pragma unroll
                for (int t = 1; t < R; ++t) {
                    const cplx<T> wv = tw[t * k * tstep];
                    v[b][t]          = INV ? cmulc(v[b][t], wv) : cmul(v[b][t], wv);
                }
            }
            dft<T, R, INV>(v[b]);
            const int o = (j / Ns) * Ns * R + k;
#pragma unroll
            for (int t = 0; t < R; ++t)
                buf[(o + t * Ns) * ld + col] = v[b][t];
        }
    }
    __syncthreads();
}

// full in-place transform of the LDS tile (ends synchronised)
template <typename T, bool INV>
__device__ void lds_stockham(cplx<T> *buf, const FftLen &L, const cplx<T> *__restrict__ tw, int ncols, int ld)
{
    int Ns = 1;
    for (int s = 0; s < L.nst; ++s) {
        const int R = L.rad[s];
        switch (R) {
        case 2: stockham_stage<T, 2, INV>(buf, L.n, ncols, ld, Ns, tw, L.tws); break;
        case 3: stockham_stage<T, 3, INV>(buf, L.n, ncols, ld, Ns, tw, L.tws); break;
        case 4: stockham_stage<T, 4, INV>(buf, L.n, ncols, ld, Ns, tw, L.tws); break;
        case 5: stockham_stage<T, 5, INV>(buf, L.n, ncols, ld, Ns, tw, L.tws); break;
        default: stockham_stage<T, 8, INV>(buf, L.n, ncols, ld, Ns, tw, L.tws); break;
        }
        Ns *= R;
    }
}

// ---- CG update fused into the forward z pass --------------------------------
// PRO_CG: the forward z pass of CG iteration i first finishes the residual
// update of iteration i-1 (solverCG.h:106-117): r -= alpha rnew, and emits per
// block the partial |r| (norm of the measure), which the reduction turns into
// the error.  Only the updated r enters the transform.  deltamid = <r, s_prev>
// needs no s here: the CG scalars form it from <d, K d> (matvec) and
// <d, K d_prev> (inverse z pass).  The matching solution update u -= alpha d
// runs in the inverse z pass of the next iteration, which reads that d anyway.
// PRO_CGF: alpha, that reduction and the one before it from the partials (CgFold).
enum { PRO_NONE = 0, PRO_CG = 1, PRO_CGF = 2 };

template <typename T>
struct ProArgs {
    const T      *rnew;     // K d of the previous iteration
    const double *alpha;    // device scalar
    int           measure;  // 0 L1, 1 L2, 2 Linf
    double       *partial;  // [gridDim.x]
    CgFold        fold;     // PRO_CGF
};

// Loads a thread issues together before the stores that follow them in the
// fused prologues / epilogues of the z passes.  Element by element, a store may
// alias the next element's loads, so the compiler keeps program order: one
// memory round trip per element.  kZGroup for the compile-time passes,
// kZGroupRt for the runtime-length ones (bounds-checked groups).
#ifndef FANS_Z_GROUP
#define FANS_Z_GROUP 16
#endif
constexpr int kZGroup = FANS_Z_GROUP;
#ifndef FANS_Z_GROUP_RT
#define FANS_Z_GROUP_RT 8
#endif
constexpr int kZGroupRt = FANS_Z_GROUP_RT;

template <typename T, int PRO>
__device__ __forceinline__ T z_load(T *__restrict__ in, int64_t gi, const ProArgs<T> &pa, T alpha, double &a0)
{
    if constexpr (PRO != PRO_NONE) {
        // r and rnew are not read again before the spectrum passes that
        // follow: streaming (non-temporal) accesses keep them from displacing
        // the freshly written spectrum in the Infinity Cache
        const T rv = __builtin_nontemporal_load(&in[gi]) - alpha * __builtin_nontemporal_load(&pa.rnew[gi]);
        __builtin_nontemporal_store(rv, &in[gi]);
        acc_norm(a0, rv, pa.measure);
        return rv;
    } else {
        return in[gi];
    }
}

template <int PRO, typename T>
__device__ __forceinline__ void z_pro_partials(const ProArgs<T> &pa, double a0, double *red)
{
    if constexpr (PRO != PRO_NONE) {
        double     v[1]  = {a0};
        const bool mx[1] = {pa.measure == 2};
        block_reduce<1>(v, mx, red);
        if (threadIdx.x == 0)
            pa.partial[blockIdx.x] = v[0];
    }
}

// r2c post-processing of the half-length transform Z (in LDS, column col):
// X[k] = (Z[k] + conj Z[M-k]) / 2 + W^k (Z[k] - conj Z[M-k]) / (2i)
template <typename T>
__device__ __forceinline__ cplx<T> r2c_untangle(cplx<T> zk, cplx<T> zc, cplx<T> w)
{
    zc              = conjg(zc);
    const cplx<T> E = cscale(zk + zc, (T) 0.5);
    const cplx<T> D = cscale(zk - zc, (T) 0.5);
    return E + cmul(w, cplx<T>{D.y, -D.x});
}
template <typename T>
__device__ __forceinline__ cplx<T> r2c_untangle(const cplx<T> *A, int ld, int col, int k, int M,
                                                const cplx<T> *__restrict__ tw)
{
    return r2c_untangle(A[(k == M ? 0 : k) * ld + col], A[(k == 0 ? 0 : M - k) * ld + col], tw[k]);
}

// ---- z pass, forward r2c ----------------------------------------------------
// LM: complex length M = nz/2 with tws = 2 into the length-nz table `tw`.
// Block b handles lines [b*lpb, b*lpb + lpb) of nz*H reals each.
template <typename T, int H, int PRO>
__global__ __launch_bounds__(256) void k_fft_z_r2c(T *__restrict__ in, cplx<T> *__restrict__ out, FftLen LM,
                                                   const cplx<T> *__restrict__ tw, int nz, int64_t nlines, int lpb,
                                                   ProArgs<T> pa, Slots sl)
{
    const int sb = slot_of(sl);
    if (sb < 0)
        return;
    if (sl.map) {  // batched launch: this slot's buffers
        in += sb * sl.field;
        out += sb * sl.spec;
        slot_pro(pa, sb, sl);
    }
    extern __shared__ char smem_raw[];
    __shared__ double red[8];
    cplx<T>      *A     = reinterpret_cast<cplx<T> *>(smem_raw);
    const int     M     = nz / 2;
    const int64_t line0 = (int64_t) blockIdx.x * lpb;
    const int     nl    = (int) ((nlines - line0) < lpb ? (nlines - line0) : lpb);
    const int     ncols = nl * H, ld = ncols + 1;
    const int     nzh   = nz * H;
    const int64_t g0    = line0 * nzh;
    T             alpha = (T) 0;
    double        a0    = 0.0;
    // places of the frequencies, behind the tile (FP64)
    unsigned short *const place = reinterpret_cast<unsigned short *>(A + M * (lpb * H + 1));
    if constexpr (sizeof(T) == 8)
        for (int k = threadIdx.x; k < M; k += blockDim.x)
            place[k] = (unsigned short) frequency_place(LM, k);
    auto place_of = [&](int k) { return sizeof(T) == 8 ? (int) place[k] : k; };
    const FastDiv dz(nzh);
    if constexpr (PRO == PRO_CG)
        alpha = (T) *pa.alpha;
    if constexpr (PRO == PRO_CGF)
        alpha = (T) fold_alpha<256>(pa.fold, red);
    if constexpr (PRO != PRO_NONE && kZGroupRt > 0) {
        // r -= alpha K d in groups (same arithmetic and order as z_load)
        constexpr int CH = kZGroupRt;
        const int     tot = nl * nzh, stp = blockDim.x;
        for (int e0 = threadIdx.x; e0 < tot; e0 += CH * stp) {
            T rv[CH], qv[CH];
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                const int e = e0 + i * stp;
                rv[i] = qv[i] = (T) 0;
                if (e < tot) {
                    rv[i] = __builtin_nontemporal_load(&in[g0 + e]);
                    qv[i] = __builtin_nontemporal_load(&pa.rnew[g0 + e]);
                }
            }
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                const int e = e0 + i * stp;
                if (e < tot) {
                    int       rem;
                    const int l = dz(e, rem), z = rem / H, c = rem - z * H;
                    const T   r = rv[i] - alpha * qv[i];
                    __builtin_nontemporal_store(r, &in[g0 + e]);
                    acc_norm(a0, r, pa.measure);
                    T *d     = reinterpret_cast<T *>(&A[(z >> 1) * ld + l * H + c]);
                    d[z & 1] = r;
                }
            }
        }
    } else {
        for (int e = threadIdx.x; e < nl * nzh; e += blockDim.x) {
            int       rem;
            const int l = dz(e, rem), z = rem / H, c = rem - z * H;
            T        *d = reinterpret_cast<T *>(&A[(z >> 1) * ld + l * H + c]);
            d[z & 1]    = z_load<T, PRO>(in, g0 + e, pa, alpha, a0);
        }
    }
    __syncthreads();
    if constexpr (sizeof(T) == 8)
        lds_fft<T, false>(A, LM, tw, ncols, ld);
    else
        lds_stockham<T, false>(A, LM, tw, ncols, ld);
    const int     Mc  = M + 1;
    const FastDiv dl(Mc * H);
    cplx<T>      *dst = out + line0 * Mc * H;
    for (int e = threadIdx.x; e < nl * Mc * H; e += blockDim.x) {
        int       rem;
        const int l = dl(e, rem), k = rem / H, c = rem - k * H, col = l * H + c;
        dst[e] = r2c_untangle(A[place_of(k == M ? 0 : k) * ld + col], A[place_of(k == 0 ? 0 : M - k) * ld + col], tw[k]);
    }
    z_pro_partials<PRO>(pa, a0, red);
}

// ---- z pass, inverse c2r with fused epilogues -------------------------------
// EPI_CGD (linear CG, solverCG.h:88-92): the new search direction
// d = s + beta d_prev with s = -result (beta from the spectral <r, s> of the x
// pass); s itself is not stored.  With qprev = K d_prev (the previous matvec's
// output) it emits per block the partial <d, K d_prev>, from which the CG
// scalars form the next deltamid.  EPI_CGDF: the same with beta, and before it
// the error and the stop test, from the partials (CgFold).
enum { EPI_STORE = 0, EPI_CG = 1, EPI_FP = 2, EPI_CGD = 3, EPI_CGDF = 4 };
constexpr bool epi_cgd(int epi) { return epi == EPI_CGD || epi == EPI_CGDF; }

template <typename T>
struct EpiArgs {
    T            *out;      // EPI_STORE: result; EPI_CG: s = -result
    const T      *r;        // EPI_CG: partial <r, s>
    double       *u;        // EPI_FP: u -= result (FP64 displacement)
    double       *partial;  // EPI_CG / EPI_CGD: one partial sum per block
    const T      *dprev;    // EPI_CGD: previous direction (read)
    const T      *qprev;    // EPI_CGD: K d_prev (nullable), partial <d, K d_prev>
    T            *dnext;    // EPI_CGD: new direction (written)
    const double *scal;     // EPI_CGD: device scalars (beta at [0])
    CgFold        fold;     // EPI_CGDF
};

// the argument blocks at RVE slot sb
template <typename T>
__device__ __forceinline__ void slot_pro(ProArgs<T> &pa, int sb, const Slots &sl)
{
    pa.rnew    = slot_ptr(pa.rnew, sb * sl.field);
    pa.alpha   = slot_ptr(pa.alpha, (int64_t) sb * kScSlot);
    pa.partial = slot_ptr(pa.partial, sb * sl.part);
    slot_fold(pa.fold, sb, sl);
}
template <typename T>
__device__ __forceinline__ void slot_epi(EpiArgs<T> &ep, int sb, const Slots &sl)
{
    ep.out     = slot_ptr(ep.out, sb * sl.field);
    ep.r       = slot_ptr(ep.r, sb * sl.field);
    ep.u       = slot_ptr(ep.u, sb * sl.field);
    ep.partial = slot_ptr(ep.partial, sb * sl.part);
    ep.dprev   = slot_ptr(ep.dprev, sb * sl.field);
    ep.qprev   = slot_ptr(ep.qprev, sb * sl.field);
    ep.dnext   = slot_ptr(ep.dnext, sb * sl.field);
    ep.scal    = slot_ptr(ep.scal, (int64_t) sb * kScSlot);
    slot_fold(ep.fold, sb, sl);
}

// c2r pre-processing of one (line, component): `line` points at kz = 0 of the
// component (stride H); the half-length transform input is
// Z[k] = (X[k] + conj X[M-k]) + i W^-k (X[k] - conj X[M-k])
template <typename T, int H>
__device__ __forceinline__ cplx<T> c2r_tangle(const cplx<T> *__restrict__ line, int k, int M,
                                              const cplx<T> *__restrict__ tw)
{
    const cplx<T> xk = line[k * H];
    const cplx<T> xm = conjg(line[(M - k) * H]);
    const cplx<T> WD = cmul(conjg(tw[k]), xk - xm);
    return (xk + xm) + cplx<T>{-WD.y, WD.x};
}

template <typename T, int EPI>
__device__ __forceinline__ void z_epilogue(const EpiArgs<T> &ep, int64_t gi, T val, double &acc, T beta)
{
    if constexpr (EPI == EPI_STORE) {
        ep.out[gi] = val;
    } else if constexpr (epi_cgd(EPI)) {
        // d_next is read by the very next pass (the matvec) and stays cached;
        // d_prev and u stream past the caches
        const T dp = __builtin_nontemporal_load(&ep.dprev[gi]);
        const T dn = beta * dp - val;
        ep.dnext[gi] = dn;
        if (ep.qprev)
            acc += (double) dn * (double) __builtin_nontemporal_load(&ep.qprev[gi]);
    } else if constexpr (EPI == EPI_CG) {
        // s is read by the very next pass (the matvec) and stays cached; r is
        // not read again this iteration
        const T sv = -val;
        ep.out[gi] = sv;
        acc += (double) __builtin_nontemporal_load(&ep.r[gi]) * (double) sv;
    } else {
        ep.u[gi] -= (double) val;
    }
}

// z_epilogue over this thread's elements e = threadIdx.x + k stp < tot in
// groups of CH, each group's global operands requested before its stores (the
// stores never alias the operands of another element: d_next and d_prev, s
// and r are distinct buffers and u is updated per element); same arithmetic
// and accumulation order as z_epilogue.  val_of(e) is element e's result.
template <typename T, int EPI, int CH, typename ValOf>
__device__ __forceinline__ void z_epilogue_grouped(const EpiArgs<T> &ep, int64_t g0, int tot, int stp, ValOf val_of,
                                                   double &acc, T beta)
{
    for (int e0 = threadIdx.x; e0 < tot; e0 += CH * stp) {
        T      pa[CH], pb[CH];
        double pu[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int     e  = e0 + i * stp;
            const int64_t gi = g0 + e;
            pa[i] = pb[i] = (T) 0;
            pu[i]         = 0.0;
            if (e < tot) {
                if constexpr (epi_cgd(EPI)) {
                    pa[i] = __builtin_nontemporal_load(&ep.dprev[gi]);
                    if (ep.qprev)
                        pb[i] = __builtin_nontemporal_load(&ep.qprev[gi]);
                } else if constexpr (EPI == EPI_CG) {
                    pb[i] = __builtin_nontemporal_load(&ep.r[gi]);
                } else if constexpr (EPI == EPI_FP) {
                    pu[i] = ep.u[gi];
                }
            }
        }
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int     e  = e0 + i * stp;
            const int64_t gi = g0 + e;
            if (e < tot) {
                const T val = val_of(e);
                if constexpr (EPI == EPI_STORE) {
                    ep.out[gi] = val;
                } else if constexpr (epi_cgd(EPI)) {
                    const T dn   = beta * pa[i] - val;
                    ep.dnext[gi] = dn;
                    if (ep.qprev)
                        acc += (double) dn * (double) pb[i];
                } else if constexpr (EPI == EPI_CG) {
                    const T sv = -val;
                    ep.out[gi] = sv;
                    acc += (double) pb[i] * (double) sv;
                } else {
                    ep.u[gi] = pu[i] - (double) val;
                }
            }
        }
    }
}

template <int EPI, typename T>
__device__ __forceinline__ void z_epi_partials(const EpiArgs<T> &ep, double acc, double *red)
{
    // (EPI_CGDF: also without qprev, a zero, which the next launch folds)
    if (EPI == EPI_CG || EPI == EPI_CGDF || (EPI == EPI_CGD && ep.qprev)) {
        double     v[1]  = {acc};
        const bool mx[1] = {false};
        block_reduce<1>(v, mx, red);
        if (threadIdx.x == 0)
            ep.partial[blockIdx.x] = v[0];
    }
}

template <typename T, int H, int EPI>
__global__ __launch_bounds__(256) void k_fft_z_c2r(const cplx<T> *__restrict__ in, FftLen LM,
                                                   const cplx<T> *__restrict__ tw, int nz, int64_t nlines, int lpb,
                                                   EpiArgs<T> ep, Slots sl)
{
    const int sb = slot_of(sl);
    if (sb < 0)
        return;
    if (sl.map) {  // batched launch: this slot's buffers
        in += sb * sl.spec;
        slot_epi(ep, sb, sl);
    }
    extern __shared__ char smem_raw[];
    __shared__ double red[8];
    cplx<T>          *A     = reinterpret_cast<cplx<T> *>(smem_raw);
    const int         M     = nz / 2, Mc = M + 1;
    const int64_t     line0 = (int64_t) blockIdx.x * lpb;
    const int         nl    = (int) ((nlines - line0) < lpb ? (nlines - line0) : lpb);
    const int         ncols = nl * H, ld = ncols + 1;
    const cplx<T>    *src   = in + line0 * Mc * H;
    const FastDiv     dl(M * H);
    FoldBeta          fb;
    if constexpr (EPI == EPI_CGDF)
        fb.template load<256>(ep.fold);
    // places of the frequencies, behind the tile (FP64)
    unsigned short *const place = reinterpret_cast<unsigned short *>(A + M * (lpb * H + 1));
    if constexpr (sizeof(T) == 8)
        for (int k = threadIdx.x; k < M; k += blockDim.x)
            place[k] = (unsigned short) frequency_place(LM, k);
    auto place_of = [&](int k) { return sizeof(T) == 8 ? (int) place[k] : k; };
    __syncthreads();
    for (int e = threadIdx.x; e < nl * M * H; e += blockDim.x) {
        int       rem;
        const int l = dl(e, rem), k = rem / H, c = rem - k * H;
        A[place_of(k) * ld + l * H + c] = c2r_tangle<T, H>(src + l * Mc * H + c, k, M, tw);
    }
    __syncthreads();
    if constexpr (sizeof(T) == 8)
        lds_fft<T, true>(A, LM, tw, ncols, ld);
    else
        lds_stockham<T, true>(A, LM, tw, ncols, ld);
    const int     nzh = nz * H;
    const int64_t g0  = line0 * nzh;
    double        acc = 0.0;
    T             beta = (T) 0;
    if constexpr (EPI == EPI_CGD)
        beta = (T) ep.scal[0];
    if constexpr (EPI == EPI_CGDF) {
        double b;
        if (!fb.template finish<256>(ep.fold, red, b))
            return;
        beta = (T) b;
    }
    const FastDiv dz(nzh);
    auto          val_of = [&](int e) {
        int           rem;
        const int     l = dz(e, rem), z = rem / H, c = rem - z * H;
        const cplx<T> v = A[(z >> 1) * ld + l * H + c];
        return (z & 1) ? v.y : v.x;
    };
    if constexpr (kZGroupRt > 0 && EPI != EPI_STORE) {
        z_epilogue_grouped<T, EPI, kZGroupRt>(ep, g0, nl * nzh, blockDim.x, val_of, acc, beta);
    } else {
        for (int e = threadIdx.x; e < nl * nzh; e += blockDim.x)
            z_epilogue<T, EPI>(ep, g0 + e, val_of(e), acc, beta);
    }
    z_epi_partials<EPI>(ep, acc, red);
}

// ---- z passes with compile-time shape ---------------------------------------
// operands of the linear CG's inverse z epilogue requested before the
// transform (0 none, 1 d_prev, 2 d_prev and K d_prev), per precision; the
// others are requested together right after it.  At 256^3: FP64 0.294 ms
// with d_prev ahead, 0.295 with none, 0.306 with both; FP32 0.134 ms with
// none, 0.136 with d_prev, 0.223 with both.
#ifndef FANS_C2R_AHEAD64
#define FANS_C2R_AHEAD64 1
#endif
#ifndef FANS_C2R_AHEAD32
#define FANS_C2R_AHEAD32 0
#endif
constexpr int kC2rAhead64 = FANS_C2R_AHEAD64;
constexpr int kC2rAhead32 = FANS_C2R_AHEAD32;

// For M = nz/2 in {16, 24, 32, 40, 48, 64, 128} the line count per block, the
// thread count and every index are compile-time constants (no runtime divisions), and the
// thread count equals the butterfly count of the first radix stage.
template <int M>
constexpr int zct_radix1()
{
    return M >= 32 ? 8 : 4;
}
template <int H, int M>
constexpr int zct_lpb()
{
    int l = 1;
    while ((M / zct_radix1<M>()) * (2 * l) * H <= 256)
        l *= 2;
    return l;
}
template <int H, int M>
constexpr int zct_threads()
{
    return (M / zct_radix1<M>()) * zct_lpb<H, M>() * H;
}

template <typename T, int R, bool INV, int N, int NC, int LD, int NS, int NT>
__device__ __forceinline__ void stockham_stage_ct(cplx<T> *__restrict__ buf, const cplx<T> *__restrict__ tw)
{
    constexpr int nb = N / R, total = nb * NC, MB = (total + NT - 1) / NT;
    constexpr int tstep = 2 * (N / (NS * R));  // into the length-2N table
    cplx<T>       v[MB][R];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const int w = threadIdx.x + b * NT;
        if (total % NT == 0 || w < total) {
            const int col = w % NC, j = w / NC;
#pragma unroll
            for (int t = 0; t < R; ++t)
                v[b][t] = buf[(j + t * nb) * LD + col];
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const int w = threadIdx.x + b * NT;
        if (total % NT == 0 || w < total) {
            const int col = w % NC, j = w / NC, k = j % NS;
            if constexpr (NS > 1) {
#pragma unroll
                for (int t = 1; t < R; ++t) {
                    const cplx<T> wv = tw[t * k * tstep];
                    v[b][t]          = INV ? cmulc(v[b][t], wv) : cmul(v[b][t], wv);
                }
            }
            dft<T, R, INV>(v[b]);
            const int o = (j / NS) * NS * R + k;
#pragma unroll
            for (int t = 0; t < R; ++t)
                buf[(o + t * NS) * LD + col] = v[b][t];
        }
    }
    __syncthreads();
}

// radix schedules: 128 = 8*4*4, 64 = 8*8, 48 = 8*3*2, 40 = 8*5, 32 = 8*4,
// 24 = 4*3*2, 16 = 4*4 (the first radix is zct_radix1)
template <typename T, bool INV, int N, int NC, int LD, int NT>
__device__ __forceinline__ void lds_fft_ct(cplx<T> *buf, const cplx<T> *__restrict__ tw)
{
    if constexpr (N == 48) {
        stockham_stage_ct<T, 8, INV, N, NC, LD, 1, NT>(buf, tw);
        stockham_stage_ct<T, 3, INV, N, NC, LD, 8, NT>(buf, tw);
        stockham_stage_ct<T, 2, INV, N, NC, LD, 24, NT>(buf, tw);
    } else if constexpr (N == 40) {
        stockham_stage_ct<T, 8, INV, N, NC, LD, 1, NT>(buf, tw);
        stockham_stage_ct<T, 5, INV, N, NC, LD, 8, NT>(buf, tw);
    } else if constexpr (N == 24) {
        stockham_stage_ct<T, 4, INV, N, NC, LD, 1, NT>(buf, tw);
        stockham_stage_ct<T, 3, INV, N, NC, LD, 4, NT>(buf, tw);
        stockham_stage_ct<T, 2, INV, N, NC, LD, 12, NT>(buf, tw);
    } else if constexpr (N == 128) {
        stockham_stage_ct<T, 8, INV, N, NC, LD, 1, NT>(buf, tw);
        stockham_stage_ct<T, 4, INV, N, NC, LD, 8, NT>(buf, tw);
        stockham_stage_ct<T, 4, INV, N, NC, LD, 32, NT>(buf, tw);
    } else if constexpr (N == 64) {
        stockham_stage_ct<T, 8, INV, N, NC, LD, 1, NT>(buf, tw);
        stockham_stage_ct<T, 8, INV, N, NC, LD, 8, NT>(buf, tw);
    } else if constexpr (N == 32) {
        stockham_stage_ct<T, 8, INV, N, NC, LD, 1, NT>(buf, tw);
        stockham_stage_ct<T, 4, INV, N, NC, LD, 8, NT>(buf, tw);
    } else {
        static_assert(N == 16, "unsupported compile-time length");
        stockham_stage_ct<T, 4, INV, N, NC, LD, 1, NT>(buf, tw);
        stockham_stage_ct<T, 4, INV, N, NC, LD, 4, NT>(buf, tw);
    }
}

// forward: lines [b*LPB, b*LPB + LPB); the host launches nlines / LPB blocks
template <typename T, int H, int M, int PRO>
__global__ __launch_bounds__((zct_threads<H, M>())) void k_fft_z_r2c_ct(T *__restrict__ in, cplx<T> *__restrict__ out,
                                                                      const cplx<T> *__restrict__ tw, ProArgs<T> pa,
                                                                      Slots sl)
{
    const int sb = slot_of(sl);
    if (sb < 0)
        return;
    if (sl.map) {  // batched launch: this slot's buffers
        in += sb * sl.field;
        out += sb * sl.spec;
        slot_pro(pa, sb, sl);
    }
    constexpr int NT = zct_threads<H, M>(), LPB = zct_lpb<H, M>();
    constexpr int NZH = 2 * M * H, NC = LPB * H, LD = NC + 1, MC = M + 1;
    __shared__ cplx<T> A[M * LD];
    __shared__ double  red[2 * ((NT + 63) / 64)];
    const int64_t      line0 = (int64_t) blockIdx.x * LPB;
    const int64_t      g0    = line0 * NZH;
    T                  alpha = (T) 0;
    double             a0    = 0.0;
    if constexpr (PRO == PRO_CG)
        alpha = (T) *pa.alpha;
    if constexpr (PRO == PRO_CGF)
        alpha = (T) fold_alpha<NT>(pa.fold, red);
    constexpr int PER = (LPB * NZH) / NT;
    constexpr int CH  = kZGroup < PER ? kZGroup : PER;
    if constexpr (PRO != PRO_NONE && kZGroup > 0 && (LPB * NZH) % NT == 0 && PER % CH == 0) {
        // r -= alpha K d in groups of CH elements: the loads of a group are in
        // flight together (same arithmetic and accumulation order as z_load)
        for (int i0 = 0; i0 < PER; i0 += CH) {
            T rv[CH], qv[CH];
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                const int64_t gi = g0 + threadIdx.x + (i0 + i) * NT;
                rv[i]            = __builtin_nontemporal_load(&in[gi]);
                qv[i]            = __builtin_nontemporal_load(&pa.rnew[gi]);
            }
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                const int e = threadIdx.x + (i0 + i) * NT;
                const int l = e / NZH, rem = e - l * NZH, z = rem / H, c = rem - z * H;
                const T   r = rv[i] - alpha * qv[i];
                __builtin_nontemporal_store(r, &in[g0 + e]);
                acc_norm(a0, r, pa.measure);
                T *d     = reinterpret_cast<T *>(&A[(z >> 1) * LD + l * H + c]);
                d[z & 1] = r;
            }
        }
    } else {
#pragma unroll 4
        for (int e = threadIdx.x; e < LPB * NZH; e += NT) {
            const int l = e / NZH, rem = e - l * NZH, z = rem / H, c = rem - z * H;
            T        *d = reinterpret_cast<T *>(&A[(z >> 1) * LD + l * H + c]);
            d[z & 1]    = z_load<T, PRO>(in, g0 + e, pa, alpha, a0);
        }
    }
    __syncthreads();
    lds_fft_ct<T, false, M, NC, LD, NT>(A, tw);
    cplx<T> *dst = out + line0 * MC * H;
#pragma unroll 4
    for (int e = threadIdx.x; e < LPB * MC * H; e += NT) {
        const int l = e / (MC * H), rem = e - l * (MC * H), k = rem / H, c = rem - k * H;
        dst[e]      = r2c_untangle(A, LD, l * H + c, k, M, tw);
    }
    z_pro_partials<PRO>(pa, a0, red);
}

template <typename T, int H, int M, int EPI>
__global__ __launch_bounds__((zct_threads<H, M>())) void k_fft_z_c2r_ct(const cplx<T> *__restrict__ in,
                                                                      const cplx<T> *__restrict__ tw, EpiArgs<T> ep,
                                                                      Slots sl)
{
    const int sb = slot_of(sl);
    if (sb < 0)
        return;
    if (sl.map) {  // batched launch: this slot's buffers
        in += sb * sl.spec;
        slot_epi(ep, sb, sl);
    }
    constexpr int NT = zct_threads<H, M>(), LPB = zct_lpb<H, M>();
    constexpr int NZH = 2 * M * H, NC = LPB * H, LD = NC + 1, MC = M + 1;
    __shared__ cplx<T> A[M * LD];
    __shared__ double  red[2 * ((NT + 63) / 64)];
    const int64_t      line0 = (int64_t) blockIdx.x * LPB;
    const cplx<T>     *src   = in + line0 * MC * H;
    const int64_t      g0    = line0 * NZH;
    // EPI_CGD: this thread's values of d_prev and K d_prev, the ones of
    // kC2rAhead* requested before the transform so that their loads overlap it,
    // at the cost of registers during it
    constexpr int  PER   = (LPB * NZH) / NT;
    constexpr int  AHEAD = sizeof(T) == 8 ? kC2rAhead64 : kC2rAhead32;
    constexpr bool PRE   = epi_cgd(EPI) && (LPB * NZH) % NT == 0;
    constexpr bool PRED = PRE && AHEAD >= 1, PREQ = PRE && AHEAD >= 2;
    T              dpv[PRE ? PER : 1], qpv[PRE ? PER : 1];
    FoldBeta       fb;
    if constexpr (EPI == EPI_CGDF)
        fb.template load<NT>(ep.fold);
    if constexpr (PRED) {
        const T *__restrict__ dp = ep.dprev;
        const T *__restrict__ qp = ep.qprev;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            dpv[i] = __builtin_nontemporal_load(&dp[g0 + threadIdx.x + i * NT]);
            if constexpr (PREQ)
                qpv[i] = qp ? __builtin_nontemporal_load(&qp[g0 + threadIdx.x + i * NT]) : (T) 0;
        }
    }
#pragma unroll 4
    for (int e = threadIdx.x; e < LPB * M * H; e += NT) {
        const int l = e / (M * H), rem = e - l * (M * H), k = rem / H, c = rem - k * H;
        A[k * LD + l * H + c] = c2r_tangle<T, H>(src + l * MC * H + c, k, M, tw);
    }
    __syncthreads();
    lds_fft_ct<T, true, M, NC, LD, NT>(A, tw);
    double acc  = 0.0;
    T      beta = (T) 0;
    if constexpr (EPI == EPI_CGD)
        beta = (T) ep.scal[0];
    if constexpr (EPI == EPI_CGDF) {
        double b;
        if (!fb.template finish<NT>(ep.fold, red, b))
            return;
        beta = (T) b;
    }
    if constexpr (PRE) {
        T *__restrict__ dn = ep.dnext;
        // the operands not requested ahead: all of this thread's values are
        // requested before the first store of d
        if constexpr (!PRED)
#pragma unroll
            for (int i = 0; i < PER; ++i)
                dpv[i] = __builtin_nontemporal_load(&ep.dprev[g0 + threadIdx.x + i * NT]);
        if constexpr (!PREQ)
            if (ep.qprev)
#pragma unroll
                for (int i = 0; i < PER; ++i)
                    qpv[i] = __builtin_nontemporal_load(&ep.qprev[g0 + threadIdx.x + i * NT]);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int     e = threadIdx.x + i * NT;
            const int     l = e / NZH, rem = e - l * NZH, z = rem / H, c = rem - z * H;
            const cplx<T> v = A[(z >> 1) * LD + l * H + c];
            const T       d = beta * dpv[i] - ((z & 1) ? v.y : v.x);
            dn[g0 + e]      = d;
            if (ep.qprev)
                acc += (double) d * (double) qpv[i];
        }
    } else {
        auto val_of = [&](int e) {
            const int     l = e / NZH, rem = e - l * NZH, z = rem / H, c = rem - z * H;
            const cplx<T> v = A[(z >> 1) * LD + l * H + c];
            return (z & 1) ? v.y : v.x;
        };
        if constexpr (kZGroup > 0 && EPI != EPI_STORE) {
            constexpr int CH = kZGroup < 8 ? kZGroup : 8;
            z_epilogue_grouped<T, EPI, CH>(ep, g0, LPB * NZH, NT, val_of, acc, beta);
        } else {
#pragma unroll 4
            for (int e = threadIdx.x; e < LPB * NZH; e += NT)
                z_epilogue<T, EPI>(ep, g0 + e, val_of(e), acc, beta);
        }
    }
    z_epi_partials<EPI>(ep, acc, red);
}

// ---- batched strided complex pass (y or x axis) ----------------------------
// data[o*ostride + i*sn + b] for i < L.n, b in [c0, c1); block (bx, o) owns
// columns [c0 + bx*bc, c0 + bx*bc + bc).  FP64, lengths without a register kernel.
// Bound by memory where the tile is 16 columns wide (125 x 120 x 150, y of 120 points:
// 24 us, 4.6 TB/s; radix 2 to 8 Stockham stages through the whole tile took 34), four
// waves per SIMD.
template <typename T, bool INV>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_fft_strided(cplx<T> *__restrict__ data, FftLen L,
                                                     const cplx<T> *__restrict__ tw, int64_t sn, int c0, int c1,
                                                     int64_t ostride, int bc, int nbx, Slots sl)
{
    const int sb = slot_of(sl);
    if (sb < 0)
        return;
    if (sl.map) {  // batched launch: this slot's buffers
        data += sb * sl.spec;
    }
    extern __shared__ char smem_raw[];
    cplx<T>      *A     = reinterpret_cast<cplx<T> *>(smem_raw);
    const int     lb    = xcd_tile_index(blockIdx.x, gridDim.x), bo = lb / nbx, bx = lb - bo * nbx;
    const int     b0    = c0 + bx * bc;
    const int     ncols = (c1 - b0) < bc ? (c1 - b0) : bc, n = L.n;
    cplx<T>      *base  = data + (int64_t) bo * ostride + b0;
    const FastDiv nc(ncols);
    auto          from_mem = [&](int p, int c) { return base[p * sn + c]; };
    auto          from_lds = [&](int p, int c) { return A[p * ncols + c]; };
    auto          to_lds   = [&](int p, int c, const cplx<T> &x) { A[p * ncols + c] = x; };
    // a place's frequency: blocks of r_last places, its digits reversed
    const int     rl = L.rad[L.nst - 1], ds = n / rl;
    const FastDiv dr(rl);
    auto          to_mem = [&](int p, int c, const cplx<T> &x) {
        int       k;
        const int q = dr(p, k);
        base[(int64_t) (block_frequency(L, q) + k * ds) * sn + c] = x;
    };
    if (L.nst == 1) {
        with_prime(rl, [&](auto r) { dif_stage<T, decltype(r)::value, INV>(n, n, nc, tw, L.tws, from_mem, to_mem); });
        return;
    }
    int m = n;
    with_radix(L.rad[0], [&](auto r) { dif_stage<T, decltype(r)::value, INV>(n, m, nc, tw, L.tws, from_mem, to_lds); });
    m /= L.rad[0];
    __syncthreads();
    for (int s = 1; s < L.nst - 1; ++s) {
        with_radix(L.rad[s],
                   [&](auto r) { dif_stage<T, decltype(r)::value, INV>(n, m, nc, tw, L.tws, from_lds, to_lds); });
        m /= L.rad[s];
        __syncthreads();
    }
    with_radix(rl, [&](auto r) { dif_stage<T, decltype(r)::value, INV>(n, m, nc, tw, L.tws, from_lds, to_mem); });
}

// the same, FP32: the whole tile through LDS; block (bx, o) = blockIdx.x, y
template <typename T, bool INV>
__global__ __launch_bounds__(256) void k_fft_strided_stockham(cplx<T> *__restrict__ data, FftLen L,
                                                     const cplx<T> *__restrict__ tw, int64_t sn, int c0, int c1,
                                                     int64_t ostride, int bc, Slots sl)
{
    const int sb = slot_of(sl);
    if (sb < 0)
        return;
    if (sl.map) {  // batched launch: this slot's buffers
        data += sb * sl.spec;
    }
    extern __shared__ char smem_raw[];
    cplx<T>  *A     = reinterpret_cast<cplx<T> *>(smem_raw);
    const int b0    = c0 + blockIdx.x * bc;
    const int ncols = (c1 - b0) < bc ? (c1 - b0) : bc, ld = ncols + 1;
    cplx<T>  *base  = data + (int64_t) blockIdx.y * ostride + b0;
    for (int w = threadIdx.x; w < L.n * ncols; w += blockDim.x) {
        const int i = w / ncols, c = w - i * ncols;
        A[i * ld + c] = base[i * sn + c];
    }
    __syncthreads();
    lds_stockham<T, INV>(A, L, tw, ncols, ld);
    for (int w = threadIdx.x; w < L.n * ncols; w += blockDim.x) {
        const int i     = w / ncols, c = w - i * ncols;
        base[i * sn + c] = A[i * ld + c];
    }
}

// ---- spectral <r, s> --------------------------------------------------------
// With s = -G * r, the unnormalised r2c / c2r pair and G holding 1/N,
// sum_x r(x) s(x) = sum over the full spectrum of conj(r^) s^ (Parseval); the
// half spectrum kz in [0, nz/2] counts the frequencies 0 < kz < nz/2 twice
// (their mirrors -kz are the complex conjugates) and kz = 0, nz/2 once.
__device__ __forceinline__ double kz_weight(int kz, int Mc) { return (kz == 0 || kz == Mc - 1) ? 1.0 : 2.0; }

constexpr int kXGreenGroup = 4;
// largest radix of the x pass: beyond 12 the pass of three components takes
// more than 168 registers (two waves per SIMD)
template <int H>
__host__ __device__ constexpr int kXGreenMaxRadix()
{
    return H == 3 ? 12 : 16;
}
// lane <- lane (quad base + S) for every lane of a quad (DPP quad_perm broadcast)
template <int S>
__device__ __forceinline__ double quad_bcast(double x)
{
    constexpr int ctrl = S * 0x55;
    const int     lo   = __builtin_amdgcn_mov_dpp(__double2loint(x), ctrl, 0xf, 0xf, true);
    const int     hi   = __builtin_amdgcn_mov_dpp(__double2hiint(x), ctrl, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
template <int S>
__device__ __forceinline__ float quad_bcast(float x)
{
    constexpr int ctrl = S * 0x55;
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), ctrl, 0xf, 0xf, true));
}

// component c of G r at stored block g with mirror signs sx, sy: for H = 3 the
// components of a frequency sit in the lanes 0..2 of a quad (lane 3 idle: c = 3
// computes a value nobody reads)
template <typename T, int H>
__device__ __forceinline__ cplx<T> green_row(const T *__restrict__ g, T sx, T sy, int c, const cplx<T> &a)
{
    if constexpr (H == 1) {
        return cscale(a, g[0]);
    } else {
        // row c of the packed symmetric 3x3 (00 01 02 11 12 22) with the mirror
        // signs of the xy (sx sy), xz (sx) and yz (sy) entries
        const int i1 = c == 0 ? 1 : (c == 1 ? 3 : 4), i2 = c == 0 ? 2 : (c == 1 ? 4 : 5), i0 = c < 2 ? c : 2;
        const T   s0 = c == 0 ? (T) 1 : (c == 1 ? sx * sy : sx);
        const T   s1 = c == 0 ? sx * sy : (c == 1 ? (T) 1 : sy);
        const T   s2 = c == 0 ? sx : (c == 1 ? sy : (T) 1);
        const T   ga = g[i0] * s0, gb = g[i1] * s1, gc = g[i2] * s2;
        const T   x0 = quad_bcast<0>(a.x), x1 = quad_bcast<1>(a.x), x2 = quad_bcast<2>(a.x);
        const T   y0 = quad_bcast<0>(a.y), y1 = quad_bcast<1>(a.y), y2 = quad_bcast<2>(a.y);
        return cplx<T>{ga * x0 + gb * x1 + gc * x2, ga * y0 + gb * y1 + gc * y2};
    }
}

// ---- x pass with the Green operator between forward and inverse ------------
// spectrum [x][y][kz][H]; logical block (bx, y) of the XCD-mapped 1-D grid (nbk
// ny blocks) owns kz in [kz_lo + bx*bk, ... + bk) and all H.
// G packed per frequency [x][y][kz][H(H+1)/2] = (00 01 02 11 12 22) or (0).
// partial (nullable): one partial of <r, s> (s = -G r) per block.
// FP64, lengths without a register kernel.  Bound by issue and latency: 240 VALU
// instructions per value at 125 points (half of them indices), 49 % of the issue slots
// at three waves per SIMD (a fourth would spill).  48^3 elastic 8.3 us (20.7 with
// Stockham stages and the Green product read back from LDS), 200 x 192 x 160
// conduction 44 (64), 96^3 elastic 18.5 (29).
template <typename T, int H>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_fft_x_green(cplx<T> *__restrict__ data, FftLen L,
                                                     const cplx<T> *__restrict__ tw, GreenView<T> gv, int kz_lo,
                                                     int kz_hi, int bk, int nbk, double *__restrict__ partial, Slots sl)
{
    const int sb = slot_of(sl);
    if (sb < 0)
        return;
    if (sl.map) {  // batched launch: this slot's buffers
        data += sb * sl.spec;
        gv.G += sb * sl.green;
        partial = slot_ptr(partial, sb * sl.part);
    }
    const int         ny = gv.ny, Mc = gv.Mc;
    __shared__ double red[8];
    double            acc = 0.0;
    extern __shared__ char smem_raw[];
    cplx<T>      *A  = reinterpret_cast<cplx<T> *>(smem_raw);
    const int     lb = xcd_tile_index(blockIdx.x, gridDim.x), yt = lb / nbk, bx = lb - yt * nbk;
    // ky and its mirror ny - ky read the same quarter-stored Green values: order
    // the rows 0, 1, ny-1, 2, ny-2, ... so that both run back to back on one XCD
    const int     y     = yt == 0 ? 0 : ((yt & 1) ? (yt + 1) >> 1 : ny - (yt >> 1));
    const int     kz0   = kz_lo + bx * bk;
    const int     nk    = (kz_hi - kz0) < bk ? (kz_hi - kz0) : bk;
    const int     ncols = nk * H, n = L.n;
    const int64_t sn    = (int64_t) ny * Mc * H;
    cplx<T>      *base  = data + ((int64_t) y * Mc + kz0) * H;
    const FastDiv nc(ncols);
    auto          from_mem = [&](int p, int c) { return base[p * sn + c]; };
    auto          to_mem   = [&](int p, int c, const cplx<T> &x) { base[p * sn + c] = x; };
    auto          from_lds = [&](int p, int c) { return A[p * ncols + c]; };
    auto          to_lds   = [&](int p, int c, const cplx<T> &x) { A[p * ncols + c] = x; };
    const bool    fy       = y >= gv.gyq;
    const T       sy       = fy ? (T) -1 : (T) 1;
    const int     kyq      = fy ? ny - y : y;
    // last forward stage, Green operator, first inverse stage on one column
    auto middle = [&](auto r, auto load, auto store) {
        constexpr int R = decltype(r)::value, HL = H == 3 ? 4 : 1;  // lanes per frequency
        const FastDiv dk(nk);
        const int     total = (n / R) * nk * HL, ds = n / R;
        for (int w = threadIdx.x; w < total; w += 256) {
            const int c = H == 3 ? w & 3 : 0;
            int       kk;
            const int q = dk(H == 3 ? w >> 2 : w, kk);
            const int col = kk * H + (c < H ? c : 0), kz = kz0 + kk;
            cplx<T>   v[R];
#pragma unroll
            for (int t = 0; t < R; ++t)
                v[t] = load(q * R + t, col);
            dft_reg<T, R, false>(v);
            const int    f  = block_frequency(L, q);
            const double wk = c < H ? kz_weight(kz, Mc) : 0.0;
#pragma unroll
            for (int k = 0; k < R; ++k) {
                // Green values of kXGreenGroup frequencies at a time: requested
                // all together they take the kernel past 256 registers
                if (k > 0 && k % kXGreenGroup == 0)
                    __builtin_amdgcn_sched_barrier(0);
                const int     kx = f + k * ds;
                const bool    fx = kx >= gv.gxq;
                const T      *g  = gv.G + (((int64_t) (fx ? gv.nx - kx : kx) * gv.gyq + kyq) * Mc + kz) * (H * (H + 1) / 2);
                const cplx<T> a  = v[k];
                v[k]             = green_row<T, H>(g, fx ? (T) -1 : (T) 1, sy, c, a);
                acc -= wk * ((double) a.x * v[k].x + (double) a.y * v[k].y);
            }
            dft_reg<T, R, true>(v);
            if (c < H)
#pragma unroll
                for (int t = 0; t < R; ++t)
                    store(q * R + t, col, v[t]);
        }
    };
    const int rl = L.rad[L.nst - 1];
    if (L.nst == 1) {
        with_prime(rl, [&](auto r) { middle(r, from_mem, to_mem); });
    } else {
        int m = n;
        with_radix<kXGreenMaxRadix<H>()>(L.rad[0],
                   [&](auto r) { dif_stage<T, decltype(r)::value, false>(n, m, nc, tw, L.tws, from_mem, to_lds); });
        m /= L.rad[0];
        __syncthreads();
        for (int s = 1; s < L.nst - 1; ++s) {
            with_radix<kXGreenMaxRadix<H>()>(L.rad[s],
                       [&](auto r) { dif_stage<T, decltype(r)::value, false>(n, m, nc, tw, L.tws, from_lds, to_lds); });
            m /= L.rad[s];
            __syncthreads();
        }
        with_radix<kXGreenMaxRadix<H>()>(rl, [&](auto r) { middle(r, from_lds, to_lds); });
        __syncthreads();
        for (int s = L.nst - 2; s > 0; --s) {
            m *= L.rad[s];
            with_radix<kXGreenMaxRadix<H>()>(L.rad[s],
                       [&](auto r) { dit_stage<T, decltype(r)::value>(n, m, nc, tw, L.tws, from_lds, to_lds); });
            __syncthreads();
        }
        with_radix<kXGreenMaxRadix<H>()>(L.rad[0], [&](auto r) { dit_stage<T, decltype(r)::value>(n, n, nc, tw, L.tws, from_lds, to_mem); });
    }
    if (partial) {
        double     v1[1] = {acc};
        const bool mx[1] = {false};
        block_reduce<1>(v1, mx, red);
        if (threadIdx.x == 0)
            partial[blockIdx.x] = v1[0];
    }
}

// stored block of frequency (kx, ky, kz) and the mirror signs sx, sy
template <typename T, int H>
__device__ __forceinline__ const T *green_at(const GreenView<T> &gv, int kx, int ky, int kz, T &sx, T &sy)
{
    const bool fx = kx >= gv.gxq, fy = ky >= gv.gyq;
    sx            = fx ? (T) -1 : (T) 1;
    sy            = fy ? (T) -1 : (T) 1;
    const int kxq = fx ? gv.nx - kx : kx, kyq = fy ? gv.ny - ky : ky;
    return gv.G + (((int64_t) kxq * gv.gyq + kyq) * gv.Mc + kz) * (H * (H + 1) / 2);
}

// FP32 x+Green pass, the whole tile through LDS; block (bx, y) = blockIdx.x, y;
// partial index blockIdx.y * gridDim.x + blockIdx.x
template <typename T, int H>
__global__ __launch_bounds__(256) void k_fft_x_green_stockham(cplx<T> *__restrict__ data, FftLen L,
                                                     const cplx<T> *__restrict__ tw, GreenView<T> gv, int kz_lo,
                                                     int kz_hi, int bk, double *__restrict__ partial, Slots sl)
{
    const int sb = slot_of(sl);
    if (sb < 0)
        return;
    if (sl.map) {  // batched launch: this slot's buffers
        data += sb * sl.spec;
        gv.G += sb * sl.green;
        partial = slot_ptr(partial, sb * sl.part);
    }
    const int ny = gv.ny, Mc = gv.Mc;
    __shared__ double red[8];
    double            acc = 0.0;
    extern __shared__ char smem_raw[];
    cplx<T>      *A     = reinterpret_cast<cplx<T> *>(smem_raw);
    const int     y     = blockIdx.y;
    const int     kz0   = kz_lo + blockIdx.x * bk;
    const int     nk    = (kz_hi - kz0) < bk ? (kz_hi - kz0) : bk;
    const int     ncols = nk * H, ld = ncols + 1;
    const int64_t sn    = (int64_t) ny * Mc * H;
    cplx<T>      *base  = data + ((int64_t) y * Mc + kz0) * H;
    for (int w = threadIdx.x; w < L.n * ncols; w += blockDim.x) {
        const int i = w / ncols, c = w - i * ncols;
        A[i * ld + c] = base[i * sn + c];
    }
    __syncthreads();
    lds_stockham<T, false>(A, L, tw, ncols, ld);
    for (int w = threadIdx.x; w < L.n * nk; w += blockDim.x) {
        const int i = w / nk, kk = w - i * nk;
        T         sx, sy;
        const T  *g = green_at<T, H>(gv, i, y, kz0 + kk, sx, sy);
        cplx<T>  *v = A + i * ld + kk * H;
        const double wk = kz_weight(kz0 + kk, Mc);
        if constexpr (H == 1) {
            const cplx<T> a = v[0];
            v[0]            = cscale(a, g[0]);
            acc -= wk * ((double) a.x * v[0].x + (double) a.y * v[0].y);
        } else {
            const cplx<T> a = v[0], b = v[1], c = v[2];
            const T       g00 = g[0], g01 = g[1] * sx * sy, g02 = g[2] * sx, g11 = g[3], g12 = g[4] * sy, g22 = g[5];
            v[0]                = cplx<T>{g00 * a.x + g01 * b.x + g02 * c.x, g00 * a.y + g01 * b.y + g02 * c.y};
            v[1]                = cplx<T>{g01 * a.x + g11 * b.x + g12 * c.x, g01 * a.y + g11 * b.y + g12 * c.y};
            v[2]                = cplx<T>{g02 * a.x + g12 * b.x + g22 * c.x, g02 * a.y + g12 * b.y + g22 * c.y};
            acc -= wk * ((double) a.x * v[0].x + (double) a.y * v[0].y + (double) b.x * v[1].x +
                         (double) b.y * v[1].y + (double) c.x * v[2].x + (double) c.y * v[2].y);
        }
    }
    __syncthreads();
    lds_stockham<T, true>(A, L, tw, ncols, ld);
    for (int w = threadIdx.x; w < L.n * ncols; w += blockDim.x) {
        const int i     = w / ncols, c = w - i * ncols;
        base[i * sn + c] = A[i * ld + c];
    }
    if (partial) {
        double     v1[1] = {acc};
        const bool mx[1] = {false};
        block_reduce<1>(v1, mx, red);
        if (threadIdx.x == 0)
            partial[blockIdx.y * gridDim.x + blockIdx.x] = v1[0];
    }
}

}  // namespace fans
