// Device scalars of the linear CG (include/solverCG.h:61-117) and their
// recurrences, shared by the reduction kernel and by the z passes that fold the
// partial sums themselves.
#pragma once
#include "common.h"

namespace fans {

// linear CG: search directions kept per iteration before the solution update
// u -= sum alpha_j d_j is applied in one pass
constexpr int kDirRing = 8;

// device scalar slots (double) -- layout shared with the host
enum {
    SC_BETA     = 0,
    SC_ALPHA    = 1,
    SC_DELTA    = 2,
    SC_DELTA0   = 3,  // delta of the previous iteration
    SC_DELTAMID = 4,
    SC_ERR      = 5,
    SC_ERR0     = 6,
    SC_DN       = 7,
    SC_TOL      = 8,
    SC_RES0     = 16,  // generic reduction results [16, 32)
    SC_ARING    = 32,  // linear CG: alpha of iteration j at SC_ARING + j % kDirRing
    SC_COUNT    = kScSlot
};

__device__ __forceinline__ double finish_norm(double v, int measure) { return measure == 1 ? sqrt(v) : v; }

// The scalars a reduction stage reads, loaded before its first store (the
// compiler cannot tell the stores to sc / is / hist from those loads, so it
// would keep each load behind the stores before it: one round trip each).
struct StageScalars {
    int    iter, errtype, nit;
    double delta, deltamid, beta, err0, tol;
};
__device__ __forceinline__ StageScalars load_stage_scalars(const double *sc, const int *is)
{
    return StageScalars{is[IS_ITER],     is[IS_ERRTYPE], is[IS_NIT], sc[SC_DELTA], sc[SC_DELTAMID],
                        sc[SC_BETA],     sc[SC_ERR0],    sc[SC_TOL]};
}

// the loop condition of solverCG.h:84 / solverFP.h:221 fails after iteration it
__device__ __forceinline__ bool cg_stop(const StageScalars &S, int it, double err)
{
    const double err_rel = it == 0 ? 100.0 : err / S.err0;
    const double e       = S.errtype == 0 ? err : err_rel;
    return !(it < S.nit && e > S.tol);
}
// records the error of iteration it and sets done on the stop test
__device__ __forceinline__ void record_error(double *sc, int *is, double *hist, const StageScalars &S, int it,
                                             double err)
{
    hist[it] = err;
    if (it == 0)
        sc[SC_ERR0] = err;
    sc[SC_ERR]  = err;
    is[IS_DONE] = cg_stop(S, it, err);
}

// alpha = delta / <d, K d> of an iteration and deltamid of the next one,
// <r - alpha K d, s> with s = d - beta d_prev (solverCG.h:87, 91 and 104):
// delta - alpha (<d, K d> - beta <K d_prev, d>), K symmetric
__device__ __forceinline__ double cg_alpha(double delta, double dn) { return delta / dn; }
__device__ __forceinline__ double cg_deltamid(double delta, double beta, double alpha, double dn, double dq)
{
    return delta - alpha * (dn - beta * dq);
}
__device__ __forceinline__ double cg_beta(double delta, double deltamid, double delta_prev)
{
    return fmax(0.0, (delta - deltamid) / delta_prev);
}

// ---- scalars folded by the z passes ------------------------------------------
// A reduction launch costs 4 to 5 us and the gap before it, three times per
// iteration, a quarter of the iteration at 48^3 (48^3 tangent 17.0 -> 14.3 ms
// without them, 32^3 conduction 4.38 -> 3.65, 96^3 elastic 5.71 -> 5.23).  While each producing kernel
// leaves at most kFoldMax partials (kFoldMax is in context.h), every workgroup of
// the consuming z pass sums them itself, in one fixed order, and its first
// workgroup stores the scalars:
//   z r2c of iteration j: alpha_(j-1) and deltamid from the matvec's and the
//     inverse z pass's partials; counts the iteration; SC_DELTA0 = delta_(j-1)
//   z c2r of iteration j: the error and the stop test from the forward z pass's
//     partials, then delta_j and beta_j from x+Green's
// No workgroup reads a scalar that its own launch stores (delta goes from
// SC_DELTA to SC_DELTA0 in one pass and back in the other), apart from the done
// flag, which every workgroup finds by itself.
struct CgFold {
    const double *p0 = nullptr, *p1 = nullptr;  // partials: r2c <d, K d>, <d, K d_prev>; c2r norm, <r, s>
    int           n0 = 0, n1 = 0;               // their counts
    double       *sc   = nullptr;
    int          *is   = nullptr;
    double       *hist = nullptr;
    int           measure = 0;
};
__device__ __forceinline__ void slot_fold(CgFold &f, int sb, const Slots &sl)
{
    f.p0   = slot_ptr(f.p0, sb * sl.part);
    f.p1   = slot_ptr(f.p1, sb * sl.part);
    f.sc   = slot_ptr(f.sc, (int64_t) sb * SC_COUNT);
    f.is   = slot_ptr(f.is, (int64_t) sb * IS_COUNT);
    f.hist = slot_ptr(f.hist, sb * sl.hist);
}
// this thread's share of n partials, kFoldLoads of them requested together
// (indices past the end read the last one and count as zero: a conditional load
// would wait for the one before it)
constexpr int kFoldLoads = 8;
template <int NT>
__device__ __forceinline__ double fold_partials(const double *__restrict__ p, int n, bool mx)
{
    double a = 0.0;
    for (int b = threadIdx.x; b < n; b += kFoldLoads * NT) {
        double x[kFoldLoads];
#pragma unroll
        for (int j = 0; j < kFoldLoads; ++j)
            x[j] = p[min(b + j * NT, n - 1)];
#pragma unroll
        for (int j = 0; j < kFoldLoads; ++j) {
            const double y = b + j * NT < n ? x[j] : 0.0;
            a              = mx ? fmax(a, y) : a + y;
        }
    }
    return a;
}
// block-wide results of two folded quantities in every thread; sm: 2 per wave
// (a last wave of fewer lanes: the shuffles read zeros from the missing ones)
template <int NT>
__device__ __forceinline__ void fold_block(double &v0, double &v1, bool mx0, double *sm)
{
    constexpr int NW = (NT + 63) / 64;
    const double  w0 = mx0 ? wave_max(v0) : wave_sum(v0), w1 = wave_sum(v1);
    if ((threadIdx.x & 63) == 0) {
        sm[threadIdx.x >> 6]      = w0;
        sm[NW + (threadIdx.x >> 6)] = w1;
    }
    __syncthreads();
    v0 = sm[0], v1 = sm[NW];
    for (int w = 1; w < NW; ++w) {
        v0 = mx0 ? fmax(v0, sm[w]) : v0 + sm[w];
        v1 += sm[NW + w];
    }
}

// z r2c: alpha of the previous iteration
template <int NT>
__device__ __forceinline__ double fold_alpha(const CgFold &f, double *sm)
{
    double       v0 = fold_partials<NT>(f.p0, f.n0, false), v1 = fold_partials<NT>(f.p1, f.n1, false);
    const double delta = f.sc[SC_DELTA], beta = f.sc[SC_BETA];
    fold_block<NT>(v0, v1, false, sm);
    const double alpha = cg_alpha(delta, v0);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const int it = f.is[IS_ITER];
        f.is[IS_ITER]                    = it + 1;
        f.sc[SC_DN]                      = v0;
        f.sc[SC_ALPHA]                   = alpha;
        f.sc[SC_ARING + it % kDirRing]   = alpha;
        f.sc[SC_DELTA0]                  = delta;
        f.sc[SC_DELTAMID]                = cg_deltamid(delta, beta, alpha, v0, v1);
    }
    return alpha;
}

// z c2r: this thread's shares and the scalars, requested at the kernel's start
struct FoldBeta {
    double       v0, v1, delta_prev, deltamid;
    StageScalars S;
    template <int NT>
    __device__ __forceinline__ void load(const CgFold &f)
    {
        v0         = fold_partials<NT>(f.p0, f.n0, f.measure == 2);
        v1         = fold_partials<NT>(f.p1, f.n1, false);
        delta_prev = f.sc[SC_DELTA0];
        deltamid   = f.sc[SC_DELTAMID];
        S          = load_stage_scalars(f.sc, f.is);
    }
    // beta of the iteration; false: the stop test holds and nothing is to be done
    template <int NT>
    __device__ __forceinline__ bool finish(const CgFold &f, double *sm, double &beta)
    {
        fold_block<NT>(v0, v1, f.measure == 2, sm);
        const bool first = blockIdx.x == 0 && threadIdx.x == 0;
        if (f.n0) {
            const double err = finish_norm(v0, f.measure);
            if (first)
                record_error(f.sc, f.is, f.hist, S, S.iter, err);
            if (cg_stop(S, S.iter, err))
                return false;
        }
        beta = cg_beta(v1, deltamid, delta_prev);
        if (first) {
            f.sc[SC_DELTA] = v1;
            f.sc[SC_BETA]  = beta;
        }
        return true;
    }
};

}  // namespace fans
