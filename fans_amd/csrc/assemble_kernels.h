// Residual assembly kernels (Solver::compute_residual_basic, solver.h:228-270,
// and the linear CG matvec of solverCG.h:94-105) for the periodic voxel grid.
//
// Both kernels march along x.  A workgroup of 256 threads owns a 16x16 (y,z)
// tile of elements (one element per thread, lanes ordered z-fastest so one
// wave holds 4 rows of 16) and emits the 15x15 nodes whose four surrounding
// elements of the current plane lie in the tile; every
// node is produced by exactly one thread in a fixed summation order, so results
// are deterministic and atomic-free.
//
// k_assemble_modal (linear materials, FP64 form): works on Walsh coefficients.  Per x
// plane each thread reads the four nodes of its y-z cell from LDS, takes their
// 2-D Walsh coefficients, and combines them with the previous plane's, kept in
// registers, to the element's 3-D coefficients; the element maps these to force
// coefficients (modal_*), whose x half goes into this plane and the next one's
// carry, and one inverse y-z transform per plane gives the corner forces.
// Against transforming all eight corners of every element this halves the LDS
// reads (24 -> 9 words per component triple), the z (DPP) and y (shuffle)
// exchanges, and takes 36 instead of about 56 additions per component.
//
// k_assemble (nonlinear models: per-Gauss-point constitutive path; linear ones in
// the mixed form, see element_forces_iso3_modal).  Per plane:
//   1. the 17x17 node plane x+1 is staged in LDS;
//   2. each thread gathers its 8 corners from LDS and computes its element;
//   3. corner forces are combined along z with DPP row_shr (in registers),
//      along y with a 16-lane shuffle (LDS only for the wave-boundary row),
//      and along x by a register carry into the next plane.
#pragma once
#include <type_traits>
#include "element_kernels.h"

namespace fans {

enum { ASM_RESID = 0, ASM_CGLIN = 1 };
constexpr int TILE = 16;  // element tile edge (y and z)
constexpr int NOUT = TILE - 1;

template <typename T>
struct AsmArgs {
    int             nx, ny, nz;
    int             cx;        // x planes per block
    int             nty, ntz;  // number of tiles in y, z
    Geom            geom;
    const uint8_t  *ms;        // phase ids [x][y][z]
    int             ms16;      // 16-bit phase ids (phase_id)
    const Phase<T> *phases;
    int             nphases;
    J2State         js;
    // ASM_RESID: in = u, out = r; norm/dot partials
    // ASM_CGLIN: in = d, out = rnew = K d; partial <d, rnew>
    const T        *in;
    T              *out;
    const T        *dotv;      // ASM_RESID optional: partial <out, dotv>
    const T        *g0;        // macroscopic gradient (n_str), device
    // ASM_RESID: [2][blocks], norm and dot; ASM_CGLIN: one dot per `grp` planes
    // and tile, [ceil(nx / grp)][tiles] (cx a multiple of grp)
    double         *partial;
    int             grp;
    int             measure;   // 0 L1, 1 L2, 2 Linf  (ASM_RESID)
    Slots           sl;        // RVE slots (done flags: finished slots return at entry)
    const T        *vk;        // per-voxel isotropic moduli (nullable, isotropic variants only):
    const T        *vg;        // bulk K and shear G, or conductivity k in vk
};

template <typename T, int H>
__device__ __forceinline__ T shfl_up16(T v)
{
    return __shfl_up(v, 16, 64);
}

// k_assemble_modal: ASM_ISO = every phase LinearElasticIsotropic (H=3) or
// LinearThermalIsotropic (H=1); ASM_ISO_CUBIC = the same on cubic voxels;
// ASM_ANISO = any linear models, the phase table holding full tensors.
// k_assemble: the isotropic two in the mixed form; ASM_GENERAL = small strain; ASM_LARGE = finite strain (F and P,
// n_str 9); ASM_GENERAL_PNL = ASM_GENERAL with power-law PseudoPlastic phases
// present; ASM_GENERAL_VISCO = ASM_GENERAL with J2ViscoPlastic phases present
// (their per-call psi / psi_bar update, see PointModel).
enum { ASM_GENERAL = 0, ASM_ISO = 1, ASM_ISO_CUBIC = 2, ASM_LARGE = 3, ASM_GENERAL_PNL = 4, ASM_GENERAL_VISCO = 5,
       ASM_ANISO = 6 };

// The per-Gauss-point FP64 residual lands just above 256 registers (one wave
// per SIMD) unless asked for two waves, which it reaches without spilling; the
// finite-strain, power-law and visco-plastic residuals and the FP64
// per-Gauss-point linear matvec would spill there, so they keep one.  The FP64
// isotropic matvec takes 132 registers (three waves per SIMD); the FP32 one fits 84
// (six), with GRP 96 (five: 256^3 184 us; at six it spills, 224; without GRP 163).
template <typename T, int MODE, int VAR, bool GRP>
constexpr int kAsmWaves()
{
    if (VAR == ASM_LARGE || VAR == ASM_GENERAL_PNL || VAR == ASM_GENERAL_VISCO ||
        (VAR == ASM_GENERAL && MODE == ASM_CGLIN && sizeof(T) == 8))
        return 1;
    if ((VAR == ASM_ISO || VAR == ASM_ISO_CUBIC) && MODE == ASM_CGLIN)
        return sizeof(T) == 8 ? 3 : GRP ? 5 : 6;
    return 2;
}

// the workgroup's buffers moved to its RVE slot
template <typename T, int H>
__device__ __forceinline__ void slot_asm(AsmArgs<T> &a, int sb)
{
    a.in      = a.in + sb * a.sl.field;
    a.out     = a.out + sb * a.sl.field;
    a.dotv    = slot_ptr(a.dotv, sb * a.sl.field);
    a.g0      = slot_ptr(a.g0, (int64_t) sb * 9);
    a.ms      = a.ms + sb * a.sl.ms;
    a.phases  = a.phases + sb * a.sl.ph;
    a.partial = slot_ptr(a.partial, sb * a.sl.part);
    a.vk      = slot_ptr(a.vk, sb * (a.sl.field / H));
    a.vg      = slot_ptr(a.vg, sb * (a.sl.field / H));
}

// waves per SIMD asked of k_assemble_modal
template <int H, int VAR>
constexpr int kModalWaves()
{
    return VAR == ASM_ANISO ? 2 : H == 1 ? 5 : 3;
}

// phases whose moduli (ASM_ANISO: tensors, in dynamic LDS) are staged per
// workgroup
constexpr int kStagedPhases = 256;
template <typename T, int H>
constexpr int kTensorLen()
{
    return H == 1 ? 9 : 21;
}

// one wave's request of SIZE bytes per lane from global memory straight to LDS:
// lane l writes a word at lds + 4 l.  Tracked by vmcnt like a load, in issue order.
template <int SIZE>
__device__ __forceinline__ void load_to_lds(const void *src, void *lds)
{
    static_assert(SIZE == 1 || SIZE == 2 || SIZE == 4, "sizes of the instruction used here");
    const auto s = (const __attribute__((address_space(1))) void *) src;
    const auto d = (__attribute__((address_space(3))) void *) lds;
    if constexpr (SIZE == 1)  // one byte (two) per lane, a zero-extended word in LDS
        __builtin_amdgcn_global_load_lds(s, d, 1, 0, 0);
    else if constexpr (SIZE == 2)
        __builtin_amdgcn_global_load_lds(s, d, 2, 0, 0);
    else
        __builtin_amdgcn_global_load_lds(s, d, 4, 0, 0);
}

// workgroup barrier that leaves up to N of the wave's own latest requests (and
// stores) in flight; every LDS access of the wave is done
template <int N>
__device__ __forceinline__ void barrier_keep()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// the H values of a node in as few stores as their alignment allows (one store
// per value cost 20 us more at 256^3)
template <typename T, int H>
__device__ __forceinline__ void store_node(T *p, const T (&v)[H])
{
    if constexpr (H == 3) {
        typedef double d2 __attribute__((ext_vector_type(2), aligned(8)));
        *reinterpret_cast<d2 *>(p) = d2{v[0], v[1]};
        p[2]                       = v[2];
    } else {
        p[0] = v[0];
    }
}

// where k_assemble_modal finds an element's material: the staged table (byte
// ids), the phase table in memory, or the voxel's own moduli (isotropic only)
enum { MAT_STAGED = 0, MAT_TABLE = 1, MAT_VOXEL = 2 };

// A staged node plane of k_assemble_modal: NL x NL nodes in words, requested by FULL
// instructions of the four waves and one of REST lanes each.
template <typename T, int H>
struct ModalPlane {
    static constexpr int NL = TILE + 1, NBUF = 4;
    static constexpr int UPN = H * (int) sizeof(T) / 4, UNITS = NL * NL * UPN;
    static constexpr int FULL = UNITS / 256, REST = (UNITS - 256 * FULL + 3) / 4, NREQ = FULL + 1;
    static_assert(REST > 0 && REST <= 64, "units of the last request");
    static constexpr int PLANE = (256 * FULL + 4 * REST) * 4 / (int) sizeof(T);
};
// a bound on the static LDS of the kernel's ASM_ANISO variants: planes, ids, y
// exchange and the small arrays
template <typename T, int H>
constexpr size_t modal_static_lds()
{
    using MP = ModalPlane<T, H>;
    return MP::NBUF * (MP::PLANE * sizeof(T) + 1024) + 2 * TILE * TILE * H * sizeof(T) + 1024;
}

// Node planes are requested three ahead, straight into four LDS buffers: two
// planes of each resident workgroup are in flight at any time, without
// registers, and one barrier per plane separates them (it waits for the requests
// of two iterations ago only).  The loop is unrolled over the buffers.
//
// What bounds it: a wave issues 185 VALU instructions per plane (156 of them
// FP64 arithmetic); without its stores and requests the 256^3 FP64 matvec takes
// 0.17 ms, with them 0.26 (0.34 before: eight-corner transforms, two barriers,
// register prefetch by one plane).  Three waves per SIMD at 156 registers.  At 48^3 and 64^3 a plane of
// a workgroup alone on its CU takes 0.8 us (1.4 before).
template <typename T, int H, int NGP, int MODE, int VAR, int MAT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kModalWaves<H, VAR>())))
void k_assemble_modal(AsmArgs<T> a)
{
    static_assert(sizeof(T) == 8, "the FP64 form's kernel");
    constexpr bool CUBIC = VAR == ASM_ISO_CUBIC, ANISO = VAR == ASM_ANISO, RES = MODE == ASM_RESID;
    static_assert(!(ANISO && MAT == MAT_VOXEL), "per-voxel moduli are isotropic");
    const int sb = slot_of(a.sl);
    if (sb < 0)
        return;
    if (a.sl.map)  // batched launch: this slot's buffers
        slot_asm<T, H>(a, sb);
    using MP         = ModalPlane<T, H>;
    constexpr int NS = H == 1 ? 3 : 6, NL = MP::NL, NBUF = MP::NBUF, UPN = MP::UPN;
    constexpr int FULL = MP::FULL, REST = MP::REST, NREQ = MP::NREQ;
    // words of an element plane's material request
    constexpr int WPT  = (int) sizeof(T) / 4, NMOD = MAT == MAT_VOXEL ? (H == 3 ? 2 : 1) * WPT : 1;
    constexpr int KEEP = NREQ + NMOD;  // requests of one plane
    __shared__ __align__(16) T   Un[NBUF][MP::PLANE];
    __shared__ __align__(16) int Mt[NBUF][NMOD][256];
    __shared__ T                 Yb[2][TILE * TILE * H];  // y exchange
    __shared__ double            red[8];
    extern __shared__ __align__(16) char dyn_lds[];

    const int t = threadIdx.x, ey = t / TILE, ez = t - ey * TILE;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const int bid  = xcd_tile_index(blockIdx.x, gridDim.x), ntile = a.nty * a.ntz;
    const int bx = bid / ntile, tile = bid - bx * ntile, ty = tile / a.ntz, tz = tile - ty * a.ntz;
    const int Y0 = ty * NOUT, Z0 = tz * NOUT, X0 = bx * a.cx;
    const int X1 = min(X0 + a.cx, a.nx);
    const int ny = a.ny, nz = a.nz, nx = a.nx;

    // periodic node index of tile position v (several wraps on grids below 16)
    auto wrap = [&](int v, int n) {
        v += v < 0 ? n : 0;
        return n <= TILE ? v % n : (v >= n ? v - n : v);
    };
    auto wrapy = [&](int v) { return wrap(Y0 - 1 + v, ny); };
    auto wrapz = [&](int v) { return wrap(Z0 - 1 + v, nz); };
    const bool own_yz = ey >= 1 && ez >= 1 && Y0 - 1 + ey < ny && Z0 - 1 + ez < nz;
    // per-thread offsets within a plane are 32-bit; the plane's base is the same
    // for the whole workgroup (scalar registers)
    const int64_t  plane   = (int64_t) ny * nz, plane_b = plane * H * (int) sizeof(T);
    const unsigned off_own = (unsigned) (wrapy(ey) * nz + wrapz(ez));
    unsigned       off_req[NREQ];  // bytes
#pragma unroll
    for (int q = 0; q < NREQ; ++q) {
        const int u = min(q < FULL ? 256 * q + t : 256 * FULL + wave * REST + lane, MP::UNITS - 1), n = u / UPN;
        off_req[q]  = ((unsigned) (wrapy(n / NL) * nz + wrapz(n % NL)) * UPN + u % UPN) * 4;
    }

    const T w = (T) a.geom.w;
    // the residual's macroscopic shift (modal_*), read from LDS where it is used
    __shared__ T sh[NS];
    if constexpr (RES) {
        const T f = CUBIC ? (T) 4 / (T) a.geom.ilx : (T) 4;
        if (t < NS)  // shear sums: sqrt(2) times the Mandel entries
            sh[t] = t < 3 ? f * a.g0[t] : f * (T) (2.0 * kSqrtHalf) * a.g0[t];
    }
    // the phase table of byte ids, times the Gauss weight: moduli, or (ANISO, in
    // dynamic LDS) tensors
    __shared__ T PL[MAT == MAT_STAGED && !ANISO ? kStagedPhases : 1][2];
    T *const     CT = reinterpret_cast<T *>(dyn_lds);
    constexpr int NT = kTensorLen<T, H>();
    if constexpr (MAT == MAT_STAGED) {
        const int np = min(a.nphases, kStagedPhases);
        if constexpr (ANISO) {
            for (int e = t; e < np * NT; e += 256)
                CT[e] = modal_tensor_entry<T, H, NGP>(a.phases[e / NT].p, e % NT, w);
        } else {
            for (int p = t; p < np; p += 256) {
                PL[p][0] = a.phases[p].p[0] * w;
                PL[p][1] = H == 3 ? a.phases[p].p[1] * w : (T) 0;
            }
        }
    }

    // request the next node plane xq into buffer BUF, and the materials of the
    // element plane below it (except for the first)
    int         xq  = X0 == 0 ? nx - 1 : X0 - 1, xm = 0;
    const char *nsrc = reinterpret_cast<const char *>(a.in) + xq * plane_b;
    int64_t     mofs = 0;
    auto        request = [&](auto bufc, auto matc) {
        constexpr int BUF = decltype(bufc)::value;
#pragma unroll
        for (int q = 0; q < FULL; ++q)
            load_to_lds<4>(nsrc + off_req[q], reinterpret_cast<char *>(Un[BUF]) + (256 * q + 64 * wave) * 4);
        if (lane < REST)
            load_to_lds<4>(nsrc + off_req[FULL],
                           reinterpret_cast<char *>(Un[BUF]) + (256 * FULL + wave * REST) * 4);
        if constexpr (decltype(matc)::value) {
            constexpr int MB = (BUF + NBUF - 1) % NBUF;
            if constexpr (MAT == MAT_VOXEL) {
#pragma unroll
                for (int q = 0; q < NMOD; ++q)
                    load_to_lds<4>(reinterpret_cast<const char *>(q < WPT ? a.vk + mofs : a.vg + mofs) +
                                              (off_own * (unsigned) sizeof(T) + 4 * (q % WPT)),
                                          &Mt[MB][q][64 * wave]);
            } else if (MAT == MAT_TABLE && a.ms16) {
                load_to_lds<2>(reinterpret_cast<const uint16_t *>(a.ms) + mofs + off_own, &Mt[MB][0][64 * wave]);
            } else {
                load_to_lds<1>(a.ms + mofs + off_own, &Mt[MB][0][64 * wave]);
            }
        }
        mofs = xq * plane;
        nsrc += plane_b;
        if (++xq == nx) {
            xq   = 0;
            nsrc = reinterpret_cast<const char *>(a.in);
        }
    };
    // 2-D Walsh coefficients of this thread's y-z cell of a staged plane (1, y,
    // z, yz)
    auto cell_walsh = [&](const T *src, T(&q)[4][H]) {
#pragma unroll
        for (int c = 0; c < H; ++c) {
            const T u0 = src[c], u1 = src[NL * H + c], u2 = src[H + c], u3 = src[(NL + 1) * H + c];
            const T s0 = u0 + u1, d0 = u0 - u1, s1 = u2 + u3, d1 = u2 - u3;
            q[0][c] = s0 + s1;
            q[1][c] = d0 + d1;
            q[2][c] = s0 - s1;
            q[3][c] = d0 - d1;
        }
    };

    // node plane X0 - 1 + i sits in buffer i % NBUF, the material of the element
    // plane above it likewise
    const int own = (ey * NL + ez) * H;
    T         qp[4][H], carry[4][H];
    double    acc0 = 0.0, acc1 = 0.0;
    request(std::integral_constant<int, 0>{}, std::false_type{});
    request(std::integral_constant<int, 1>{}, std::true_type{});
    barrier_keep<0>();
    request(std::integral_constant<int, 2>{}, std::true_type{});
    if (X0 + 2 <= X1)
        request(std::integral_constant<int, 3>{}, std::true_type{});
    cell_walsh(&Un[0][own], qp);
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int c = 0; c < H; ++c)
            carry[n][c] = (T) 0;
    int      xe   = X0 - 1;             // element plane between node planes xe and xe + 1
    int      left = RES ? 0 : a.grp + 1;  // planes to the next partial
    T       *dst  = a.out + (int64_t) (X0 - 1) * plane * H;
    const T *dot  = RES && a.dotv ? a.dotv + (int64_t) (X0 - 1) * plane * H : nullptr;
    double  *part = RES ? nullptr : a.partial + (int64_t) (X0 / a.grp) * ntile + tile;
    auto     step = [&](auto bc) {
        constexpr int B = decltype(bc)::value;  // iteration % NBUF
        T             wc[8][H], b[8][H];
        {
            T qc[4][H];
            cell_walsh(&Un[(B + 1) % NBUF][own], qc);
#pragma unroll
            for (int c = 0; c < H; ++c) {
                wc[1][c] = qp[0][c] - qc[0][c];
#pragma unroll
                for (int n = 1; n < 4; ++n) {
                    wc[2 * n][c]     = qp[n][c] + qc[n][c];
                    wc[2 * n + 1][c] = qp[n][c] - qc[n][c];
                }
#pragma unroll
                for (int n = 0; n < 4; ++n)
                    qp[n][c] = qc[n][c];
            }
        }
        const int *mt = &Mt[B][0][t];
        if constexpr (ANISO) {
            if constexpr (MAT == MAT_STAGED) {
                modal_aniso<T, H, NGP, RES>(wc, a.geom, CT + mt[0] * NT, sh, b);
            } else {
                T C[NT];
#pragma unroll
                for (int e = 0; e < NT; ++e)
                    C[e] = modal_tensor_entry<T, H, NGP>(a.phases[mt[0]].p, e, w);
                modal_aniso<T, H, NGP, RES>(wc, a.geom, C, sh, b);
            }
        } else {
            T lw, mw = (T) 0;
            if constexpr (MAT == MAT_VOXEL) {  // bulk and shear modulus -> lambda, mu
                lw = staged_value<T>(mt) * w;
                if constexpr (H == 3) {
                    mw = staged_value<T>(mt + 256 * WPT) * w;
                    lw -= (T) (2.0 / 3.0) * mw;
                }
            } else if constexpr (MAT == MAT_STAGED) {
                lw = PL[mt[0]][0];
                mw = PL[mt[0]][1];
            } else {
                lw = a.phases[mt[0]].p[0] * w;
                mw = H == 3 ? a.phases[mt[0]].p[1] * w : (T) 0;
            }
            if constexpr (H == 3)
                modal_iso3<T, NGP, CUBIC, RES>(wc, a.geom, lw, mw, sh, b);
            else
                modal_iso1<T, NGP, CUBIC, RES>(wc, a.geom, lw, sh, b);
        }
        if constexpr (NGP == 1)
#pragma unroll
            for (int c = 0; c < H; ++c)
                b[3][c] = b[5][c] = b[6][c] = b[7][c] = (T) 0;
        T P0[H], dv[H];
#pragma unroll
        for (int c = 0; c < H; ++c) {
            // x transform: this plane's force coefficients and the next one's
            const T t0 = carry[0][c] + b[1][c], t1 = carry[1][c] + (b[2][c] + b[3][c]);
            const T t2 = carry[2][c] + (b[4][c] + b[5][c]), t3 = carry[3][c] + (b[6][c] + b[7][c]);
            carry[0][c] = -b[1][c];
            carry[1][c] = b[2][c] - b[3][c];
            carry[2][c] = b[4][c] - b[5][c];
            carry[3][c] = b[6][c] - b[7][c];
            // y-z transform, z combined: node (., ez) <- az = 0 corners of this
            // element + az = 1 corners of element ez - 1; rows ey and ey + 1
            const T s0 = t0 + t1, d0 = t0 - t1, s1 = t2 + t3, d1 = t2 - t3;
            P0[c]              = (s0 + s1) + dpp_row_shr1(s0 - s1);
            Yb[B & 1][t * H + c] = (d0 + d1) + dpp_row_shr1(d0 - d1);
            if constexpr (!RES)
                dv[c] = Un[B][own + c];  // own node of plane xe
        }
        // after it: plane xe + 2 is staged, and no thread reads plane xe any more
        if (xe + 3 <= X1)
            barrier_keep<KEEP>();
        else
            barrier_keep<0>();
        if (xe >= X0 && own_yz) {
            T res[H];
#pragma unroll
            for (int c = 0; c < H; ++c) {
                // y: row ey's own part + row (ey - 1)'s
                res[c] = P0[c] + Yb[B & 1][(t - TILE) * H + c];
                if constexpr (!RES) {
                    acc0 += (double) dv[c] * (double) res[c];
                } else {
                    acc_norm(acc0, res[c], a.measure);
                    if (dot)
                        acc1 += (double) res[c] * (double) dot[off_own * H + c];
                }
            }
            store_node<T, H>(dst + off_own * H, res);
        }
        if (xe + 4 <= X1)
            request(bc, std::true_type{});
        ++xe;
        dst += plane * H;
        if constexpr (!RES) {
            // one partial per grp planes, the same for every cx
            if (--left == 0 || xe == X1) {
                double     v[1]  = {acc0};
                const bool mx[1] = {false};
                block_reduce<1>(v, mx, red);
                if (t == 0)
                    *part = v[0];
                part += ntile;
                acc0 = 0.0;
                left = a.grp;
            }
        } else if (dot) {
            dot += plane * H;
        }
        return xe < X1;
    };
    while (step(std::integral_constant<int, 0>{}) && step(std::integral_constant<int, 1>{}) &&
           step(std::integral_constant<int, 2>{}) && step(std::integral_constant<int, 3>{}))
        ;
    if constexpr (RES) {
        if (a.partial) {
            double     v[2]  = {acc0, acc1};
            const bool mx[2] = {a.measure == 2, false};
            block_reduce<2>(v, mx, red);
            if (t == 0) {
                a.partial[blockIdx.x]             = v[0];
                a.partial[gridDim.x + blockIdx.x] = v[1];
            }
        }
    }
}

// GRP (matvec): one partial per a.grp planes instead of one per workgroup, for
// workgroups of several times a.grp planes
template <typename T, int H, int NGP, int MODE, int VAR, bool GRP = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kAsmWaves<T, MODE, VAR, GRP>()))) void k_assemble(AsmArgs<T> a)
{
    constexpr bool ISO = VAR == ASM_ISO || VAR == ASM_ISO_CUBIC, CUBIC = VAR == ASM_ISO_CUBIC;
    const int sb = slot_of(a.sl);
    if (sb < 0)
        return;
    if (a.sl.map)  // batched launch: this slot's buffers
        slot_asm<T, H>(a, sb);
    constexpr int NL = TILE + 1;  // node tile edge
    constexpr int NS = nstr_of<H, VAR == ASM_LARGE>();
    __shared__ T      Un[2][NL * NL * H];
    __shared__ T      Yb[4][TILE * 2 * H];  // last row of each wave for the y exchange
    __shared__ double red[8];

    const int t = threadIdx.x, ey = t / TILE, ez = t - ey * TILE;
    const int wave = t >> 6, lane = t & 63;
    int       bid  = xcd_tile_index(blockIdx.x, gridDim.x);
    const int tz   = bid % a.ntz;
    bid /= a.ntz;
    const int     ty = bid % a.nty;
    const int     bx = bid / a.nty;
    const int     Y0 = ty * NOUT, Z0 = tz * NOUT, X0 = bx * a.cx;
    const int     X1 = min(X0 + a.cx, a.nx);
    const int     ny = a.ny, nz = a.nz, nx = a.nx;
    const int64_t plane = (int64_t) ny * nz;

    // periodic node index of tile position v (several wraps on grids below 16)
    auto wrapy = [&](int v) { return ((Y0 - 1 + v) % ny + ny) % ny; };
    auto wrapz = [&](int v) { return ((Z0 - 1 + v) % nz + nz) % nz; };
    const int  my_y   = Y0 - 1 + ey, my_z = Z0 - 1 + ez;
    const bool own_yz = ey >= 1 && ez >= 1 && my_y < ny && my_z < nz;
    // node-plane slots of this thread: its own node (ey, ez) and, for 33 threads
    // spread over the waves, one of the extra row/column 16 nodes
    const int  ext    = (t % 7 == 0 && t / 7 < 2 * NL - 1) ? t / 7 : -1;
    const int  e_a    = ext < 0 ? 0 : (ext < NL ? TILE : ext - NL);
    const int  e_b    = ext < 0 ? 0 : (ext < NL ? ext : TILE);
    const int64_t off_own = (int64_t) wrapy(ey) * nz + wrapz(ez);
    const int64_t off_ext = (int64_t) wrapy(e_a) * nz + wrapz(e_b);
    // J2 state slot of this thread's element within an x plane of the state
    // layout: the tile's 16 slots are its 16 element columns in z
    static_assert(NOUT == kStateTile && TILE == 16, "the J2 state layout follows the stencil tiles");
    const int64_t splane = (int64_t) ny * a.ntz * 16;
    const int64_t sl_own = ((int64_t) wrapy(ey) * a.ntz + tz) * 16 + ez;
    // elements next to an owned node; the others (rows of the last tile past
    // the grid edge when 15 does not divide it) only feed unowned sums
    const bool el_needed = Y0 - 1 + max(ey, 1) < ny && Z0 - 1 + max(ez, 1) < nz;

    T      carry[H];
    double acc0 = 0.0, acc1 = 0.0;
#pragma unroll
    for (int c = 0; c < H; ++c)
        carry[c] = (T) 0;
    T g0[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i)
        g0[i] = (MODE == ASM_RESID) ? a.g0[i] : (T) 0;
    const T w = (T) a.geom.w;
    // isotropic moduli of the first 256 phases, staged once per block (ids
    // beyond read the phase table)
    __shared__ T PL[256][2];
    if constexpr (ISO) {
        for (int p = t; p < min(a.nphases, 256); p += blockDim.x) {
            PL[p][0] = a.phases[p].p[0];
            PL[p][1] = H == 3 ? a.phases[p].p[1] : (T) 0;
        }
    }
    // per-Gauss-point residual: model kind of the first 256 phases, staged once
    // per block
    constexpr bool PM = !ISO && VAR != ASM_LARGE && MODE == ASM_RESID;
    __shared__ int PK[PM ? 256 : 1];
    if constexpr (PM)
        for (int p = t; p < min(a.nphases, 256); p += blockDim.x)
            PK[p] = a.phases[p].kind;
    auto kind_of = [&](int ph) { return ph < 256 ? PK[ph] : a.phases[ph].kind; };

    // node plane x+1: fetch (global) then commit (LDS); the phase id of the
    // next element plane is loaded one plane ahead.  Addresses are a
    // per-thread base (loop invariant) plus a per-plane offset that is the
    // same for the whole workgroup (scalar arithmetic).
    const int64_t planeH = plane * H;
    const T *const in_own = a.in + off_own * H, *const in_ext = a.in + off_ext * H;
    T    pf_own[H], pf_ext[H];
    auto fetch_plane = [&](int xp) {
        const int     xg = xp < 0 ? xp + nx : (xp >= nx ? xp - nx : xp);
        const int64_t po = xg * planeH;
#pragma unroll
        for (int c = 0; c < H; ++c)
            pf_own[c] = in_own[po + c];
        if (ext >= 0)
#pragma unroll
            for (int c = 0; c < H; ++c)
                pf_ext[c] = in_ext[po + c];
    };
    auto commit_plane = [&](int buf) {
#pragma unroll
        for (int c = 0; c < H; ++c)
            Un[buf][(ey * NL + ez) * H + c] = pf_own[c];
        if (ext >= 0)
#pragma unroll
            for (int c = 0; c < H; ++c)
                Un[buf][(e_a * NL + e_b) * H + c] = pf_ext[c];
    };
    const uint8_t *const ms_own = a.ms + (a.ms16 ? 2 : 1) * off_own;
    auto phase_of = [&](int xe) {
        const int xg = xe < 0 ? xe + nx : xe;
        return phase_id(ms_own, a.ms16, xg * plane);
    };

    fetch_plane(X0 - 1);
    commit_plane(0);
    fetch_plane(X0);
    int                   ph_next = phase_of(X0 - 1);
    PointModel<T, H, NGP, VAR == ASM_GENERAL_PNL || VAR == ASM_GENERAL_VISCO, VAR == ASM_GENERAL_VISCO> pm;
    bool pm_pre = false;  // point 0 of the coming element requested
    int           left = a.grp;
    double       *part = GRP ? a.partial + ((int64_t) (X0 / a.grp) * a.nty + ty) * a.ntz + tz : nullptr;
    for (int i = 0; X0 - 1 + i < X1; ++i) {
        const int xe = X0 - 1 + i;
        commit_plane((i + 1) & 1);
        const int ph = ph_next;
        if (xe + 1 < X1)
            ph_next = phase_of(xe + 1);
        __syncthreads();
        T u[8][H];
#pragma unroll
        for (int cr = 0; cr < 8; ++cr) {
            const int ax = cr & 1, ay = (cr >> 1) & 1, az = cr >> 2;
            const T  *src = &Un[(i + ax) & 1][((ey + ay) * NL + ez + az) * H];
#pragma unroll
            for (int c = 0; c < H; ++c)
                u[cr][c] = src[c];
        }
        T dv[H];  // d at node plane xe (CG mode)
#pragma unroll
        for (int c = 0; c < H; ++c)
            dv[c] = u[0][c];
        const int     xg = xe < 0 ? xe + nx : xe;
        const int64_t el = xg * plane + off_own;
        T             f[8][H];
        if constexpr (ISO) {
            if constexpr (H == 3) {
                T lam = ph < 256 ? PL[ph][0] : a.phases[ph].p[0], mu = ph < 256 ? PL[ph][1] : a.phases[ph].p[1];
                if (a.vk) {
                    mu  = a.vg[el];
                    lam = a.vk[el] - (T) (2.0 / 3.0) * mu;
                }
                const T lw = lam * w, mw = mu * w;
                T       T0[3][3];
                if constexpr (MODE == ASM_RESID) {
                    const T r = (T) kSqrtHalf, tr = g0[0] + g0[1] + g0[2];
                    const T E[3][3] = {{g0[0], r * g0[3], r * g0[4]}, {r * g0[3], g0[1], r * g0[5]},
                                       {r * g0[4], r * g0[5], g0[2]}};
#pragma unroll
                    for (int p = 0; p < 3; ++p)
#pragma unroll
                        for (int q = 0; q < 3; ++q)
                            T0[p][q] = (T) 2 * mw * E[p][q] + (p == q ? lw * tr : (T) 0);
                } else {
#pragma unroll
                    for (int p = 0; p < 3; ++p)
#pragma unroll
                        for (int q = 0; q < 3; ++q)
                            T0[p][q] = (T) 0;
                }
                element_forces_iso3_modal<T, NGP, CUBIC>(reinterpret_cast<const T(&)[8][3]>(u), a.geom, lw, mw, T0,
                                            reinterpret_cast<T(&)[8][3]>(f));
            } else {
                const T kw    = (a.vk ? a.vk[el] : (ph < 256 ? PL[ph][0] : a.phases[ph].p[0])) * w;
                const T T0[3] = {kw * g0[0], kw * g0[1], kw * g0[2]};
                element_forces_iso1_modal<T, NGP, CUBIC>(reinterpret_cast<const T(&)[8][1]>(u), a.geom, kw, T0,
                                            reinterpret_cast<T(&)[8][1]>(f));
            }
        } else {
            const Phase<T> &P = a.phases[ph];
            // the linear matvec sees linear models only: no state to prefetch
            if constexpr (NS == 9) {
                auto mat = [&](int gp, const T(&e)[NS], T(&s)[NS]) {
                    material_point_ns<T, H, NS>(P, e, s);
                };
                element_forces<T, H, NGP, NS>(u, a.geom, g0, mat, f);
            } else if constexpr (MODE == ASM_CGLIN) {
                auto mat = [&](int gp, const T(&e)[NS], T(&s)[NS]) { linear_point<T, H>(P, e, s); };
                element_forces<T, H, NGP, NS>(u, a.geom, g0, mat, f);
            } else {
                // the next element of this thread's row is xe + 1 (phase ph_next),
                // 0 <= xe + 1 < X1 <= nx: no wrap (xe = -1 itself wraps to nx - 1)
                // an element feeding no owned node reads no state (elastic stand-in)
                const double *sn = nullptr;
                if (xe + 1 < X1 && el_needed)
                    sn = decltype(pm)::state_of(kind_of(ph_next), a.js, (int64_t) (xe + 1) * splane + sl_own);
                // owned elements of this block's x range are evaluated here and
                // nowhere else in the pass: they carry the per-call state updates
                pm.begin(P, el_needed ? kind_of(ph) : (int) MODEL_ELASTIC_ISO, a.js, (int64_t) xg * splane + sl_own, sn,
                         pm_pre, own_yz && xe >= X0);
                pm_pre = true;
                auto mat = [&](int gp, const T(&e)[NS], T(&s)[NS]) { pm.eval(gp, e, s); };
                element_forces<T, H, NGP, NS>(u, a.geom, g0, mat, f);
            }
        }
        // the loads of the plane after next fly during the exchange and the
        // stores (the element's registers are free again here)
        if (xe + 2 <= X1)
            fetch_plane(xe + 2);
        // z: node (ey,ez) <- az=0 corners of element ez + az=1 corners of element ez-1
        T P2[2][2][H];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int c = 0; c < H; ++c)
                P2[q & 1][q >> 1][c] = f[q][c] + dpp_row_shr1(f[q + 4][c]);
        // y: node (ey,ez) <- ay=0 of own row + ay=1 of row ey-1 (lane-16, or previous wave)
        if (lane >= 48)
#pragma unroll
            for (int ax = 0; ax < 2; ++ax)
#pragma unroll
                for (int c = 0; c < H; ++c)
                    Yb[wave][(ez * 2 + ax) * H + c] = P2[ax][1][c];
        T up[2][H];
#pragma unroll
        for (int ax = 0; ax < 2; ++ax)
#pragma unroll
            for (int c = 0; c < H; ++c)
                up[ax][c] = shfl_up16<T, H>(P2[ax][1][c]);
        __syncthreads();
        if (lane < 16 && wave > 0)
#pragma unroll
            for (int ax = 0; ax < 2; ++ax)
#pragma unroll
                for (int c = 0; c < H; ++c)
                    up[ax][c] = Yb[wave - 1][(ez * 2 + ax) * H + c];
        if (i >= 1 && own_yz) {
            const int64_t po = xe * planeH;
#pragma unroll
            for (int c = 0; c < H; ++c) {
                const T res            = carry[c] + P2[0][0][c] + up[0][c];
                a.out[off_own * H + po + c] = res;
                if constexpr (MODE == ASM_CGLIN) {
                    acc0 += (double) dv[c] * (double) res;
                } else {
                    const double ar = fabs((double) res);
                    if (a.measure == 2)
                        acc0 = fmax(acc0, ar);
                    else if (a.measure == 1)
                        acc0 += ar * ar;
                    else
                        acc0 += ar;
                    if (a.dotv)
                        acc1 += (double) res * (double) a.dotv[off_own * H + po + c];
                }
            }
        }
#pragma unroll
        for (int c = 0; c < H; ++c)
            carry[c] = P2[1][0][c] + up[1][c];
        if constexpr (GRP) {
            if (i >= 1 && (--left == 0 || xe + 1 == X1)) {
                double     v[1]  = {acc0};
                const bool mx[1] = {false};
                block_reduce<1>(v, mx, red);
                if (t == 0)
                    *part = v[0];
                part += a.nty * a.ntz;
                acc0 = 0.0;
                left = a.grp;
            }
        }
    }
    if (!GRP && a.partial) {
        double     v[2]  = {acc0, acc1};
        const bool mx[2] = {MODE == ASM_RESID && a.measure == 2, false};
        block_reduce<2>(v, mx, red);
        if (t == 0) {
            if (MODE == ASM_CGLIN) {
                a.partial[((int64_t) bx * a.nty + ty) * a.ntz + tz] = v[0];
            } else {
                a.partial[blockIdx.x]             = v[0];
                a.partial[gridDim.x + blockIdx.x] = v[1];
            }
        }
    }
}

}  // namespace fans
