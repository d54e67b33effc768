// Point-parallel kernels: wall planes of a stage, CFL reduction, BCON,
// stand-alone fluxes, diagnostics and small bookkeeping kernels.
//
// The wall kernel evaluates the one-sided stencils of the two z walls and
// then applies BCON (3dmhdsub.h:720-873) to the freshly updated wall values,
// reading the new values two planes inward that the interior stage kernel has
// already written.
#pragma once
// FP64 arithmetic follows the reference's operation order, so nothing is
// contracted into FMA; the translation unit of the FP32 (mixed-form) kernels
// alone allows contraction within an expression.
#ifdef MHD3D_FP32_FORM_TU
#pragma clang fp contract(on)
#else
#pragma clang fp contract(off)
#endif

#include <type_traits>

#include "flux_point.hpp"
#include "mhd3d_types.hpp"

namespace mhd {

// Background profiles of the mixed form (index k * nz + z).
// FP32: RO0, TT0, D1z(TT0), D2z(TT0), RO0*GRAV - D1z(P0), then BX0 BY0 BZ0,
// their D1z and their D2z (one-sided on the wall planes for BX0 and BY0).
enum { BG_R0 = 0, BG_T0 = 1, BG_DZT0 = 2, BG_D2ZT0 = 3, BG_HB = 4, BG_B0 = 5, BG_DZB = 8,
       BG_D2ZB = 11, NBGF = 14 };
// FP64: RO0, TT0, BX0 BY0 BZ0.
enum { BG64_R0 = 0, BG64_T0 = 1, BG64_B0 = 2, NBG64 = 5 };

// Index of the FP64 background of field f (RO, TT, BX, BY, BZ), or -1.
__host__ __device__ __forceinline__ int bg64_slot(int f)
{
    return f == 3 ? BG64_R0 : (f == 4 ? BG64_T0 : (f >= 5 ? BG64_B0 + (f - 5) : -1));
}

// A value every thread of a workgroup reads at the same address (a plane's
// metric term or background value, the plane's TSTEP record), read through
// the constant address space: the compiler then issues a scalar load, which
// waits on its own counter instead of the in-order vector-memory counter
// the stencil loads of the next plane are counted on.  Only for memory no
// kernel writes while it runs.
template <typename T>
__device__ __forceinline__ T uniform_load(const T* p)
{
    return *(const __attribute__((address_space(4))) T*)p;
}

// State accessor that reads the register straight from global memory and
// forms 1/RO, u, v, w and P on the fly (3dmhdsub.h:267-276).  TI is the type
// the register is stored in, T the type the fluxes are evaluated in.
// GHOST_COPY (the off-default kernels): with nz_ghost_copy != 0 (= nz), RO
// on a z ghost plane reads the plane two in, as fluxes() copies it there
// under iD != 0 or lRem before forming P and 1/RO (3dmhdsub.h:230-239).
// BG: the register holds the mixed form's FP32 copy (RO, TT, B as
// deviations from the FP64 background bg64 of each plane, in the layout of
// StageArgs::bg64) and the accessor adds the background back.
template <typename T, typename TI = T, bool GHOST_COPY = false, bool BG = false>
struct GAcc {
    static constexpr bool kNeighbourRO = true;   // ro() at any offset
    const TI* __restrict__ U;
    int64_t fs, plane;
    int pitch, nPx, nPy, x, y, z;
    int nz_ghost_copy = 0;
    const double* __restrict__ bg64 = nullptr;   // BG only
    int nzb = 0;                                 // BG only: planes of bg64
    __device__ __forceinline__ T ld(int f, int dx, int dy, int dz) const
    {
        const int xx = wrapi(x + dx, nPx), yy = wrapi(y + dy, nPy);
        const TI v = U[f * fs + (int64_t)(z + dz) * plane + (int64_t)yy * pitch + xx];
        if constexpr (BG) {
            const int k = bg64_slot(f);
            return k < 0 ? T(v) : T(double(v) + uniform_load(bg64 + k * nzb + (z + dz)));
        }
        return T(v);
    }
    __device__ __forceinline__ T ru(int a, int b, int c) const { return ld(0, a, b, c); }
    __device__ __forceinline__ T rv(int a, int b, int c) const { return ld(1, a, b, c); }
    __device__ __forceinline__ T rw(int a, int b, int c) const { return ld(2, a, b, c); }
    __device__ __forceinline__ T ro(int a, int b, int c) const
    {
        if (GHOST_COPY && nz_ghost_copy) {
            const int zz = z + c;
            if (zz == 0) c += 2;
            else if (zz == nz_ghost_copy - 1) c -= 2;
        }
        return ld(3, a, b, c);
    }
    __device__ __forceinline__ T tt(int a, int b, int c) const { return ld(4, a, b, c); }
    __device__ __forceinline__ T bx(int a, int b, int c) const { return ld(5, a, b, c); }
    __device__ __forceinline__ T by(int a, int b, int c) const { return ld(6, a, b, c); }
    __device__ __forceinline__ T bz(int a, int b, int c) const { return ld(7, a, b, c); }
    __device__ __forceinline__ T ri(int a, int b, int c) const { return T(1) / ro(a, b, c); }
    __device__ __forceinline__ T u(int a, int b, int c) const { return ru(a, b, c) * ri(a, b, c); }
    __device__ __forceinline__ T v(int a, int b, int c) const { return rv(a, b, c) * ri(a, b, c); }
    __device__ __forceinline__ T w(int a, int b, int c) const { return rw(a, b, c) * ri(a, b, c); }
    __device__ __forceinline__ T p(int a, int b, int c) const { return ro(a, b, c) * tt(a, b, c); }
};

struct CflPart;

// Scalars of one domain on the device (the CTIM/ITER globals of the
// reference and the DT guard state).
struct DevScalars {
    double dt;          // DT of the current step
    double timc;        // TIMC (3dmhdsub.h:151)
    double dt_last;     // DT of the last completed step
    double nit;         // nIt
    double umach;
    double wmin[4];
    unsigned int nonfinite;
    unsigned int halted;   // HALT_GUARD: the DT guard stopped this domain;
                           // HALT_STOP: it reached its step budget nit_stop
    double dt_min;         // DT guard threshold (0: no guard)
    double nit_call0;      // nIt at the start of the current step call
    double nit_stop;       // stop after this many steps in all (0: no budget)
    unsigned int arrived;  // blocks of a closing stage-3 launch that are done (0 between launches)
    unsigned int pad;
};

// HALT_EXIT: the reference's program exits at this point (RLAX, 3dmhdsub.h:
// 344,416,427-439); the kernels of the domain do nothing until a new state.
enum : unsigned int { HALT_GUARD = 1u, HALT_STOP = 2u, HALT_EXIT = 4u };


// Global-memory accessor of the mixed form's wall kernel: reads the FP64
// state (TI = double, stage 1; deviations are formed in FP64, then rounded)
// or the FP32 deviation copy (TI = float), and gives the deviation-form
// values flux_point<..., DEV = true> asks for.
template <typename TI>
struct GAccDev {
    static constexpr bool kNeighbourRO = true;
    const TI* __restrict__ U;
    int64_t fs, plane;
    int pitch, nPx, nPy, x, y, z, nz;
    const float* __restrict__ bgf;
    const double* __restrict__ bg64;
    __device__ __forceinline__ float raw(int f, int dx, int dy, int dz) const
    {
        const int xx = wrapi(x + dx, nPx), yy = wrapi(y + dy, nPy);
        const TI v = U[f * fs + (int64_t)(z + dz) * plane + (int64_t)yy * pitch + xx];
        if constexpr (std::is_same<TI, double>::value) {
            const int k = bg64_slot(f);
            return k < 0 ? float(v) : float(v - bg64[k * nz + z + dz]);
        } else {
            return v;
        }
    }
    __device__ __forceinline__ float ru(int a, int b, int c) const { return raw(0, a, b, c); }
    __device__ __forceinline__ float rv(int a, int b, int c) const { return raw(1, a, b, c); }
    __device__ __forceinline__ float rw(int a, int b, int c) const { return raw(2, a, b, c); }
    __device__ __forceinline__ float ro(int a, int b, int c) const { return bgf[BG_R0 * nz + z + c] + raw(3, a, b, c); }
    __device__ __forceinline__ float tt(int a, int b, int c) const { return raw(4, a, b, c); }
    __device__ __forceinline__ float bx(int a, int b, int c) const { return raw(5, a, b, c); }
    __device__ __forceinline__ float by(int a, int b, int c) const { return raw(6, a, b, c); }
    __device__ __forceinline__ float bz(int a, int b, int c) const { return raw(7, a, b, c); }
    __device__ __forceinline__ float ri(int a, int b, int c) const { return 1.0f / ro(a, b, c); }
    __device__ __forceinline__ float u(int a, int b, int c) const { return ru(a, b, c) * ri(a, b, c); }
    __device__ __forceinline__ float v(int a, int b, int c) const { return rv(a, b, c) * ri(a, b, c); }
    __device__ __forceinline__ float w(int a, int b, int c) const { return rw(a, b, c) * ri(a, b, c); }
    __device__ __forceinline__ float p(int a, int b, int c) const
    {
        const float R0 = bgf[BG_R0 * nz + z + c], T0 = bgf[BG_T0 * nz + z + c];
        const float r = raw(3, a, b, c), t = raw(4, a, b, c);
        return (R0 * t + r * T0) + r * t;
    }
    __device__ __forceinline__ float hb() const { return bgf[BG_HB * nz + z]; }
    __device__ __forceinline__ float dzt0() const { return bgf[BG_DZT0 * nz + z]; }
    __device__ __forceinline__ float d2zt0() const { return bgf[BG_D2ZT0 * nz + z]; }
    __device__ __forceinline__ float rodev() const { return raw(3, 0, 0, 0); }
    __device__ __forceinline__ float ttfull() const { return bgf[BG_T0 * nz + z] + raw(4, 0, 0, 0); }
    __device__ __forceinline__ float bfull(int k) const { return bgf[(BG_B0 + k) * nz + z] + raw(5 + k, 0, 0, 0); }
    __device__ __forceinline__ float dzb(int k) const { return bgf[(BG_DZB + k) * nz + z]; }
    __device__ __forceinline__ float d2zb(int k) const { return bgf[(BG_D2ZB + k) * nz + z]; }
};


struct StageArgs {
    Geom g;
    Phys c;
    Metric m;
    const double* __restrict__ Uin;
    double* __restrict__ Uout;
    double* __restrict__ Z;
    const double* __restrict__ dt;
    // the domain's scalars (DT guard flag); null: no guard
    const DevScalars* ds;
    // mixed form only: the FP32 copies of the stage values that stages 2 and
    // 3 take their stencils from (Uin32) and that stages 1 and 2 write
    // (Uout32); Uin (read by stage 1) and Uout (written by stage 3) are then
    // the FP64 state, and stages 1-2 write no FP64 U
    const float* __restrict__ Uin32;
    float* __restrict__ Uout32;
    // mixed form only: the z-only background, bgf[k * nz + z] (BG_*) and
    // bg64[k * nz + z] (BG64_*); the FP32 copies hold RO - RO0(z), TT - TT0(z)
    // and B - B0(z) in place of RO, TT and B
    const float* __restrict__ bgf;
    const double* __restrict__ bg64;
    // stage 3 only: when non-null, the kernel also evaluates the CFL limits
    // of the new state (the TSTEP of the next step, 3dmhdsub.h:36-106) and
    // writes one partial record per block at cfl_parts[cfl_base + block]
    CflPart* cfl_parts;
    int cfl_base;
    // off-default branches (FP64 point and wall kernels only)
    ExtArgs x;
};

// Forward: whether the DT guard has stopped the domain (defined below).
__device__ __forceinline__ bool domain_halted(const StageArgs& a);


// Background subtracted from field f of plane z when the FP32 copy is written.
__device__ __forceinline__ double bg_sub(const StageArgs& a, int f, int z)
{
    const int k = bg64_slot(f);
    return k < 0 ? 0.0 : uniform_load(a.bg64 + k * a.g.nz + z);
}

__device__ __forceinline__ PointMetric point_metric(const Metric& m, int xg, int yg, int zg)
{
    PointMetric pm;
    pm.dxx = m.dxxdx[xg];
    pm.d2xx = m.d2xxdx2[xg];
    pm.dyy = m.dyydy[yg];
    pm.d2yy = m.d2yydy2[yg];
    pm.dzz = m.dzzdz[zg];
    pm.d2zz = m.d2zzdz2[zg];
    pm.kap = m.RKAPA[zg];
    pm.dkap = m.DKAPA[zg];
    return pm;
}

// Off-default inputs of point (x, y, z) at field index i (ExtArgs -> ExtPt):
// the horizontal means of planes z-1..z+1, the density-diffusion weight
// wwz[z] (iD 1: 1.0f/ROM[z], iD 2: the host table, 3dmhdsub.h:243-252), the
// lRem mean-profile term HRAD[z] from TTM (:322-325, same products), the
// carried-over FT (lShr), the RLAX correction of the plane and the heat-loss
// factors (iTCon 2).
template <int EXTM = EXT_INTERIOR>
__device__ __forceinline__ void ext_point(const StageArgs& a, int x, int y, int z, int64_t i, ExtPt& e)
{
    const ExtArgs& X = a.x;
    e.flags = X.flags;
    if ((EXTM & (EXT_DH | EXT_DV)) && (X.flags & (EXT_DH | EXT_DV))) {
        e.rom[0] = X.means[z - 1];
        e.rom[1] = X.means[z];
        e.rom[2] = X.means[z + 1];
        e.wwz = X.iD == 1 ? 1.0 / e.rom[1] : X.wwz2[z];
        e.cdh = X.cdh;
        e.cdv = X.cdv;
    }
    if (ext_on<EXTM, EXT_REM>(X.flags)) {
        const double* t = X.means + a.g.nz;
        const double tm = t[z - 1], t0 = t[z], tp = t[z + 1];
        e.ttm[0] = tm;
        e.ttm[1] = t0;
        e.ttm[2] = tp;
        const double dzz = a.m.dzzdz[z];
        double h = (((tp - 2.0 * t0) + tm) * a.c.h2z * dzz * dzz + (tp - tm) * a.c.hz * a.m.d2zzdz2[z]) *
                   a.m.RKAPA[z];
        h += (tp - tm) * a.c.hz * dzz * a.m.DKAPA[z];
        e.hrad = h;
    }
    if (ext_on<EXTM, EXT_SHR>(X.flags)) e.ft_old = X.ft[i];
    if (ext_on<EXTM, EXT_RLAX>(X.flags)) {
        e.corr = X.relax[z];
        e.rscale = X.relax[a.g.nz];
    }
    if (ext_on<EXTM, EXT_HEAT>(X.flags)) {
        e.heat_amp = X.heat_amp;
        e.hx = X.heat_x[x + 1];
        e.hy = X.heat_y[y + 1];
        e.hz = X.heat_z[z];
    }
}

template <typename T>
__device__ __forceinline__ double fsel(const FluxOutT<T>& o, int f)
{
    switch (f) {
    case 0: return o.FU;
    case 1: return o.FV;
    case 2: return o.FW;
    case 3: return o.FR;
    case 4: return o.FT;
    case 5: return o.B1;
    case 6: return o.B2;
    default: return o.B3;
    }
}

// Per-point TSTEP quantities from the state values (3dmhdsub.h:41-88), with
// the scalars from K (Phys or CflRec, same field names), DD the point's grid
// spacing and KC the plane's conduction denominator.
template <typename K>
__device__ __forceinline__ void cfl_core(const K& k, bool mag, double RU, double RV, double RW,
                                         double RO, double TT, double BX, double BY, double BZ,
                                         double DD, double KC, double w[5], double& um)
{
    double UU = (RU * RU + RV * RV + RW * RW) / (RO * RO);
    um = k.OGAMMA * UU / TT;
    if (mag) {
        const double Q = k.GAMMA * TT + (BX * BX + BY * BY + BZ * BZ) * k.OBETA / RO;
        UU += Q + 2.0 * sqrt(UU * Q);
    } else {
        UU += k.GAMMA * TT + 2.0 * sqrt(k.GAMMA * UU * TT);
    }
    w[0] = DD / sqrt(UU);
    w[1] = 0.5 * DD * DD * k.REPR * k.CV * RO / KC;
    w[2] = 0.375 * DD * DD * k.RE * RO;
    w[3] = mag ? 0.5 * DD * DD * k.RM : 1e99;
    // non-finite probe of the point's state: NaN or +-Inf if any field is
    w[4] = ((RU + RV) + (RW + RO)) + ((TT + BX) + (BY + BZ));
}

__device__ __forceinline__ void cfl_values(const Phys& c, const Metric& m, bool mag, double RU,
                                           double RV, double RW, double RO, double TT,
                                           double BX, double BY, double BZ, int xg, int yg,
                                           int z, double w[5], double& um)
{
    double DD = ref_min(m.DDY[yg], m.DDZ[z]);
    if (c.xdim) DD = ref_min(DD, m.DDX[xg]);
    cfl_core(c, mag, RU, RV, RW, RO, TT, BX, BY, BZ, DD, m.KCFL[z], w, um);
}

// The same values with plane z's record r and the column's part of the grid
// spacing, ddxy = DDY[yg] (min DDX[xg] when x is resolved).  DD is the
// minimum of the same finite spacings as in cfl_values, so it is the same
// double.
__device__ __forceinline__ void cfl_values_rec(const CflRec& r, bool mag, double RU, double RV,
                                               double RW, double RO, double TT, double BX,
                                               double BY, double BZ, double ddxy, double w[5],
                                               double& um)
{
    cfl_core(r, mag, RU, RV, RW, RO, TT, BX, BY, BZ, ref_min(ddxy, r.DDZ), r.KCFL, w, um);
}

__device__ __forceinline__ void cfl_point(const Geom& g, const Phys& c, const Metric& m,
                                          const double* __restrict__ U, bool mag, int x, int y,
                                          int z, double w[5], double& um)
{
    const int64_t i = (int64_t)z * g.plane + (int64_t)y * g.pitch + x;
    const int64_t fs = g.fs;
    const double bx = mag ? U[5 * fs + i] : 0.0;
    const double by = mag ? U[6 * fs + i] : 0.0;
    const double bz = mag ? U[7 * fs + i] : 0.0;
    cfl_values(c, m, mag, U[i], U[fs + i], U[2 * fs + i], U[3 * fs + i], U[4 * fs + i], bx, by,
               bz, x + 1, y + 1, z, w, um);
}

// Running CFL extrema of one thread; NaN candidates never replace the
// running value (std::min/std::max of 3dmhdutils.h:61-95).
struct CflAcc {
    double w[4] = {1e99, 1e99, 1e99, 1e99};
    double um = 0.0, bad = 0.0;
    // wp[4]: the point's non-finite probe (cfl_core).  Only NaN/Inf in the
    // state sets the flag: a finite state whose limits are NaN (a negative
    // temperature under the square root) is what the reference steps on
    __device__ __forceinline__ void add(const double wp[5], double up)
    {
        for (int k = 0; k < 4; ++k) w[k] = ref_min(w[k], wp[k]);
        um = ref_max(um, up);
        if (!(wp[4] - wp[4] == 0.0)) bad = 1.0;
    }
};

__device__ __forceinline__ double wave_min(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = ref_min(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ double wave_max(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = ref_max(v, __shfl_xor(v, o, 64));
    return v;
}

// One partial record per block: minima of WW1, WW2, WW3, VV and max of
// OGAMMA*UU/TT over the block's points, plus a non-finite flag.
struct CflPart {
    double w[4];
    double um;
    double bad;
};

// Block reduction of CflAcc into part[b] (wave shuffles, then LDS: sh,
// 6 x 16 doubles, which a kernel may lend from its own buffer once every
// thread is past its last use of it).
__device__ __forceinline__ void cfl_block_reduce(CflAcc& a, CflPart* part, int b, double (*sh)[16])
{
    for (int k = 0; k < 4; ++k) a.w[k] = wave_min(a.w[k]);
    a.um = wave_max(a.um);
    a.bad = wave_max(a.bad);
    const int tid = (threadIdx.z * blockDim.y + threadIdx.y) * blockDim.x + threadIdx.x;
    const int wv = tid >> 6, lane = tid & 63;
    if (lane == 0) {
        for (int k = 0; k < 4; ++k) sh[k][wv] = a.w[k];
        sh[4][wv] = a.um;
        sh[5][wv] = a.bad;
    }
    __syncthreads();
    if (tid == 0) {
        const int nw = (blockDim.x * blockDim.y * blockDim.z + 63) / 64;
        for (int j = 1; j < nw; ++j) {
            for (int k = 0; k < 4; ++k) a.w[k] = ref_min(a.w[k], sh[k][j]);
            a.um = ref_max(a.um, sh[4][j]);
            a.bad = ref_max(a.bad, sh[5][j]);
        }
        for (int k = 0; k < 4; ++k) part[b].w[k] = a.w[k];
        part[b].um = a.um;
        part[b].bad = a.bad;
    }
}

__device__ __forceinline__ void cfl_block_reduce(CflAcc& a, CflPart* part, int b)
{
    __shared__ double sh[6][16];
    cfl_block_reduce(a, part, b, sh);
}

// The DT guard of the reference's driver (3dmhd.cpp:292): after a step whose
// DT fell below dt_min the run halts -- here every later kernel of the
// domain returns at once, leaving the state of that step.
__device__ __forceinline__ void clock_and_guard(DevScalars* s)
{
    s->timc += s->dt;
    s->nit += 1.0;
    s->dt_last = s->dt;
    if (s->dt_min > 0.0 && s->dt < s->dt_min) s->halted |= HALT_GUARD;
    if (s->nit_stop > 0.0 && s->nit >= s->nit_stop) s->halted |= HALT_STOP;
}

// Reduces the per-block partials in a fixed order (one block of 256 threads:
// strided per-thread reduction, then the block reduction) and forms
// DT = SFF * min(...) as 3dmhdsub.h:101-105.  sh: shared memory the caller
// lends; load(p) reads one record.
template <typename LD>
__device__ __forceinline__ void cfl_finalize_block(const CflPart* part, int nparts, DevScalars* s, const Phys& c,
                                                   int mag, double (*sh)[256], LD load)
{
    const int t = threadIdx.y * blockDim.x + threadIdx.x;
    double w[4] = {1e99, 1e99, 1e99, 1e99};
    double um = 0.0, bad = 0.0;
    for (int b = t; b < nparts; b += 256) {
        const CflPart r = load(part + b);
        for (int k = 0; k < 4; ++k) w[k] = ref_min(w[k], r.w[k]);
        um = ref_max(um, r.um);
        bad = ref_max(bad, r.bad);
    }
    for (int k = 0; k < 4; ++k) sh[k][t] = w[k];
    sh[4][t] = um;
    sh[5][t] = bad;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (t < st) {
            for (int k = 0; k < 4; ++k) sh[k][t] = ref_min(sh[k][t], sh[k][t + st]);
            sh[4][t] = ref_max(sh[4][t], sh[4][t + st]);
            sh[5][t] = ref_max(sh[5][t], sh[5][t + st]);
        }
        __syncthreads();
    }
    if (t == 0) {
        for (int k = 0; k < 4; ++k) w[k] = sh[k][0];
        s->umach = sqrt(sh[4][0]);
        for (int k = 0; k < 4; ++k) s->wmin[k] = w[k];
        if (sh[5][0] != 0.0) s->nonfinite = 1u;
        if (mag)
            s->dt = c.SFF * ref_min(ref_min(w[0], w[1]), ref_min(w[2], w[3]));
        else
            s->dt = c.SFF * ref_min(ref_min(w[0], w[1]), w[2]);
    }
}

__device__ __forceinline__ void cfl_finalize_block(const CflPart* __restrict__ part, int nparts,
                                                   DevScalars* s, const Phys& c, int mag)
{
    __shared__ double sh[6][256];
    cfl_finalize_block(part, nparts, s, c, mag, sh, [](const CflPart* p) { return *p; });
}

// What the launches of a step do besides at the ends of the step and of a step
// call: first (stage 1) starts the call's bookkeeping as call_begin_kernel,
// close (the last launch of stage 3, with nparts TSTEP records in all) closes
// the step as step_close_kernel, last publishes the scalars to the host's
// pinned copy `host`.  Launches of their own for these took 13 of 62 us a step
// call on 32^3.
struct StepEnds {
    DevScalars* ds;
    DevScalars* host;
    int first, close, last, nparts;
};

// A TSTEP record that another block of the same launch reads, moved with
// device-scope accesses: they pass by the caches that are not coherent
// between XCDs, so no block has to write back its whole L2 (a device-scope
// release in each of 352 blocks took 20 us of a 53 us launch).
__device__ __forceinline__ void store_part(CflPart* p, const CflPart& v)
{
    const double* s = reinterpret_cast<const double*>(&v);
    double* d = reinterpret_cast<double*>(p);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(CflPart) / sizeof(double)); ++k)
        __hip_atomic_store(d + k, s[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ CflPart load_part(const CflPart* p)
{
    CflPart v;
    double* d = reinterpret_cast<double*>(&v);
    const double* s = reinterpret_cast<const double*>(p);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(CflPart) / sizeof(double)); ++k)
        d[k] = __hip_atomic_load(s + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return v;
}

// Shared memory step_end_block needs.
constexpr int STEP_END_LDS = (int)sizeof(double) * 6 * 256 + (int)sizeof(CflPart) + 16;

// End of a stage-3 block of a closing launch of nblocks blocks: its record (in
// place `slot`), then the count of blocks done; the last one closes the step (clock, DT guard, step budget,
// the next DT).  Every block of the grid comes here once, none of them waits
// for another.  lds: STEP_END_LDS bytes no thread uses any more.
__device__ __forceinline__ void step_end_block(CflAcc& cfl, CflPart* parts, int slot, int nblocks, const StepEnds& e,
                                               const Phys& c, int mag, char* lds)
{
    constexpr int RED = (int)sizeof(double) * 6 * 256;
    const int t = threadIdx.y * blockDim.x + threadIdx.x;
    CflPart* rec = reinterpret_cast<CflPart*>(lds + RED);
    int* last = reinterpret_cast<int*>(lds + RED + sizeof(CflPart));
    __syncthreads();
    if (parts) cfl_block_reduce(cfl, rec, 0, reinterpret_cast<double (*)[16]>(lds));   // thread 0 writes rec
    if (t == 0) {
        if (parts) store_part(parts + slot, *rec);
        // the record has reached the device's point of coherence before this block counts as done
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        *last = __hip_atomic_fetch_add(&e.ds->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                (unsigned)nblocks - 1u;
    }
    __syncthreads();
    if (!*last) return;
    if (t == 0) {
        e.ds->arrived = 0u;
        clock_and_guard(e.ds);
    }
    __syncthreads();
    if (parts && !(e.ds->halted & HALT_GUARD))
        cfl_finalize_block(parts, e.nparts, e.ds, c, mag, reinterpret_cast<double (*)[256]>(lds),
                           [](const CflPart* q) { return load_part(q); });
    if (e.last && t == 0) *e.host = *e.ds;   // thread 0 wrote the scalars
}

// ---------------------------------------------------------------------------
// Interior planes of one RK stage, one thread per point (baseline form).
// Stage k: F = fluxes(Uin); Uout = Zin + GAM_k*DT*F; Z = Uout + ZETA_k*DT*F
// (step_block_GAM / step_block_ZETA, 3dmhdsub.h:168-192; Zin = Uin for k = 1).
// EXT: with the off-default branches of a.x (the only kernel that has them
// between the walls).
template <bool MAG, bool ROT, int STAGE, bool EXT = false>
__global__ void __launch_bounds__(256) stage_point_kernel(StageArgs a)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const int z = blockIdx.z + 2;   // planes 2 .. nPz-1
    if (domain_halted(a)) return;
    if (x >= a.g.nPx || y >= a.g.nPy || z > a.g.nPz - 1) return;
    GAcc<double> acc{a.Uin, a.g.fs, a.g.plane, a.g.pitch, a.g.nPx, a.g.nPy, x, y, z};
    const PointMetric pm = point_metric(a.m, x + 1, y + 1, z);
    const int64_t i = (int64_t)z * a.g.plane + (int64_t)y * a.g.pitch + x;
    FluxOut o;
    ExtPt e;
    if constexpr (EXT) ext_point(a, x, y, z, i, e);
    flux_point<MAG, ROT, 0, double, false, EXT>(acc, a.c, pm, o, &e);
    if constexpr (EXT) {
        if (a.x.flags & EXT_SHR) a.x.ft[i] = o.FT;
    }
    const double DT = *a.dt;
    const double cg = a.c.GAM[STAGE - 1] * DT;
    const double cz = STAGE < 3 ? a.c.ZETA[STAGE - 1] * DT : 0.0;
    constexpr int NF = MAG ? NF_MAG : NF_HYDRO;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        const double F = fsel(o, f);
        const double zin = STAGE == 1 ? a.Uin[f * a.g.fs + i] : a.Z[f * a.g.fs + i];
        const double un = zin + cg * F;
        a.Uout[f * a.g.fs + i] = un;
        if (STAGE < 3) a.Z[f * a.g.fs + i] = un + cz * F;
    }
}

// ---------------------------------------------------------------------------
// BCON() (3dmhdsub.h:720-873) of one wall column.  un[] holds the wall values
// RU..TT[, BX..BZ] of the column (RO final); inward(f, k) gives field f one
// (k = 1) or two (k = 2) planes inward, read only by the branches that need
// it; timt = TIMT of the step.  Covers lShr (moving walls, :721-743,820-826),
// the iTCon 0/1 Gaussian plume with TP != 0 (:744-776), iTCon 0/2/4, 1 and 3
// and izCon 0/1 incl. the lRem wall temperatures (:777-862), and BZ = 0
// (iBCon 0).  EXT = false: the default branches only (the off-default ones
// compiled out of the default kernels).
template <bool EXT, typename In>
__device__ __forceinline__ void bcon_point(const Phys& c, const Metric& m, const ExtArgs& xa,
                                           bool mag, int nPx, bool top, int x, int y, int z,
                                           double timt, const In& inward, double* un)
{
    if (EXT && xa.lShr) {
        const double RRT = 1.0, RRB = -1.0, RPP = 0.0;   // :722-726
        un[0] = 0.0;
        un[1] = (top ? RRT : RRB) * cos(RPP * timt) * un[3];
    } else {
        const double ro1 = inward(3, 1), ro2 = inward(3, 2);
        un[0] = un[3] * (c.C43 * inward(0, 1) / ro1 - c.C13 * inward(0, 2) / ro2);
        un[1] = un[3] * (c.C43 * inward(1, 1) / ro1 - c.C13 * inward(1, 2) / ro2);
    }
    un[2] = 0.0;
    if (top) {
        if (EXT && (xa.flags & EXT_PLUME)) {
            const double gx = xa.plume_x[x + 1], gy = xa.plume_y[y + 1], HH = xa.HH;
            if (c.iTCon == 0) {
                un[4] = 1.0 - (1.0 - xa.tpr) * gx / HH * gy / HH;
            } else {
                const double DZ = xa.ORZD / m.dzzdz[z];
                un[4] = c.C43 * inward(4, 1) - c.C13 * inward(4, 2) -
                        c.C23 * DZ * (c.THETA - (c.THETA - xa.tpr) * gx / HH * gy / HH);
            }
        } else if (c.iTCon == 0 || c.iTCon == 2 || c.iTCon == 4) {
            if (EXT && xa.lRem) {
                un[4] = xa.TU;
            } else {
                un[4] = 1.0;
                if (c.iTCon == 4 && (x + 1) < (nPx + 2) / 2) un[4] = 1.0 - c.TP;
            }
        } else if (c.iTCon == 1) {
            if (EXT && xa.lRem) {
                un[4] = c.C43 * inward(4, 1) - c.C13 * inward(4, 2) + xa.DZTU;
            } else {
                const double DZ = c.ORZF / m.dzzdz[z];
                un[4] = c.C43 * inward(4, 1) - c.C13 * inward(4, 2) - c.C23 * DZ * c.THETA;
            }
        }
    } else {
        if (c.izCon == 0) {
            un[4] = c.TB;
        } else if (EXT && xa.lRem) {
            un[4] = c.C43 * inward(4, 1) - c.C13 * inward(4, 2) + xa.DZTB;
        } else {
            const double DZ = c.ORZF / m.dzzdz[z];
            un[4] = c.C43 * inward(4, 1) - c.C13 * inward(4, 2) - c.C23 * DZ * c.THETA / m.RKAPA[z];
        }
    }
    if (mag && c.iBCon == 0) un[7] = 0.0;
}

// ---------------------------------------------------------------------------
// One wall point of one RK stage: fluxes with the one-sided wall stencils, the
// GAM update, BCON on the updated wall values, then the ZETA register; stage 3
// adds the point to the CFL accumulator.  BCON reads the new values one and
// two planes inward in the same column, so the caller must have updated them.
// T = double: the FP64 form.  T = float: the mixed form (fluxes in FP32, in
// deviation form, from the FP64 state at stage 1 and from the FP32 stage copy
// at stages 2-3; the update, BCON and the Z register in FP64; BCON reads the
// new inward planes from the FP32 copy at stages 1-2 and from the FP64 state
// at stage 3).
// FULL = false: only RO (and BX, BY) of the wall are advanced by their
// fluxes.  BCON replaces RU, RV, RW, TT and BZ there from planes inward and
// constants, and their Z register is read by nothing but the update BCON
// replaces, so their fluxes -- the viscous, conduction, heating and Lorentz
// terms of the wall -- have no reader.  FULL = true where one has: iTCon 3,
// whose top wall keeps the TT its flux gives, and lShr, whose FT register
// carries over (walls_full).  us a wall launch, every flux -> these,
// FP64 MHD (MI355X, rocprofv3, stages 1 / 2): 32^3 12.1 / 12.4 -> 5.2 / 6.3,
// 64^3 13.9 / 14.4 -> 5.8 / 7.3, 256x256x128 28.5 / 29.7 -> 14.2 / 15.0.
template <typename T, bool MAG, bool ROT, int STAGE, bool EXT = false, bool S32 = false, bool FULL = true>
__device__ __forceinline__ void wall_point(const StageArgs& a, int x, int y, bool top, CflAcc& cfl)
{
    constexpr bool F64 = std::is_same<T, double>::value;
    static_assert(F64 || !EXT, "the off-default branches are evaluated in FP64");
    static_assert(F64 || !S32, "S32: FP64 fluxes from the mixed form's FP32 copies");
    constexpr int NF = MAG ? NF_MAG : NF_HYDRO;
    auto kept = [](int f) { return FULL || f == 3 || f == 5 || f == 6; };
    const int z = top ? 1 : a.g.nPz;
    const int zi1 = top ? z + 1 : z - 1;   // first plane inward
    const int zi2 = top ? z + 2 : z - 2;   // second plane inward
    const PointMetric pm = point_metric(a.m, x + 1, y + 1, z);
    // the mixed form's stage 1 reads the FP64 state: its wall fluxes are
    // evaluated in FP64 too (faster than forming FP32 deviations at every
    // stencil read, and no less accurate)
    using TO = typename std::conditional<F64 || STAGE == 1, double, T>::type;
    FluxOutT<TO> o;
    if constexpr (F64 || STAGE == 1) {
        auto eval = [&](auto& acc) {
            ExtPt e;
            if constexpr (EXT) {
                ext_point(a, x, y, z, (int64_t)z * a.g.plane + (int64_t)y * a.g.pitch + x, e);
                if (a.x.flags & EXT_ROCOPY) acc.nz_ghost_copy = a.g.nz;
            }
            if (top)
                flux_point<MAG, ROT, 1, double, false, EXT>(acc, a.c, pm, o, &e);
            else
                flux_point<MAG, ROT, 2, double, false, EXT>(acc, a.c, pm, o, &e);
            if constexpr (EXT && FULL) {
                if (a.x.flags & EXT_SHR) a.x.ft[(int64_t)z * a.g.plane + (int64_t)y * a.g.pitch + x] = o.FT;
            }
        };
        if constexpr (S32 && STAGE > 1) {
            // the FP32 copy of the stage value, its FP64 background added back
            GAcc<double, float, EXT, true> acc{a.Uin32, a.g.fs, a.g.plane, a.g.pitch, a.g.nPx, a.g.nPy, x, y, z};
            acc.bg64 = a.bg64;
            acc.nzb = a.g.nz;
            eval(acc);
        } else {
            GAcc<double, double, EXT> acc{a.Uin, a.g.fs, a.g.plane, a.g.pitch, a.g.nPx, a.g.nPy, x, y, z};
            eval(acc);
        }
    } else {
        GAccDev<float> acc{a.Uin32, a.g.fs, a.g.plane, a.g.pitch, a.g.nPx, a.g.nPy, x, y, z,
                           a.g.nz, a.bgf, a.bg64};
        if (top)
            flux_point<MAG, ROT, 1, float, true>(acc, a.c, pm, o);
        else
            flux_point<MAG, ROT, 2, float, true>(acc, a.c, pm, o);
    }
    const double DT = *a.dt;
    const double cg = a.c.GAM[STAGE - 1] * DT;
    const double cz = STAGE < 3 ? a.c.ZETA[STAGE - 1] * DT : 0.0;
    const int64_t row = (int64_t)y * a.g.pitch + x;
    const int64_t i = (int64_t)z * a.g.plane + row;
    const int64_t i1 = (int64_t)zi1 * a.g.plane + row;
    const int64_t i2 = (int64_t)zi2 * a.g.plane + row;
    const int64_t fs = a.g.fs;
    double un[NF] = {};
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        if (!kept(f)) continue;
        const double zin = STAGE == 1 ? a.Uin[f * fs + i] : a.Z[f * fs + i];
        un[f] = zin + cg * fsel(o, f);
    }
    // BCON (3dmhdsub.h:727-872) on the updated planes inward
    const bool new64 = (F64 && !S32) || STAGE == 3;
    auto Un = [&](int f, int64_t j, int zj) -> double {
        if (new64) return a.Uout[f * fs + j];
        return double(a.Uout32[f * fs + j]) + bg_sub(a, f, zj);
    };
    const Phys& c = a.c;
    const double timt = (EXT && a.x.lShr) ? a.x.TIMI + a.ds->timc : 0.0;
    auto inward = [&](int f, int k) { return k == 1 ? Un(f, i1, zi1) : Un(f, i2, zi2); };
    bcon_point<EXT>(c, a.m, a.x, MAG, a.g.nPx, top, x, y, z, timt, inward, un);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        if (new64)
            a.Uout[f * fs + i] = un[f];
        else
            a.Uout32[f * fs + i] = float(un[f] - bg_sub(a, f, z));
        if (STAGE < 3 && kept(f)) a.Z[f * fs + i] = un[f] + cz * fsel(o, f);
    }
    if (STAGE == 3 && a.cfl_parts) {
        double wp[5], up;
        cfl_values(c, a.m, MAG, un[0], un[1], un[2], un[3], un[4], MAG ? un[5] : 0.0,
                   MAG ? un[6] : 0.0, MAG ? un[7] : 0.0, x + 1, y + 1, z, wp, up);
        cfl.add(wp, up);
    }
}

// Wall planes of one RK stage as a launch of their own, after the interior's
// (where the stage launch does not take them itself, see walls_in_stage); in
// stage 3 it closes the step where e says so.
// Latency-bound (two planes of one-sided stencils from global memory): built
// for three waves per SIMD (FP64) or two (the mixed form's deviation
// stencils), so the register allocator keeps the occupancy; the off-default
// variant needs the registers of one wave.
template <typename T, bool MAG, bool ROT, int STAGE, bool EXT = false, bool S32 = false, bool FULL = true>
__global__ void __launch_bounds__(256, EXT ? 1 : (sizeof(T) == 4 ? 2 : 3)) stage_wall_kernel(StageArgs a, StepEnds e)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const bool top = blockIdx.z == 0;
    const int b = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    if (domain_halted(a)) {
        if (STAGE == 3 && e.last && b == 0 && threadIdx.x == 0 && threadIdx.y == 0) *e.host = *e.ds;
        return;
    }
    // every thread reaches the block reduction below; threads outside the
    // domain only contribute the identity
    CflAcc cfl;
    if (x < a.g.nPx && y < a.g.nPy) wall_point<T, MAG, ROT, STAGE, EXT, S32, FULL>(a, x, y, top, cfl);
    if constexpr (STAGE == 3) {
        __shared__ __align__(16) char lds[STEP_END_LDS];
        if (e.close)
            step_end_block(cfl, a.cfl_parts, a.cfl_base + b, gridDim.x * gridDim.y * gridDim.z, e, a.c, MAG ? 1 : 0,
                           lds);
        else if (a.cfl_parts)
            cfl_block_reduce(cfl, a.cfl_parts, a.cfl_base + b, reinterpret_cast<double (*)[16]>(lds));
    }
}

// ---------------------------------------------------------------------------
// Stand-alone fluxes() into F (all interior planes incl. walls).
// (EXT: with the off-default branches; the carried-over FT of lShr is read,
// not replaced.)
template <bool MAG, bool ROT, bool EXT = false>
__global__ void __launch_bounds__(256) flux_only_kernel(StageArgs a, double* __restrict__ F)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const int z = blockIdx.z + 1;   // planes 1 .. nPz
    if (x >= a.g.nPx || y >= a.g.nPy || z > a.g.nPz) return;
    GAcc<double, double, EXT> acc{a.Uin, a.g.fs, a.g.plane, a.g.pitch, a.g.nPx, a.g.nPy, x, y, z};
    const PointMetric pm = point_metric(a.m, x + 1, y + 1, z);
    const int64_t i = (int64_t)z * a.g.plane + (int64_t)y * a.g.pitch + x;
    FluxOut o;
    ExtPt e;
    if constexpr (EXT) {
        ext_point(a, x, y, z, i, e);
        if (a.x.flags & EXT_ROCOPY) acc.nz_ghost_copy = a.g.nz;
    }
    if (z == 1)
        flux_point<MAG, ROT, 1, double, false, EXT>(acc, a.c, pm, o, &e);
    else if (z == a.g.nPz)
        flux_point<MAG, ROT, 2, double, false, EXT>(acc, a.c, pm, o, &e);
    else
        flux_point<MAG, ROT, 0, double, false, EXT>(acc, a.c, pm, o, &e);
    constexpr int NF = MAG ? NF_MAG : NF_HYDRO;
#pragma unroll
    for (int f = 0; f < NF; ++f) F[f * a.g.fs + i] = fsel(o, f);
}

// ---------------------------------------------------------------------------
// BCON() on a register in place (3dmhdsub.h:720-873).
template <bool MAG, bool EXT>
__global__ void bcon_kernel(Geom g, Phys c, Metric m, ExtArgs xa, const DevScalars* ds,
                            double* __restrict__ U)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const bool top = blockIdx.z == 0;
    if (x >= g.nPx || y >= g.nPy) return;
    const int z = top ? 1 : g.nPz;
    const int64_t row = (int64_t)y * g.pitch + x;
    const int64_t i = (int64_t)z * g.plane + row;
    const int64_t i1 = (int64_t)(top ? z + 1 : z - 1) * g.plane + row;
    const int64_t i2 = (int64_t)(top ? z + 2 : z - 2) * g.plane + row;
    const int64_t fs = g.fs;
    constexpr int NF = MAG ? NF_MAG : NF_HYDRO;
    double un[NF_MAG] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int f = 0; f < NF; ++f) un[f] = U[f * fs + i];
    const double timt = (EXT && xa.lShr) ? xa.TIMI + ds->timc : 0.0;
    auto inward = [&](int f, int k) { return U[f * fs + (k == 1 ? i1 : i2)]; };
    bcon_point<EXT>(c, m, xa, MAG, g.nPx, top, x, y, z, timt, inward, un);
    U[0 * fs + i] = un[0];
    U[1 * fs + i] = un[1];
    U[2 * fs + i] = un[2];
    U[4 * fs + i] = un[4];
    if (MAG) U[7 * fs + i] = un[7];
}

// ---------------------------------------------------------------------------
// TSTEP (3dmhdsub.h:36-106): per-point CFL limits, then a wave + block
// reduction into one partial record per block; cfl_finalize_kernel reduces
// the partials.  Min and max are exact, so the result does not depend on the
// reduction order.

template <bool MAG>
__global__ void __launch_bounds__(256) cfl_kernel(Geom g, Phys c, Metric m,
                                                  const double* __restrict__ U,
                                                  CflPart* __restrict__ part)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    CflAcc acc;
    if (x < g.nPx && y < g.nPy) {
        for (int z = 1 + blockIdx.z; z <= g.nPz; z += gridDim.z) {
            double wp[5], up;
            cfl_point(g, c, m, U, MAG, x, y, z, wp, up);
            acc.add(wp, up);
        }
    }
    const int b = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    cfl_block_reduce(acc, part, b);
}

MHD_TU_LOCAL __global__ void __launch_bounds__(256) cfl_finalize_kernel(const CflPart* __restrict__ part,
                                                           int nparts, DevScalars* s, Phys c,
                                                           int mag)
{
    if (s->halted) return;
    cfl_finalize_block(part, nparts, s, c, mag);
}

__device__ __forceinline__ bool domain_halted(const StageArgs& a) { return a.ds && a.ds->halted; }

MHD_TU_LOCAL __global__ void set_dt_kernel(DevScalars* s, double dt) { s->dt = dt; }

MHD_TU_LOCAL __global__ void clock_kernel(DevScalars* s)
{
    if (s->halted) return;
    clock_and_guard(s);
}

// The close of a step whose TSTEP ran inside stage 3: the clock, the DT
// guard and the step budget (thread 0), then -- unless the guard halted the
// run -- the next DT and the non-finite flag
// from the stage-3 partials, in one launch instead of clock_kernel followed
// by cfl_finalize_kernel (same order, same effect).
MHD_TU_LOCAL __global__ void __launch_bounds__(256) step_close_kernel(const CflPart* __restrict__ part,
                                                         int nparts, DevScalars* s, Phys c,
                                                         int mag)
{
    if (s->halted) return;
    __syncthreads();   // every thread has read the flag before thread 0 may set it
    if (threadIdx.x == 0) clock_and_guard(s);
    __syncthreads();
    if (s->halted & HALT_GUARD) return;
    cfl_finalize_block(part, nparts, s, c, mag);
}

MHD_TU_LOCAL __global__ void set_guard_kernel(DevScalars* s, double dt_min)
{
    s->dt_min = dt_min;
    s->halted &= ~HALT_GUARD;
}

MHD_TU_LOCAL __global__ void clear_halt_kernel(DevScalars* s) { s->halted = 0u; }

// Start of a step call: the non-finite flag of this call, and nIt at its
// start (the steps a call actually took decide which register holds the
// state when the DT guard or the step budget stopped the domain early).
MHD_TU_LOCAL __global__ void call_begin_kernel(DevScalars* s)
{
    s->nonfinite = 0u;
    s->nit_call0 = s->nit;
}

// Step budget of a domain: it stops after nit_stop steps in all.
MHD_TU_LOCAL __global__ void set_stop_kernel(DevScalars* s, double nit_stop)
{
    s->nit_stop = nit_stop;
    s->halted &= ~HALT_STOP;
    if (nit_stop > 0.0 && s->nit >= nit_stop) s->halted |= HALT_STOP;
}

// horizontal_mean (3dmhdsub.h:698-718): the sum over a plane's interior in
// the reference's order -- y outer, x inner, one running double -- so it
// rounds exactly as there.  A sum in that order is one chain of dependent
// additions; here it is walked by wave 0 of the block, while PM_P producer
// waves form the summands: the plane is a flat sequence of groups of
// PM_G * 64 summands, producer wave w forms chunks w-1, w-1+PM_P, ... of 64
// (lane l: summand 64c + l) of the next group into one half of an LDS double
// buffer while wave 0 adds the current group from the other half, from
// uniform-address LDS reads that reach every lane at once.  A summand that
// costs loads and a division (the convective flux of RLAX) is then off the
// chain's path: the additions are the only serial work.  value(y, x) forms
// the summand of interior point (x, y); the sum is returned to wave 0.
constexpr int PM_G = 16;
constexpr int PM_P = 2;
constexpr int PM_T = 64 * (1 + PM_P);
static_assert(PM_G % PM_P == 0, "a producer's summands form one arithmetic progression");

template <typename V>
__device__ __forceinline__ double ordered_plane_sum(const Geom& g, V value, double (*buf)[PM_G * 64])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nPx = g.nPx;
    const int64_t N = (int64_t)nPx * g.nPy;
    const int64_t ngroups = (N + PM_G * 64 - 1) / (PM_G * 64);
    // a producer lane's summands: f = 64 (w-1) + lane + 64 PM_P j, j = 0, 1, ...
    // (with PM_G a multiple of PM_P the stride holds across groups)
    const int f0 = 64 * (w > 0 ? w - 1 : 0) + lane;
    int64_t f = f0;
    int y = f0 / nPx, x = f0 - (f0 / nPx) * nPx;
    const int qy = 64 * PM_P / nPx, qx = 64 * PM_P - qy * nPx;
    auto produce = [&](int64_t gi) {
        double* b = buf[gi & 1];
#pragma unroll
        for (int d = 0; d < PM_G / PM_P; ++d) {
            b[(d * PM_P + w - 1) * 64 + lane] = f < N ? value(y, x) : 0.0;
            f += 64 * PM_P;
            x += qx;
            y += qy;
            if (x >= nPx) {
                x -= nPx;
                ++y;
            }
        }
    };
    if (w > 0) produce(0);
    __syncthreads();
    double s = 0.0;
    for (int64_t gi = 0; gi < ngroups; ++gi) {
        if (w > 0) {
            if (gi + 1 < ngroups) produce(gi + 1);
        } else {
            const double* b = buf[gi & 1];
            const int64_t base = gi * (PM_G * 64);
            if (base + PM_G * 64 <= N) {
                // batches of 16 values: the reads of batch j+1 are issued
                // before the additions of batch j, so LDS latency stays hidden
                const double2* b2 = reinterpret_cast<const double2*>(b);
                constexpr int NB = PM_G * 64 / 16;
                double2 r[2][8];
#pragma unroll
                for (int i = 0; i < 8; ++i) r[0][i] = b2[i];
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    if (j + 1 < NB) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) r[(j + 1) & 1][i] = b2[(j + 1) * 8 + i];
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        s += r[j & 1][i].x;
                        s += r[j & 1][i].y;
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                const int n = (int)(N - base);
                for (int j = 0; j < n; ++j) s += b[j];
            }
        }
        // the half just added is the one the producers fill next
        __syncthreads();
    }
    return s;
}

// Plane sum of the mixed form: each of the block's PT_T threads sums a fixed
// strided subset of the plane in FP64, in order, then a fixed pairwise tree
// combines the partial sums.  The same doubles on every run, alone or in an
// ensemble, in microseconds instead of one dependent chain of nPx*nPy
// additions; not the reference's sequential order, which the FP64 form keeps
// for bit identity (the mixed form is held to 1e-5 per field, not to the
// bit, and a tree of partial sums is the more accurate of the two).
constexpr int PT_T = 256;

template <typename V>
__device__ __forceinline__ double tree_plane_sum(const Geom& g, V value, double* red)
{
    const int t = threadIdx.x;
    const int nPx = g.nPx;
    const int64_t N = (int64_t)nPx * g.nPy;
    int y = t / nPx, x = t - (t / nPx) * nPx;
    const int qy = PT_T / nPx, qx = PT_T - qy * nPx;
    double s = 0.0;
    for (int64_t f = t; f < N; f += PT_T) {
        s += value(y, x);
        x += qx;
        y += qy;
        if (x >= nPx) {
            x -= nPx;
            ++y;
        }
    }
    red[t] = s;
    __syncthreads();
    for (int w = PT_T / 2; w > 0; w >>= 1) {
        if (t < w) red[t] += red[t + w];
        __syncthreads();
    }
    return red[0];
}

// The sequential sum of ordered_plane_sum -- the same double, bit for bit --
// by a block of PW_T walker threads.  While the running sum s stays inside one
// binade, |s| in (2^e, 2^(e+1)), every value it takes is a multiple of that
// binade's grid u = 2^(e-52): s = M*u with the integer M in (2^52, 2^53).
// Adding v then gives M' = M + RNE(v/u) (the exact sum's nearest grid
// point) unless v/u is a halfway case k + 1/2, where the tie goes to the
// even one of M + k and M + k + 1.  So the running value is M plus a prefix
// sum of integer increments, with one bit of sequential state, the parity of
// M: a halfway summand leaves M even, any other flips the parity by its
// increment's.  A round takes the next PW_C summands, PW_R consecutive ones
// per thread, forms their increments, runs the parity through the block
// (within a wave by ballots, across waves from each wave's published map
// and its totals for either incoming parity), and accepts the summands in
// order up to the first one with |v| >= 2^e or whose prefix P takes M + P
// out of the open binade; that one is added in FP64 (s' = u*(M + P) + v, the
// chain's own rounding) and the next round starts after it.  The increments
// and their sums are integers held in doubles: the accepted prefixes lie in
// an interval of width 2^52 and |increment| <= 2^52 + 1, so every partial
// sum formed before the first rejected summand is exact, and so is that
// summand's own range test (rounding is monotone and the bounds are
// doubles); sums after it may round and are never used.  A plane of
// positive values (RO, TT) needs one FP64 addition per binade its sum
// crosses: ~11 for 512 x 512 summands.  The first PW_K0 summands, a zero or
// non-normal running sum, and planes that keep leaving the binade (sums of
// both signs near zero) are walked as the plain chain, a resident chunk at
// a time.
//
// The plane streams through LDS as chunks of PW_C summands in a ring of
// PW_SLOTS chunks: at a round starting in chunk a, chunks a .. a+2 are
// resident; meanwhile PW_T producer threads of the same block (their own
// waves, at the same barriers) load chunk a+3 and store it after the round in
// the slot of chunk a-1, so that its addresses and loads are not in the
// walkers' path.  us a step of iD with lRem, FP64 hydro: 192x192x96 646 ->
// 626 (a launch 62 -> 56), 256x256x128 1250 -> 1236, 512x512x256 9440 -> 9240;
// held to 128 VGPRs, as a plane count beyond the CUs needs two blocks on one
// (256x256x128 with 130: 1377).  The chunk after the
// plane's last is stored as zeros, summands that add nothing, so a round
// reads its PW_C summands unchecked.  Ring index r of summand f is
// f mod PW_RING, stored at r + r/8 so that the threads' strided reads of 8
// consecutive summands hit distinct banks.  value(y, x) forms the summand of
// interior point (x, y); the sum is returned to every thread.
constexpr int PW_T = 256;              // walker threads
constexpr int PW_B = 2 * PW_T;         // and as many producers
constexpr int PW_W = PW_T / 64;
constexpr int PW_R = 8;
constexpr int PW_C = PW_T * PW_R;
constexpr int PW_SLOTS = 4;
constexpr int PW_RING = PW_SLOTS * PW_C;
constexpr int PW_LDS = PW_RING + PW_RING / 8;
constexpr int PW_K0 = 128;

struct PwShared {
    double ring[PW_LDS];
    double tot[2][PW_W];       // each wave's total of increments for an incoming parity 0, 1
    int64_t brk_f[PW_W];       // each wave's first rejected summand (INT64_MAX: none)
    double brk_s[PW_W];        // the running sum after it
    unsigned par[PW_W];        // each wave's parity map: bit 0 passes the incoming parity
                               // through, bit 1 is xor-ed onto it (or replaces it)
};

__device__ __forceinline__ int pw_slot(int64_t f)
{
    const int r = (int)(f & (PW_RING - 1));
    return r + (r >> 3);
}

// Parity of an integer-valued double below 2^53 in magnitude.
__device__ __forceinline__ int pw_odd(double k)
{
    const double h = k * 0.5;
    return h != floor(h) ? 1 : 0;
}

// DPP move of a double (both halves), 0 where the source lane is outside
// the pattern or its row is masked off.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double pw_dpp(double x)
{
    const uint64_t b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROW_MASK, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROW_MASK, 0xf, true);
    return __longlong_as_double((long long)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
}

// Exclusive prefix sum over the 64 lanes of a wave: row_shr 1, 2, 4, 8
// within rows of 16, row_bcast 15 (rows 1, 3) and 31 (rows 2, 3) for the
// inclusive sum, then wave_shr 1.  incl receives the inclusive sum.
__device__ __forceinline__ double pw_wave_scan(double x, double& incl)
{
    x += pw_dpp<0x111, 0xf>(x);
    x += pw_dpp<0x112, 0xf>(x);
    x += pw_dpp<0x114, 0xf>(x);
    x += pw_dpp<0x118, 0xf>(x);
    x += pw_dpp<0x142, 0xa>(x);
    x += pw_dpp<0x143, 0xc>(x);
    incl = x;
    return pw_dpp<0x138, 0xf>(x);
}

// s += the summands [p, end) in order, from the ring (every thread alike).
__device__ __forceinline__ double pw_chain(const double* ring, double s, int64_t p, int64_t end)
{
    for (; p + 16 <= end; p += 16) {
        double r[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) r[i] = ring[pw_slot(p + i)];
#pragma unroll
        for (int i = 0; i < 16; ++i) s += r[i];
    }
    for (; p < end; ++p) s += ring[pw_slot(p)];
    return s;
}

template <typename V>
__device__ __forceinline__ double walk_plane_sum(const Geom& g, V value, PwShared& sh)
{
    const bool producer = __builtin_amdgcn_readfirstlane((int)threadIdx.x) >= PW_T;   // whole waves
    const int t = threadIdx.x & (PW_T - 1), lane = t & 63, w = t >> 6;
    const int nPx = g.nPx;
    const int64_t N = (int64_t)nPx * g.nPy;
    const int64_t nch = (N + PW_C - 1) / PW_C;
    // producers: (y, x) of this thread's summand in the next chunk to load: steps of
    // PW_T summands within a chunk, PW_C from one chunk to the next
    const int qy = PW_T / nPx, qx = PW_T - qy * nPx;
    const int cy = PW_C / nPx, cx = PW_C - cy * nPx;
    int ly = t / nPx, lx = t - (t / nPx) * nPx;
    int64_t lf = t;
    double pre[PW_R];
    auto load_next = [&]() {
        int y = ly, x = lx;
        int64_t f = lf;
#pragma unroll
        for (int j = 0; j < PW_R; ++j) {
            pre[j] = f < N ? value(y, x) : 0.0;
            f += PW_T;
            x += qx;
            y += qy;
            if (x >= nPx) {
                x -= nPx;
                ++y;
            }
        }
        lf += PW_C;
        lx += cx;
        ly += cy;
        if (lx >= nPx) {
            lx -= nPx;
            ++ly;
        }
    };
    // chunk c from registers, or zeros past the last
    auto store_chunk = [&](int64_t c) {
        const bool z = c >= nch;
#pragma unroll
        for (int j = 0; j < PW_R; ++j) sh.ring[pw_slot(c * PW_C + t + j * PW_T)] = z ? 0.0 : pre[j];
    };
    if (producer) {
        for (int c = 0; c < 3; ++c) {
            if (c < nch) load_next();
            store_chunk(c);
        }
    }
    int64_t hi = 2;   // highest chunk stored in the ring
    __syncthreads();
    int64_t p = N < PW_K0 ? N : PW_K0;
    double s = pw_chain(sh.ring, 0.0, 0, p);
    int breaks = 0;
    const int64_t budget = 64 + N / 4096;
    const uint64_t below = (uint64_t(1) << lane) - 1;
    while (p < N) {
        const int64_t a = p / PW_C;
        const bool fetch = hi == a + 2 && a + 3 <= nch;
        if (producer && fetch && a + 3 < nch) load_next();
        const double as = fabs(s);
        if (!(as >= 0x1p-1021 && as < __builtin_inf()) || breaks >= budget) {
            const int64_t end = (a + 1) * PW_C < N ? (a + 1) * PW_C : N;
            s = pw_chain(sh.ring, s, p, end);
            p = end;
            __syncthreads();
        } else {
            int e;
            (void)frexp(as, &e);
            e -= 1;   // |s| in [2^e, 2^(e+1))
            const double lim = ldexp(1.0, e);
            const double u = ldexp(1.0, e - 52);
            const double M = ldexp(s, 52 - e);   // s / u, |M| in [2^52, 2^53)
            // accepted prefixes P: M + P in (2^52, 2^53), or its negative
            const double plo = s > 0.0 ? 0x1p52 - M : -0x1p53 - M;
            const double phi = s > 0.0 ? 0x1p53 - M : -0x1p52 - M;
            double T = 0.0;   // the round's whole increment
            // Each branch is taken by whole waves and passes two barriers, which
            // the hardware counts by wave, not by place: a barrier added to one
            // branch belongs into the other as well.  (With the barriers outside
            // the branches the walkers' values stay live for the producers too: a
            // step of iD with lRem 206 -> 209 us on 96x96x64, 627 -> 631 on
            // 192x192x96, 1237 -> 1246 on 256x256x128.)
            if (producer) {
                __syncthreads();   // the walkers' totals and parity maps
                int pin = pw_odd(M);
#pragma unroll
                for (int ww = 0; ww < PW_W; ++ww) {
                    T += pin ? sh.tot[1][ww] : sh.tot[0][ww];
                    const unsigned pm = sh.par[ww];
                    pin = (pm & 1u) ? (pin ^ (int)(pm >> 1)) : (int)(pm >> 1);
                }
                __syncthreads();   // the first rejected summand
            } else {
                const int64_t f0 = p + (int64_t)t * PW_R;
                double v[PW_R], q[PW_R];
                unsigned flag = 0;       // summands rejected
                unsigned halfm = 0;      // halfway cases
                double acc = 0.0;
#pragma unroll
                for (int i = 0; i < PW_R; ++i) {
                    v[i] = sh.ring[pw_slot(f0 + i)];
                    const double sc = ldexp(v[i], 52 - e);
                    const double r = rint(sc);
                    const bool half = fabs(sc - r) == 0.5;
                    if (!(fabs(v[i]) < lim)) flag |= 1u << i;
                    if (half) halfm |= 1u << i;
                    acc += half ? sc - 0.5 : r;   // the floor for a halfway case
                    q[i] = acc;
                }
                // The parity of the running integer M flips by the parity of a sum
                // of increments, so a thread without halfway cases passes on its
                // incoming parity flipped by that of its total.  With them (rare
                // but for planes of equal or dyadic values): the first one's
                // rounding bit is the incoming parity ^ g2, added as bf once the
                // parity is known; it leaves M even, so each later one's bit is
                // the parity of the increments since the tie before it, and the
                // parity passed on is that of the increments after the last tie.
                const bool seen = halfm != 0;
                unsigned after = 0;      // summands from the first halfway case on
                int g2 = 0, gam;
                if (!seen) {
                    gam = pw_odd(acc);
                } else {
                    const int fh = __builtin_ctz(halfm);
                    after = ~0u << fh;
                    double q0L = 0.0, add = 0.0;   // the prefix at the last tie; later rounding bits
#pragma unroll
                    for (int i = 0; i < PW_R; ++i) {
                        const double q0 = q[i];
                        if (i == fh) {
                            g2 = pw_odd(q0);
                            q0L = q0;
                        } else if (i > fh && ((halfm >> i) & 1u)) {
                            add += (double)pw_odd(q0 - q0L);
                            q0L = q0;
                        }
                        q[i] = q0 + add;
                    }
                    gam = pw_odd(acc - q0L);
                    acc = q[PW_R - 1];
                }
                // incoming parity of this lane: base ^ (dep & the wave's incoming parity)
                const uint64_t Rm = __ballot(seen);
                const uint64_t Xb = __ballot(gam);
                const uint64_t Rb = Rm & below;
                int base, dep;
                if (Rb) {
                    const int r = 63 - __clzll((long long)Rb);
                    base = __popcll(Xb & below & ~((uint64_t(1) << r) - 1)) & 1;
                    dep = 0;
                } else {
                    base = __popcll(Xb & below) & 1;
                    dep = 1;
                }
                const int b0 = base ^ g2;   // the first halfway case's bit for an incoming parity 0
                double incl;
                double E = pw_wave_scan(acc + (seen ? (double)b0 : 0.0), incl);
                // for an incoming parity 1 the lanes with seen && dep add 1 - 2*b0 instead of b0
                // (counts as signed ints: __popcll is unsigned)
                const uint64_t up1 = __ballot(seen && dep && !b0), dn1 = __ballot(seen && dep && b0);
                if (lane == 63) {
                    sh.tot[0][w] = incl;
                    sh.tot[1][w] = incl + (double)((int)__popcll(up1) - (int)__popcll(dn1));
                }
                if (lane == 0) {
                    int xw;
                    if (Rm) {
                        const int r = 63 - __clzll((long long)Rm);
                        xw = __popcll(Xb & ~((uint64_t(1) << r) - 1)) & 1;
                    } else {
                        xw = __popcll(Xb) & 1;
                    }
                    sh.par[w] = (Rm ? 0u : 1u) | ((unsigned)xw << 1);
                }
                __syncthreads();
                int pin = pw_odd(M), mine = 0;
                double Ew = 0.0;
#pragma unroll
                for (int ww = 0; ww < PW_W; ++ww) {
                    if (ww == w) mine = pin;
                    const double tw = pin ? sh.tot[1][ww] : sh.tot[0][ww];
                    if (ww < w) Ew += tw;
                    T += tw;
                    const unsigned pm = sh.par[ww];
                    pin = (pm & 1u) ? (pin ^ (int)(pm >> 1)) : (int)(pm >> 1);
                }
                if (mine) E += (double)((int)__popcll(up1 & below) - (int)__popcll(dn1 & below));
                E += Ew;
                const double bf = seen ? (double)(base ^ (dep & mine) ^ g2) : 0.0;
                const double lo = plo - E, up = phi - E;
#pragma unroll
                for (int i = 0; i < PW_R; ++i) {
                    q[i] += ((after >> i) & 1u) ? bf : 0.0;
                    if (!(q[i] > lo && q[i] < up)) flag |= 1u << i;
                }
                const uint64_t bal = __ballot(flag != 0);
                if (bal) {
                    if (lane == __builtin_ctzll(bal)) {
                        const int j = __builtin_ctz(flag);
                        double before = E, vj = 0.0;
#pragma unroll
                        for (int i = 0; i < PW_R; ++i) {
                            if (i < j) before = E + q[i];
                            if (i == j) vj = v[i];
                        }
                        sh.brk_s[w] = (M + before) * u + vj;
                        sh.brk_f[w] = f0 + j;
                    }
                } else if (lane == 0) {
                    sh.brk_f[w] = INT64_MAX;
                }
                __syncthreads();
            }
            int64_t bfi = INT64_MAX;
            double bs = 0.0;
#pragma unroll
            for (int ww = 0; ww < PW_W; ++ww) {
                const int64_t fw = sh.brk_f[ww];
                if (fw < bfi) {
                    bfi = fw;
                    bs = sh.brk_s[ww];
                }
            }
            if (bfi != INT64_MAX) {
                s = bs;
                p = bfi + 1;
                ++breaks;
            } else {
                s = (M + T) * u;
                p = p + PW_C < N ? p + PW_C : N;
            }
        }
        // chunk a+3 into the slot of chunk a-1, read from the round at a+2 on
        if (fetch) {
            if (producer) store_chunk(a + 3);
            hi = a + 3;
        }
    }
    return s;
}

// Horizontal means of RO (blockIdx.y = 0) and TT (1) on every plane of
// register U, into out[k * nz + z], divided by float(nPx*nPy) as there.  For
// RO the z ghost planes take the planes two in, which fluxes() copies there
// before taking the mean (3dmhdsub.h:230-239).  TI = float: U is the mixed
// form's FP32 copy, whose values are deviations from bg64 (added back).
// SUM(g, value) sums the plane: the reference's order (FP64 form) or the
// tree of the mixed form.
template <typename TI, typename SUM>
__device__ __forceinline__ void plane_mean_body(const Geom& g, const TI* __restrict__ U,
                                                const double* __restrict__ bg64, int want_ro,
                                                int want_tt, double* __restrict__ out, SUM sum)
{
    const int z = blockIdx.x, k = blockIdx.y;
    if (k == 0 ? !want_ro : !want_tt) return;
    int zs = z;
    if (k == 0) zs = z == 0 ? 2 : (z == g.nz - 1 ? g.nz - 3 : z);
    const TI* __restrict__ p = U + (int64_t)(3 + k) * g.fs + (int64_t)zs * g.plane;
    double b = 0.0;
    if constexpr (std::is_same<TI, float>::value) b = bg64[(k == 0 ? BG64_R0 : BG64_T0) * g.nz + zs];
    const double s = sum(g, [&](int y, int x) -> double {
        if constexpr (std::is_same<TI, float>::value)
            return double(p[(int64_t)y * g.pitch + x]) + b;
        else
            return p[(int64_t)y * g.pitch + x];
    });
    if (threadIdx.x == 0) out[k * g.nz + z] = s / (double)(float)(g.nPx * g.nPy);
}

// PW_B threads per plane, the reference's order (walk_plane_sum).
template <typename TI>
__global__ void __launch_bounds__(PW_B, 4)
plane_mean_walk_kernel(Geom g, const TI* __restrict__ U, const double* __restrict__ bg64, int want_ro,
                       int want_tt, double* __restrict__ out)
{
    __shared__ PwShared sh;
    plane_mean_body(g, U, bg64, want_ro, want_tt, out,
                    [&](const Geom& gg, auto value) { return walk_plane_sum(gg, value, sh); });
}

// PT_T threads per plane, the tree of the mixed form.
template <typename TI>
__global__ void __launch_bounds__(PT_T)
plane_mean_tree_kernel(Geom g, const TI* __restrict__ U, const double* __restrict__ bg64, int want_ro,
                       int want_tt, double* __restrict__ out)
{
    __shared__ double red[PT_T];
    plane_mean_body(g, U, bg64, want_ro, want_tt, out,
                    [&](const Geom& gg, auto value) { return tree_plane_sum(gg, value, red); });
}

// FCONM of the RLAX relaxation (3dmhdsub.h:349-353): horizontal_mean of the
// convective flux WW2 = RW*WW1*(-2.5) + RW*UU*UU*(-0.5) + RW*VV*VV*(-0.5) +
// RW*WW*WW*(-0.5) on the interior planes 1..nPz (blockIdx.x + 1), with
// UU = RU * (1/RO) etc. (:268,274-277) and WW1 = TT - TTM(z) (:297-301) --
// or, under lShr, whose `#if !lShr` block skips that, the pressure RO*TT
// left there at :267.  Products in the reference's order (func_mul2,
// func_mul3: ((a*b)*c)*s).  Skipped while the domain is stopped when
// `stopped` is set (a stage), evaluated regardless otherwise (mhd3d_fluxes).
// SUM as for plane_mean_body.
template <typename TI, typename SUM>
__device__ __forceinline__ void conv_flux_mean_body(const Geom& g, const TI* __restrict__ U,
                                                    const double* __restrict__ bg64,
                                                    const double* __restrict__ ttm, int shr,
                                                    const DevScalars* __restrict__ ds, int stopped,
                                                    double* __restrict__ fconm, SUM sum)
{
    if (stopped && ds->halted) return;
    const int z = blockIdx.x + 1;
    const int64_t o = (int64_t)z * g.plane;
    const TI* __restrict__ ru = U + o;
    const TI* __restrict__ rv = U + g.fs + o;
    const TI* __restrict__ rw = U + 2 * g.fs + o;
    const TI* __restrict__ ro = U + 3 * g.fs + o;
    const TI* __restrict__ tt = U + 4 * g.fs + o;
    const double tm = ttm[z];
    // TI = float: the mixed form's FP32 copy, RO and TT as deviations from bg64
    [[maybe_unused]] double r0 = 0.0, t0 = 0.0;
    if constexpr (std::is_same<TI, float>::value) {
        r0 = bg64[BG64_R0 * g.nz + z];
        t0 = bg64[BG64_T0 * g.nz + z];
    }
    const double s = sum(g, [&](int y, int x) -> double {
        const int64_t i = (int64_t)y * g.pitch + x;
        double r = double(ro[i]), t = double(tt[i]);
        if constexpr (std::is_same<TI, float>::value) {
            r += r0;
            t += t0;
        }
        const double w = double(rw[i]);
        const double ri = 1.0 / r;
        const double uu = double(ru[i]) * ri, vv = double(rv[i]) * ri, ww = w * ri;
        const double w1 = shr ? r * t : t - tm;
        double v = (w * w1) * -2.5;
        v += ((w * uu) * uu) * -0.5;
        v += ((w * vv) * vv) * -0.5;
        v += ((w * ww) * ww) * -0.5;
        return v;
    });
    if (threadIdx.x == 0) fconm[z] = s / (double)(float)(g.nPx * g.nPy);
}

// PM_T threads per plane: wave 0 walks the chain, PM_P waves form the summands.
template <typename TI>
__global__ void __launch_bounds__(PM_T)
conv_flux_mean_kernel(Geom g, const TI* __restrict__ U, const double* __restrict__ bg64,
                      const double* __restrict__ ttm, int shr, const DevScalars* __restrict__ ds,
                      int stopped, double* __restrict__ fconm)
{
    __shared__ __align__(16) double buf[2][PM_G * 64];
    conv_flux_mean_body(g, U, bg64, ttm, shr, ds, stopped, fconm,
                        [&](const Geom& gg, auto value) { return ordered_plane_sum(gg, value, buf); });
}

template <typename TI>
__global__ void __launch_bounds__(PT_T)
conv_flux_mean_tree_kernel(Geom g, const TI* __restrict__ U, const double* __restrict__ bg64,
                           const double* __restrict__ ttm, int shr, const DevScalars* __restrict__ ds,
                           int stopped, double* __restrict__ fconm)
{
    __shared__ double red[PT_T];
    conv_flux_mean_body(g, U, bg64, ttm, shr, ds, stopped, fconm,
                        [&](const Geom& gg, auto value) { return tree_plane_sum(gg, value, red); });
}

// The statics of fluxes() that the relaxation keeps between calls
// (3dmhdsub.h:195-198) and the exit point reached, on the device.
struct RelaxState {
    double TFAC, TTM_MAX, TTM_MIN;
    double icall;              // ICALL (an exact integer in a double)
    unsigned int exited;       // 0; 1: "yk not implement" (:427-439); 2: "Relax: check boundary temperature" (:344,416)
    unsigned int exit_stage;   // the RK stage (1-3) whose fluxes() call exited; 0 outside a step
};

// Host-formed constants of the relaxation.
struct RelaxArgs {
    double RLAX, TSTART, TOFF, REPR, FTOT, hz, TIMI;
    int combo;   // 1: iTCon 0 / izCon 1; 2: iTCon 1 / izCon 0; 0: other walls
    int P, nRz;  // z ranks of the reference run and their planes
    const double* __restrict__ dzzdz;
    const double* __restrict__ RKAPA;
    const double* __restrict__ ZEE;
};

// FRADM of global plane z (3dmhdsub.h:356-365): the central difference of
// TTM, one-sided on the two walls of the domain.
__device__ __forceinline__ double relax_fradm(const RelaxArgs& r, const double* __restrict__ TTM, int z, int nPz)
{
    double d;
    if (z == 1)
        d = -3.0 * TTM[z] + 4.0 * TTM[z + 1] - TTM[z + 2];
    else if (z == nPz)
        d = 3.0 * TTM[z] - 4.0 * TTM[z - 1] + TTM[z - 2];
    else
        d = TTM[z + 1] - TTM[z - 1];
    return d * r.hz * r.dzzdz[z] * r.RKAPA[z] / r.REPR;
}

// The relaxation's host-side logic of fluxes() (3dmhdsub.h:322-441), for a
// reference run on P z ranks of nRz planes (rank q's local plane l is global
// plane q*nRz + l): the TFAC update from the wall-plane mean, ALPHA from
// FCONM and FRADM, the per-rank trapezoid scans of CORRECT over planes
// 1..nRz+1 (the rank's upper ghost plane with FCONM = 0 -- WW2 is never
// written on z ghost planes -- and FRADM of the next rank's first plane, 0
// on the last rank, which receives none), the end values summed across
// ranks as :405-421 do, and the exit test.  The block forms every plane's
// ALPHA and the ZEE differences at once (they depend on no scan); thread 0
// then runs the scans in the reference's order from them, and the block
// writes out[z] = CORRECT (planes 1..nPz); out[nz] = RLAX*TFAC; endval holds
// P values.  Work arrays: RELAX_WORK(nz, P) doubles, in dynamic LDS
// (use_lds) or at wk.  `stage` (1-3) marks a call inside a step: the domain
// then stops at once at an exit (the stage's kernels do nothing); with stage
// 0 (mhd3d_fluxes) the state records the exit and the host stops the domain
// after the fluxes.
#define RELAX_WORK(nz, P) (3 * (size_t)(nz) + 4 + 2 * (size_t)(P))
MHD_TU_LOCAL __global__ void __launch_bounds__(256)
relax_kernel(RelaxArgs r, Geom g, const double* __restrict__ TTM, const double* __restrict__ FCONM,
             DevScalars* ds, RelaxState* rs, double* __restrict__ out, double* __restrict__ endval, int stage,
             double* __restrict__ wk, int use_lds)
{
    extern __shared__ double relax_lds[];
    if (stage && ds->halted) return;
    const int t = threadIdx.x, nt = blockDim.x;
    const int nPz = g.nPz, P = r.P, nRz = r.nRz, nz = g.nz;
    double* A = use_lds ? relax_lds : wk;   // ALPHA of plane z, 1..nPz
    double* C = A + (nz + 1);               // CORRECT of plane z before the ranks' sums
    double* DZ = C + (nz + 1);              // ZEE[z] - ZEE[z-1], z = 2..nPz+1
    double* G = DZ + (nz + 2);              // ALPHA of rank q's upper ghost plane
    double* S = G + P;                      // the sum of end values rank q adds
    const double DT = ds->dt;
    const double TIMT = r.TIMI + ds->timc;
    const bool active = (TIMT > r.TSTART) && (rs->TFAC > (double)1e-4f);
    if (active && r.combo != 1 && r.combo != 2) {
        if (t == 0) {
            rs->exited = 2;
            rs->exit_stage = stage;
            if (stage) ds->halted |= HALT_EXIT;
        }
        return;
    }
    if (active) {
        for (int z = 1 + t; z <= nPz; z += nt) {
            double a = 1.0 - (FCONM[z] + relax_fradm(r, TTM, z, nPz)) / r.FTOT;
            A[z] = a / (1.0 + 4.0 * fabs(a));
        }
        for (int z = 2 + t; z <= nPz + 1; z += nt) DZ[z] = r.ZEE[z] - r.ZEE[z - 1];
        for (int q = t; q < P; q += nt) {
            const int z = (q + 1) * nRz + 1;
            const double fr = q < P - 1 ? relax_fradm(r, TTM, z, nPz) : 0.0;
            double a = 1.0 - (0.0 + fr) / r.FTOT;
            G[q] = a / (1.0 + 4.0 * fabs(a));
        }
    }
    // every thread has read TFAC and formed its values before thread 0 goes on
    __syncthreads();
    if (t == 0) {
        if (active) {
            const double step = DT / (3.0 * r.TOFF);
            if (r.combo == 1) {
                if (TTM[nPz] <= rs->TTM_MAX) {
                    rs->TFAC -= step;
                } else {
                    rs->TTM_MAX = TTM[nPz];
                    rs->TFAC += step;
                    if (2.0 < rs->TFAC) rs->TFAC = 2.0;
                }
            } else {
                if (TTM[1] >= rs->TTM_MIN) {
                    rs->TFAC -= step;
                } else {
                    rs->TTM_MIN = TTM[1];
                    rs->TFAC += step;
                    if (2.0 < rs->TFAC) rs->TFAC = 2.0;
                }
            }
            // per-rank scans (the rank's sum of the ranks' end values follows)
            for (int q = 0; q < P; ++q) {
                const int g0 = q * nRz;
                double aprev = 0.0, c = 0.0;
                for (int l = 1; l <= nRz + 1; ++l) {
                    const int z = g0 + l;
                    const double a = l <= nRz ? A[z] : G[q];
                    if (l > 1) c = c + 0.5 * (a + aprev) * DZ[z];
                    if (l <= nRz) C[z] = c;
                    aprev = a;
                }
                endval[q] = c;
            }
            for (int q = 0; q < P; ++q) {
                double SUM = 0.0;
                if (r.combo == 1) {
                    for (int k = 0; k < q; ++k) SUM += endval[k];
                } else {
                    for (int k = P - 1; k >= q; --k) {
                        SUM -= endval[k];
                        SUM -= endval[k];
                    }
                }
                S[q] = SUM;
            }
        }
        out[nz] = r.RLAX * rs->TFAC;
        if (r.combo != 0 && fmod(TIMT, 25.0) <= DT && fmod(rs->icall, 3.0) == 0.0) {
            rs->exited = 1;
            rs->exit_stage = stage;
            if (stage) ds->halted |= HALT_EXIT;
        }
        rs->icall += 1.0;
    }
    __syncthreads();
    // CORRECT, then the ranks' sum added to it (:405-421)
    for (int z = 1 + t; z <= nPz; z += nt) out[z] = active ? C[z] + S[(z - 1) / nRz] : 0.0;
}

// Stops the domain at a recorded exit (after an mhd3d_fluxes call).
MHD_TU_LOCAL __global__ void relax_stop_kernel(DevScalars* ds, const RelaxState* rs)
{
    if (rs->exited) ds->halted |= HALT_EXIT;
}

// A new state runs again: the exit record is cleared (the other statics --
// TFAC, the temperature range, the call count -- persist, as the function
// statics of a process do).
MHD_TU_LOCAL __global__ void relax_clear_exit_kernel(RelaxState* rs)
{
    rs->exited = 0u;
    rs->exit_stage = 0u;
}

// Non-finite scan of a register (interior incl. walls): one thread per
// (x, y) column, looping over z.
MHD_TU_LOCAL __global__ void __launch_bounds__(256) nonfinite_kernel(Geom g, int nf,
                                                        const double* __restrict__ U,
                                                        DevScalars* s)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    if (x >= g.nPx || y >= g.nPy) return;
    bool bad = false;
    for (int z = 1 + blockIdx.z; z <= g.nPz; z += gridDim.z) {
        const int64_t i = (int64_t)z * g.plane + (int64_t)y * g.pitch + x;
        for (int f = 0; f < nf; ++f) {
            const double v = U[f * g.fs + i];
            if (!(v - v == 0.0)) bad = true;
        }
    }
    if (bad) atomicOr(&s->nonfinite, 1u);
}

MHD_TU_LOCAL __global__ void clear_flag_kernel(DevScalars* s) { s->nonfinite = 0u; }

// Counter-based uniform deviate in [-1, 1) for (seed, field, z, y, x):
// the splitmix64 finaliser of the packed key (x, y < 2^18, z < 2^20).
__host__ __device__ inline double hash_uniform(unsigned long long seed, int f, int z, int y, int x)
{
    unsigned long long k = seed * 0x9E3779B97F4A7C15ull ^ ((unsigned long long)f << 56) ^
                           ((unsigned long long)z << 36) ^ ((unsigned long long)y << 18) ^
                           (unsigned long long)x;
    k += 0x9E3779B97F4A7C15ull;
    k = (k ^ (k >> 30)) * 0xBF58476D1CE4E5B9ull;
    k = (k ^ (k >> 27)) * 0x94D049BB133111EBull;
    k ^= k >> 31;
    return (double)(k >> 11) * (2.0 / 9007199254740992.0) - 1.0;
}

// Synthetic stratified state on the device: RO, TT from the z profiles;
// RU, RV, RW = RO * amp * u on the planes between the walls; with lMag
// BX = b0 + b_amp*u, BY, BZ = b_amp*u on planes 1..nPz (BZ = 0 on the walls),
// ghost planes copies of the walls.  u = hash_uniform(seed, field, z, y, x).
MHD_TU_LOCAL __global__ void __launch_bounds__(256) init_stratified_kernel(Geom g, int nf, double* __restrict__ U,
                                                              const double* __restrict__ Tz,
                                                              const double* __restrict__ Rz,
                                                              unsigned long long seed, double amp,
                                                              double b0, double b_amp)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const int z = blockIdx.z;
    if (x >= g.nPx || y >= g.nPy) return;
    const int64_t i = (int64_t)z * g.plane + (int64_t)y * g.pitch + x;
    const double ro = Rz[z];
    U[3 * g.fs + i] = ro;
    U[4 * g.fs + i] = Tz[z];
    const bool inner = z >= 2 && z <= g.nPz - 1;
    for (int f = 0; f < 3; ++f)
        U[f * g.fs + i] = inner ? ro * amp * hash_uniform(seed, f, z, y, x) : 0.0;
    if (nf == NF_MAG) {
        const int zz = z == 0 ? 1 : (z == g.nz - 1 ? g.nPz : z);
        const bool wall = zz == 1 || zz == g.nPz;
        U[5 * g.fs + i] = b0 + b_amp * hash_uniform(seed, 5, zz, y, x);
        U[6 * g.fs + i] = b_amp * hash_uniform(seed, 6, zz, y, x);
        U[7 * g.fs + i] = wall ? 0.0 : b_amp * hash_uniform(seed, 7, zz, y, x);
    }
}

// Plain streaming copy (HBM byte-counter calibration): dst[i] = src[i].
MHD_TU_LOCAL __global__ void __launch_bounds__(256) calibration_copy_kernel(const double* __restrict__ src,
                                                               double* __restrict__ dst, int64_t n)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// Streaming ceiling of the memory system: each thread moves U 16-byte
// vectors per array and iteration (global_load_dwordx4, U independent loads
// in flight per input array), NR input arrays summed into NW output arrays
// of n vectors each (NR:NW = 1:2, 2:2, 2:1 are the read/write mixes of the
// three RK stages).  NW = 0: read only; the sum is kept alive by a store the
// data never triggers.
typedef double dvec2 __attribute__((ext_vector_type(2)));

template <int NR, int NW, int U>
__global__ void __launch_bounds__(256) stream_ceiling_kernel(const dvec2* __restrict__ in,
                                                             dvec2* __restrict__ out, int64_t n)
{
    const int64_t T = (int64_t)gridDim.x * blockDim.x;
    dvec2 acc = {0.0, 0.0};
    for (int64_t i0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i0 < n; i0 += T * U) {
        dvec2 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = dvec2{0.0, 0.0};
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t i = i0 + u * T;
                if (i < n) v[u] += in[r * n + i];
            }
        if constexpr (NW == 0) {
#pragma unroll
            for (int u = 0; u < U; ++u) acc += v[u];
        } else {
#pragma unroll
            for (int w = 0; w < NW; ++w)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int64_t i = i0 + u * T;
                    if (i < n) out[w * n + i] = v[u] * (double)(w + 1);
                }
        }
    }
    if constexpr (NW == 0)
        if (acc.x == -1.2345e300) out[0] = acc;
}

// FP32 copy of a register in the mixed form's deviation layout:
// dst = (float)(src - background) for RO, TT, BX, BY, BZ, (float)src otherwise.
MHD_TU_LOCAL __global__ void __launch_bounds__(256) to_f32_dev_kernel(const double* __restrict__ src,
                                                         float* __restrict__ dst, Geom g, int nf,
                                                         const double* __restrict__ bg64)
{
    const int64_t n = g.fs * nf;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int f = (int)(i / g.fs);
        const int64_t j = i - (int64_t)f * g.fs;
        const int z = (int)(j / g.plane);
        double v = src[i];
        const int k = bg64_slot(f);
        if (z < g.nz && k >= 0) v -= bg64[k * g.nz + z];
        dst[i] = float(v);
    }
}

}  // namespace mhd

namespace mhd {

// Global FP64 diagnostics: total mass and total energy, each point weighted
// by its cell volume DDX[x] * DDY[y] * DDZ[z] (DDX = 1 when x is not
// resolved), and max |div B|.  Deterministic: fixed per-block partials,
// summed in block order.
MHD_TU_LOCAL __global__ void __launch_bounds__(256) diag_kernel(Geom g, Phys c, Metric m, int nf,
                                                   const double* __restrict__ U,
                                                   double* __restrict__ part)
{
    __shared__ double sh[3][256];
    double ms = 0.0, en = 0.0, db = 0.0;
    const int64_t npts = (int64_t)g.nPz * g.nPy * g.nPx;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < npts;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int x = (int)(t % g.nPx);
        const int y = (int)((t / g.nPx) % g.nPy);
        const int z = (int)(t / ((int64_t)g.nPx * g.nPy)) + 1;
        const int64_t i = (int64_t)z * g.plane + (int64_t)y * g.pitch + x;
        const double RU = U[i], RV = U[g.fs + i], RW = U[2 * g.fs + i];
        const double RO = U[3 * g.fs + i], TT = U[4 * g.fs + i];
        const double dV = (c.xdim ? m.DDX[x + 1] : 1.0) * m.DDY[y + 1] * m.DDZ[z];
        ms += RO * dV;
        double e = 0.5 * (RU * RU + RV * RV + RW * RW) / RO + c.CV * RO * TT;
        if (nf == NF_MAG) {
            const double BX = U[5 * g.fs + i], BY = U[6 * g.fs + i], BZ = U[7 * g.fs + i];
            e += 0.5 * c.OBETA * (BX * BX + BY * BY + BZ * BZ);
            if (z > 1 && z < g.nPz) {
                const int xp = wrapi(x + 1, g.nPx), xm = wrapi(x - 1, g.nPx);
                const int yp = wrapi(y + 1, g.nPy), ym = wrapi(y - 1, g.nPy);
                const int64_t r = (int64_t)z * g.plane;
                const double dbx = (U[5 * g.fs + r + (int64_t)y * g.pitch + xp] -
                                    U[5 * g.fs + r + (int64_t)y * g.pitch + xm]) * m.dxxdx[x + 1] * c.hx;
                const double dby = (U[6 * g.fs + r + (int64_t)yp * g.pitch + x] -
                                    U[6 * g.fs + r + (int64_t)ym * g.pitch + x]) * m.dyydy[y + 1] * c.hy;
                const double dbz = (U[7 * g.fs + i + g.plane] - U[7 * g.fs + i - g.plane]) *
                                   m.dzzdz[z] * c.hz;
                db = fmax(db, fabs(dbx + dby + dbz));
            }
        }
        en += e * dV;
    }
    sh[0][threadIdx.x] = ms;
    sh[1][threadIdx.x] = en;
    sh[2][threadIdx.x] = db;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + s];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + s];
            sh[2][threadIdx.x] = fmax(sh[2][threadIdx.x], sh[2][threadIdx.x + s]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[3 * blockIdx.x + 0] = sh[0][0];
        part[3 * blockIdx.x + 1] = sh[1][0];
        part[3 * blockIdx.x + 2] = sh[2][0];
    }
}

MHD_TU_LOCAL __global__ void diag_finalize_kernel(const double* part, int n, double* out)
{
    if (threadIdx.x != 0) return;
    double a = 0.0, b = 0.0, c = 0.0;
    for (int k = 0; k < n; ++k) {
        a += part[3 * k];
        b += part[3 * k + 1];
        c = fmax(c, part[3 * k + 2]);
    }
    out[0] = a;
    out[1] = b;
    out[2] = c;
}

}  // namespace mhd
