#pragma once
// Temporally blocked 1-D Yee/CPML/ADE/Kerr stencil for gfx950.
//
// One wavefront (64 lanes) owns a tile of 64*K consecutive cells of one
// simulation; lane l holds cells base + l*K .. base + l*K + K-1 in registers.
// The tile advances S steps per launch without touching memory: the only
// neighbour traffic per step is one DPP wave shift of H (for the E half) and
// one of E (for the H half).  Each step shrinks the valid region by one cell
// on each side, so a tile loaded over [out0-S, out0+U+S) with U = 64K-2S
// writes back exactly its interior [out0, out0+U).  State is ping-ponged
// between two buffers so neighbouring tiles never read what another tile of
// the same launch wrote.
//
// Per cell and step, in the order of IntegratorLinLor1D / IntegratorNL1D
// (Solver_Engine.py:297-316):
//   ADE polarisation (ADE_PolarisationCurrent_Ex, BaseFDTD11.py:609-633)
//   E update + CPML psi_E (ADE_ExUpdate :663-669, CPML_Psi_e_Update :364-376)
//   soft source / TFSF (Solver_Engine.py:307-310)
//   slab: D update + E creation (ADE_DxUpdate :750-760, ADE_ExCreate :712-725,
//         AcubicFinder/NonLinExUpdate :803-877)
//   H update + CPML psi_H (ADE_HyUpdate :640-656, CPML_Psi_m_Update :381-393)
//   probes / snapshots (probeSim :16-54, vidMake :57-68)
#include <hip/hip_ext.h>

#include <type_traits>

#include "device_common.hpp"

namespace fdtd {

template <typename R, int K>
__device__ __forceinline__ R pick(const R (&a)[K], int j) {
    R v = a[0];
#pragma unroll
    for (int i = 1; i < K; ++i) v = (i == j) ? a[i] : v;
    return v;
}

// Wave-uniform lane broadcast / insert (v_readlane / v_writelane).
__device__ __forceinline__ float lane_read(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ double lane_read(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// Lane of the calling thread in its wave (a tile runs as one wave of a
// multi-wave workgroup).
__device__ __forceinline__ int wave_lane() { return (int)(threadIdx.x & 63u); }

constexpr int kChunks = 4;    // S <= 255: a launch spans at most 4 x 64 steps

// Kerr small-z series y(z) = sum_k (-1)^k C(3k,k)/(2k+1) z^k; FP64 keeps 14
// terms, FP32 8 (truncation < 5e-10 relative for z < 0.01, below FP32 rounding).
template <typename R>
__device__ __forceinline__ double kerr_series(double z) {
    double y;
    if constexpr (sizeof(R) == 8) {
        y = 300830572.0;
        y = fma(y, -z, 50067108.0);
        y = fma(y, -z, 8414640.0);
        y = fma(y, -z, 1430715.0);
        y = fma(y, -z, 246675.0);
        y = fma(y, -z, 43263.0);
        y = fma(y, -z, 7752.0);
        y = fma(y, -z, 1428.0);
    } else {
        y = 1428.0;
    }
    y = fma(y, -z, 273.0);
    y = fma(y, -z, 55.0);
    y = fma(y, -z, 12.0);
    y = fma(y, -z, 3.0);
    y = fma(y, -z, 1.0);
    y = fma(y, -z, 1.0);
    return y;
}

constexpr double kKerrSeriesCut = 0.01;

// FP32 mode: the root is x (1 + delta) with x = u/eps in FP64 and the small
// correction delta = y - 1 = -z (1 - 3z + 12z^2 - 55z^3 + 273z^4) in FP32
// (z < 0.01: |delta| < 0.01; the first term left out, 1428 z^6, and the rest
// of the alternating tail stay below 1.5e-9 relative, 1/40 of an FP32 ulp;
// one FMA fewer per slab cell and step than with the z^5 term: config 2
// 12.73 against 12.80 us per launch).  The series/closed-form choice stays
// on z.
__device__ __forceinline__ float kerr_delta_f32(float z) {
    float t = 273.0f;
    t = fmaf(t, -z, 55.0f);
    t = fmaf(t, -z, 12.0f);
    t = fmaf(t, -z, 3.0f);
    t = fmaf(t, -z, 1.0f);
    return -z * t;
}
// z of the small-z test: FP32 in the FP32 mode, where z only selects the
// branch (the 1e-5 bar leaves no need for an FP64 copy).
template <typename R>
using KerrZ = typename std::conditional<sizeof(R) == 4, float, double>::type;

template <typename R>
__device__ __forceinline__ R kerr_series_e(KerrZ<R> x, double kz, KerrZ<R>& z) {
    if constexpr (sizeof(R) == 4) {
        // E = x (1 + delta) rounded once in FP32: E is stored in FP32 and
        // formed again from D - P every step, so nothing accumulates
        const float zf = (float)kz * x * x;
        z = zf;
        return fmaf(x, kerr_delta_f32(zf), x);
    } else {
        z = kz * x * x;
        return (R)(x * kerr_series<R>(z));
    }
}

// ADE + D update for one slab cell (no branches: ade == 0 is encoded as
// zero coefficients).  FP64 keeps the reference form P' = A P + B Pm + C E
// (ADE_PolarisationCurrent_Ex :620-631); FP32 keeps the velocity form
// V' = -B V - (1-A-B) P + C E, P += V' (sA = -B, sB = 1-A-B).
// HASJ: the step carries a current (general tiles); otherwise Jv is zero and
// the jD * Jv term is left out (jD * 0 is not folded under IEEE rules).
template <typename R, bool KAHAN, bool HASJ>
__device__ __forceinline__ KerrZ<R> slab_u(R kD, R jD, R dH, R Jv, R E, R& D, R& cD, R& P, R& Pm, R& cP,
                                           R sA, R sB, R sC) {
    if constexpr (sizeof(R) == 4) {
        const R Vn = __builtin_fmaf(sC, E, __builtin_fmaf(sA, Pm, -(sB * P)));
        Pm = Vn;
        if (KAHAN) kahan_add(P, cP, Vn); else P = P + Vn;
    } else {
        const R Pn = fmr(sA, P, fmr(sB, Pm, sC * E));
        Pm = P;
        P = Pn;
    }
    const R g = HASJ ? fmr(-jD, Jv, dH) : dH;
    if (KAHAN) kahan_fma(D, cD, g, kD); else D = fmr(g, kD, D);
    // FP32: u = (D - cD) - (P - cP) from the compensated values, in FP32.
    // D - P is exact when D and P are within a factor 2 (the cancelling case)
    // and otherwise rounded relative to a u of their size, so the rounded sum
    // is within ~1e-7 of u itself.  FP64: cD = cP = 0.
    if constexpr (sizeof(R) == 4)
        return KAHAN ? (D - P) + (cP - cD) : (D - P);
    else
        return D - P;
}

// E of a slab cell from u = D - P (per KIND); ie = 1/e.
template <typename R, int KIND>
__device__ __forceinline__ R slab_e_simple(const SimDev<R>& sd, double u, R D, R ie) {
    if constexpr (KIND == SLAB_KERR_REF) {
        const double dd = (double)D / sd.kerr_e0;
        const double A = cubic_root0_1728(sd.kerr_a, sd.kerr_b, sd.kerr_c, sd.cub, -(fabs(dd) * fabs(dd)));
        return (R)((double)D / (sd.kerr_e0 * sd.kerr_lin + sd.kerr_e0 * sd.kerr_chi3 * A));
    } else {
#pragma clang fp contract(off)
        // FP32: u comes from a float; the product rounds as it does through FP64 (48 bits are exact there)
        return (R)u * ie;
    }
}

// Cells whose z reached the series cut take the closed form; one wave-level
// test per step keeps the common path free of per-cell branches.
template <typename R, int K>
__device__ __forceinline__ void kerr_fixup(R (&E)[K], const KerrZ<R> (&x)[K], const KerrZ<R> (&z)[K],
                                           const double (&ied)[K], double chi3) {
    using Z = KerrZ<R>;
    constexpr Z cut = (Z)kKerrSeriesCut;
    Z zmax = z[0];
#pragma unroll
    for (int j = 1; j < K; ++j) zmax = zmax > z[j] ? zmax : z[j];
    if (__any(zmax >= cut)) {
#pragma unroll
        for (int j = 0; j < K; ++j)
            if (z[j] >= cut) E[j] = (R)kerr_root_e((double)x[j] / ied[j], 1.0 / ied[j], chi3);
    }
}

// Register-resident state of one lane's K cells.  Kept as separate arrays
// passed by reference (one struct of ~25 arrays is not scalar-replaced and
// would live in scratch memory).
#define TILE_PARAMS                                                                                      \
    R(&E)[K], R(&H)[K], R(&cE)[K], R(&cH)[K], R(&ke)[K], R(&kh)[K], R(&D)[K], R(&P)[K], R(&Pm)[K],  \
        R(&cD)[K], R(&cP)[K], R(&sA)[K], R(&sB)[K], R(&sC)[K], R(&ie)[K], double(&ied)[K],            \
        double(&kz)[K], R(&psE)[K], R(&psH)[K], R(&bE)[K], R(&cEc)[K], R(&CbE)[K], R(&bH)[K],           \
        R(&cHc)[K], R(&C2H)[K], const unsigned slab_mask, const unsigned interior_mask
#define TILE_ARGS                                                                                       \
    E, H, cE, cH, ke, kh, D, P, Pm, cD, cP, sA, sB, sC, ie, ied, kz, psE, psH, bE, cEc, CbE, bH, cHc, C2H, \
        slab_mask, interior_mask

// Uniform per-launch values of one tile.
template <typename R>
struct TileCtx {
    int lane, t0, base, N, s_lo, s_hi, t_first, T;
    long long gstep0, t_begin;
    int src_lane, src_j, tf_lane, tf_j;
    int npr, pr_rel[2], pr_t0[2], pr_t1[2], pr_id[2];
    unsigned probe_bits;
    int nprobe, snap_interval, snap_rows;
    R kD, jD;
    double chi3;
    const R *srcE, *srcH, *Jc;
    double* Hprev;          // energy: H' before the launch's last H update, or null
    const double* pS;       // beam CIC sums (J' formed here), or null: J' read from Jc
    int pcmin, pcmax;
    bool jpre;              // J' of the lane's cells formed at set-up (K <= 2): Jpre
    double Jpre[2];
    double* probe_out;      // FP64 samples (FP32 fields: hi - c of the Kahan pair)
    R* snap;
    R (*prl)[2][64];        // the wave's LDS rows of probe samples: [probe][E, cE][step in the chunk]
    // workgroup halo exchange (M_GROUP): this wave's place in its workgroup,
    // the exchange period in steps (= halo cells on an inner side) and the
    // emulated vacuum cells (E-form Kerr slab-boundary tiles)
    int wv, hx;
    unsigned emu_mask;
    unsigned first_mask;    // FP32 resident tiles: cells that are a lane's first one in the one-block tiles
};

// What a tile's step loop has to handle (compile-time, one loop per class).
enum : int {
    M_PURE_SLAB = 1,   // every cell is a slab cell
    M_MIXED = 2,       // slab and interior cells: selects per cell
    M_STRIP = 4,       // CPML psi (coefficients are zero off the strips)
    M_SRC = 8,         // soft source / TFSF cell in the tile
    M_PROBE = 16,      // up to two probes in the tile's interior
    M_GENERAL = 32,    // current J, snapshots, more than two probes
    M_GROUP = 64,      // the workgroup's four windows exchange inner halos every hx steps
};

// Inner halos of a workgroup's four adjacent windows (M_GROUP).  Window w
// starts 64K - 2hx cells after window w - 1, so its first hx cells are the
// owned cells hx .. 2hx - 1 from the end of window w - 1, and its last hx
// cells are the owned cells hx .. 2hx - 1 of window w + 1.  Between
// exchanges each window recomputes its halos itself; the invalid front that
// enters at a window edge moves one cell per step, so after hx steps it has
// just reached the owned cells and the halos are replaced by the owners'
// values.  Every state array of a cell goes across (E, H and their Kahan
// compensations, D, P, Pm, cD, cP, psi_E, psi_H); an emulated vacuum cell
// (D-form Kerr tiles) sends the compensation of its E, E - (D - cD), as the
// write-back stores it, and the receiver emulates its halo cells again.
// Double buffered: a buffer is written again only after the next barrier,
// which every wave reaches after reading it.  All four waves run the same
// steps (one simulation per workgroup), so they pass the same barriers.
constexpr int kTileWaves = 4;        // tiles (waves) per workgroup
constexpr int kHaloMaxLanes = 8;     // hx / K lanes per inner side
template <typename R, int K, bool KAHAN>
__device__ __forceinline__ void halo_exchange(TILE_PARAMS, const TileCtx<R>& c, int buf) {
    constexpr int NV = 11;
    __shared__ R xb[2][4][2][NV][kHaloMaxLanes][K];
    constexpr int st = kHaloMaxLanes * K;    // between the arrays of one (buffer, wave, side)
    const int hl = c.hx / K;
    const int lane = c.lane;
    const int w = c.wv;
    // side 0: cells hx .. 2hx-1 (the left neighbour's right halo); side 1:
    // cells 64K-2hx .. 64K-hx-1 (the right neighbour's left halo)
    int side = -1, q = 0;
    if (w > 0 && lane >= hl && lane < 2 * hl) { side = 0; q = lane - hl; }
    if (w < 3 && lane >= 64 - 2 * hl && lane < 64 - hl) { side = 1; q = lane - (64 - 2 * hl); }
    if (side >= 0) {
#pragma unroll
        for (int j = 0; j < K; ++j) {
            R ce = cE[j];
            if (KAHAN && ((c.emu_mask >> j) & 1u)) ce = (R)((double)E[j] - ((double)D[j] - (double)cD[j]));
            R* o = &xb[buf][w][side][0][q][j];
            o[0 * st] = E[j]; o[1 * st] = H[j]; o[2 * st] = ce; o[3 * st] = cH[j];
            o[4 * st] = D[j]; o[5 * st] = P[j]; o[6 * st] = Pm[j]; o[7 * st] = cD[j];
            o[8 * st] = cP[j]; o[9 * st] = psE[j]; o[10 * st] = psH[j];
        }
    }
    __syncthreads();
    int from = -1, fside = 0, fq = 0;
    if (w > 0 && lane < hl) { from = w - 1; fside = 1; fq = lane; }
    if (w < 3 && lane >= 64 - hl) { from = w + 1; fside = 0; fq = lane - (64 - hl); }
    if (from >= 0) {
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const R* o = &xb[buf][from][fside][0][fq][j];
            E[j] = o[0 * st]; H[j] = o[1 * st]; cE[j] = o[2 * st]; cH[j] = o[3 * st];
            D[j] = o[4 * st]; P[j] = o[5 * st]; Pm[j] = o[6 * st]; cD[j] = o[7 * st];
            cP[j] = o[8 * st]; psE[j] = o[9 * st]; psH[j] = o[10 * st];
            if ((c.emu_mask >> j) & 1u) {
                D[j] = E[j];
                cD[j] = cE[j];
                P[j] = Pm[j] = cP[j] = R(0);
            }
        }
    }
}

// Slab E half for all K cells of a pure-slab lane (straight-line: the K FP64
// chains interleave).
template <typename R, int K, bool KAHAN, int KIND, bool HASJ>
__device__ __forceinline__ void e_pure_slab(TILE_PARAMS, const TileCtx<R>& c, const SimDev<R>& sd,
                                            const R (&dH)[K], const R (&Jv)[K]) {
    KerrZ<R> x[K], z[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const KerrZ<R> u = slab_u<R, KAHAN, HASJ>(c.kD, c.jD, dH[j], Jv[j], E[j], D[j], cD[j], P[j], Pm[j],
                                            cP[j], sA[j], sB[j], sC[j]);
        if constexpr (KIND == SLAB_KERR_E) {
            x[j] = u * ie[j];          // ie = 1/eps_inf in R (FP64: the same value as ied)
            E[j] = kerr_series_e<R>(x[j], kz[j], z[j]);
        } else {
            E[j] = slab_e_simple<R, KIND>(sd, (double)u, D[j], ie[j]);
        }
    }
    if constexpr (KIND == SLAB_KERR_E) kerr_fixup<R, K>(E, x, z, ied, c.chi3);
}

// psi' = b psi + c d of the CPML.  FP64 fuses b psi.  FP32 fuses it too (FORM 0),
// except in the E half of the even steps of a block (FORM 1): there the cells
// that are not a lane's first one in the one-block tiles fuse c d.  That is how
// the one-block loops were first compiled; one-block and resident tiles both
// write it out, so that a result does not depend on which of them ran (the
// tests hold them to the same bits).  FORM < 0 leaves the choice to the
// compiler: the halo-exchange instance, which stands alone.
template <int FORM, typename R>
__device__ __forceinline__ R psi_next(R b, R psi, R c, R d, bool first) {
    if constexpr (FORM < 0 || sizeof(R) == 8) {
        return fmr(b, psi, c * d);
    } else {
        const R v = __builtin_fmaf(b, psi, c * d);
        if constexpr (FORM == 0) return v;
        else return first ? v : __builtin_fmaf(c, d, b * psi);
    }
}

// Mixed tile: every cell takes the interior update (+ CPML psi), slab cells
// then take E from D - P through selects.
template <typename R, int K, bool KAHAN, int KIND, bool STRIP, bool HASJ, int FORM = -1>
__device__ __forceinline__ void e_mixed(TILE_PARAMS, const TileCtx<R>& c, const SimDev<R>& sd,
                                        const R (&dH)[K], const R (&Jv)[K]) {
    R Ev[K], cEv[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        Ev[j] = E[j]; cEv[j] = cE[j];
        const R a = dH[j] - Jv[j];
        if (KAHAN) kahan_fma(Ev[j], cEv[j], a, ke[j]); else Ev[j] = fmr(a, ke[j], Ev[j]);
        if (STRIP) {
            psE[j] = psi_next<FORM>(bE[j], psE[j], cEc[j], dH[j], (c.first_mask >> j) & 1u);
            Ev[j] = fmr(-CbE[j], psE[j], Ev[j]);
        }
    }
    KerrZ<R> x[K], z[K];
    R Es[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const bool sl = (slab_mask >> j) & 1u;
        R Dn = D[j], cDn = cD[j], Pn = P[j], Pmn = Pm[j], cPn = cP[j];
        const KerrZ<R> u = slab_u<R, KAHAN, HASJ>(c.kD, c.jD, dH[j], Jv[j], E[j], Dn, cDn, Pn, Pmn, cPn, sA[j],
                                            sB[j], sC[j]);
        if constexpr (KIND == SLAB_KERR_E) {
            x[j] = u * ie[j];
            Es[j] = kerr_series_e<R>(x[j], sl ? kz[j] : 0.0, z[j]);
        } else {
            x[j] = 0;
            z[j] = 0;
            Es[j] = slab_e_simple<R, KIND>(sd, (double)u, Dn, ie[j]);
        }
        D[j] = sl ? Dn : D[j]; cD[j] = sl ? cDn : cD[j];
        P[j] = sl ? Pn : P[j]; Pm[j] = sl ? Pmn : Pm[j]; cP[j] = sl ? cPn : cP[j];
    }
    if constexpr (KIND == SLAB_KERR_E) kerr_fixup<R, K>(Es, x, z, ied, c.chi3);
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const bool sl = (slab_mask >> j) & 1u;
        E[j] = sl ? Es[j] : Ev[j];
        cE[j] = sl ? cE[j] : cEv[j];
    }
}

// Source and TFSF values of up to 64 steps, one step per lane.
template <typename R>
struct SrcChunk {
    R E, H;
    __device__ __forceinline__ void load(const TileCtx<R>& c, int t_first, int n) {
        E = (c.lane < n && c.src_lane >= 0) ? c.srcE[t_first + c.lane] : R(0);
        H = (c.lane < n && c.tf_lane >= 0) ? c.srcH[t_first + c.lane] : R(0);
    }
};

// Steps c.s_lo .. c.s_hi-1.  pre: the source values, when the caller has
// loaded them (a resident tile does while it waits for its halos).
template <typename R, int K, bool KAHAN, int KIND, int MODE>
__device__ __forceinline__ void run_steps(TILE_PARAMS, const TileCtx<R>& c, const SimDev<R>& sd,
                                          const SrcChunk<R>* pre = nullptr) {
    constexpr bool SLAB_CODE = (MODE & (M_PURE_SLAB | M_MIXED)) != 0 && KIND >= SLAB_LINEAR;
    constexpr bool STRIP = (MODE & M_STRIP) != 0;
    constexpr bool SRC = (MODE & M_SRC) != 0;
    constexpr bool PROBE = (MODE & M_PROBE) != 0;
    constexpr bool GEN = (MODE & M_GENERAL) != 0;
    constexpr bool GROUP = (MODE & M_GROUP) != 0;
    int xleft = c.hx, xbuf = 0;      // steps to the next halo exchange, its buffer
    // source values of this launch, one step per lane (read back with
    // v_readlane): no global memory access on the per-step path
    // (chunk q of 64 steps sits in srcEc[0] while it runs; the arrays rotate
    // at chunk ends so every index is a compile-time constant)
    // The source and TFSF cells enter through 0/1 masks per lane and cell:
    // E + 1*v is E + v exactly and E + 0*v is E, so the injection needs no
    // branch on the lane or the cell.
    // Probe samples of the current 64 steps: the lane holding the probe cell
    // writes the field and (FP32) its Kahan compensation into the wave's LDS
    // rows c.prl, step j of the chunk at index j (one masked LDS store per
    // value, against a v_readlane, its wait states and a select per value
    // when the samples were gathered lane by lane in registers: config 2
    // launches 12.78 against 13.27 us); at the chunk's end lane j reads step
    // j back, combines the pair in FP64 and stores it
    R srcEc[kChunks], srcHc[kChunks], ms[K], mt[K];
    if constexpr (SRC) {
#pragma unroll
        for (int j = 0; j < K; ++j) {
            ms[j] = (c.src_lane >= 0 && c.lane == c.src_lane && j == c.src_j) ? R(1) : R(0);
            mt[j] = (c.tf_lane >= 0 && c.lane == c.tf_lane && j == c.tf_j) ? R(1) : R(0);
        }
#pragma unroll
        for (int q = 0; q < kChunks; ++q) {
            if (pre) {
                srcEc[q] = q == 0 ? pre->E : R(0);      // at most 64 steps
                srcHc[q] = q == 0 ? pre->H : R(0);
                continue;
            }
            const int ix = q * 64 + c.lane;
            const bool in = ix < (c.s_hi - c.s_lo);
            srcEc[q] = (in && c.src_lane >= 0) ? c.srcE[c.t_first + ix] : R(0);
            srcHc[q] = (in && c.tf_lane >= 0) ? c.srcH[c.t_first + ix] : R(0);
        }
    }
    // the step body, called twice per loop trip: with two copies the
    // loop-carried registers alternate instead of being moved back each step
    auto step = [&](const int s, auto form) {
        constexpr int FORM = decltype(form)::value;
        const int ix = s - c.s_lo;
        R Jv[K];
#pragma unroll
        for (int j = 0; j < K; ++j) Jv[j] = R(0);
        if constexpr (GEN) {
            if (c.pS && c.jpre) {
#pragma unroll
                for (int j = 0; j < K; ++j) Jv[j] = (R)c.Jpre[j < 2 ? j : 0];
            } else if (c.pS) {
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    const int n = c.base + j;
                    if (n >= 0 && n <= c.N) Jv[j] = (R)j_from_sums(c.pS, c.pcmin, c.pcmax, n);
                }
            } else if (c.Jc) {
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    const int n = c.base + j;
                    if (n >= 0 && n <= c.N) Jv[j] = c.Jc[n];
                }
            }
        }
        // ---------------- E half ----------------
        const R Hl = shr1(H[K - 1]);
        R dH[K];
#pragma unroll
        for (int j = 0; j < K; ++j) dH[j] = H[j] - ((j == 0) ? Hl : H[j - 1]);
        if constexpr (SLAB_CODE && (MODE & M_PURE_SLAB) && !STRIP) {
            e_pure_slab<R, K, KAHAN, KIND, GEN>(TILE_ARGS, c, sd, dH, Jv);
        } else if constexpr (SLAB_CODE) {
            e_mixed<R, K, KAHAN, KIND, STRIP, GEN, FORM>(TILE_ARGS, c, sd, dH, Jv);
        } else {
#pragma unroll
            for (int j = 0; j < K; ++j) {
                const R a = dH[j] - Jv[j];
                if (KAHAN) kahan_fma(E[j], cE[j], a, ke[j]); else E[j] = fmr(a, ke[j], E[j]);
                if (STRIP) {
                    psE[j] = psi_next<FORM>(bE[j], psE[j], cEc[j], dH[j], (c.first_mask >> j) & 1u);
                    E[j] = fmr(-CbE[j], psE[j], E[j]);
                }
            }
        }
        if constexpr (SRC) {
            const R sv = lane_read(srcEc[0], ix & 63);
#pragma unroll
            for (int j = 0; j < K; ++j) E[j] = fmr(ms[j], sv, E[j]);
            // ---------------- H half (TFSF correction first) ----------------
            const R hv = lane_read(srcHc[0], ix & 63);
#pragma unroll
            for (int j = 0; j < K; ++j) H[j] = fmr(-mt[j], hv, H[j]);
        }
        if constexpr (GEN) {
            // energy: the interior's H' before the launch's last H update
            if (c.Hprev && s == c.s_hi - 1) {
#pragma unroll
                for (int j = 0; j < K; ++j)
                    if ((interior_mask >> j) & 1u)
                        c.Hprev[c.base + j] = (double)H[j] - (KAHAN ? (double)cH[j] : 0.0);
            }
        }
        const R Er = shl1(E[0]);
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const R dE = ((j == K - 1) ? Er : E[j + 1]) - E[j];
            if (KAHAN) kahan_fma(H[j], cH[j], dE, kh[j]); else H[j] = fmr(dE, kh[j], H[j]);
            if (STRIP) {
                psH[j] = psi_next<GROUP ? -1 : 0>(bH[j], psH[j], cHc[j], dE, true);
                H[j] = fmr(C2H[j], psH[j], H[j]);
            }
        }
        // ---------------- probes / snapshots ----------------
        if constexpr (PROBE && !GEN) {
#pragma unroll
            for (int k = 0; k < 2; ++k)
                if (k < c.npr && c.lane == c.pr_rel[k] / K) {
                    c.prl[k][0][ix & 63] = pick<R, K>(E, c.pr_rel[k] % K);
                    if (KAHAN) c.prl[k][1][ix & 63] = pick<R, K>(cE, c.pr_rel[k] % K);
                }
        }
        // end of a 64-step chunk: flush probe samples, rotate source chunks
        if constexpr (PROBE || SRC) {
            if (((ix & 63) == 63) || s == c.s_hi - 1) {
                if constexpr (PROBE && !GEN) {
                    // the owning lanes' LDS stores come before the other lanes' reads
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    const int tt = c.t_first + (ix & ~63) + c.lane;
#pragma unroll
                    for (int k = 0; k < 2; ++k)
                        if (k < c.npr && c.lane <= (ix & 63) && tt >= c.pr_t0[k] && tt <= c.pr_t1[k])
                            // FP64 in both precisions: an FP32 field as hi - c of
                            // its Kahan pair (the value fdtd_read_field returns)
                            c.probe_out[(long long)c.pr_id[k] * c.T + tt] =
                                KAHAN ? (double)c.prl[k][0][c.lane] - (double)c.prl[k][1][c.lane]
                                      : (double)c.prl[k][0][c.lane];
                    // and the reads before the next chunk's stores
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                }
                if constexpr (SRC) {
#pragma unroll
                    for (int q = 0; q + 1 < kChunks; ++q) { srcEc[q] = srcEc[q + 1]; srcHc[q] = srcHc[q + 1]; }
                }
            }
        }
        if constexpr (GEN) {
            const int t = c.t_first + ix;
            if (c.probe_bits) {
                for (int p = 0; p < c.nprobe; ++p) {
                    if (!((c.probe_bits >> p) & 1u)) continue;
                    if (t < sd.probe_t0[p] || t > sd.probe_t1[p]) continue;
                    const int rel = sd.probe_cell[p] - c.t0;
                    if (c.lane == rel / K)
                        c.probe_out[(long long)p * c.T + t] =
                            KAHAN ? (double)pick<R, K>(E, rel % K) - (double)pick<R, K>(cE, rel % K)
                                  : (double)pick<R, K>(E, rel % K);
                }
            }
            if (c.snap_interval > 0 && t > 0 && (t % c.snap_interval) == 0) {
                const int row = t / c.snap_interval;
                if (row < c.snap_rows) {
#pragma unroll
                    for (int j = 0; j < K; ++j)
                        if ((interior_mask >> j) & 1u)
                            c.snap[(long long)row * (c.N + 1) + c.base + j] = E[j];
                }
            }
        }
        if constexpr (GROUP) {
            if (--xleft == 0) {
                xleft = c.hx;
                if (s + 1 < c.s_hi) {
                    halo_exchange<R, K, KAHAN>(TILE_ARGS, c, xbuf);
                    xbuf ^= 1;
                }
            }
        }
    };
    using Even = std::integral_constant<int, GROUP ? -1 : 1>;
    using Odd = std::integral_constant<int, GROUP ? -1 : 0>;
    int s = c.s_lo;
    for (; s + 1 < c.s_hi; s += 2) {
        step(s, Even{});
        step(s + 1, Odd{});
    }
    if (s < c.s_hi) step(s, Even{});
}

// Steps of a resident tile: the arithmetic of run_steps, cell by cell
// and in its order, with the rest of the loop cut to what a block of at most
// 64 steps needs.  The slowest tile of a launch sets the pace of all of them,
// and with run_steps that was one tile at the grid's end: a CPML strip tile
// of one cell per lane took 150 ns a step in FP64, a slab tile 57.  So here a tile
// without source or probe has a class of its own, probe rows are written
// without a branch (lanes that hold no probe write a spare word of their own)
// and go out after the loop, and one chunk of source values needs no
// rotation.  odd: the n steps begin at an odd step of their block (psi_next).
constexpr int kResMaxS = 60;

// Every vector store this wave has issued is in memory (and the compiler moves
// none across).  A release fence at workgroup scope does not say so: on gfx950
// it waits for LDS alone, since the waves of a workgroup share their L1.  One
// at agent scope would write back an L2 besides.
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <typename R, int K, bool KAHAN, int KIND, int MODE>
__device__ __forceinline__ void res_steps(TILE_PARAMS, const TileCtx<R>& c, const SimDev<R>& sd,
                                          const SrcChunk<R>& src, R* spare, const int n, const bool odd) {
    constexpr bool SLAB_CODE = (MODE & (M_PURE_SLAB | M_MIXED)) != 0 && KIND >= SLAB_LINEAR;
    constexpr bool STRIP = (MODE & M_STRIP) != 0;
    constexpr bool SRC = (MODE & M_SRC) != 0;
    constexpr bool PROBE = (MODE & M_PROBE) != 0;
    R ms[K], mt[K], Jv[K];
#pragma unroll
    for (int j = 0; j < K; ++j) Jv[j] = R(0);
    if constexpr (SRC) {
#pragma unroll
        for (int j = 0; j < K; ++j) {
            ms[j] = (c.src_lane >= 0 && c.lane == c.src_lane && j == c.src_j) ? R(1) : R(0);
            mt[j] = (c.tf_lane >= 0 && c.lane == c.tf_lane && j == c.tf_j) ? R(1) : R(0);
        }
    }
    // a probe's rows: E, then (FP32) its Kahan compensation 64 words on
    R* row[2];
    int inc[2];
    if constexpr (PROBE) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const bool mine = k < c.npr && c.lane == c.pr_rel[k] / K;
            row[k] = mine ? &c.prl[k][0][0] : spare + c.lane;
            inc[k] = mine ? 1 : 0;
        }
    }
    auto step = [&](const int s, auto form) {
        constexpr int FORM = decltype(form)::value;
        const R Hl = shr1(H[K - 1]);
        R dH[K];
#pragma unroll
        for (int j = 0; j < K; ++j) dH[j] = H[j] - ((j == 0) ? Hl : H[j - 1]);
        if constexpr (SLAB_CODE && (MODE & M_PURE_SLAB) && !STRIP) {
            e_pure_slab<R, K, KAHAN, KIND, false>(TILE_ARGS, c, sd, dH, Jv);
        } else if constexpr (SLAB_CODE) {
            e_mixed<R, K, KAHAN, KIND, STRIP, false, FORM>(TILE_ARGS, c, sd, dH, Jv);
        } else {
#pragma unroll
            for (int j = 0; j < K; ++j) {
                if (KAHAN) kahan_fma(E[j], cE[j], dH[j], ke[j]); else E[j] = fmr(dH[j], ke[j], E[j]);
                if (STRIP) {
                    psE[j] = psi_next<FORM>(bE[j], psE[j], cEc[j], dH[j], (c.first_mask >> j) & 1u);
                    E[j] = fmr(-CbE[j], psE[j], E[j]);
                }
            }
        }
        if constexpr (SRC) {
            const R sv = lane_read(src.E, s);
#pragma unroll
            for (int j = 0; j < K; ++j) E[j] = fmr(ms[j], sv, E[j]);
            if (c.tf_lane >= 0) {
                const R hv = lane_read(src.H, s);
#pragma unroll
                for (int j = 0; j < K; ++j) H[j] = fmr(-mt[j], hv, H[j]);
            }
        }
        const R Er = shl1(E[0]);
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const R dE = ((j == K - 1) ? Er : E[j + 1]) - E[j];
            if (KAHAN) kahan_fma(H[j], cH[j], dE, kh[j]); else H[j] = fmr(dE, kh[j], H[j]);
            if (STRIP) {
                psH[j] = psi_next<0>(bH[j], psH[j], cHc[j], dE, true);
                H[j] = fmr(C2H[j], psH[j], H[j]);
            }
        }
        if constexpr (PROBE) {
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                row[k][0] = pick<R, K>(E, c.pr_rel[k] % K);
                if (KAHAN) row[k][64] = pick<R, K>(cE, c.pr_rel[k] % K);
                row[k] += inc[k];
            }
        }
    };
    int s = 0;
    // (after an odd cut the first step here is an odd one of its block)
    if constexpr (STRIP && sizeof(R) == 4)
        if (odd) step(s++, std::integral_constant<int, 0>{});
    for (; s + 1 < n; s += 2) {
        step(s, std::integral_constant<int, 1>{});
        step(s + 1, std::integral_constant<int, 0>{});
    }
    if (s < n) step(s, std::integral_constant<int, 1>{});
    // the words emptied after the last hand-off, before the next one sends (ResArgs); they are a
    // block old here, while the probe samples and the snapshot rows to come need no wait
    stores_done();
    if constexpr (PROBE) {
        // the owning lanes' LDS stores come before the other lanes' reads
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int tt = c.t_first + c.lane;
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (k < c.npr && c.lane < n && tt >= c.pr_t0[k] && tt <= c.pr_t1[k])
                c.probe_out[(long long)c.pr_id[k] * c.T + tt] =
                    KAHAN ? (double)c.prl[k][0][c.lane] - (double)c.prl[k][1][c.lane] : (double)c.prl[k][0][c.lane];
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// Device-coherent loads and stores of the resident hand-off: relaxed atomics
// at agent scope are issued with the device-scope cache bits, so each access
// is coherent across the XCDs' L2 caches by itself, and no fence has to write
// back or invalidate a whole L2 (an agent-scope fence per block and tile made
// a 42-step block take 55 us against 12.8 us for a one-block launch).
__device__ __forceinline__ unsigned long long ld_dev(const unsigned long long* p) {
    return __hip_atomic_load(const_cast<unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Mailbox words: a value (FP64) or a pair of values (FP32).
__device__ __forceinline__ unsigned long long pack2(double a, double) { return (unsigned long long)__double_as_longlong(a); }
__device__ __forceinline__ unsigned long long pack2(float a, float b) {
    return ((unsigned long long)__float_as_uint(b) << 32) | __float_as_uint(a);
}
__device__ __forceinline__ void unpack2(unsigned long long w, double& a, double&) { a = __longlong_as_double((long long)w); }
__device__ __forceinline__ void unpack2(unsigned long long w, float& a, float& b) {
    a = __uint_as_float((unsigned)(w & 0xffffffffull));
    b = __uint_as_float((unsigned)(w >> 32));
}

// One tile: 64 lanes x K cells, S steps (the whole per-tile program); with
// RES, tile rt of a resident launch (ResArgs): all of the launch's steps, in
// blocks of S with the hand-off between them (a separate instance: the
// one-block kernel keeps its own register allocation).
template <typename R, int K, bool KAHAN, int KIND, bool RES, bool GROUP = false>
__device__ __forceinline__ void tile_body(const SimDev<R>& sd, int out0_, long long launch_idx, long long gstep0,
                                          int nsteps, int S, const PersistArgs& pa, const int4 rt, const ResArgs& ra) {
    constexpr bool DFORM = KIND >= SLAB_LINEAR;
    const int lane = wave_lane();
    // the window [t0, t0 + 64K) and the cells it owns (writes back, probes):
    // a tile entry holds the first owned cell, the window reaching S cells
    // to either side; with GROUP it holds the window start, and wave w of the
    // workgroup owns all but its outer halo of S cells (first and last wave)
    // and its inner halos of hx cells
    const int wv = GROUP ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;
    const int hx = GROUP ? pa.halo : 0;
    const int t0 = GROUP ? out0_ : out0_ - S;
    const int out0 = GROUP ? t0 + (wv == 0 ? S : hx) : out0_;
    const int U = RES ? rt.z - rt.y
                  : GROUP ? 64 * K - (wv == 0 ? S : hx) - (wv == kTileWaves - 1 ? S : hx) : 64 * K - 2 * S;
    const int N = sd.N;
    const int par = (int)((launch_idx - sd.launch_begin) & 1);
    const int F = sd.F, Rr = sd.Rr, Ls = sd.Ls, Rs = sd.Rs;

    // Everything the step loop reads from the descriptor is copied into
    // registers: the loop's global stores (probes, snapshots) could alias the
    // descriptor, so the compiler would otherwise reload it every step.
    TileCtx<R> c;
    // probe sample rows, one set per wave of the 256-thread workgroup
    __shared__ R pr_rows[kTileWaves][2][2][64];
    const int wvi = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    c.prl = pr_rows[wvi];
    c.lane = lane;
    c.t0 = t0;
    c.wv = wv;
    c.hx = hx;
    c.emu_mask = 0;
    c.first_mask = RES ? 0 : 1;
    c.base = c.t0 + lane * K;
    c.N = N;
    c.T = sd.T;
    c.gstep0 = gstep0;
    c.t_begin = sd.t_begin;
    c.kD = sd.kD; c.jD = sd.jD; c.chi3 = sd.kerr_chi3;
    c.nprobe = sd.nprobe; c.snap_interval = sd.snap_interval; c.snap_rows = sd.snap_rows;
    c.srcE = sd.srcE; c.srcH = sd.srcH; c.Jc = sd.J; c.probe_out = sd.probe_out; c.snap = sd.snap;
    c.Hprev = sd.Hprev;
    c.pS = sd.pS;
    c.pcmin = 1;
    c.pcmax = 0;
    c.jpre = false;
    c.Jpre[0] = c.Jpre[1] = 0.0;
    if (c.pS) {
        // J' of a launch is the same at each of its steps (the sums of this
        // launch's push).  With K <= 2 it is formed here: the sums come in
        // from clamped cells without waiting for the live range, which only
        // masks them afterwards (the sum of j_from_sums, in its order).
        double raw[K <= 2 ? K : 1][4];
        if constexpr (K <= 2 && !RES) {
#pragma unroll
            for (int j = 0; j < K; ++j)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const int cc = min(max(c.base + j - 2 + w, 0), N + 1);
                    raw[j][w] = c.pS[4 * (size_t)cc + (3 - w)];
                }
        }
        c.pcmin = sd.prange[par][0];
        c.pcmax = sd.prange[par][1];
        if constexpr (K <= 2 && !RES) {
            c.jpre = true;
#pragma unroll
            for (int j = 0; j < K; ++j) {
                const int n = c.base + j;
                double t = 0.0;
                if (n >= 0 && n <= N) {
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const int cc = n - 2 + w;
                        const double v = (c.pcmin <= c.pcmax && cc >= c.pcmin - 1 && cc <= c.pcmax + 1) ? raw[j][w]
                                                                                                       : 0.0;
                        t = w == 0 ? v : t + v;
                    }
                }
                c.Jpre[j] = t;
            }
        }
    }

    R E[K], H[K], cE[K], cH[K], ke[K], kh[K];
    R D[K], P[K], Pm[K], cD[K], cP[K], sA[K], sB[K], sC[K], ie[K];
    double ied[K], kz[K];
    R psE[K], psH[K], bE[K], cEc[K], CbE[K], bH[K], cHc[K], C2H[K];
    unsigned slab_mask = 0, strip_mask = 0, interior_mask = 0;
    const R* Ein = sd.E[par];
    const R* Hin = sd.H[par];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const int n = c.base + j;
        // a resident tile may own fewer cells than its window holds; the rest stays zero
        const bool valid = (n >= 0) && (n <= N) && (!RES || n < out0 + U + S);
        E[j] = valid ? Ein[n] : R(0);
        H[j] = valid ? Hin[n] : R(0);
        cE[j] = cH[j] = R(0);
        if (KAHAN && valid) { cE[j] = sd.cE[par][n]; cH[j] = sd.cH[par][n]; }
        ke[j] = valid ? sd.ke0 : R(0);
        kh[j] = valid ? sd.kh0 : R(0);
        D[j] = P[j] = Pm[j] = cD[j] = cP[j] = sA[j] = sB[j] = sC[j] = R(0);
        ie[j] = R(1);
        psE[j] = psH[j] = bE[j] = cEc[j] = CbE[j] = bH[j] = cHc[j] = C2H[j] = R(0);
        const bool inslab = valid && n >= F && n < Rr;
        if (KIND == SLAB_DIEL && inslab) { ke[j] = sd.keS; kh[j] = sd.khS; }
        if (DFORM && inslab) {
            const int i = n - F;
            slab_mask |= 1u << j;
            D[j] = sd.D[par][i]; P[j] = sd.P[par][i]; Pm[j] = sd.Pm[par][i];
            if (KAHAN) { cD[j] = sd.cD[par][i]; cP[j] = sd.cP[par][i]; }
            sA[j] = sd.sl_A[i]; sB[j] = sd.sl_B[i]; sC[j] = sd.sl_C[i]; ie[j] = sd.sl_e[i];
        }
        if (valid && (n < Ls || n >= Rs)) {
            const int i = n < Ls ? n : Ls + (n - Rs);
            strip_mask |= 1u << j;
            ke[j] = sd.s_ke[i]; kh[j] = sd.s_kh[i];
            bE[j] = sd.s_bE[i]; cEc[j] = sd.s_cE[i]; CbE[j] = sd.s_CbE[i];
            bH[j] = sd.s_bH[i]; cHc[j] = sd.s_cH[i]; C2H[j] = sd.s_C2H[i];
            psE[j] = sd.psiE[par][i]; psH[j] = sd.psiH[par][i];
        }
        if (valid && n >= out0 && n < out0 + U) interior_mask |= 1u << j;
        if constexpr (RES && sizeof(R) == 4)
            if ((n + S) % ra.formK == 0) c.first_mask |= 1u << j;
        ied[j] = (double)ie[j];
        kz[j] = c.chi3 * ied[j];
    }
    constexpr unsigned full = (K >= 32) ? 0xffffffffu : ((1u << K) - 1u);
    // tile classes (wave-uniform)
    const bool tile_strip = __any(strip_mask != 0);
    const bool pure_slab = DFORM && __all(slab_mask == full);
    const bool any_slab = DFORM && __any(slab_mask != 0);
    const int tile_end = c.t0 + 64 * K;
    const int src = sd.src_cell;
    // (a resident tile's idle cells take no source)
    const int src_end = RES ? min(tile_end, out0 + U + S) : tile_end;
    const bool tile_src = src >= c.t0 && src < src_end;
    c.src_lane = tile_src ? (src - c.t0) / K : -1;
    c.src_j = tile_src ? (src - c.t0) % K : 0;
    const bool tile_tf = sd.tfsf && (src - 1) >= c.t0 && (src - 1) < src_end;
    c.tf_lane = tile_tf ? (src - 1 - c.t0) / K : -1;
    c.tf_j = tile_tf ? (src - 1 - c.t0) % K : 0;
    c.probe_bits = 0;
    for (int p = 0; p < c.nprobe; ++p) {
        const int cc = sd.probe_cell[p];
        if (cc >= out0 && cc < out0 + U && cc <= N) c.probe_bits |= 1u << p;
    }
    c.npr = __popc(c.probe_bits);
    // first two probes of the tile (constant indices keep TileCtx in registers)
    c.pr_rel[0] = c.pr_rel[1] = c.pr_id[0] = c.pr_id[1] = c.pr_t0[0] = c.pr_t0[1] = 0;
    c.pr_t1[0] = c.pr_t1[1] = -1;
    {
        bool have0 = false;
        for (int p = 0; p < c.nprobe; ++p) {
            if (!((c.probe_bits >> p) & 1u)) continue;
            const int rel = sd.probe_cell[p] - c.t0, a = sd.probe_t0[p], z = sd.probe_t1[p];
            if (!have0) { c.pr_rel[0] = rel; c.pr_t0[0] = a; c.pr_t1[0] = z; c.pr_id[0] = p; have0 = true; }
            else { c.pr_rel[1] = rel; c.pr_t0[1] = a; c.pr_t1[1] = z; c.pr_id[1] = p; break; }
        }
    }

    // one lean loop per tile class.  With a beam, J' is formed from the CIC
    // sums of this step's live range [cmin, cmax] and is zero off the nodes
    // cmin-2 .. cmax+3; a tile whose window misses them runs without J.
    bool needJ = c.Jc != nullptr;
    if (c.pS) needJ = c.pcmin <= c.pcmax && c.t0 + 64 * K - 1 >= c.pcmin - 2 && c.t0 <= c.pcmax + 3;
    const bool gen = needJ || c.snap_interval > 0 || c.npr > 2 || c.Hprev != nullptr;
    const bool extras = tile_strip || tile_src || tile_tf || c.npr > 0;
    // A slab-boundary tile of the E-form Kerr slab runs the pure-slab loop:
    // a vacuum cell is a slab cell with D = E, P = 0, eps = 1, chi3 = 0 when
    // the D and E updates share the coefficient (kD == ke0, jD == 1); FP64
    // then gives the vacuum update bit for bit.
    unsigned emu_mask = 0;
    bool emu_tile = false;
    auto emulate = [&](int j) {
        D[j] = E[j];
        cD[j] = cE[j];
        P[j] = Pm[j] = cP[j] = R(0);
    };
    if constexpr (KIND == SLAB_KERR_E || (RES && KIND == SLAB_LINEAR)) {
        const bool all_valid = __all(c.base >= 0 && c.base + K - 1 <= N);
        emu_tile = any_slab && !pure_slab && !extras && !gen && all_valid && sd.ke0 == sd.kD && sd.jD == R(1);
        // FP32 rounds an emulated cell's E as D - cD, so a resident tile
        // emulates where the one-block tile that owns its cells does
        if constexpr (RES && sizeof(R) == 4) emu_tile = (rt.x & kResEmu) != 0;
        if (emu_tile) {
#pragma unroll
            for (int j = 0; j < K; ++j) {
                if ((slab_mask >> j) & 1u) continue;
                emu_mask |= 1u << j;
                emulate(j);
                sA[j] = sB[j] = sC[j] = R(0);
                ie[j] = R(1);
                ied[j] = 1.0;
                kz[j] = 0.0;
            }
        }
    }

    // the launch's steps of this simulation: local steps 0 .. total-1, the
    // first at the simulation's step t0s
    const long long lo = max(0LL, (long long)sd.t_begin - gstep0);
    const int total = (int)max(0LL, min((long long)nsteps, (long long)c.T + sd.t_begin - gstep0) - lo);
    const int t0s = (int)(gstep0 + lo - sd.t_begin);
    c.emu_mask = emu_mask;
    auto run = [&](const SrcChunk<R>* pre) {
        constexpr int GM = GROUP ? M_GROUP : 0;
        if (gen || RES)      // resident tiles: the general class only (FP64)
            run_steps<R, K, KAHAN, KIND, M_MIXED | M_STRIP | M_SRC | M_GENERAL | GM>(TILE_ARGS, c, sd, pre);
        else if ((pure_slab || emu_tile) && !extras)
            run_steps<R, K, KAHAN, KIND, M_PURE_SLAB | GM>(TILE_ARGS, c, sd, pre);
        else if (!any_slab && !extras)
            run_steps<R, K, KAHAN, KIND, GM>(TILE_ARGS, c, sd, pre);
        else if (!any_slab)
            run_steps<R, K, KAHAN, KIND, M_STRIP | M_SRC | M_PROBE | GM>(TILE_ARGS, c, sd, pre);
        else
            run_steps<R, K, KAHAN, KIND, M_MIXED | M_STRIP | M_SRC | M_PROBE | GM>(TILE_ARGS, c, sd, pre);
    };
    // the compensation of E (FP32); an emulated vacuum cell carries it in cD: E - cE = D - cD
    auto comp_e = [&](int j) {
        return ((emu_mask >> j) & 1u) ? (R)((double)E[j] - ((double)D[j] - (double)cD[j])) : cE[j];
    };
    if constexpr (!RES) {
        c.s_lo = (int)lo;
        c.s_hi = (int)lo + total;
        c.t_first = t0s;
        run(nullptr);
    } else {
        // the words of this lane's cells: sent cells are owned and within S of
        // a neighbour, received cells are the valid ones off the interior;
        // lanes without one address the mailbox's spare cell, which is never
        // empty, so the loads need no branch
        const int spare = ra.stride - 1;
        const bool has_l = out0 > 0, has_r = out0 + U <= N;
        const bool any_strip = tile_strip;
        unsigned send = 0;
        int rv[K], rs[K], rp[K];
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const int n = c.base + j;
            const bool own = (interior_mask >> j) & 1u;
            if (ra.box && own && ((has_l && n < out0 + S) || (has_r && n >= out0 + U - S))) send |= 1u << j;
            const bool rec = !own && n >= 0 && n <= N && n < out0 + U + S;
            rv[j] = rec ? rt.w + n : spare;
            rs[j] = rec && ((slab_mask >> j) & 1u) ? rt.w + n : spare;
            rp[j] = rec && ((strip_mask >> j) & 1u) ? rt.w + n : spare;
        }
        constexpr int NV = kResValues<R>;
        const size_t slot_words = (size_t)NV * ra.stride;
        // every word of a cell this tile sends: w(v) is the word of value v
        auto words = [&](int j, auto&& f) {
            const int n = rt.w + c.base + j;
            f(0, n); f(1, n);
            if ((slab_mask >> j) & 1u) { f(2, n); f(3, n); f(4, n); }
            if ((strip_mask >> j) & 1u) { f(5, n); if (NV > 6) f(NV - 1, n); }
        };
        auto empty = [&](unsigned long long* slot) {
#pragma unroll
            for (int j = 0; j < K; ++j)
                if ((send >> j) & 1u)
                    words(j, [&](int v, int n) { st_dev(slot + (size_t)v * ra.stride + n, kResEmpty); });
        };
        // what the launch before this one left in the other set
        for (int q = 0; q < 3; ++q) empty(ra.other + q * slot_words);
        SrcChunk<R> sc;
        const int snap_interval = c.snap_interval;
        c.snap_interval = 0;
        c.s_lo = 0;
        sc.load(c, t0s, min(S, total));
        int q = 0;           // hand-offs so far; q3 = q % 3
        int q3 = 0;
        for (int k0 = 0; k0 < total;) {
            // A block is cut at its snapshot steps: the lean loops run up to
            // and including a snapshot step, then the row is stored from
            // registers (t = 0 takes none).
            const int kbeg = k0, kend = min(k0 + S, total);
            bool fresh = true;
            while (k0 < kend) {
                int k1 = kend;
                bool row = false;
                if (snap_interval > 0) {
                    const int ks = snap_step(t0s, k0, kend, snap_interval);
                    if (ks < kend) {
                        k1 = ks + 1;
                        row = (t0s + ks) / snap_interval < c.snap_rows;
                    }
                }
                c.t_first = t0s + k0;
                c.s_hi = k1 - k0;
                if (!fresh) sc.load(c, c.t_first, c.s_hi);
                fresh = false;
                {
                    __shared__ R spare_rows[kTileWaves][2][64];
                    R* sp = &spare_rows[wvi][0][0];
                    const int n = c.s_hi;
                    const bool odd = (k0 - kbeg) & 1;
                    const bool srcs = tile_src || tile_tf, prb = c.npr > 0, ends = srcs || prb;
                    if constexpr (K == 4)      // light tiles: plain cells only
                        res_steps<R, K, KAHAN, KIND, 0>(TILE_ARGS, c, sd, sc, sp, n, odd);
                    else if (sizeof(R) == 8 && gen) {
                        run(&sc);
                        stores_done();
                    }
                    else if ((pure_slab || emu_tile) && !extras)
                        res_steps<R, K, KAHAN, KIND, M_PURE_SLAB>(TILE_ARGS, c, sd, sc, sp, n, odd);
                    else if (!any_slab && !extras)
                        res_steps<R, K, KAHAN, KIND, 0>(TILE_ARGS, c, sd, sc, sp, n, odd);
                    else if (!any_slab && !ends)
                        res_steps<R, K, KAHAN, KIND, M_STRIP>(TILE_ARGS, c, sd, sc, sp, n, odd);
                    else if (!any_slab && !prb)
                        res_steps<R, K, KAHAN, KIND, M_STRIP | M_SRC>(TILE_ARGS, c, sd, sc, sp, n, odd);
                    else if (!any_slab && !srcs)
                        res_steps<R, K, KAHAN, KIND, M_STRIP | M_PROBE>(TILE_ARGS, c, sd, sc, sp, n, odd);
                    else if (!any_slab)
                        res_steps<R, K, KAHAN, KIND, M_STRIP | M_SRC | M_PROBE>(TILE_ARGS, c, sd, sc, sp, n, odd);
                    else if (!ends)
                        res_steps<R, K, KAHAN, KIND, M_MIXED | M_STRIP>(TILE_ARGS, c, sd, sc, sp, n, odd);
                    else
                        res_steps<R, K, KAHAN, KIND, M_MIXED | M_STRIP | M_SRC | M_PROBE>(TILE_ARGS, c, sd, sc, sp, n,
                                                                                          odd);
                }
                if (row) {
                    R* o = c.snap + (long long)((t0s + k1 - 1) / snap_interval) * (N + 1) + c.base;
#pragma unroll
                    for (int j = 0; j < K; ++j)
                        if ((interior_mask >> j) & 1u) o[j] = E[j];
                }
                k0 = k1;
            }
            if (k0 >= total || !ra.box) break;      // one block: nothing to hand over
            // ---- hand-off q ----
            unsigned long long* slot = ra.box + q3 * slot_words;
            // (the words emptied after hand-off q - 1 are in memory: the steps end with stores_done)
#pragma unroll
            for (int j = 0; j < K; ++j) {
                if (!((send >> j) & 1u)) continue;
                unsigned long long* o = slot + rt.w + c.base + j;
                const size_t st = (size_t)ra.stride;
                st_dev(o, pack2(E[j], KAHAN ? comp_e(j) : R(0)));
                st_dev(o + st, pack2(H[j], cH[j]));
                if ((slab_mask >> j) & 1u) {
                    st_dev(o + 2 * st, pack2(D[j], cD[j]));
                    st_dev(o + 3 * st, pack2(P[j], cP[j]));
                    st_dev(o + 4 * st, pack2(Pm[j], R(0)));
                }
                if ((strip_mask >> j) & 1u) {
                    st_dev(o + 5 * st, pack2(psE[j], psH[j]));
                    if constexpr (sizeof(R) == 8) st_dev(o + 6 * st, pack2(psH[j], R(0)));
                }
            }
            sc.load(c, t0s + k0, min(S, total - k0));
            int polls = 0;
            unsigned long long w[K][NV];
            for (;;) {
                bool here = true;
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    const size_t st = (size_t)ra.stride;
                    w[j][0] = ld_dev(slot + rv[j]);
                    w[j][1] = ld_dev(slot + st + rv[j]);
                    if (any_slab) {
#pragma unroll
                        for (int v = 2; v < 5; ++v) w[j][v] = ld_dev(slot + v * st + rs[j]);
                    }
                    if (any_strip) {
#pragma unroll
                        for (int v = 5; v < NV; ++v) w[j][v] = ld_dev(slot + v * st + rp[j]);
                    }
                }
#pragma unroll
                for (int j = 0; j < K; ++j) {
                    here = here && w[j][0] != kResEmpty && w[j][1] != kResEmpty;
                    if (any_slab) here = here && w[j][2] != kResEmpty && w[j][3] != kResEmpty && w[j][4] != kResEmpty;
                    if (any_strip) here = here && w[j][5] != kResEmpty && w[j][NV - 1] != kResEmpty;
                }
                if (__all(here)) break;
                if (++polls > ra.max_polls) {
                    if (lane == 0) {
                        __hip_atomic_store(ra.err, ra.ordinal, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        __hip_atomic_store(ra.herr, ra.ordinal, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    }
                    return;
                }
            }
#pragma unroll
            for (int j = 0; j < K; ++j) {
                R none;
                if (rv[j] != spare) {
                    unpack2(w[j][0], E[j], cE[j]);
                    unpack2(w[j][1], H[j], cH[j]);
                    if ((emu_mask >> j) & 1u) emulate(j);
                } else if (KAHAN && ((emu_mask >> j) & 1u)) {
                    // a block of its own would read E and its compensation back: (D, cD) is the same
                    // value, but where |cD| is half a unit of D in the last place E is not D
                    cE[j] = comp_e(j);
                    emulate(j);
                }
                if (any_slab && rs[j] != spare) {
                    unpack2(w[j][2], D[j], cD[j]);
                    unpack2(w[j][3], P[j], cP[j]);
                    unpack2(w[j][4], Pm[j], none);
                }
                if (any_strip && rp[j] != spare) {
                    unpack2(w[j][5], psE[j], psH[j]);
                    if constexpr (sizeof(R) == 8) unpack2(w[j][NV - 1], psH[j], none);
                }
            }
            // hand-off q - 1 has been read by everyone who needs it
            if (q > 0) empty(ra.box + (q3 == 0 ? 2 : q3 - 1) * slot_words);
            ++q;
            q3 = q3 == 2 ? 0 : q3 + 1;
        }
    }

    // ---------------- write back the interior ----------------
    const int po = par ^ 1;
#pragma unroll
    for (int j = 0; j < K; ++j) {
        if (!((interior_mask >> j) & 1u)) continue;
        const int n = c.base + j;
        sd.E[po][n] = E[j];
        sd.H[po][n] = H[j];
        if (KAHAN) {
            sd.cE[po][n] = comp_e(j);
            sd.cH[po][n] = cH[j];
        }
        if ((slab_mask >> j) & 1u) {
            const int i = n - F;
            sd.D[po][i] = D[j]; sd.P[po][i] = P[j]; sd.Pm[po][i] = Pm[j];
            if (KAHAN) { sd.cD[po][i] = cD[j]; sd.cP[po][i] = cP[j]; }
        }
        if ((strip_mask >> j) & 1u) {
            const int i = n < Ls ? n : Ls + (n - Rs);
            sd.psiE[po][i] = psE[j]; sd.psiH[po][i] = psH[j];
        }
    }
}

// Tile t runs as wave t % kTileWaves of workgroup t / kTileWaves, and
// consecutive workgroups go round-robin to the 8 XCDs (workgroup b runs on
// XCD b % 8), so the costly slab tiles, which are contiguous along the grid,
// spread over every XCD.  (A contiguous run of tiles per XCD keeps
// neighbours in one L2 but put all of config 2's slab on three XCDs: 25.4 us
// launches against 18.0 us here.)  Four tiles per workgroup rather than one
// cut the workgroups to dispatch by four: config 2 235.5 -> 244.0 Gcell/s
// (FP32), 239.5 -> 243.4 (FP64); two or eight per workgroup measured ~198
// (FP32) and ~181 (FP64).  A tile entry is (sim | narrow << 24, first
// interior cell): narrow tiles hold KW/2 cells per lane, the others KW, so
// tiles with costly slab cells can be made narrower than plain ones within
// one launch.
template <typename R, int KW, bool KAHAN, int KIND, bool GROUP = false>
__device__ __forceinline__ void field_tile(const SimDev<R>* __restrict__ sims, const int2* __restrict__ tiles,
                                           int tid, long long launch_idx, long long gstep0, int nsteps, int S,
                                           const PersistArgs& pa) {
    const int2 tl = tiles[tid];
    const SimDev<R>& sd = sims[tl.x & 0xffffff];
    const int4 rt{0, 0, 0, 0};
    const ResArgs ra{};
    if constexpr (KW > 1 && !GROUP) {
        if (tl.x & kTileNarrow) {
            tile_body<R, KW / 2, KAHAN, KIND, false>(sd, tl.y, launch_idx, gstep0, nsteps, S, pa, rt, ra);
            return;
        }
    }
    tile_body<R, KW, KAHAN, KIND, false, GROUP>(sd, tl.y, launch_idx, gstep0, nsteps, S, pa, rt, ra);
}

// GROUP: the halo-exchange instance; its tile list holds whole workgroups
// (ntiles a multiple of kTileWaves, every wave of a workgroup from one
// simulation), so every wave reaches the exchange barriers.
template <typename R, int KW, bool KAHAN, int KIND, bool GROUP = false>
__global__ __launch_bounds__(64 * kTileWaves) void stencil_tiles(const SimDev<R>* __restrict__ sims,
                                                                 const int2* __restrict__ tiles, int ntiles,
                                                                 long long launch_idx, long long gstep0,
                                                                 int nsteps, int S, PersistArgs pa) {
    // wave-uniform tile index, so the descriptors come in through scalar loads
    const int tid = kTileWaves * (int)blockIdx.x + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (tid >= ntiles) return;
    field_tile<R, KW, KAHAN, KIND, GROUP>(sims, tiles, tid, launch_idx, gstep0, nsteps, S, pa);
}

// Resident launch: tile t is wave t % 4 of workgroup t / 4, W workgroups fit
// on a CU, and a whole run is one launch.  A tile keeps its window in registers
// from the first step to the last; every S steps it hands its edge cells to its
// neighbours through the mailbox (tile_body) and reads theirs.
//
// Bound: the instruction stream of the slowest tile plus its hand-off.  A
// Lorentz run of 2,000 cells (one cell per lane, S = 28): 95-100 ns per step of
// the source and slab tiles and 1.25 us per hand-off (0.25 to send, one trip
// over the fabric to read), 150 ns per step in all; one launch per block took
// 459 ns.  A Kerr grid of 65,536 cells, two cells per lane, S = 48: 146-152 ns
// per step and 1.75 us per hand-off, 226 ns per step (FP32) against 273; FP64
// 305 against 503.  XCDs run at clocks that differ by a tenth, and the slowest
// one sets the pace of all tiles.
//
// Tiles hold 1 or 2 cells per lane, plain ones up to 4: light tiles (plain
// cells alone) take 46, 60 and 77-85 ns per step at 1, 2 and 4 cells per lane,
// so wide ones leave waves for narrow slab tiles.
//
// With ra.box null the launch is one block of at most S steps: nothing is
// handed over and the tiles need not be on the device together.
template <typename R, bool KAHAN, int KIND, int W>
__global__ __launch_bounds__(64 * kTileWaves, W) void stencil_resident(const SimDev<R>* __restrict__ sims,
                                                                       const int4* __restrict__ tiles, int ntiles,
                                                                       long long launch_idx, long long gstep0,
                                                                       ResArgs ra) {
    const int tid = kTileWaves * (int)blockIdx.x + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (tid >= ntiles) return;
    const int4 rt = tiles[tid];
    const SimDev<R>& sd = sims[rt.x & 0xffffff];
    if (*ra.err) return;      // an earlier launch gave up: the host runs these steps again
    const PersistArgs pa{0};
    auto body = [&](auto k, auto kind) {
        tile_body<R, decltype(k)::value, KAHAN, decltype(kind)::value, true>(sd, rt.y, launch_idx, gstep0, ra.nsteps,
                                                                             ra.S, pa, rt, ra);
    };
    using std::integral_constant;
    using Kind = integral_constant<int, KIND>;
    using Plain = integral_constant<int, SLAB_DIEL>;
    using K1 = integral_constant<int, 1>;
    using K2 = integral_constant<int, 2>;
    using K4 = integral_constant<int, 4>;
    const bool plain = KIND == SLAB_DIEL || (rt.x & kResPlain);
    if (!plain) {
        if (rt.x & kResK2) body(K2{}, Kind{});
        else body(K1{}, Kind{});
    } else if (rt.x & kResK4) {
        body(K4{}, Plain{});
    } else if (rt.x & kResK2) {
        body(K2{}, Plain{});
    } else {
        body(K1{}, Plain{});
    }
}

template <typename R, bool KAHAN, int KIND>
hipError_t launch_resident_kind(const SimDev<R>* sims, const int4* tiles, int ntiles, long long launch_idx,
                                long long gstep0, int W, const ResArgs& ra, hipStream_t st) {
    const dim3 grid((ntiles + kTileWaves - 1) / kTileWaves), block(64 * kTileWaves);
    if (W == 1)
        hipLaunchKernelGGL((stencil_resident<R, KAHAN, KIND, 1>), grid, block, 0, st, sims, tiles, ntiles, launch_idx,
                           gstep0, ra);
    else
        hipLaunchKernelGGL((stencil_resident<R, KAHAN, KIND, 2>), grid, block, 0, st, sims, tiles, ntiles, launch_idx,
                           gstep0, ra);
    return hipGetLastError();
}

// Workgroups of the resident kernel that one CU holds at once (register and
// LDS limits).
template <typename R, bool KAHAN, int KIND>
int resident_per_cu(int W) {
    int nb = 0;
    const hipError_t e =
        W == 1 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, stencil_resident<R, KAHAN, KIND, 1>, 64 * kTileWaves, 0)
               : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, stencil_resident<R, KAHAN, KIND, 2>, 64 * kTileWaves, 0);
    return e == hipSuccess ? nb : 0;
}

// Host-side launcher (called from host.hip).
// With profiling events the launch goes through hipExtLaunchKernelGGL, which
// stamps ev0/ev1 from the kernel's own dispatch packet (kernel execution time
// only, the figure a kernel trace reports).
template <typename R, int K, bool KAHAN, int KIND, bool GROUP = false>
static hipError_t launch_kp(const SimDev<R>* sims, const int2* tiles, int ntiles, long long launch_idx,
                            long long gstep0, int nsteps, int S, const PersistArgs& pa, hipStream_t st,
                            hipEvent_t ev0, hipEvent_t ev1) {
    if (GROUP && ntiles % kTileWaves) return hipErrorInvalidValue;
    const int grid = (ntiles + kTileWaves - 1) / kTileWaves;
    if (ev0 || ev1)
        hipExtLaunchKernelGGL((stencil_tiles<R, K, KAHAN, KIND, GROUP>), dim3(grid), dim3(64 * kTileWaves), 0, st, ev0,
                              ev1, 0, sims, tiles, ntiles, launch_idx, gstep0, nsteps, S, pa);
    else
        hipLaunchKernelGGL((stencil_tiles<R, K, KAHAN, KIND, GROUP>), dim3(grid), dim3(64 * kTileWaves), 0, st, sims,
                           tiles, ntiles, launch_idx, gstep0, nsteps, S, pa);
    return hipGetLastError();
}

template <typename R, int K, bool KAHAN, int KIND>
static hipError_t launch_k(const SimDev<R>* sims, const int2* tiles, int ntiles, long long launch_idx,
                           long long gstep0, int nsteps, int S, const PersistArgs& pa, hipStream_t st,
                           hipEvent_t ev0, hipEvent_t ev1) {
    if (pa.halo > 0) {
        // halo-exchange instances: K = 2 and 4 (hx / K <= kHaloMaxLanes)
        if constexpr (K == 2 || K == 4) {
            if (pa.halo % K || pa.halo / K > kHaloMaxLanes) return hipErrorInvalidValue;
            return launch_kp<R, K, KAHAN, KIND, true>(sims, tiles, ntiles, launch_idx, gstep0, nsteps, S, pa, st, ev0,
                                                     ev1);
        }
        return hipErrorInvalidValue;
    }
    return launch_kp<R, K, KAHAN, KIND>(sims, tiles, ntiles, launch_idx, gstep0, nsteps, S, pa, st, ev0, ev1);
}

template <typename R, bool KAHAN, int KIND>
hipError_t launch_kind(const SimDev<R>* sims, const int2* tiles, int ntiles, long long launch_idx,
                       long long gstep0, int nsteps, int K, int S, const PersistArgs& pa, hipStream_t st,
                       hipEvent_t ev0, hipEvent_t ev1) {
    switch (K) {
        case 1: return launch_k<R, 1, KAHAN, KIND>(sims, tiles, ntiles, launch_idx, gstep0, nsteps, S, pa, st, ev0, ev1);
        case 2: return launch_k<R, 2, KAHAN, KIND>(sims, tiles, ntiles, launch_idx, gstep0, nsteps, S, pa, st, ev0, ev1);
        case 4: return launch_k<R, 4, KAHAN, KIND>(sims, tiles, ntiles, launch_idx, gstep0, nsteps, S, pa, st, ev0, ev1);
        case 8: return launch_k<R, 8, KAHAN, KIND>(sims, tiles, ntiles, launch_idx, gstep0, nsteps, S, pa, st, ev0, ev1);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace fdtd
