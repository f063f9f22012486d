// Device-side types and helpers shared by the stencil and PIC kernels (gfx950).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fdtd {

constexpr int kMaxProbes = 16;

// What the reference's cubic a x^3 + b x^2 + c x + d shares between cells (d
// alone varies): f, g = g0 + g1 d, h = g^2/4 + F, the shift b/(3a), and
// for three real roots 1/(2i) and 2 i^(1/3) with i = sqrt(-F).
struct CubicConst {
    double f, g0, g1, F, shift, inv2i, twoj;
};

// Per-simulation descriptor as the kernels see it.  One per simulation,
// read by the tile kernel with wave-uniform (scalar) loads.  State arrays
// are ping-ponged: a launch reads [par] and writes [par^1].
template <typename R>
struct SimDev {
    int32_t N, T, Ls, Rs, F, Rr;
    int32_t slab_kind, ade, src_cell, tfsf;
    int32_t nprobe, snap_interval, snap_rows, has_current;
    int64_t launch_begin;     // global launch index of this simulation's first launch
    int64_t t_begin;          // global step at which the simulation's step 0 runs
    int32_t probe_cell[kMaxProbes], probe_t0[kMaxProbes], probe_t1[kMaxProbes];
    R ke0, kh0, keS, khS, kD, jD;
    double kerr_a, kerr_b, kerr_c, kerr_e0, kerr_lin, kerr_chi3;
    CubicConst cub;
    R *E[2], *H[2], *cE[2], *cH[2];             // N+1 cells
    R *D[2], *P[2], *Pm[2], *cD[2], *cP[2];     // R-F slab cells (Pm holds V in FP32)
    R *psiE[2], *psiH[2];                       // strip cells
    const R *s_ke, *s_kh, *s_bE, *s_cE, *s_CbE, *s_bH, *s_cH, *s_C2H;
    const R *sl_A, *sl_B, *sl_C, *sl_e;         // FP64: A,B,C ; FP32: -B, 1-A-B, C
    const R *srcE, *srcH;
    double *probe_out;                          // nprobe x T, FP64 (an FP32 field as hi - c of its
                                                // Kahan pair)
    R *snap;                                    // snap_rows x (N+1)
    double* Hprev;                              // N+1 or null: H' before the last H update of a launch
                                                // (compensated, FP64), for the energy sum
    const R *J;                                 // N+1 (PIC current, read every step)
    // with a beam attached the field step forms J' itself from the beam's
    // per-cell CIC sums (j_from_sums), so it does not wait for the scatter
    const double* pS;                           // 4 per cell, or null
    const int32_t* prange[2];                   // the beam's live range per parity
};

// One simulation's energy sum (energy.hip): the launch's final E, H (and
// FP32 compensations), H' before its last H update, and where W goes.
template <typename R>
struct EnergyJob {
    const R *E, *H, *cE, *cH;         // cE, cH null in FP64
    const double* Hprev;
    double* out;
    int N;
};

enum SlabKind { SLAB_NONE = 0, SLAB_DIEL = 1, SLAB_LINEAR = 2, SLAB_KERR_REF = 3, SLAB_KERR_E = 4 };

// Halo option of a one-block field launch.
struct PersistArgs {
    int halo;        // > 0: the workgroup halo-exchange instance, exchange period (cells = steps)
};

// A resident field launch: nsteps steps of every simulation in one launch, in
// blocks of S.  Every tile is one wave that keeps its window in registers for
// the whole launch; after a block it hands its edge cells to the tiles whose
// halos they are, through the mailbox, and takes its own halo cells from
// there.  The host launches no more tiles than the device holds at once.
//
// Mailbox: u64 words [set 2][slot 3][value kResValues][cell].  A word holds
// the value itself (FP64) or a pair of values (FP32: a field and its Kahan
// compensation), and kResEmpty, a signalling NaN pattern that no arithmetic
// produces, while nothing is there, so one load brings a value and tells that
// it has come.  Hand-off q of a launch uses slot q % 3; a tile empties the
// words of hand-off q - 1 once it has received hand-off q (its readers sent q
// after they had read q - 1), two blocks before they are written again, and
// waits until those stores are in memory (stores_done) before its next sends: a
// neighbour that has hand-off q + 1 may poll the slot for q + 2, and must not
// find q - 1 there.  Launches alternate the sets:
// each empties what the launch before it left in the other one.
//
// A wait of more than max_polls loads of the halo (each goes to memory and
// back, about 0.5 us; the tiles are not all resident: something else holds the
// device) sets *err and *herr to the launch's ordinal and ends the tile; the other tiles end the same way
// and a later launch that finds *err set returns at once.  The launch reads
// the buffers of its parity and writes only the other ones, so the host runs
// the steps again from there with one-block launches.
struct ResArgs {
    unsigned long long* box;     // this launch's set
    unsigned long long* other;   // the other set
    int stride;                  // cells of the mailbox (all simulations, with one spare)
    int nsteps, S;
    int formK;                   // FP32: cells per lane of the one-block tiles (psi_next)
    int ordinal;
    int32_t* err;                // device
    int32_t* herr;               // host memory
    int max_polls;
};
// Flags of a one-block tile entry beside the simulation's index.
constexpr int kTileNarrow = 1 << 24;     // half the cells per lane
constexpr int kTilePlain = 1 << 25;      // no D-form slab, in a launch of a slab kind (field_scatter)
// Tile of a resident launch: x = simulation | flags, y, z = first owned cell
// and the one after the last, w = the simulation's first cell in the mailbox.
constexpr int kResK2 = 1 << 24, kResK4 = 1 << 25;   // cells per lane: 1, 2 or 4
constexpr int kResPlain = 1 << 26;                  // no D-form slab cell in its window: the plain bodies
constexpr int kResEmu = 1 << 27;                    // FP32: the vacuum cells of the window are emulated slab cells
constexpr unsigned long long kResEmpty = 0x7ff45ea17fb45ea1ull;
template <typename R>
constexpr int kResValues = sizeof(R) == 8 ? 7 : 6;   // FP64 E H D P Pm psiE psiH; FP32 pairs E H D P, Pm, psiE|psiH

// First local step k in [k0, kend) of a launch that began at step t0s whose
// step t0s + k stores a snapshot row (a positive multiple of interval), or
// kend.  interval may be any positive int: no sum here passes t0s + kend.
__host__ __device__ inline int snap_step(int t0s, int k0, int kend, int interval) {
    const int k = t0s + k0 > 0 ? k0 : 1 - t0s;         // step 0 stores none
    const int past = (t0s + k) % interval;
    const int wait = past ? interval - past : 0;
    return k < kend && wait < kend - k ? k + wait : kend;
}

// Particle beam of one simulation.  Particles are kept sorted by cell
// (stable), structure of arrays, ping-ponged per step like the fields;
// start[c] is the first particle of cell c (start[N+1] = np).  Live
// particles occupy cells [2, N-3]; cells 1 and N-2 park absorbed ones, which
// keep their index from then on.
constexpr int kPicGMax = 64;        // cells per push/count group (LDS tables; the last group of a
                                    // range may take one more)
// push/count waves per workgroup (a CU holds a limited number of workgroups;
// single-wave workgroups would cap the resident waves; 8 measured slower:
// config 3 push/count 13.0 against 11.6 us); the host pads the work list to
// whole workgroups of this many waves
constexpr int kPushWaves = 4;
constexpr int kXMove = 8;           // move_block threads per push/count block boundary
constexpr int kBatch = 2;           // chunks of 64 particles fetched per memory round trip
// pic_push_group: waves per group, and chunks of 64 particles each holds in
// registers across the group's counts.  8 x 3 chunks hold 1,536 particles,
// half as many again as a group aims at.
constexpr int kMcWaves = 8;
constexpr int kMcHold = 3;
// pic_push_cell's LDS rows (dynamic shared memory): one pushed 64-particle
// chunk each (id, move and rank, frac, ux, uy, uz), xr rows for each of a
// wave's two cells; at most 8 in FP32, 4 in FP64 (about 96 KiB per workgroup)
template <typename R>
constexpr size_t kOvfRowBytes = 64 * (2 * sizeof(int32_t) + 4 * sizeof(R));
template <typename R>
constexpr int kPushCellMaxRows = sizeof(R) == 4 ? 8 : 4;
template <typename R>
struct BeamDev {
    int64_t launch_begin;  // the simulation's, copied: the parity without a load of the sim descriptor
    int32_t sim, N, np, G;
    int32_t nwaves;      // push/count waves of this beam (grid-stride over cell groups; one-cell
                         // groups: whole workgroups of kPushWaves waves)
    int32_t nnode;       // scatter node blocks of this beam (grid-stride over nodes)
    int32_t nmove;       // node blocks for its staged movers and parked particles (move_block)
    R a;                 // q dt / (2 m c)
    R jscale;            // Z0 q w c: J' of one particle per unit u_x/gamma
    R Sc;                // c dt / dz
    int32_t* cell[2];    // multi-cell beams only (a one-cell beam's cells follow from start[])
    R *frac[2], *ux[2], *uy[2], *uz[2];
    int32_t* id[2];
    int32_t* start[2];   // N+2
    int32_t* range[2];   // [cmin, cmax] of the live particles' cells (empty: cmin > cmax)
    int32_t* urange[2];  // union of the live ranges so far (where J and start[] can change)
    int32_t* park;       // [2]: the previous step's start[2] and start[N-2] (push/count -> scatter):
                         // particles below / at or above them are parked and in both buffers already
    // per-cell results of the push/count pass, valid on the live range +-1
    int32_t *cup, *cdown;  // particles moving up / down out of the cell
    double* S;             // 4 per cell: J' sums onto nodes c-1, c, c+1, c+2
    int32_t* err;        // set when an index check fails (never expected)
};

// J'[m] of a beam from its per-cell CIC sums S (4 per cell: onto nodes
// c-1 .. c+2), which exist on the live range [cmin, cmax] +-1 this step:
// J'[m] = S+2(m-2) + S+1(m-1) + S0(m) + S-1(m+1), summed in this order.
template <typename P>
__device__ __forceinline__ double j_from_sums(P S, int cmin, int cmax, int m) {
    auto Sq = [&](int c, int w) {
        return (cmin <= cmax && c >= cmin - 1 && c <= cmax + 1) ? S[4 * (size_t)c + w] : 0.0;
    };
    return Sq(m - 2, 3) + Sq(m - 1, 2) + Sq(m, 1) + Sq(m + 1, 0);
}

// ---- cross-lane shifts inside one wavefront (DPP, GFX9 wave_shr/wave_shl) ----
// shr1: lane i receives lane i-1 (lane 0 receives 0); shl1: lane i receives lane i+1.
__device__ __forceinline__ int dpp_shr1_i(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, false); }
__device__ __forceinline__ int dpp_shl1_i(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, false); }
__device__ __forceinline__ float shr1(float v) { return __int_as_float(dpp_shr1_i(__float_as_int(v))); }
__device__ __forceinline__ float shl1(float v) { return __int_as_float(dpp_shl1_i(__float_as_int(v))); }
__device__ __forceinline__ double shr1(double v) {
    long long b = __double_as_longlong(v);
    int lo = dpp_shr1_i((int)(b & 0xffffffffll)), hi = dpp_shr1_i((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double shl1(double v) {
    long long b = __double_as_longlong(v);
    int lo = dpp_shl1_i((int)(b & 0xffffffffll)), hi = dpp_shl1_i((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Kahan-compensated s += inc; (s - c) is the compensated value.
template <typename R>
__device__ __forceinline__ void kahan_add(R& s, R& c, R inc) {
    R y = inc - c;
    R t = s + y;
    c = (t - s) - y;
    s = t;
}

// a * b + c.  FP64: rounded once (an explicit FMA); the FP64 translation
// units are compiled without FMA contraction (-ffp-contract=off), so every
// fused product is one written out here and a cell's update is the same
// sequence of roundings in every tile class and every (K, S) tiling.  FP32:
// the plain expression, fused as the compiler chooses (the FP32 field units
// keep contraction on; their results are held to a tolerance, and the
// compensated sums absorb the difference).
__device__ __forceinline__ double fmr(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmr(float a, float b, float c) { return a * b + c; }

// Kahan-compensated s += a * b (FP64: a * b - c rounded once).
template <typename R>
__device__ __forceinline__ void kahan_fma(R& s, R& c, R a, R b) {
    R y = fmr(a, b, -c);
    R t = s + y;
    c = (t - s) - y;
    s = t;
}

// ---- Kerr, reference path: Re(roots[0]) of a x^3 + b x^2 + c x + d (FP64) ----
// Restates the 1728.org closed form vendored at CubicEquationSolver.py:29-105
// (branch order and tests kept), as consumed by Nonlin_Cubic_Solver
// (BaseFDTD11.py:834-838): only roots[0] is used, |d| <= 1e-8 gives 0.
__host__ __device__ inline CubicConst cubic_const(double a, double b, double c) {
    CubicConst k{};
    if (a == 0.0) return k;
    k.f = ((3.0 * c / a) - (pow(b, 2.0) / pow(a, 2.0))) / 3.0;
    k.g0 = (((2.0 * pow(b, 3.0)) / pow(a, 3.0)) - ((9.0 * b * c) / pow(a, 2.0))) / 27.0;
    k.g1 = 1.0 / a;
    k.F = pow(k.f, 3.0) / 27.0;
    k.shift = b / (3.0 * a);
    const double i = k.F < 0.0 ? sqrt(-k.F) : 0.0;         // F > 0: one real root whatever d is
    k.inv2i = i > 0.0 ? 1.0 / (2.0 * i) : 0.0;
    k.twoj = 2.0 * cbrt(i);
    return k;
}

// The root from those constants.  Bound by its FP64 operations, which every
// slab cell spends once per step: a cell pays two cube roots (or an acos and a
// polynomial) and one square root; the powers of a, b and f are
// not its own.  S + U takes each cube root of its own sum, as the reference
// does.  19,250 steps of a 7,700-cell slab, one cell per lane: 17.2 ms with the
// divisions by a and 27, 16.4 ms without them, 73 ms when each cell formed f, h
// and the roots through pow and cos.  Over random coefficients the distance to
// the 128-bit root is smaller than that form's in the mean (0.0003 to 0.99 of
// it by range), and at worst the same or less; where both are near a
// cancellation the worst of 100,000 lies between 0.92 and 1.06 of it from seed
// to seed.
__device__ __forceinline__ double cubic_root0_1728(double a, double b, double c, const CubicConst& k, double d) {
    if (!(fabs(d) > 1e-8)) return 0.0;
    if (a == 0.0 && b == 0.0) return (-d * 1.0) / c;
    if (a == 0.0) {
        const double disc = c * c - 4.0 * b * d;
        if (disc >= 0.0) return (-c + sqrt(disc)) / (2.0 * b);
        return -c / (2.0 * b);               // real part of the complex pair
    }
    const double g = fma(k.g1, d, k.g0);
    const double h = fma(0.25 * g, g, k.F);
    if (h <= 0.0) {
        if (k.f == 0.0 && g == 0.0 && h == 0.0) return -cbrt(d / a);
        // 2 i^(1/3) cos(acos(-g/(2i))/3): the angle lies in [0, pi/3], where the
        // cosine's Taylor series to x^20 leaves 3e-21
        const double x = acos(fmin(1.0, fmax(-1.0, -g * k.inv2i))) * (1.0 / 3.0);
        const double q = -x * x;
        double t = 1.0 / 2432902008176640000.0;
        t = fma(t, q, 1.0 / 6402373705728000.0);
        t = fma(t, q, 1.0 / 20922789888000.0);
        t = fma(t, q, 1.0 / 87178291200.0);
        t = fma(t, q, 1.0 / 479001600.0);
        t = fma(t, q, 1.0 / 3628800.0);
        t = fma(t, q, 1.0 / 40320.0);
        t = fma(t, q, 1.0 / 720.0);
        t = fma(t, q, 1.0 / 24.0);
        t = fma(t, q, 1.0 / 2.0);
        t = fma(t, q, 1.0);
        return k.twoj * t - k.shift;
    }
    const double sh = sqrt(h);
    return (cbrt(sh - 0.5 * g) + cbrt(-0.5 * g - sh)) - k.shift;
}

// ---- Kerr, physical path: real root of chi3 E^3 + eps E = u (chi3 >= 0), FP64 ----
// With x = u/eps and z = chi3 x^2/eps (27 z / 4 is the ratio q^2/(4 p^3/27) that
// sets the sign of the depressed cubic's discriminant), E = x*y where
// y = 1 - z y^3.  For |z| < 0.01 y is the alternating Fuss-Catalan series
// sum_k (-1)^k C(3k,k)/(2k+1) z^k (14 terms, error < 1e-16); otherwise the
// hyperbolic closed form E = -2 s sinh(asinh(3q/(2p s))/3), s = sqrt(p/3).
__device__ inline double kerr_root_e(double u, double eps, double chi3) {
    const double x = u / eps;
    if (chi3 == 0.0) return x;
    const double z = chi3 * x * x / eps;
    if (z < 0.01) {
        double y = 300830572.0;
        y = fma(y, -z, 50067108.0);
        y = fma(y, -z, 8414640.0);
        y = fma(y, -z, 1430715.0);
        y = fma(y, -z, 246675.0);
        y = fma(y, -z, 43263.0);
        y = fma(y, -z, 7752.0);
        y = fma(y, -z, 1428.0);
        y = fma(y, -z, 273.0);
        y = fma(y, -z, 55.0);
        y = fma(y, -z, 12.0);
        y = fma(y, -z, 3.0);
        y = fma(y, -z, 1.0);
        y = fma(y, -z, 1.0);
        return x * y;
    }
    const double p = eps / chi3, q = -u / chi3;
    const double s = sqrt(p / 3.0);
    return -2.0 * s * sinh(asinh((1.5 * q / p) / s) / 3.0);
}

}  // namespace fdtd
