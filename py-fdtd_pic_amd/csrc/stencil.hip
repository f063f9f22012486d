// Field-step launchers (called from host.hip): dispatch on the slab kind to
// the instances compiled in stencil_<precision>_<kind>.hip.
#include <algorithm>

#include "field_scatter.hpp"

namespace fdtd {

extern template hipError_t launch_kind<float, true, SLAB_DIEL>(const SimDev<float>*, const int2*, int, long long, long long, int, int, int, const PersistArgs&, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_kind<float, true, SLAB_LINEAR>(const SimDev<float>*, const int2*, int, long long, long long, int, int, int, const PersistArgs&, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_kind<float, true, SLAB_KERR_E>(const SimDev<float>*, const int2*, int, long long, long long, int, int, int, const PersistArgs&, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_kind<double, false, SLAB_DIEL>(const SimDev<double>*, const int2*, int, long long, long long, int, int, int, const PersistArgs&, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_kind<double, false, SLAB_LINEAR>(const SimDev<double>*, const int2*, int, long long, long long, int, int, int, const PersistArgs&, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_kind<double, false, SLAB_KERR_E>(const SimDev<double>*, const int2*, int, long long, long long, int, int, int, const PersistArgs&, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_kind<double, false, SLAB_KERR_REF>(const SimDev<double>*, const int2*, int, long long, long long, int, int, int, const PersistArgs&, hipStream_t, hipEvent_t, hipEvent_t);

extern template hipError_t launch_resident_kind<float, true, SLAB_DIEL>(const SimDev<float>*, const int4*, int, long long, long long, int, const ResArgs&, hipStream_t);
extern template int resident_per_cu<float, true, SLAB_DIEL>(int);
extern template hipError_t launch_resident_kind<float, true, SLAB_LINEAR>(const SimDev<float>*, const int4*, int, long long, long long, int, const ResArgs&, hipStream_t);
extern template int resident_per_cu<float, true, SLAB_LINEAR>(int);
extern template hipError_t launch_resident_kind<float, true, SLAB_KERR_E>(const SimDev<float>*, const int4*, int, long long, long long, int, const ResArgs&, hipStream_t);
extern template int resident_per_cu<float, true, SLAB_KERR_E>(int);
extern template hipError_t launch_resident_kind<double, false, SLAB_DIEL>(const SimDev<double>*, const int4*, int, long long, long long, int, const ResArgs&, hipStream_t);
extern template int resident_per_cu<double, false, SLAB_DIEL>(int);
extern template hipError_t launch_resident_kind<double, false, SLAB_LINEAR>(const SimDev<double>*, const int4*, int, long long, long long, int, const ResArgs&, hipStream_t);
extern template int resident_per_cu<double, false, SLAB_LINEAR>(int);
extern template hipError_t launch_resident_kind<double, false, SLAB_KERR_E>(const SimDev<double>*, const int4*, int, long long, long long, int, const ResArgs&, hipStream_t);
extern template int resident_per_cu<double, false, SLAB_KERR_E>(int);
extern template hipError_t launch_resident_kind<double, false, SLAB_KERR_REF>(const SimDev<double>*, const int4*, int, long long, long long, int, const ResArgs&, hipStream_t);
extern template int resident_per_cu<double, false, SLAB_KERR_REF>(int);

extern template hipError_t launch_fused_kind<float, true, SLAB_DIEL>(const SimDev<float>*, const int2*, int, long long, long long, int, int, int, const BeamDev<float>*, const int2*, int, int, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_fused_kind<float, true, SLAB_LINEAR>(const SimDev<float>*, const int2*, int, long long, long long, int, int, int, const BeamDev<float>*, const int2*, int, int, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_fused_kind<float, true, SLAB_KERR_E>(const SimDev<float>*, const int2*, int, long long, long long, int, int, int, const BeamDev<float>*, const int2*, int, int, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_fused_kind<double, false, SLAB_DIEL>(const SimDev<double>*, const int2*, int, long long, long long, int, int, int, const BeamDev<double>*, const int2*, int, int, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_fused_kind<double, false, SLAB_LINEAR>(const SimDev<double>*, const int2*, int, long long, long long, int, int, int, const BeamDev<double>*, const int2*, int, int, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_fused_kind<double, false, SLAB_KERR_E>(const SimDev<double>*, const int2*, int, long long, long long, int, int, int, const BeamDev<double>*, const int2*, int, int, hipStream_t, hipEvent_t, hipEvent_t);
extern template hipError_t launch_fused_kind<double, false, SLAB_KERR_REF>(const SimDev<double>*, const int2*, int, long long, long long, int, int, int, const BeamDev<double>*, const int2*, int, int, hipStream_t, hipEvent_t, hipEvent_t);

// kind: 0 (no D-form slab: NONE or DIEL share the DIEL kernel), SLAB_LINEAR,
// SLAB_KERR_REF (FP64 only), SLAB_KERR_E.
template <typename R, bool KAHAN>
hipError_t launch_stencil(const SimDev<R>* sims, const int2* tiles, int ntiles, long long launch_idx,
                          long long gstep0, int nsteps, int K, int S, int kind, const PersistArgs& pa,
                          hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
#define FDTD_FIELD(KIND) \
    launch_kind<R, KAHAN, KIND>(sims, tiles, ntiles, launch_idx, gstep0, nsteps, K, S, pa, st, ev0, ev1)
    switch (kind) {
        case SLAB_NONE:
        case SLAB_DIEL: return FDTD_FIELD(SLAB_DIEL);
        case SLAB_LINEAR: return FDTD_FIELD(SLAB_LINEAR);
        case SLAB_KERR_E: return FDTD_FIELD(SLAB_KERR_E);
        case SLAB_KERR_REF:
            if constexpr (sizeof(R) == 8) return FDTD_FIELD(SLAB_KERR_REF);
            return hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
#undef FDTD_FIELD
}

template hipError_t launch_stencil<double, false>(const SimDev<double>*, const int2*, int, long long,
                                                  long long, int, int, int, int, const PersistArgs&, hipStream_t,
                                                  hipEvent_t, hipEvent_t);
template hipError_t launch_stencil<float, true>(const SimDev<float>*, const int2*, int, long long,
                                                long long, int, int, int, int, const PersistArgs&, hipStream_t,
                                                hipEvent_t, hipEvent_t);

// Empties the mailbox of resident launches: `values` rows of `stride` words;
// the spare word at a row's end always holds something.
__global__ __launch_bounds__(256) void box_empty(unsigned long long* __restrict__ box, size_t values, int stride) {
    const size_t n = values * (size_t)stride;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        box[i] = i % (size_t)stride == (size_t)stride - 1 ? 0ull : kResEmpty;
}
hipError_t launch_box_empty(unsigned long long* box, size_t values, int stride, hipStream_t st) {
    const size_t n = values * (size_t)stride;
    hipLaunchKernelGGL(box_empty, dim3((unsigned)std::min<size_t>((n + 255) / 256, 2048)), dim3(256), 0, st, box, values,
                       stride);
    return hipGetLastError();
}

// A resident launch of every simulation (kinds as launch_stencil: the kind of
// the D-form slabs, beside which simulations without one run too).
template <typename R, bool KAHAN>
hipError_t launch_resident(const SimDev<R>* sims, const int4* tiles, int ntiles, long long launch_idx,
                           long long gstep0, int kind, int W, const ResArgs& ra, hipStream_t st) {
#define FDTD_RES(KIND) launch_resident_kind<R, KAHAN, KIND>(sims, tiles, ntiles, launch_idx, gstep0, W, ra, st)
    switch (kind) {
        case SLAB_NONE:
        case SLAB_DIEL: return FDTD_RES(SLAB_DIEL);
        case SLAB_LINEAR: return FDTD_RES(SLAB_LINEAR);
        case SLAB_KERR_E: return FDTD_RES(SLAB_KERR_E);
        case SLAB_KERR_REF:
            if constexpr (sizeof(R) == 8) return FDTD_RES(SLAB_KERR_REF);
            return hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
#undef FDTD_RES
}
template hipError_t launch_resident<double, false>(const SimDev<double>*, const int4*, int, long long, long long, int,
                                                   int, const ResArgs&, hipStream_t);
template hipError_t launch_resident<float, true>(const SimDev<float>*, const int4*, int, long long, long long, int,
                                                 int, const ResArgs&, hipStream_t);

// Resident workgroups one CU holds at once, for a slab kind.
template <typename R, bool KAHAN>
int resident_capacity_per_cu(int kind, int W) {
    switch (kind) {
        case SLAB_NONE:
        case SLAB_DIEL: return resident_per_cu<R, KAHAN, SLAB_DIEL>(W);
        case SLAB_LINEAR: return resident_per_cu<R, KAHAN, SLAB_LINEAR>(W);
        case SLAB_KERR_E: return resident_per_cu<R, KAHAN, SLAB_KERR_E>(W);
        case SLAB_KERR_REF:
            if constexpr (sizeof(R) == 8) return resident_per_cu<R, KAHAN, SLAB_KERR_REF>(W);
            return 0;
        default: return 0;
    }
}

template int resident_capacity_per_cu<double, false>(int, int);
template int resident_capacity_per_cu<float, true>(int, int);

// The field step of one tile group and the particle scatter in one launch
// (field_scatter.hpp); same kinds as launch_stencil.
template <typename R, bool KAHAN>
hipError_t launch_field_scatter(const SimDev<R>* sims, const int2* tiles, int ntiles, long long launch_idx,
                                long long gstep0, int nsteps, int K, int S, int kind, const BeamDev<R>* beams,
                                const int2* sblocks, int nsblocks, int nfirst, hipStream_t st, hipEvent_t ev0,
                                hipEvent_t ev1) {
#define FDTD_FUSED(KIND) \
    launch_fused_kind<R, KAHAN, KIND>(sims, tiles, ntiles, launch_idx, gstep0, nsteps, K, S, beams, sblocks, nsblocks, \
                                      nfirst, st, ev0, ev1)
    switch (kind) {
        case SLAB_NONE:
        case SLAB_DIEL: return FDTD_FUSED(SLAB_DIEL);
        case SLAB_LINEAR: return FDTD_FUSED(SLAB_LINEAR);
        case SLAB_KERR_E: return FDTD_FUSED(SLAB_KERR_E);
        case SLAB_KERR_REF:
            if constexpr (sizeof(R) == 8) return FDTD_FUSED(SLAB_KERR_REF);
            return hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
#undef FDTD_FUSED
}

template hipError_t launch_field_scatter<double, false>(const SimDev<double>*, const int2*, int, long long, long long,
                                                        int, int, int, int, const BeamDev<double>*, const int2*, int,
                                                        int, hipStream_t, hipEvent_t, hipEvent_t);
template hipError_t launch_field_scatter<float, true>(const SimDev<float>*, const int2*, int, long long, long long,
                                                      int, int, int, int, const BeamDev<float>*, const int2*, int,
                                                      int, hipStream_t, hipEvent_t, hipEvent_t);

}  // namespace fdtd
