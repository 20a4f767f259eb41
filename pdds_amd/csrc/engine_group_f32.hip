// engine_group_f32.hip -- the group path kernel's FP32 instantiations and launchers.
#include "../../include/pdds_engine.h"
#include "engine_group.h"

namespace pdds {

template <int PDE> static hipError_t group_f32(bool mixed, int lanes, const PathLaunch &l, const PathKernelArgs &a) {
    if constexpr (const_motion<PDE>()) {
        if (lanes == 16)
            return mixed ? l.go(group_kernel<float, PDE, true, 16>, a, NoOut{}) : l.go(group_kernel<float, PDE, false, 16>, a, NoOut{});
        if (lanes == 1)
            return mixed ? l.go(group_kernel<float, PDE, true, 1>, a, NoOut{}) : l.go(group_kernel<float, PDE, false, 1>, a, NoOut{});
    }
    return mixed ? l.go(group_kernel<float, PDE, true, 4>, a, NoOut{}) : l.go(group_kernel<float, PDE, false, 4>, a, NoOut{});
}

hipError_t launch_group_f32(int pde, bool mixed, int lanes, const PathLaunch &l, const PathKernelArgs &a) {
    if (a.pp.refl) return hipErrorInvalidValue;
    switch (pde) {
        case PDE_SINSIN: return group_f32<PDE_SINSIN>(mixed, lanes, l, a);
        case PDE_VARCOEF: return group_f32<PDE_VARCOEF>(mixed, lanes, l, a);
        case PDE_VARCOEF_LUT: return group_f32<PDE_VARCOEF_LUT>(mixed, lanes, l, a);
        case PDE_HELMHOLTZ: return group_f32<PDE_HELMHOLTZ>(mixed, lanes, l, a);
        case PDE_TABLE: return group_f32<PDE_TABLE>(mixed, lanes, l, a);
        default: return hipErrorInvalidValue;
    }
}

template <int PDE> static hipError_t group_records_f32(const PathLaunch &l, const PathKernelArgs &a, const PathOut &o) {
    return l.go(group_kernel<float, PDE, false, 4, false, PathOut>, a, o);
}

// one phase, without reflecting sides; not the coefficient LUT, whose records take one lane to a path
hipError_t launch_group_records_f32(int pde, const PathLaunch &l, const PathKernelArgs &a, const PathOut &o) {
    if (a.pp.refl || o.phase2) return hipErrorInvalidValue;
    switch (pde) {
        case PDE_SINSIN: return group_records_f32<PDE_SINSIN>(l, a, o);
        case PDE_VARCOEF: return group_records_f32<PDE_VARCOEF>(l, a, o);
        case PDE_HELMHOLTZ: return group_records_f32<PDE_HELMHOLTZ>(l, a, o);
        case PDE_TABLE: return group_records_f32<PDE_TABLE>(l, a, o);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace pdds
