// engine_group_f64.hip -- the group path kernel's FP64 instantiations and launchers.
#include "../../include/pdds_engine.h"
#include "engine_group.h"

namespace pdds {

// Lanes that carry one path of a launch of the group kernel.  One lane is the cheapest per step (the
// step-ordered sums are repeated by every lane of a group), 16 finish a path soonest.  With one lane
// a card holds 1024 to 2048 paths per CU; it pays once every lane has several paths one after
// another, and below that a launch lasts as long as its longest path.  Measured on 256 CUs:
// FP32 Helmholtz server burst (15.5 M paths) 83 ms with one lane, 119 with four; FP32 Poisson
// assembly (0.6 M) 3.4 and 3.5; FP64 Helmholtz assembly (1.9 M) 2.5 and 3.1, FP64 recorded run
// (0.77 M) 4.0 and 3.6; with four and sixteen lanes: 140 k FP32 paths 1.25 and 1.16 ms, 5000 FP64
// paths 0.73 and 0.58, 4000 0.34 and 0.29.
// Lanes that read a table repeat the reads of their path's other lanes, which pays while a launch lasts as
// long as its longest path.  By groups and by one lane in the persistent kernel: the tabulated problem's
// 32 reads of 16 bytes a step (h = 2e-4; 4 x 4 subdomains, 128 x 128 texels) FP64 6 10^4 paths 3.4 and 4.0 ms,
// 1.2 10^5 4.3 and 4.4, 2 10^5 5.2 and 5.2; FP32 2.7 and 3.0, 5.1 and 5.1, 6.2 and 5.6, and with 512 x 512
// texels on 8 x 8 1.0 and 0.73, 1.6 and 0.96, 2.2 and 1.15.  The LUT's 20 reads (4 x 4 subdomains and points
// on the whole square, 64 x 64 samples, h = 1e-3 of the domain): FP64 6.5 10^4 paths 14.5 and 16.8, 5.2 and
// 5.1, 10^5 15.9 and 16.9, 6.7 and 6.7, 1.3 10^5 17.1 and 19.3, 6.6 and 6.8, 5 10^5 27 and 23, 13.5 and 10.2;
// FP32 11.5 and 15.0, 2.7 and 3.0, 12.5 and 14.9, 4.0 and 3.1, 13.7 and 15.2, 4.2 and 3.2, 20 and 19, 9.1 and
// 6.6; with 512 x 512 samples 10^5 FP64 17.4 and 17.3, 8.3 and 7.0, FP32 13.7 and 15.4, 6.4 and 3.7.
int group_lanes(int pde, int precision, bool refl, int n_cu, int64_t paths) {
    const bool fp64 = precision == PDDS_FP64;
    const bool moves = pde == PDE_SINSIN || pde == PDE_HELMHOLTZ || pde == PDE_MONEGROS;   // const_motion
    if (!fp64 && (refl || pde == PDE_MONEGROS)) return 0;
    if ((!moves || refl) && paths > (int64_t)n_cu * 2048) return 0;
    if (pde == PDE_TABLE && paths > (int64_t)n_cu * (fp64 ? 512 : 256)) return 0;
    if (pde == PDE_VARCOEF_LUT && paths > (int64_t)n_cu * (fp64 ? 384 : 256)) return 0;
    if (!moves) return 4;
    if (refl) return paths > (int64_t)n_cu * 32 ? 4 : 16;
    if (paths >= (int64_t)n_cu * (fp64 ? 4096 : 2048)) return 1;
    return paths > (int64_t)n_cu * 32 ? 4 : 16;
}

template <int PDE> static hipError_t group_f64(bool mixed, int lanes, const PathLaunch &l, const PathKernelArgs &a) {
    if constexpr (const_motion<PDE>()) {
        if (a.pp.refl)
            return lanes == 16 ? l.go(group_kernel<double, PDE, false, 16, true>, a, NoOut{})
                               : l.go(group_kernel<double, PDE, false, 4, true>, a, NoOut{});
        if (lanes == 16)
            return mixed ? l.go(group_kernel<double, PDE, true, 16>, a, NoOut{}) : l.go(group_kernel<double, PDE, false, 16>, a, NoOut{});
        if (lanes == 1)
            return mixed ? l.go(group_kernel<double, PDE, true, 1>, a, NoOut{}) : l.go(group_kernel<double, PDE, false, 1>, a, NoOut{});
    } else if (a.pp.refl) {
        return l.go(group_kernel<double, PDE, false, 4, true>, a, NoOut{});
    }
    return mixed ? l.go(group_kernel<double, PDE, true, 4>, a, NoOut{}) : l.go(group_kernel<double, PDE, false, 4>, a, NoOut{});
}

hipError_t launch_group_f64(int pde, bool mixed, int lanes, const PathLaunch &l, const PathKernelArgs &a) {
    if (mixed && a.pp.refl) return hipErrorInvalidValue;
    switch (pde) {
        case PDE_MONEGROS: return group_f64<PDE_MONEGROS>(mixed, lanes, l, a);
        case PDE_SINSIN: return group_f64<PDE_SINSIN>(mixed, lanes, l, a);
        case PDE_VARCOEF: return group_f64<PDE_VARCOEF>(mixed, lanes, l, a);
        case PDE_VARCOEF_LUT: return group_f64<PDE_VARCOEF_LUT>(mixed, lanes, l, a);
        case PDE_HELMHOLTZ: return group_f64<PDE_HELMHOLTZ>(mixed, lanes, l, a);
        case PDE_TABLE: return group_f64<PDE_TABLE>(mixed, lanes, l, a);
        default: return hipErrorInvalidValue;
    }
}

template <int PDE> static hipError_t group_records_f64(const PathLaunch &l, const PathKernelArgs &a, const PathOut &o) {
    return a.pp.refl ? l.go(group_kernel<double, PDE, false, 4, true, PathOut>, a, o)
                     : l.go(group_kernel<double, PDE, false, 4, false, PathOut>, a, o);
}

hipError_t launch_group_records_f64(int pde, const PathLaunch &l, const PathKernelArgs &a, const PathOut &o) {
    switch (pde) {
        case PDE_MONEGROS: return group_records_f64<PDE_MONEGROS>(l, a, o);
        case PDE_SINSIN: return group_records_f64<PDE_SINSIN>(l, a, o);
        case PDE_VARCOEF: return group_records_f64<PDE_VARCOEF>(l, a, o);
        case PDE_VARCOEF_LUT: return group_records_f64<PDE_VARCOEF_LUT>(l, a, o);
        case PDE_HELMHOLTZ: return group_records_f64<PDE_HELMHOLTZ>(l, a, o);
        case PDE_TABLE: return group_records_f64<PDE_TABLE>(l, a, o);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace pdds
