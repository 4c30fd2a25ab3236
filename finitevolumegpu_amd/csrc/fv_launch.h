// Launch helpers shared by the two arithmetic-policy translation units.
#pragma once

#include <hip/hip_runtime.h>

#include "fv_ensemble.h"
#include "fv_step.h"
#include "fv_substep.h"

namespace fvmi {

enum SchemeId : int { SCHEME_KP07 = 0, SCHEME_HLL2 = 1, SCHEME_WAF = 2, SCHEME_EULER = 3 };

// Columns per lane of each scheme's march in each arithmetic policy (the kC
// of its policy struct) and the output columns of one of its strips.
inline int scheme_cols_per_lane(int scheme, int math) {
    static_assert(SweKP07<MathFast>::kC == FVMI_SWE_COLS && SweHLL2<MathFast>::kC == FVMI_SWE_COLS &&
                      SweWAF<MathFast>::kC == 1 && EulerKP07<MathFast>::kC == 2 &&
                      SweKP07<MathExact>::kC == FVMI_SWE_COLS && SweHLL2<MathExact>::kC == FVMI_SWE_COLS &&
                      SweWAF<MathExact>::kC == 1 && EulerKP07<MathExact>::kC == 1,
                  "scheme_cols_per_lane follows the policy structs");
    if (scheme == SCHEME_WAF) return 1;
    if (scheme == SCHEME_EULER) return math == FVMI_MATH_EXACT ? 1 : 2;
    return FVMI_SWE_COLS;
}
inline int scheme_strip_cols(int scheme, int math) {
    return scheme_cols_per_lane(scheme, math) == 2 ? strip_cols<2>() : strip_cols<1>();
}

// The whole-step kernels (one column per lane).
using StepKP07 = SweKP07<MathFast, 1>;
using StepHLL2 = SweHLL2<MathFast, 1>;
using StepEuler = EulerKP07<MathFast, 1>;

// Whether a whole step of this grid can be one launch (fv_step.h, fv_rk2.h).
inline bool step_grid_fits(const SubstepArgs& a) {
    if (a.nx < kStepMinSide || a.ny < kStepMinSide) return false;
    if (a.seg_rows > 0 && a.seg_rows < kStepMinSegRows) return false;
    const int w = a.bc & 0xF, e = (a.bc >> 8) & 0xF, s = (a.bc >> 16) & 0xF, n = (a.bc >> 24) & 0xF;
    if (w == BC_DIRICHLET || e == BC_DIRICHLET || s == BC_DIRICHLET || n == BC_DIRICHLET) return false;
    // a periodic edge opposite to another kind wraps to cells whose own
    // neighbours are that kind's ghosts, which the images marched along are not
    return (w == BC_PERIODIC) == (e == BC_PERIODIC) && (s == BC_PERIODIC) == (n == BC_PERIODIC);
}

// Whether a dimensionally split step is.  Fast arithmetic only: the exact kernels
// and WAF are bound by VALU issue already as substeps (4096^2: 177 us for
// KP07_dimsplit, 262 for WAF, against 79 us for their bytes), so that the wider
// halo is expected to cost more than the memory passes saved (a whole exact step has
// not been built and timed).
inline bool step_is_fused(int scheme, int math, const SubstepArgs& a) {
    return math != FVMI_MATH_EXACT && scheme != SCHEME_WAF && step_grid_fits(a);
}

// Costs of the schemes' segments (fitted to steps of one simulator at 256^2 to
// 2000^2 over segments of 2 to 40 rows).  Of a split step's two substeps one has
// the CFL minimum.
inline SegmentCost substep_cost(int math) {
    return {4, 2, math == FVMI_MATH_EXACT ? 0.5f : 0.25f, 0.005f};
}
// Percent of the equal segments' waves that the round-weighted split of a whole
// step has to put to work.  8192^2 (24 of 27 segments a strip, 89 %), rounds and
// equal segments, one simulator and three in turn: KP07_dimsplit 756 and 711 us,
// 715 and 683, HLL2 949 and 883, 894 and 826, Euler 1239 and 1183, 1140 and 1049,
// KP07 653 and 618, 621 and 622; 9500x7000 KP07_dimsplit 773 and 683; 7500^2 (93 %)
// even; 5500^2 (98 %) 317 and 323.  The weights and the shortest part are those of
// the substep kernel; at 3000^2 equal segments were 4 % faster than these rounds.
constexpr int kStepMinFill = 93;
inline SegmentCost step_cost() { return {2 * kStepHalo, kStepMinSegRows, 0.45f, 0.01f}; }

// Fills the decomposition fields of `a` (sub-area, launch shape, device size)
// and returns the grid size to launch.  seg_rows == 0 picks the shape:
//   * the round-weighted plan (round_segment) when `round_ok`, the workgroups
//     have 4 waves, the XCD remap is on and every strip holds row groups long
//     enough for their shortest part to have `min_part` rows;
//   * otherwise segments of equal length (balanced_segment_rows): at most
//     `waves_per_simd` waves on every SIMD of the device (one more would run
//     after all the others).
inline int plan_substep(SubstepArgs& a, int cu_count, const SegmentCost& cost, bool round_ok = false,
                        int min_fill = 0, int waves_per_simd = 4, int min_part = 16) {
    const int wx = a.x1 - a.x0;
    a.rows_per_strip = a.y1 - a.y0;
    a.strips_x = (wx + a.strip_cols - 1) / a.strip_cols;
    a.round_plan = 0;
    a.xcds = 8;
    a.cus_per_xcd = cu_count / 8;
    a.gps = a.grows = 0;
    int gps = 0, grows = 0;
    if (round_ok && a.seg_rows <= 0 && a.xcd_remap &&
        round_split_fits(a.strips_x, a.rows_per_strip, a.waves_per_block, cu_count, min_part, min_fill, gps, grows)) {
        a.round_plan = 1;
        a.gps = gps;
        a.grows = grows;
        a.seg_rows = grows / kRounds;  // nominal, for reporting
        a.segs_per_strip = gps * kRounds;
        a.num_waves = a.strips_x * gps * kRounds;
        a.num_blocks = kRounds * cu_count;
        return a.num_blocks;
    }
    if (a.seg_rows <= 0)
        a.seg_rows = balanced_segment_rows(a.rows_per_strip, a.strips_x, cu_count, waves_per_simd, cost);
    a.segs_per_strip = (a.rows_per_strip + a.seg_rows - 1) / a.seg_rows;
    a.num_waves = a.strips_x * a.segs_per_strip;
    a.num_blocks = (a.num_waves + a.waves_per_block - 1) / a.waves_per_block;
    int grid = a.num_blocks;
    if (a.xcd_remap) grid = ((grid + 7) / 8) * 8;
    return grid;
}

// The plan of a whole step.  Equal segments of a large grid fill the device once,
// so that a lone launch ends with SIMDs at one wave; for Euler, whose rows cost most,
// segments above this length are halved.  One simulator, and three in turn, as they
// are, halved, and the two substep launches: 7300^2 920, 872 and 907 us, 835, 855
// and 953; 8192^2 1180, 1117 and 1134, 1061, 1110 and 1227; 10000^2 1783, 1658 and
// 1684, 1561, 1583 and 1846.  KP07_dimsplit and HLL2 8192^2 gain 2 and 3 % alone and
// lose 4 and 2 % in turn: theirs stay.
constexpr int kEulerMaxRows = 200;
inline int plan_whole_step(SubstepArgs& a, int scheme, int cu_count) {
    const bool chosen = a.seg_rows <= 0;
    const int grid = plan_substep(a, cu_count, step_cost(), true, kStepMinFill);
    if (!chosen || scheme != SCHEME_EULER || a.round_plan || a.seg_rows <= kEulerMaxRows) return grid;
    a.seg_rows = (a.seg_rows + 1) / 2;
    return plan_substep(a, cu_count, step_cost());
}

inline unsigned substep_lds(const SubstepArgs& a) {
    return block_cfl_bytes(block_cfl(a.round_plan, a.step == 1 ? a.cfl : nullptr));
}

// One scheme's kernel (each translation unit instantiates the ones it owns).
template <class S, class M>
hipError_t launch_substep_scheme(const SubstepArgs& a, int grid, hipStream_t stream) {
    hipLaunchKernelGGL((substep_kernel<S, M>), dim3(grid), dim3(kLanes * a.waves_per_block), substep_lds(a), stream, a);
    return hipGetLastError();
}

template <class M>
hipError_t launch_substep(int scheme, SubstepArgs a, int grid, hipStream_t stream) {
    const dim3 block(kLanes * a.waves_per_block);
    const unsigned lds = substep_lds(a);
    switch (scheme) {
        case SCHEME_KP07:
            hipLaunchKernelGGL((substep_kernel<SweKP07<M>, M>), dim3(grid), block, lds, stream, a);
            break;
        case SCHEME_HLL2:
            hipLaunchKernelGGL((substep_kernel<SweHLL2<M>, M>), dim3(grid), block, lds, stream, a);
            break;
        case SCHEME_WAF:
            hipLaunchKernelGGL((substep_kernel<SweWAF<M>, M>), dim3(grid), block, lds, stream, a);
            break;
        case SCHEME_EULER:
            hipLaunchKernelGGL((substep_kernel<EulerKP07<M>, M>), dim3(grid), block, lds, stream, a);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <class S, class M>
hipError_t launch_step_scheme(const SubstepArgs& a, int grid, hipStream_t stream) {
    hipLaunchKernelGGL((step_kernel<S, M>), dim3(grid), dim3(kLanes * a.waves_per_block),
                       block_cfl_bytes(block_cfl(a.round_plan, a.cfl)), stream, a);
    return hipGetLastError();
}

template <class S, class M>
hipError_t launch_ensemble_scheme(const EnsembleArgs& e, int grid, hipStream_t stream) {
    hipLaunchKernelGGL((ensemble_kernel<S, M, false>), dim3(grid), dim3(kLanes * e.waves_per_block), 0, stream, e);
    return hipGetLastError();
}

template <class S, class M>
hipError_t launch_ensemble_step_scheme(const EnsembleArgs& e, int grid, hipStream_t stream) {
    hipLaunchKernelGGL((ensemble_kernel<S, M, true>), dim3(grid), dim3(kLanes * e.waves_per_block), 0, stream, e);
    return hipGetLastError();
}

template <class M>
hipError_t launch_ensemble_substep(int scheme, EnsembleArgs e, int grid, hipStream_t stream) {
    const dim3 block(kLanes * e.waves_per_block);
    switch (scheme) {
        case SCHEME_KP07:
            hipLaunchKernelGGL((ensemble_kernel<SweKP07<M>, M, false>), dim3(grid), block, 0, stream, e);
            break;
        case SCHEME_HLL2:
            hipLaunchKernelGGL((ensemble_kernel<SweHLL2<M>, M, false>), dim3(grid), block, 0, stream, e);
            break;
        case SCHEME_WAF:
            hipLaunchKernelGGL((ensemble_kernel<SweWAF<M>, M, false>), dim3(grid), block, 0, stream, e);
            break;
        case SCHEME_EULER:
            hipLaunchKernelGGL((ensemble_kernel<EulerKP07<M>, M, false>), dim3(grid), block, 0, stream, e);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Defined in fv_kernels_exact.hip and fv_kernels_fast.hip (whole steps: KP07_dimsplit,
// HLL2 and Euler in fast arithmetic).
hipError_t launch_ensemble_exact(int scheme, const EnsembleArgs& e, int grid, hipStream_t stream);
hipError_t launch_ensemble_fast(int scheme, const EnsembleArgs& e, int grid, hipStream_t stream);
hipError_t launch_substep_exact(int scheme, const SubstepArgs& a, int grid, hipStream_t stream);
hipError_t launch_substep_fast(int scheme, const SubstepArgs& a, int grid, hipStream_t stream);
hipError_t launch_step_fast(int scheme, const SubstepArgs& a, int grid, hipStream_t stream);
hipError_t launch_ensemble_step_fast(int scheme, const EnsembleArgs& e, int grid, hipStream_t stream);
// Defined in fv_kernels_fast_ilp.hip: the shallow-water schemes of the above, and the
// two Runge-Kutta stages of KP07 in fast arithmetic.
hipError_t launch_step_fast_ilp(int scheme, const SubstepArgs& a, int grid, hipStream_t stream);
hipError_t launch_ensemble_step_fast_ilp(int scheme, const EnsembleArgs& e, int grid, hipStream_t stream);
hipError_t launch_rk2_step(const SubstepArgs& a, int grid, hipStream_t stream);
hipError_t launch_substep_fast_ilp(int scheme, const SubstepArgs& a, int grid, hipStream_t stream);
hipError_t launch_ensemble_fast_ilp(int scheme, const EnsembleArgs& e, int grid, hipStream_t stream);

}  // namespace fvmi
