// Fused dimensionally split substep: ghost fill + first sweep + second sweep
// (+ gravity) + store + CFL minimum, one pass over HBM.
//
// Replaces the tile kernels KP07DimsplitKernel (GPUSimulators/cuda/SWE2D_KP07_dimsplit.cu:123-205),
// HLL2Kernel (SWE2D_HLL2.cu:126-214), WAFKernel (SWE2D_WAF.cu:103-176) and the
// Euler KP07DimsplitKernel (EE2D_KP07_dimsplit.cu:126-247).
//
// Work decomposition (gfx950, 64-lane wavefronts).  A wavefront owns a
// "strip" of output columns x `tile_rows` output rows, C padded columns per
// lane: with C = 1 lane c holds padded column x0+c (x0 = 60*strip), lanes
// 2..61 are the strip's own 60 columns and lanes 0,1,62,63 its x halo; with
// C = 2 lane c holds columns x0+2c, x0+2c+1 (x0 = 124*strip), lanes 1..62 the
// strip's own 124 columns and lanes 0, 63 the halo, each row read and written
// with 8-byte accesses.  The wave marches down the strip one padded row at a
// time (tile_rows+4 rows including the 2+2 y halo):
//   * the x sweep of a row is done across lanes, neighbours exchanged with
//     cross-lane moves, no LDS and no barrier;
//   * the y sweep is done per lane with a register window of the last 3
//     (slope schemes) or 4 (WAF) rows, so every y flux is computed once.
// The reference's "X then Y" (step 0) / "Y then X" (step 1) order, its
// extended first sweep over the halo lines, and its read/write masks are
// preserved exactly (GPUSimulators/cuda/common.h:320-475).
//
// Ghost cells are not materialised: each load maps its padded index through the
// boundary rule (periodic wrap, mirror with sign, or the memory value) so the
// kernel reads the values that readBlock + handleReflectiveBoundary would have
// produced, in global form (correct for every grid size, unlike the tile code's
// nx%bw==1 case).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fv_fast.h"
#include "fv_math.h"

namespace fvmi {

enum : int { BC_DIRICHLET = 0, BC_NEUMANN = 1, BC_PERIODIC = 2, BC_REFLECTIVE = 3, BC_OUTFLOW = 4 };

constexpr int kLanes = 64;

// A wavefront marches a strip of the domain, C padded columns per lane.  The
// lanes at each end that hold the strip's 2-column x halo are not written:
// halo_lanes<C>() of them, leaving strip_cols<C>() output columns (60 for one
// column per lane, 124 for two).
template <int C, int Halo = 2>
__host__ __device__ constexpr int halo_lanes() {
    return (Halo + C - 1) / C;
}
template <int C, int Halo = 2>
__host__ __device__ constexpr int strip_cols() {
    return (kLanes - 2 * halo_lanes<C, Halo>()) * C;
}

struct SubstepArgs {
    int nx, ny;
    float dx, dy, dt, g, theta, gamma;
    int step, bc;
    // interior sub-area [x0,x1) x [y0,y1) to update (0,0,nx,ny = whole domain)
    int x0, y0, x1, y1;
    const float* in[4];
    int in_pitch[4];  // bytes
    float* out[4];
    int out_pitch[4];
    float* cfl;  // two-slot CFL buffer: a step-1 launch minimises slot 1, every launch resets slot 1-step; may be null
    int cfl_slot;  // whole-step launch: the slot it minimises (it resets the other)
    // Work decomposition: the sub-area is cut into strips of strip_cols columns and every
    // strip into `segs_per_strip` segments of `seg_rows` rows (the last one
    // shorter), one per wavefront.  Segment j starts at the same row in every
    // strip, so the waves of neighbouring strips (on the same XCD) read the
    // cache lines they share at about the same time.
    int seg_rows;
    int segs_per_strip;
    int strip_cols;  // output columns per strip (strip_cols<S::kC>() of the scheme launched)
    int strips_x;
    int rows_per_strip;  // y1 - y0
    int num_waves;       // strips_x * segs_per_strip
    int waves_per_block;
    int num_blocks;  // logical blocks = ceil(num_waves / waves_per_block)
    int xcd_remap;
    // Round-weighted plan (round_plan = 1, see round_segment): the grid is
    // kRounds blocks per CU; strips are cut into gps row groups of grows rows
    // (the last one shorter), and part k of a group goes to a wave of dispatch
    // round k.
    int round_plan;
    int xcds, cus_per_xcd;
    int gps, grows;
    // derived constants for the fast policy (set by the host launcher)
    float hg, sqrt_g, inv_g, inv_dx, inv_dy, dtdx, dtdy;
    float half_theta;  // theta / 2
    float inv_2theta;  // 1 / (2 theta), 0 for theta <= 0
    float g_theta;     // g theta
};

// What a launch of equal segments costs, in us, with w waves on a SIMD:
// row_us (rows + halo_rows) (1 + w) + block_us * workgroups.  A wave alone on its
// SIMD waits for its own results; each further one adds about half that time to a
// row of all of them (KP07_dimsplit whole steps, rows of 0.41 us: 5.4, 8.6, 11.2
// and 13.9 cycles an instruction for one to four waves).  The second term is the
// CFL minimum's atomics, one after the other (reduce_cfl).
struct SegmentCost {
    int halo_rows;   // rows a segment sweeps and does not store
    int min_rows;    // shortest segment
    float row_us;
    float block_us;
};

// Rows per segment of the equal-segment plan: of the longest segments that put
// one, two .. waves_per_simd waves on every SIMD, the cheapest; more waves only
// for 3 % or more, since their halo rows are work that another stream's launches
// would have to wait for.  A multiple of the device's SIMDs just exceeded is what
// it avoids: KP07_dimsplit 1500^2 with 40 rows (1026 waves for 1024 SIMDs) and 20,
// a step of one simulator: 57.9 and 35.8 us, KP07 2048x1500 51 and 44, Euler exact
// 256^2 with 4 and 2 rows 19.9 and 16.5, HLL 512^2 with 24 and 6 13.9 and 8.8.
inline int balanced_segment_rows(int rows, int strips, int cu_count, int waves_per_simd, const SegmentCost& c) {
    int best = rows;  // also where there are more strips than waves
    float best_cost = 0.0f;
    for (int w = 1; w <= waves_per_simd; ++w) {
        const int k = cu_count * 4 * w / strips;
        if (k < 1) continue;
        int seg = (rows + k - 1) / k;
        if (seg < c.min_rows) seg = c.min_rows;
        const long long waves = (long long)strips * ((rows + seg - 1) / seg);
        const int per_simd = (int)((waves + 4LL * cu_count - 1) / (4LL * cu_count));
        const float cost =
            c.row_us * (float)(seg + c.halo_rows) * (float)(1 + per_simd) + c.block_us * 0.25f * (float)waves;
        if (best_cost == 0.0f || cost < 0.97f * best_cost) {
            best = seg;
            best_cost = cost;
        }
    }
    return best;
}

// the slope constants from g and theta
__host__ __device__ inline void set_slope_constants(SubstepArgs& a) {
    a.half_theta = 0.5f * a.theta;
    a.inv_2theta = a.theta > 0.0f ? 0.5f / a.theta : 0.0f;
    a.g_theta = a.g * a.theta;
}

struct AxisMap {
    int idx;
    bool mirrored;
};

// Memory index read for padded index k along an axis of n interior cells
// (common.h:247-288 and the mirror rules of :133-239).  Indices past the padded
// array are clamped as readBlock does (those lanes/rows are never stored).
// GC ghost cells a side: ghost k < GC mirrors cell 2*GC-1-k (bc*Reflective,
// common.h:133-239, for any gc), periodic wraps by n.
// Deep: two more images a side (k from -GC to n + 3 GC - 1) on periodic edges;
// elsewhere those indices read some cell of the array.
template <int GC, bool Deep = false>
__device__ __forceinline__ AxisMap map_axis_gc(int k, int n, int bc_lo, int bc_hi) {
    if (k < GC) {
        if (bc_lo == BC_PERIODIC) return {k + n, false};
        if (bc_lo == BC_REFLECTIVE) return {2 * GC - 1 - k, true};
        if (bc_lo == BC_OUTFLOW) return {GC, false};
        // the two columns before a strip that starts at padded column 0 (u_first_col
        // in fv_unsplit.h) read those after it
        return {k < 0 ? k + 2 * GC : k, false};
    }
    if (k >= n + GC) {
        const int k_max = n + 2 * GC - 1 + (Deep && bc_hi == BC_PERIODIC ? 2 : 0);
        if (k > k_max) k = k_max;
        if (bc_hi == BC_PERIODIC) return {k - n, false};
        if (bc_hi == BC_REFLECTIVE) return {2 * (n + GC) - 1 - k, true};
        if (bc_hi == BC_OUTFLOW) return {n + GC - 1, false};
        return {k, false};
    }
    return {k, false};
}

// The same map along y in affine, branch-free form for the row march (the row
// index is wave-uniform, so the selects stay scalar): a ghost row k < GC reads
// memory row lo_a*k + lo_b, a ghost row k >= n+GC (clamped to the padded
// array) hi_a*k + hi_b, an interior row itself.  A mirroring side flips the
// sign of the y momentum (sign-bit mask).
struct RowMap {
    int lo_a, lo_b, hi_a, hi_b;
    int n_gc;   // n + GC, the first ghost row of the high side
    int k_max;  // n + 2 GC - 1, the last padded row (Deep, periodic: two more images)
    unsigned lo_sign, hi_sign;
};

template <int GC>
__device__ __forceinline__ void row_map_side(int bc, int n, bool hi, int& a, int& b, unsigned& sign) {
    a = 1;
    b = 0;
    sign = 0u;
    if (bc == BC_PERIODIC) {
        b = hi ? -n : n;
    } else if (bc == BC_REFLECTIVE) {
        a = -1;
        b = hi ? 2 * (n + GC) - 1 : 2 * GC - 1;
        sign = 0x80000000u;
    } else if (bc == BC_OUTFLOW) {
        a = 0;
        b = hi ? n + GC - 1 : GC;
    }
}

template <int GC, bool Deep = false>
__device__ __forceinline__ RowMap make_row_map(int n, int bc_lo, int bc_hi) {
    RowMap m;
    row_map_side<GC>(bc_lo, n, false, m.lo_a, m.lo_b, m.lo_sign);
    row_map_side<GC>(bc_hi, n, true, m.hi_a, m.hi_b, m.hi_sign);
    m.n_gc = n + GC;
    m.k_max = n + 2 * GC - 1 + (Deep && bc_hi == BC_PERIODIC ? 2 : 0);
    return m;
}

// memory row of padded row k (wave-uniform) and the y-momentum sign mask
template <int GC>
__device__ __forceinline__ int map_row(const RowMap& m, int k, unsigned& sign) {
    const bool lo = k < GC, hi = k >= m.n_gc;
    // every candidate is computed, then selected (no branches)
    const int lo_row = m.lo_a * k + m.lo_b;
    const int hi_row = m.hi_a * min(k, m.k_max) + m.hi_b;
    int row = hi ? hi_row : k;
    row = lo ? lo_row : row;
    unsigned sg = hi ? m.hi_sign : 0u;
    sg = lo ? m.lo_sign : sg;
    sign = __builtin_amdgcn_readfirstlane(sg);
    return __builtin_amdgcn_readfirstlane(row);
}

// Cross-lane operations on N values at once (the value held by lane - 1 or
// lane + 1: wave_shr:1, wave_shl:1), as one run of DPP instructions: a lone one
// among other VALU instructions costs several times its place in a run (see
// FVMI_TRANS_RUN in fv_math.h).  s_nop 1: a DPP operand that the
// instruction before has written needs two wait states, which the compiler
// does not see inside the block.  Lane 0 (63) takes 0 for its missing
// neighbour.
#define FVMI_DPP_MOV(o, x, ctrl) "v_mov_b32_dpp %" #o ", %" #x " " ctrl " row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
#define FVMI_DPP_SUB(o, x, y, ctrl) \
    "v_sub_f32_dpp %" #o ", %" #x ", %" #y " " ctrl " row_mask:0xf bank_mask:0xf bound_ctrl:0\n\t"
#define FVMI_OUT3 "=&v"(o[0]), "=&v"(o[1]), "=&v"(o[2])
#define FVMI_OUT4 FVMI_OUT3, "=&v"(o[3])
#define FVMI_OUT6 FVMI_OUT4, "=&v"(o[4]), "=&v"(o[5])
#define FVMI_OUT8 FVMI_OUT6, "=&v"(o[6]), "=&v"(o[7])
#define FVMI_IN3(v) "v"(v[0]), "v"(v[1]), "v"(v[2])
#define FVMI_IN4(v) FVMI_IN3(v), "v"(v[3])
#define FVMI_IN6(v) FVMI_IN4(v), "v"(v[4]), "v"(v[5])
#define FVMI_IN8(v) FVMI_IN6(v), "v"(v[6]), "v"(v[7])
#define FVMI_DPP_MOV_RUN(name, ctrl) \
    template <int N> \
    __device__ __forceinline__ void name(const float (&x)[N], float (&o)[N]) { \
        static_assert(N == 3 || N == 4 || N == 6 || N == 8, "runs of 3, 4, 6 or 8"); \
        if constexpr (N == 3) \
            asm("s_nop 1\n\t" \
                FVMI_DPP_MOV(0, 3, ctrl) FVMI_DPP_MOV(1, 4, ctrl) FVMI_DPP_MOV(2, 5, ctrl) \
                : FVMI_OUT3 : FVMI_IN3(x)); \
        if constexpr (N == 4) \
            asm("s_nop 1\n\t" \
                FVMI_DPP_MOV(0, 4, ctrl) FVMI_DPP_MOV(1, 5, ctrl) FVMI_DPP_MOV(2, 6, ctrl) \
                FVMI_DPP_MOV(3, 7, ctrl) \
                : FVMI_OUT4 : FVMI_IN4(x)); \
        if constexpr (N == 6) \
            asm("s_nop 1\n\t" \
                FVMI_DPP_MOV(0, 6, ctrl) FVMI_DPP_MOV(1, 7, ctrl) FVMI_DPP_MOV(2, 8, ctrl) \
                FVMI_DPP_MOV(3, 9, ctrl) FVMI_DPP_MOV(4, 10, ctrl) FVMI_DPP_MOV(5, 11, ctrl) \
                : FVMI_OUT6 : FVMI_IN6(x)); \
        if constexpr (N == 8) \
            asm("s_nop 1\n\t" \
                FVMI_DPP_MOV(0, 8, ctrl) FVMI_DPP_MOV(1, 9, ctrl) FVMI_DPP_MOV(2, 10, ctrl) \
                FVMI_DPP_MOV(3, 11, ctrl) FVMI_DPP_MOV(4, 12, ctrl) FVMI_DPP_MOV(5, 13, ctrl) \
                FVMI_DPP_MOV(6, 14, ctrl) FVMI_DPP_MOV(7, 15, ctrl) \
                : FVMI_OUT8 : FVMI_IN8(x)); \
    }
#define FVMI_DPP_SUB_RUN(name, ctrl) \
    template <int N> \
    __device__ __forceinline__ void name(const float (&x)[N], const float (&y)[N], float (&o)[N]) { \
        static_assert(N == 3 || N == 4 || N == 6 || N == 8, "runs of 3, 4, 6 or 8"); \
        if constexpr (N == 3) \
            asm("s_nop 1\n\t" \
                FVMI_DPP_SUB(0, 3, 6, ctrl) FVMI_DPP_SUB(1, 4, 7, ctrl) FVMI_DPP_SUB(2, 5, 8, ctrl) \
                : FVMI_OUT3 : FVMI_IN3(x), FVMI_IN3(y)); \
        if constexpr (N == 4) \
            asm("s_nop 1\n\t" \
                FVMI_DPP_SUB(0, 4, 8, ctrl) FVMI_DPP_SUB(1, 5, 9, ctrl) FVMI_DPP_SUB(2, 6, 10, ctrl) \
                FVMI_DPP_SUB(3, 7, 11, ctrl) \
                : FVMI_OUT4 : FVMI_IN4(x), FVMI_IN4(y)); \
        if constexpr (N == 6) \
            asm("s_nop 1\n\t" \
                FVMI_DPP_SUB(0, 6, 12, ctrl) FVMI_DPP_SUB(1, 7, 13, ctrl) FVMI_DPP_SUB(2, 8, 14, ctrl) \
                FVMI_DPP_SUB(3, 9, 15, ctrl) FVMI_DPP_SUB(4, 10, 16, ctrl) FVMI_DPP_SUB(5, 11, 17, ctrl) \
                : FVMI_OUT6 : FVMI_IN6(x), FVMI_IN6(y)); \
        if constexpr (N == 8) \
            asm("s_nop 1\n\t" \
                FVMI_DPP_SUB(0, 8, 16, ctrl) FVMI_DPP_SUB(1, 9, 17, ctrl) FVMI_DPP_SUB(2, 10, 18, ctrl) \
                FVMI_DPP_SUB(3, 11, 19, ctrl) FVMI_DPP_SUB(4, 12, 20, ctrl) FVMI_DPP_SUB(5, 13, 21, ctrl) \
                FVMI_DPP_SUB(6, 14, 22, ctrl) FVMI_DPP_SUB(7, 15, 23, ctrl) \
                : FVMI_OUT8 : FVMI_IN8(x), FVMI_IN8(y)); \
    }
FVMI_DPP_MOV_RUN(all_from_left, "wave_shr:1")    // o = x of lane - 1
FVMI_DPP_MOV_RUN(all_from_right, "wave_shl:1")   // o = x of lane + 1
FVMI_DPP_SUB_RUN(left_minus_all, "wave_shr:1")   // o = x of lane - 1, minus y
FVMI_DPP_SUB_RUN(right_minus_all, "wave_shl:1")  // o = x of lane + 1, minus y

// the WafCell of lane+1
__device__ __forceinline__ WafCell waf_from_right(const WafCell& p) {
    const float x[6] = {p.h, p.hu, p.hv, p.u, p.v, p.c}, y[3] = {p.ih, p.f1, p.f2};
    float o[6], w[3];
    all_from_right<6>(x, o);
    all_from_right<3>(y, w);
    return {o[0], o[1], o[2], o[3], o[4], o[5], w[0], w[1], w[2]};
}

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = fminf(v, __shfl_xor(v, off, kLanes));
    return v;
}

// A CFL accumulator that has seen no cell.
template <class M>
__device__ __forceinline__ float no_cfl() {
    return M::exact ? __builtin_inff() : 0.0f;
}

// The CFL minimum of a workgroup and the number of its waves that have added
// to it, in the launch's dynamic LDS.
struct BlockCfl {
    unsigned least, waves;
};

// Whether the waves of a workgroup take their CFL minimum to memory together.
// Atomics on one address take about 10 ns each, one after the other, and where
// the segments are of equal length they all come at the end: with one per wave,
// and with one per workgroup, a step of one simulator: KP07_dimsplit 256^2 12.6
// and 10.3 us, 512^2 20.6 and 14.3, 1000^2 31.7 and 23.8 (11.8 and 21.6 at the
// last two without the minimum), Euler 512^2 exact 32.6 and 25.3, HLL2 2047^2 81
// and 73, HLL 1000^2 20.8 and 15.4.  The parts of the round-weighted split end at
// different times: KP07_dimsplit 4096^2 188 and 187 us, and with three simulators
// on three streams 177 and 179 a step (a workgroup with LDS starts later beside
// another launch's last ones).  The first-order schemes' shorter rows gain there
// too, HLL 4096^2 120 and 102 us alone, 98 and 98 in turn (fv_unsplit.h shares
// always; part of it is a row kept in registers, see store_row).
__host__ __device__ inline bool block_cfl(bool round_plan, const float* cfl) { return !round_plan && cfl != nullptr; }

inline unsigned block_cfl_bytes(bool shared) { return shared ? sizeof(BlockCfl) : 0; }

__device__ __forceinline__ void begin_cfl(bool shared) {
    extern __shared__ BlockCfl block[];
    if (!shared) return;
    if (threadIdx.x == 0) block->least = 0x7f800000u, block->waves = 0;  // +inf
    __syncthreads();
}

// The accumulator of a wave (also of one without a segment) into the launch's
// CFL minimum; the last wave of a workgroup with `shared` does it for all.
template <class M>
__device__ __forceinline__ void reduce_cfl(bool shared, float* slot, float acc, int lane) {
    extern __shared__ BlockCfl block[];
    float dt_min = acc;
    if constexpr (!M::exact) dt_min = (acc > 0.0f) ? fast::rcp(acc) : __builtin_inff();
    const float m = wave_min(dt_min);
    if (lane != 0) return;
    unsigned least = m < __builtin_inff() ? __float_as_uint(m) : 0x7f800000u;
    if (shared) {
        __hip_atomic_fetch_min(&block->least, least, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const unsigned before =
            __hip_atomic_fetch_add(&block->waves, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (before != blockDim.x / kLanes - 1) return;
        least = __hip_atomic_load(&block->least, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (least < 0x7f800000u) atomicMin(reinterpret_cast<unsigned int*>(slot), least);
}

// Rows loaded ahead of the row being processed.  Each wave keeps a ring of
// row slots in registers: the rows its y stencil still needs plus this many
// rows in flight, so a load is issued kRowPrefetch rows of work before its
// first use.
#ifndef FVMI_ROW_PREFETCH
#define FVMI_ROW_PREFETCH 2
#endif
constexpr int kRowPrefetch = FVMI_ROW_PREFETCH;
static_assert(kRowPrefetch >= 1 && kRowPrefetch <= 3, "row prefetch distance 1..3");

// ---------------------------------------------------------------------------
// Scheme policies
// ---------------------------------------------------------------------------

// Scheme policies.  pred_diff = F(QL) - F(QR) for the half-step predictor;
// flux_x / flux_y the interface fluxes; cell_dt (exact) or cell_rate = 1/dt
// (fast) the CFL quantity of an updated cell.
// kPinRows: the march pins each prefetched row at its first use (use_row);
// kCarryDiff: the y sweep of the fast policy carries one row's forward
// difference over as the next row's backward difference; kPrefetch: rows
// loaded ahead (kRowPrefetch unless a scheme sets its own).  Measured at 4096^2 (SWE) and 8192^2 (Euler):
// pinning takes the WAF substep from 210 to 197 us and HLL2 about 1 % faster,
// KP07_dimsplit even; the Euler kernel is 7 % (carry) and 20-25 % (pinned rows)
// slower with them, so it keeps neither, and 1.5 % faster with one row ahead
// instead of two.
// Columns per lane, rows loaded ahead and row pinning of the KP07_dimsplit and
// HLL2 marches (build-time choices; the defaults are the measured best).
// Measured at 4096^2 per substep, same box: one column, 3 rows ahead, pinned
// rows: KP07_dimsplit 113.0 us, HLL2 132.1; two columns (8-byte accesses):
// 1 row ahead 111.3-112.7 and 156-159 us, 2 rows ahead 132-146 and 153-176 us.
#ifndef FVMI_SWE_COLS
#define FVMI_SWE_COLS 1
#endif
#ifndef FVMI_SWE_PREFETCH
#define FVMI_SWE_PREFETCH 3
#endif
#ifndef FVMI_SWE_PIN
#define FVMI_SWE_PIN 1
#endif

template <class M>
struct SweBase {
    static constexpr int NV = 3;
    static constexpr bool kEuler = false;
    static constexpr bool kPinRows = FVMI_SWE_PIN != 0;
    static constexpr bool kCarryDiff = true;
    static constexpr int kPrefetch = kRowPrefetch;
    __device__ static void pred_diff(const float QL[3], const float QR[3], const SubstepArgs& a, float D[3]) {
        float FL[3], FR[3];
        swe_F<M>(QL, a.g, FL);
        swe_F<M>(QR, a.g, FR);
#pragma unroll
        for (int k = 0; k < 3; ++k) D[k] = FL[k] - FR[k];
    }
    // fast policy: faces QL/QR = c -/+ (theta/2) m of the cell c with limited
    // slope m (in units of theta), r = 1/(QL0 QR0)
    __device__ static void pred_diff_fast(const float QL[3], const float QR[3], float r, const float c[3],
                                          const float m[3], const SubstepArgs& a, float D[3]) {
        fast::swe_pred_diff(QL, QR, r, c[0], m[0], a.g_theta, D);
    }
    __device__ static float cell_dt(const float q[3], const SubstepArgs& a) { return swe_cell_dt<M>(q, a.dx, a.dy, a.g); }
    __device__ static float cell_rate(const float q[3], const SubstepArgs& a) {
        return fast::swe_cell_rate(q, a.sqrt_g, a.inv_dx, a.inv_dy);
    }
};

// Cols: columns per lane.  flux_x / flux_y take the interfaces of a lane's
// columns at once.
template <class M, int Cols = FVMI_SWE_COLS>
struct SweKP07 : SweBase<M> {
    using Pair = SweKP07<M, 2>;  // two rows side by side (Rows of x_sweep_row)
    static constexpr int kPrefetch = FVMI_SWE_PREFETCH;
    static constexpr bool kSlopes = true;
    static constexpr int kC = Cols;
    __device__ static void flux(const float (&l)[kC][3], const float (&r)[kC][3], const SubstepArgs& a,
                                float (&o)[kC][3]) {
        if constexpr (M::exact) {
#pragma unroll
            for (int c = 0; c < kC; ++c) swe_cu_flux(l[c], r[c], a.g, o[c]);
        } else {
            fast::swe_cu_flux<kC>(l, r, a.hg, a.sqrt_g, o);
        }
    }
    __device__ static void flux_x(const float (&l)[kC][3], const float (&r)[kC][3], const SubstepArgs& a,
                                  float (&o)[kC][3]) {
        flux(l, r, a, o);
    }
    __device__ static void flux_y(const float (&l)[kC][3], const float (&r)[kC][3], const SubstepArgs& a,
                                  float (&o)[kC][3]) {
        flux(l, r, a, o);
    }
};

template <class M, int Cols = FVMI_SWE_COLS>
struct SweHLL2 : SweBase<M> {
    using Pair = SweHLL2<M, 2>;  // two rows side by side (Rows of x_sweep_row)
    static constexpr int kPrefetch = FVMI_SWE_PREFETCH;
    static constexpr bool kSlopes = true;
    static constexpr int kC = Cols;
    __device__ static void flux(const float (&l)[kC][3], const float (&r)[kC][3], const SubstepArgs& a,
                                float (&o)[kC][3]) {
        if constexpr (M::exact) {
#pragma unroll
            for (int c = 0; c < kC; ++c) swe_hll_flux(l[c], r[c], a.g, o[c]);
        } else {
            fast::swe_hll_flux<kC>(l, r, a.hg, a.sqrt_g, o);
        }
    }
    __device__ static void flux_x(const float (&l)[kC][3], const float (&r)[kC][3], const SubstepArgs& a,
                                  float (&o)[kC][3]) {
        flux(l, r, a, o);
    }
    __device__ static void flux_y(const float (&l)[kC][3], const float (&r)[kC][3], const SubstepArgs& a,
                                  float (&o)[kC][3]) {
        flux(l, r, a, o);
    }
};

template <class M>
struct SweWAF : SweBase<M> {
    // the flux is assembled by the march from shared pieces (waf_cell,
    // waf_hstar, waf_flux_core in fv_math.h)
    static constexpr bool kSlopes = false;
    static constexpr int kC = 1;  // columns per lane (its march needs the registers of two)
};

template <class M, int Cols = (M::exact ? 1 : 2)>
struct EulerKP07 {
    using Pair = EulerKP07<M, 2>;
    static constexpr int NV = 4;
    static constexpr bool kSlopes = true;
    // columns per lane: two in fast arithmetic (8-byte accesses: 8192^2 step
    // 1.263 -> 1.157 ms); the exact arithmetic's division sequences need the
    // registers of the second column
    static constexpr int kC = Cols;
    static constexpr bool kEuler = true;
    static constexpr bool kPinRows = false;
    static constexpr bool kCarryDiff = false;
    static constexpr int kPrefetch = 1;
    // The predictor passes gamma in the pressure slot: EE2D_KP07_dimsplit.cu:57-58, 102-103.
    __device__ static void pred_diff(const float QL[4], const float QR[4], const SubstepArgs& a, float D[4]) {
        float FL[4], FR[4];
        euler_F<M>(QL, a.gamma, FL);
        euler_F<M>(QR, a.gamma, FR);
#pragma unroll
        for (int k = 0; k < 4; ++k) D[k] = FL[k] - FR[k];
    }
    __device__ static void pred_diff_fast(const float QL[4], const float QR[4], float r, const float c[4],
                                          const float m[4], const SubstepArgs& a, float D[4]) {
        (void)c;
        (void)m;
        fast::euler_pred_diff(QL, QR, r, a.gamma, D);
    }
    __device__ static void flux_x(const float (&l)[kC][4], const float (&r)[kC][4], const SubstepArgs& a,
                                  float (&o)[kC][4]) {
        if constexpr (M::exact) {
#pragma unroll
            for (int c = 0; c < kC; ++c) euler_hll_flux(l[c], r[c], a.gamma, o[c]);
        } else {
            fast::euler_hll_flux<kC>(l, r, a.gamma, o);
        }
    }
    __device__ static void flux_y(const float (&l)[kC][4], const float (&r)[kC][4], const SubstepArgs& a,
                                  float (&o)[kC][4]) {
        if constexpr (M::exact) {
#pragma unroll
            for (int c = 0; c < kC; ++c) euler_cu_flux(l[c], r[c], a.gamma, o[c]);
        } else {
            fast::euler_cu_flux<kC>(l, r, a.gamma, o);
        }
    }
    __device__ static float cell_dt(const float q[4], const SubstepArgs& a) {
        return euler_cell_dt<M>(q, a.dx, a.dy, a.gamma);
    }
    __device__ static float cell_rate(const float q[4], const SubstepArgs& a) {
        return fast::euler_cell_rate(q, a.gamma, a.inv_dx, a.inv_dy);
    }
};

// ---------------------------------------------------------------------------
// Sweep pieces
// ---------------------------------------------------------------------------

// y-sweep order: (rho, normal = y momentum, tangential = x momentum[, E])
template <int NV>
__device__ __forceinline__ void to_y(const float q[NV], float o[NV]) {
    o[0] = q[0];
    o[1] = q[2];
    o[2] = q[1];
    if constexpr (NV == 4) o[3] = q[3];
}

// Fast-policy reconstruction + half-step predictor of a lane's cells from
// their backward and forward differences, b(c, k) = q - l and f(c, k) = r - q
// of variable k (callables, so that each difference is formed where it is used):
//   minmod(theta b, (b + f)/2, theta f) = theta minmod(b, (b + f)/(2 theta), f)
// for theta > 0, so each neighbour enters once and the y sweep reuses the
// forward difference of one row as the backward difference of the next.
template <class S, class B, class F>
__device__ __forceinline__ void reconstruct_fast(B b, F f, const float (&q)[S::kC][S::NV], const SubstepArgs& a,
                                                 float kk, float (&qbl)[S::kC][S::NV], float (&qbr)[S::kC][S::NV]) {
    constexpr int NV = S::NV;
    constexpr int C = S::kC;
    float QL[C][NV], QR[C][NV], m[C][NV], p[C], r[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const float bk = b(c, k), fk = f(c, k);
            m[c][k] =
                __builtin_amdgcn_fmed3f(__builtin_amdgcn_fmed3f(bk, fk, 0.0f), (bk + fk) * a.inv_2theta, 0.0f);
            QL[c][k] = __builtin_fmaf(-a.half_theta, m[c][k], q[c][k]);
            QR[c][k] = __builtin_fmaf(a.half_theta, m[c][k], q[c][k]);
        }
        p[c] = QL[c][0] * QR[c][0];
    }
    rcp_all<C>(p, r);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        float D[NV];
        S::pred_diff_fast(QL[c], QR[c], r[c], q[c], m[c], a, D);
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            qbl[c][k] = QL[c][k] + kk * D[k];
            qbr[c][k] = QR[c][k] + kk * D[k];
        }
    }
}

// Difference of two neighbouring values as the limiter takes it: times
// theta in the exact policy (minmod_slope in fv_math.h).
template <class M>
__device__ __forceinline__ float limiter_diff(float lo, float hi, const SubstepArgs& a) {
    return M::exact ? (hi - lo) * a.theta : hi - lo;
}

// Reconstruction + half-step predictor of a lane's cells (computeFluxF,
// SWE2D_KP07_dimsplit.cu:42-58) from their backward and forward differences
// b(c, k), f(c, k) (limiter_diff) and, in the exact policy, cd(c, k) = right -
// left; gives the predicted left-face (qbl) and right-face (qbr) states.
template <class S, class M, class B, class F, class D2>
__device__ __forceinline__ void reconstruct(B b, F f, D2 cd, const float (&q)[S::kC][S::NV], const SubstepArgs& a,
                                            float kk, float (&qbl)[S::kC][S::NV], float (&qbr)[S::kC][S::NV]) {
    constexpr int NV = S::NV;
    if constexpr (M::exact) {
#pragma unroll
        for (int c = 0; c < S::kC; ++c) {
            float QL[NV], QR[NV], D[NV];
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const float hs = 0.5f * minmod_slope(b(c, k), 0.5f * cd(c, k), f(c, k));
                QL[k] = q[c][k] - hs;
                QR[k] = q[c][k] + hs;
            }
            S::pred_diff(QL, QR, a, D);
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                qbl[c][k] = QL[k] + kk * D[k];
                qbr[c][k] = QR[k] + kk * D[k];
            }
        }
    } else {
        reconstruct_fast<S>(b, f, q, a, kk, qbl, qbr);
    }
}

// evolveF/evolveG, common.h:450, 471: q plus the flux difference df = f_in -
// f_out times dt/d; dtd = dt/d (fast policy only).  SignedZero: the increment
// keeps the sign of a zero (WAF).
template <class M, bool SignedZero = false>
__device__ __forceinline__ float evolve(float q, float df, float dt, float d, float dtd) {
    if constexpr (M::exact) {
        return q + (SignedZero ? M::div(df * dt, d) : M::quot(df * dt, d));
    } else {
        return q + df * dtd;
    }
}

// x sweep of rows held across the 64 lanes (valid on the strip's output
// columns).  q[c]: column c of the lane's C columns of one row, or, with Rows,
// the lane's column of row c of C independent rows swept side by side.  The
// cross-lane operations and the transcendentals of all C come in runs.
template <class S, class M, bool Rows = false>
__device__ __forceinline__ void x_sweep_row(float (&q)[S::kC][S::NV], const SubstepArgs& a) {
    constexpr int NV = S::NV;
    constexpr int C = S::kC;
    // values that cross a lane's ends: the first and last column of each row
    constexpr int E = Rows ? C : 1;
    constexpr int N = E * NV;
    const auto first = [](const float (&x)[C][NV], float (&o)[N]) {
#pragma unroll
        for (int i = 0; i < N; ++i) o[i] = x[Rows ? i / NV : 0][i % NV];
    };
    const auto last = [](const float (&x)[C][NV], float (&o)[N]) {
#pragma unroll
        for (int i = 0; i < N; ++i) o[i] = x[Rows ? i / NV : C - 1][i % NV];
    };
    const auto end = [](const float (&x)[N], int c, int k) { return x[(Rows ? c : 0) * NV + k]; };
    float F[C][NV];
    if constexpr (S::kSlopes) {
        const float kk = M::exact ? M::div(a.dt, 2.0f * a.dx) : 0.5f * a.dtdx;
        float qbl[C][NV], qbr[C][NV];
        float q_first[N], q_last[N], d_hi[N], d_lo[N];
        first(q, q_first);
        last(q, q_last);
        right_minus_all<N>(q_first, q_last, d_hi);  // forward difference of the last column
        if constexpr (M::exact) {
            static_assert(Rows || C == 1, "exact arithmetic marches one column per lane");
            float q_lo[N], cd[N];
            all_from_left<N>(q_last, q_lo);
            right_minus_all<N>(q_first, q_lo, cd);
#pragma unroll
            for (int i = 0; i < N; ++i) d_hi[i] *= a.theta;  // limiter_diff
            all_from_left<N>(d_hi, d_lo);
            reconstruct<S, M>([&](int c, int k) { return end(d_lo, c, k); },
                              [&](int c, int k) { return end(d_hi, c, k); },
                              [&](int c, int k) { return end(cd, c, k); }, q, a, kk, qbl, qbr);
        } else {
            all_from_left<N>(d_hi, d_lo);  // backward difference of the first column
            const auto f = [&](int c, int k) { return Rows || c == C - 1 ? end(d_hi, c, k) : q[c + 1][k] - q[c][k]; };
            const auto b = [&](int c, int k) { return Rows || c == 0 ? end(d_lo, c, k) : q[c][k] - q[c - 1][k]; };
            reconstruct_fast<S>(b, f, q, a, kk, qbl, qbr);
        }
        float qbl_first[N], qbl_hi[N], qr[C][NV];  // qr: left faces of the right neighbours
        first(qbl, qbl_first);
        all_from_right<N>(qbl_first, qbl_hi);
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < NV; ++k) qr[c][k] = Rows || c == C - 1 ? end(qbl_hi, c, k) : qbl[c + 1][k];
        S::flux_x(qbr, qr, a, F);  // interfaces (c, c+1)
    } else {
        // WAF: the cell's quantities, and the h* and limiter denominators of
        // its right interface, once; the neighbours' through DPP
        static_assert(C == 1, "WAF marches one column per lane");
        const WafCell P = waf_cell<M>(q[0], a.g, a.hg, a.sqrt_g);
        const WafCell R = waf_from_right(P);
        const float hd = waf_hstar<M>(P, R, a.g, a.inv_g);
        const WafDen D = waf_den<M>(P, R, hd);
        const float d[3] = {D.d1, D.d2, D.d3};
        float dl[3], dr[3];
        all_from_left<3>(d, dl);
        all_from_right<3>(d, dr);
        waf_flux_core<M>(P, R, WafDen{dl[0], dl[1], dl[2]}, D, WafDen{dr[0], dr[1], dr[2]}, hd, a.dx, a.dt, a.dtdx,
                         F[0]);
    }
    float F_first[N], F_last[N], dF[N];
    first(F, F_first);
    last(F, F_last);
    left_minus_all<N>(F_last, F_first, dF);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const float df = Rows || c == 0 ? end(dF, c, k) : F[c - 1][k] - F[c][k];
            q[c][k] = evolve<M, !S::kSlopes>(q[c][k], df, a.dt, a.dx, a.dtdx);
        }
}

// ---------------------------------------------------------------------------
// The kernel
// ---------------------------------------------------------------------------

// Raw buffer descriptor of one padded field (dword3 = 32-bit data format,
// the value used for raw buffers on gfx9).  Reads past `bytes` return 0 and
// writes past it are dropped by the hardware.
//
// Lanes that must not write use the vector offset kMaskedOffset (2 GiB).  The
// host keeps every field below 2 GiB, so that offset is out of range whether
// or not the scalar (row) offset, itself below 2 GiB, is added to it.
constexpr int kMaskedOffset = static_cast<int>(0x80000000u);
__device__ __forceinline__ __amdgpu_buffer_rsrc_t field_rsrc(const void* base, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

typedef unsigned fvmi_v2u __attribute__((ext_vector_type(2)));

// Per-wave constants of a strip of C columns per lane.  Lane L holds padded
// columns wstart + C L + c; halo_lanes<C>() lanes at each end hold the x halo.
//
// Loads (C = 2): one 8-byte load per field and row at pair_off; its words are
// the lane's two columns in order, or reversed (pair_rev) where both columns
// are mirrored ghost columns.  A lane whose two mapped columns are not such a
// pair at an 8-byte offset (zero-gradient ghosts, a periodic or mirrored
// ghost next to an interior column when nx is odd, the columns past the
// domain) loads each column with a 4-byte load instead (fix_off); waves
// without such a lane (wave_fix false) skip those loads.
// Stores (C = 2): an 8-byte store of the two columns where both are written
// and 8-byte aligned (store_off), else 4-byte stores of the written ones
// (single_off; only in waves with such a lane, wave_single).
template <int C>
struct Strip {
    int lane;
    int col[C];          // padded column of each column of this lane
    int row0;            // padded row of r = 0
    int r_end;           // rows r in [0, r_end)
    int lane_off[C];     // byte offset of each column after the boundary map
    unsigned xsign[C];   // sign-bit mask of the x momentum (mirrored ghost column)
    bool lane_out[C];    // column written
    int store_off;       // C = 1: the column, C = 2: the pair (8-byte store); kMaskedOffset if not
    int pair_off;        // C = 2: offset of the 8-byte load (kMaskedOffset for fix lanes)
    bool pair_rev;       // C = 2: the pair's words are (column 1, column 0)
    bool lane_fix;       // C = 2: this lane loads its columns one by one
    bool wave_fix;       // C = 2: some lane of the wave does
    int fix_off[2];      // C = 2: the 4-byte loads of a fix lane (kMaskedOffset elsewhere)
    int single_off[2];   // C = 2: 4-byte stores of written columns not in a full aligned pair
    bool wave_single;    // C = 2: some lane of the wave has such a column
    RowMap ymap;
    __amdgpu_buffer_rsrc_t rin[4], rout[4];
};

// x mirrors flip the x momentum, y mirrors the y momentum
template <int C, int NV>
__device__ __forceinline__ void apply_signs(const Strip<C>& st, unsigned ysign, float (&v)[C][NV]) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
        v[c][1] = __uint_as_float(__float_as_uint(v[c][1]) ^ st.xsign[c]);
        v[c][2] = __uint_as_float(__float_as_uint(v[c][2]) ^ ysign);
    }
}

// Issues the loads of padded row r and returns the sign-bit mask of its y
// momentum.  Pinned: the raw words are returned and use_row applies the mirror
// signs at the row's first use; otherwise they are applied here.
template <int C, int NV, bool Pinned, bool Edge = false, int GC = 2, class Args>
__device__ __forceinline__ unsigned load_row_raw(const Args& a, const Strip<C>& st, int r, float (&v)[C][NV]) {
    // Row offsets are wave-uniform (SGPR soffset); the lane adds its column
    // offset (VGPR voffset): no per-lane address arithmetic.
    unsigned ysign;
    const int row = map_row<GC>(st.ymap, __builtin_amdgcn_readfirstlane(st.row0 + r), ysign);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int soff = row * a.in_pitch[k];
        if constexpr (C == 1) {
            // the b32 buffer builtins move raw 32-bit words
            v[0][k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(st.rin[k], st.lane_off[0], soff, 0));
        } else {
            static_assert(C == 2, "one or two columns per lane");
            const fvmi_v2u x = __builtin_amdgcn_raw_buffer_load_b64(st.rin[k], st.pair_off, soff, 0);
            // (with one ghost cell a side no pair is reversed)
            unsigned w0 = GC > 1 && st.pair_rev ? x.y : x.x;
            unsigned w1 = GC > 1 && st.pair_rev ? x.x : x.y;
            if constexpr (Edge) {
                const unsigned f0 = __builtin_amdgcn_raw_buffer_load_b32(st.rin[k], st.fix_off[0], soff, 0);
                const unsigned f1 = __builtin_amdgcn_raw_buffer_load_b32(st.rin[k], st.fix_off[1], soff, 0);
                w0 = st.lane_fix ? f0 : w0;
                w1 = st.lane_fix ? f1 : w1;
            }
            v[0][k] = __uint_as_float(w0);
            v[1][k] = __uint_as_float(w1);
        }
    }
    if constexpr (!Pinned) apply_signs<C, NV>(st, ysign, v);
    return ysign;
}

// First use of a row loaded by load_row_raw.  Pinned: an empty volatile
// statement takes the loaded words and hands them on; being volatile it stays
// behind every load and store issued before it in program order, so the
// instruction scheduler cannot hoist the row's consumers (and the wait for its
// data) above the later rows' loads, and each load keeps its distance of
// kRowPrefetch rows of work.  The mirror signs are applied after it.
template <int C, int NV, bool Pinned>
__device__ __forceinline__ void use_row(const Strip<C>& st, unsigned ysign, float (&v)[C][NV]) {
    if constexpr (Pinned) {
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < NV; ++k) asm volatile("" : "+v"(v[c][k]));
        apply_signs<C, NV>(st, ysign, v);
    }
}

template <int C, int NV, bool Edge = false, class Args>
__device__ __forceinline__ void store_row(const Args& a, const Strip<C>& st, int r, const float (&q)[C][NV]) {
    const int prow = __builtin_amdgcn_readfirstlane(st.row0 + r);
    // every lane stores; the halo lanes' offset is out of range and the
    // hardware drops their writes (no branch around the stores)
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int soff = prow * a.out_pitch[k];
        if constexpr (C == 1) {
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(q[0][k]), st.rout[k], st.store_off, soff, 0);
        } else {
            // the optimiser widens a lone load of q[0][k] to a pair, which keeps q
            // in memory (LDS or scratch) for the whole march: stop it here
            unsigned lo = __float_as_uint(q[0][k]), hi = __float_as_uint(q[1][k]);
            asm("" : "+v"(lo));
            const fvmi_v2u x = {lo, hi};
            __builtin_amdgcn_raw_buffer_store_b64(x, st.rout[k], st.store_off, soff, 0);
        }
    }
    if constexpr (C == 2 && Edge) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const int soff = prow * a.out_pitch[k];
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(q[0][k]), st.rout[k], st.single_off[0], soff, 0);
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(q[1][k]), st.rout[k], st.single_off[1], soff, 0);
        }
    }
}

// CFL accumulator: the exact policy keeps min(dt) as the reference's writeCfl
// does; the fast policy keeps max(1/dt) (one reciprocal per segment, taken in
// reduce_cfl).
template <class S, class M>
__device__ __forceinline__ void accumulate_cfl(const float (&q)[S::kC][S::NV], const SubstepArgs& a,
                                               const Strip<S::kC>& st, float& acc) {
#pragma unroll
    for (int c = 0; c < S::kC; ++c) {
        if constexpr (M::exact) {
            const float cd = S::cell_dt(q[c], a);
            acc = st.lane_out[c] ? fminf(acc, cd) : acc;
        } else {
            const float rate = S::cell_rate(q[c], a);
            acc = st.lane_out[c] ? fmaxf(acc, rate) : acc;
        }
    }
}

// One row step of the y sweep for slope schemes.  Loop-carried state (per
// column): qbt, the predicted top face of row r-2, and g, the flux through its
// bottom interface; both are replaced by the values of row r-1 (in place:
// reads precede writes).  w0, w1, w2: rows r-2, r-1, r (x swept when the x
// sweep comes first).  dq (unless the fast policy's kCarryDiff is off):
// y-order limiter_diff of rows r-2 and r-1 on entry, of rows r-1 and r on exit.
// With `emit`, outq is row r-2 after the y sweep.
template <class S, class M>
__device__ __forceinline__ void y_sweep_step(const SubstepArgs& a, float kky, const float (&w0)[S::kC][S::NV],
                                             const float (&w1)[S::kC][S::NV], const float (&w2)[S::kC][S::NV],
                                             float (&qbt)[S::kC][S::NV], float (&g)[S::kC][S::NV],
                                             float (&dq)[S::kC][S::NV], bool emit, float (&outq)[S::kC][S::NV]) {
    constexpr int NV = S::NV;
    constexpr int C = S::kC;
    float y0[C][NV], y1[C][NV], y2[C][NV], qbb[C][NV], qbt_next[C][NV], G[C][NV];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        to_y<NV>(w0[c], y0[c]);
        to_y<NV>(w1[c], y1[c]);
        to_y<NV>(w2[c], y2[c]);
    }
    if constexpr (!M::exact && !S::kCarryDiff) {
        reconstruct_fast<S>([&](int c, int k) { return y1[c][k] - y0[c][k]; },
                            [&](int c, int k) { return y2[c][k] - y1[c][k]; }, y1, a, kky, qbb,
                            qbt_next);  // faces of row r-1
    } else {
        float f[C][NV];
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < NV; ++k) f[c][k] = limiter_diff<M>(y1[c][k], y2[c][k], a);
        reconstruct<S, M>([&](int c, int k) { return dq[c][k]; }, [&](int c, int k) { return f[c][k]; },
                          [&](int c, int k) { return y2[c][k] - y0[c][k]; }, y1, a, kky, qbb,
                          qbt_next);  // faces of row r-1
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < NV; ++k) dq[c][k] = f[c][k];
    }
    S::flux_y(qbt, qbb, a, G);  // interface (r-2, r-1)
#pragma unroll
    for (int c = 0; c < C; ++c) {
        if (emit) {
#pragma unroll
            for (int k = 0; k < NV; ++k) y0[c][k] = evolve<M>(y0[c][k], g[c][k] - G[c][k], a.dt, a.dy, a.dtdy);
            to_y<NV>(y0[c], outq[c]);
        }
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            qbt[c][k] = qbt_next[c][k];
            g[c][k] = G[c][k];
        }
    }
}

// The y sweep's carried state from the first three rows of a march: the faces
// of row 1 (its top face in qbt) and its difference to row 2.
template <class S, class M>
__device__ __forceinline__ void y_sweep_begin(const SubstepArgs& a, float kky, const float (&w0)[S::kC][S::NV],
                                              const float (&w1)[S::kC][S::NV], const float (&w2)[S::kC][S::NV],
                                              float (&qbt)[S::kC][S::NV], float (&g)[S::kC][S::NV],
                                              float (&dq)[S::kC][S::NV]) {
    constexpr int NV = S::NV;
    constexpr int C = S::kC;
    float y0[C][NV], y1[C][NV], y2[C][NV], qbb[C][NV];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        to_y<NV>(w0[c], y0[c]);
        to_y<NV>(w1[c], y1[c]);
        to_y<NV>(w2[c], y2[c]);
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            dq[c][k] = limiter_diff<M>(y1[c][k], y2[c][k], a);
            g[c][k] = 0.0f;
        }
    }
    reconstruct<S, M>([&](int c, int k) { return limiter_diff<M>(y0[c][k], y1[c][k], a); },
                      [&](int c, int k) { return dq[c][k]; },
                      [&](int c, int k) { return y2[c][k] - y0[c][k]; }, y1, a, kky, qbb, qbt);
}

// gravity source after both sweeps of a substep, EE2D_KP07_dimsplit.cu:197-205
template <class S>
__device__ __forceinline__ void gravity_source(const SubstepArgs& a, float (&q)[S::kC][S::NV]) {
    if constexpr (S::kEuler) {
        if (a.g > 0.0f) {
#pragma unroll
            for (int c = 0; c < S::kC; ++c) {
                const float rho_v = q[c][2];
                q[c][2] -= a.g * q[c][0] * a.dt;
                q[c][3] -= a.g * rho_v * a.dt;
            }
        }
    }
}

// One row of a substep's march: the x and y sweeps in the substep's order,
// gravity, store and CFL of row r-2.  w2 holds raw row r on entry.
template <class S, class M, bool XFirst, bool Edge>
__device__ __forceinline__ void slope_row(const SubstepArgs& a, const Strip<S::kC>& st, float kky,
                                          const float (&w0)[S::kC][S::NV], const float (&w1)[S::kC][S::NV],
                                          float (&w2)[S::kC][S::NV], float (&qbt)[S::kC][S::NV],
                                          float (&g)[S::kC][S::NV], float (&dq)[S::kC][S::NV], int r, bool emit,
                                          float& dt_min) {
    constexpr int NV = S::NV;
    constexpr int C = S::kC;
    if constexpr (XFirst) x_sweep_row<S, M>(w2, a);
    float outq[C][NV];
    y_sweep_step<S, M>(a, kky, w0, w1, w2, qbt, g, dq, emit, outq);
    if (emit) {
        if constexpr (!XFirst) x_sweep_row<S, M>(outq, a);
        gravity_source<S>(a, outq);
        store_row<C, NV, Edge>(a, st, r - 2, outq);
        // the CFL minimum is taken after the y-then-x substep only: it is what
        // computeDt reads after a full step (the last launch's values)
        if constexpr (!XFirst) accumulate_cfl<S, M>(outq, a, st, dt_min);
    }
}

// WAF: the y window holds 3 rows (r-2 .. r) and there is no slope state.
// Each ring slot carries its row's WafCells (sweep-y view), computed once when
// the row is ready; hd carries h* of the interface (r-2, r-1) and dd[0], dd[1]
// the limiter denominators of the interfaces (r-3, r-2) and (r-2, r-1); g is
// the flux through the bottom interface of row r-2.  All carried values are
// replaced in place.
template <class S, class M, bool XFirst, bool Edge>
__device__ __forceinline__ void waf_row(const SubstepArgs& a, const Strip<S::kC>& st, const float (&w1)[S::kC][3],
                                        float (&w3)[S::kC][3], const WafCell (&c1)[S::kC],
                                        const WafCell (&c2)[S::kC], WafCell (&c3)[S::kC], float (&hd)[S::kC],
                                        WafDen (&dd)[2][S::kC], float (&g)[S::kC][3], int r, bool emit,
                                        float& dt_min) {
    constexpr int C = S::kC;
    // w1: row r-2 (x swept when XFirst), w3: raw row r on entry
    if constexpr (XFirst) x_sweep_row<S, M>(w3, a);
    float outq[C][3];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        {
            float y3[3];
            to_y<3>(w3[c], y3);
            c3[c] = waf_cell<M>(y3, a.g, a.hg, a.sqrt_g);
        }
        const float hd_r = waf_hstar<M>(c2[c], c3[c], a.g, a.inv_g);  // interface (r-1, r)
        const WafDen Dn = waf_den<M>(c2[c], c3[c], hd_r);
        float G[3];
        waf_flux_core<M>(c1[c], c2[c], dd[0][c], dd[1][c], Dn, hd[c], a.dy, a.dt, a.dtdy, G);  // interface (r-2, r-1)
        if (emit) {
            float y1[3];
            to_y<3>(w1[c], y1);
#pragma unroll
            for (int k = 0; k < 3; ++k) y1[k] = evolve<M, true>(y1[k], g[c][k] - G[k], a.dt, a.dy, a.dtdy);
            to_y<3>(y1, outq[c]);
        }
        hd[c] = hd_r;
        dd[0][c] = dd[1][c];
        dd[1][c] = Dn;
#pragma unroll
        for (int k = 0; k < 3; ++k) g[c][k] = G[k];
    }
    if (emit) {
        if constexpr (!XFirst) x_sweep_row<S, M>(outq, a);
        store_row<C, 3, Edge>(a, st, r - 2, outq);
        // the CFL minimum is taken after the y-then-x substep only: it is what
        // computeDt reads after a full step (the last launch's values)
        if constexpr (!XFirst) accumulate_cfl<S, M>(outq, a, st, dt_min);
    }
}

// Row march of a slope scheme over one segment.  Row m of the segment lives in
// ring slot m % N; the steady loop is unrolled N times so that every slot index
// is a compile-time constant (the ring stays in registers, nothing is copied).
// Edge: the wave has lanes whose columns need 4-byte loads or stores (see
// Strip); the other waves' marches carry no code for them.
template <class S, class M, bool XFirst, bool Edge>
__device__ __forceinline__ float march_slopes(const SubstepArgs& a, const Strip<S::kC>& st) {
    constexpr int NV = S::NV;
    constexpr int C = S::kC;
    constexpr int PF = S::kPrefetch;
    constexpr int N = PF + 3;  // rows r-2, r-1, r and PF rows in flight
    const float kky = M::exact ? M::div(a.dt, 2.0f * a.dy) : 0.5f * a.dtdy;
    float dt_min = M::exact ? __builtin_inff() : 0.0f;
    float ring[N][C][NV], P[C][NV], G[C][NV], dq[C][NV];
    unsigned ys[N];  // y-momentum sign mask of each slot's row
    const int last = st.r_end - 1;  // r_end >= 5
    // prologue: rows 0 .. N-1; faces of row 1; then step r = 3 (flux (1,2), no output)
#pragma unroll
    for (int m = 0; m < N; ++m) ys[m] = load_row_raw<C, NV, S::kPinRows, Edge>(a, st, min(m, last), ring[m]);
#pragma unroll
    for (int m = 0; m < 3; ++m) use_row<C, NV, S::kPinRows>(st, ys[m], ring[m]);
    if constexpr (XFirst) {
        x_sweep_row<S, M>(ring[0], a);
        x_sweep_row<S, M>(ring[1], a);
        x_sweep_row<S, M>(ring[2], a);
    }
    y_sweep_begin<S, M>(a, kky, ring[0], ring[1], ring[2], P, G, dq);  // faces of row 1
    ys[(3 + PF) % N] = load_row_raw<C, NV, S::kPinRows, Edge>(a, st, min(3 + PF, last), ring[(3 + PF) % N]);
    use_row<C, NV, S::kPinRows>(st, ys[3 % N], ring[3 % N]);
    slope_row<S, M, XFirst, Edge>(a, st, kky, ring[1], ring[2], ring[3 % N], P, G, dq, 3, false, dt_min);
    // steady state: r = 4, 4 + N, ...; the step of row rr loads row rr + PF into
    // the slot of row rr - 3, whose last use was the previous step.  Whole
    // groups of N rows run without branches; the remainder (< N rows) keeps
    // the same compile-time slots behind wave-uniform tests.
    auto step = [&](int u, int rr) {
        ys[(4 + u + PF) % N] =
            load_row_raw<C, NV, S::kPinRows, Edge>(a, st, min(rr + PF, last), ring[(4 + u + PF) % N]);
        use_row<C, NV, S::kPinRows>(st, ys[(4 + u) % N], ring[(4 + u) % N]);
        slope_row<S, M, XFirst, Edge>(a, st, kky, ring[(2 + u) % N], ring[(3 + u) % N], ring[(4 + u) % N], P, G, dq, rr,
                                true, dt_min);
    };
    int r = 4;
    for (; r + N <= st.r_end; r += N) {
#pragma unroll
        for (int u = 0; u < N; ++u) step(u, r + u);
    }
#pragma unroll
    for (int u = 0; u < N - 1; ++u)
        if (r + u < st.r_end) step(u, r + u);
    return dt_min;
}

// Row march of WAF (3-row window): row m and its WafCells in ring slot m % N.
template <class S, class M, bool XFirst, bool Edge>
__device__ __forceinline__ float march_waf(const SubstepArgs& a, const Strip<S::kC>& st) {
    constexpr int C = S::kC;
    constexpr int PF = S::kPrefetch;
    constexpr int N = PF + 3;  // rows r-2 .. r and PF rows in flight
    float dt_min = M::exact ? __builtin_inff() : 0.0f;
    float ring[N][C][3], G[C][3], hd[C];
    WafCell cell[N][C];
    WafDen dd[2][C];
    unsigned ys[N];  // y-momentum sign mask of each slot's row
    const int last = st.r_end - 1;  // r_end >= 5
    // prologue: rows 0 .. N-1; interfaces (0, 1) and (1, 2); row 3 + PF; then
    // step r = 3 (flux (1,2), no output)
#pragma unroll
    for (int m = 0; m < N; ++m) ys[m] = load_row_raw<C, 3, S::kPinRows, Edge>(a, st, min(m, last), ring[m]);
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        use_row<C, 3, S::kPinRows>(st, ys[m], ring[m]);
        if constexpr (XFirst) x_sweep_row<S, M>(ring[m], a);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            float y[3];
            to_y<3>(ring[m][c], y);
            cell[m][c] = waf_cell<M>(y, a.g, a.hg, a.sqrt_g);
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float hd01 = waf_hstar<M>(cell[0][c], cell[1][c], a.g, a.inv_g);
        hd[c] = waf_hstar<M>(cell[1][c], cell[2][c], a.g, a.inv_g);
        dd[0][c] = waf_den<M>(cell[0][c], cell[1][c], hd01);
        dd[1][c] = waf_den<M>(cell[1][c], cell[2][c], hd[c]);
#pragma unroll
        for (int k = 0; k < 3; ++k) G[c][k] = 0.0f;
    }
    // row 3 + PF into the slot of row 0, whose last use was above
    ys[(3 + PF) % N] = load_row_raw<C, 3, S::kPinRows, Edge>(a, st, min(3 + PF, last), ring[(3 + PF) % N]);
    use_row<C, 3, S::kPinRows>(st, ys[3], ring[3]);
    waf_row<S, M, XFirst, Edge>(a, st, ring[1], ring[3], cell[1], cell[2], cell[3], hd, dd, G, 3, false, dt_min);
    // steady state: r = 4, 4 + N, ...; the step of row rr loads row rr + PF into
    // the slot of row rr - 3, whose last use was the previous step
    auto step = [&](int u, int rr) {
        ys[(4 + u + PF) % N] = load_row_raw<C, 3, S::kPinRows, Edge>(a, st, min(rr + PF, last), ring[(4 + u + PF) % N]);
        use_row<C, 3, S::kPinRows>(st, ys[(4 + u) % N], ring[(4 + u) % N]);
        waf_row<S, M, XFirst, Edge>(a, st, ring[(2 + u) % N], ring[(4 + u) % N], cell[(2 + u) % N], cell[(3 + u) % N],
                              cell[(4 + u) % N], hd, dd, G, rr, true, dt_min);
    };
    int r = 4;
    for (; r + N <= st.r_end; r += N) {
#pragma unroll
        for (int u = 0; u < N; ++u) step(u, r + u);
    }
#pragma unroll
    for (int u = 0; u < N - 1; ++u)
        if (r + u < st.r_end) step(u, r + u);
    return dt_min;
}

// The column constants of a strip whose lane 0, column 0 is padded column
// `wstart`; H lanes at each end are halo, and only columns [lo, hi) are written.
template <int C, int GC, bool Deep>
__device__ __forceinline__ void setup_columns(Strip<C>& st, int lane, int wstart, int H, int nx, int bc, int lo,
                                              int hi) {
    st.lane = lane;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        st.col[c] = wstart + C * lane + c;
        const AxisMap mx = map_axis_gc<GC, Deep>(st.col[c], nx, bc & 0xF, (bc >> 8) & 0xF);
        st.lane_off[c] = mx.idx * (int)sizeof(float);
        st.xsign[c] = mx.mirrored ? 0x80000000u : 0u;
        st.lane_out[c] = lane >= H && lane < kLanes - H && st.col[c] >= lo && st.col[c] < hi;
    }
    if constexpr (C == 1) {
        st.store_off = st.lane_out[0] ? st.col[0] * (int)sizeof(float) : kMaskedOffset;
    } else {
        const int o0 = st.lane_off[0], o1 = st.lane_off[1];
        const bool fwd = o1 == o0 + 4, rev = GC > 1 && o1 == o0 - 4;
        const int base = rev ? o1 : o0;
        st.pair_rev = rev;
        st.lane_fix = !(fwd || rev) || (base & 7) != 0;
        st.pair_off = st.lane_fix ? kMaskedOffset : base;
        st.fix_off[0] = st.lane_fix ? o0 : kMaskedOffset;
        st.fix_off[1] = st.lane_fix ? o1 : kMaskedOffset;
        st.wave_fix = __builtin_amdgcn_ballot_w64(st.lane_fix) != 0;
        const int s0 = st.col[0] * (int)sizeof(float);
        const bool full = st.lane_out[0] && st.lane_out[1] && (s0 & 7) == 0;
        st.store_off = full ? s0 : kMaskedOffset;
        st.single_off[0] = (!full && st.lane_out[0]) ? s0 : kMaskedOffset;
        st.single_off[1] = (!full && st.lane_out[1]) ? s0 + 4 : kMaskedOffset;
        st.wave_single = __builtin_amdgcn_ballot_w64(!full && (st.lane_out[0] || st.lane_out[1])) != 0;
    }
}

// The fields' buffer descriptors, of `rows` padded rows each.
template <int NV, int C, class Args>
__device__ __forceinline__ void setup_fields(const Args& a, Strip<C>& st, int rows) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        st.rin[k] = field_rsrc(a.in[k], (unsigned)rows * (unsigned)a.in_pitch[k]);
        st.rout[k] = field_rsrc(a.out[k], (unsigned)rows * (unsigned)a.out_pitch[k]);
    }
}

// Halo: cells of halo a side, 2 for a substep and 4 for a whole step.
template <class S, class M, int Halo = 2>
__device__ __forceinline__ void setup_strip(const SubstepArgs& a, Strip<S::kC>& st, int lane, int strip_x, int row_in,
                                            int count) {
    constexpr int C = S::kC;
    constexpr int H = halo_lanes<C, Halo>();
    constexpr bool Deep = Halo > 2;
    st.row0 = __builtin_amdgcn_readfirstlane(a.y0 + row_in + 2 - Halo);  // padded row of r = 0
    st.r_end = __builtin_amdgcn_readfirstlane(count + 2 * Halo);         // output rows r = 2 Halo .. r_end-1
    st.ymap = make_row_map<2, Deep>(a.ny, (a.bc >> 16) & 0xF, (a.bc >> 24) & 0xF);
    const int first = a.x0 + strip_cols<C, Halo>() * strip_x + 2;  // padded column of the first output
    setup_columns<C, 2, Deep>(st, lane, first - H * C, H, a.nx, a.bc, first, a.x1 + 2);
    setup_fields<S::NV>(a, st, a.ny + 4);
}

// The march of one segment: sweep order by step, and the edge variant only
// for waves that need it (a wave-uniform choice made once per segment).
template <class S, class M>
__device__ __forceinline__ float march(const SubstepArgs& a, const Strip<S::kC>& st) {
    if constexpr (S::kC == 2) {
        if (st.wave_fix || st.wave_single) {
            if constexpr (S::kSlopes)
                return (a.step == 0) ? march_slopes<S, M, true, true>(a, st) : march_slopes<S, M, false, true>(a, st);
            else
                return (a.step == 0) ? march_waf<S, M, true, true>(a, st) : march_waf<S, M, false, true>(a, st);
        }
    }
    if constexpr (S::kSlopes)
        return (a.step == 0) ? march_slopes<S, M, true, false>(a, st) : march_slopes<S, M, false, false>(a, st);
    else
        return (a.step == 0) ? march_waf<S, M, true, false>(a, st) : march_waf<S, M, false, false>(a, st);
}

// at least this many waves per SIMD must fit (the plan asks for four)
#ifndef FVMI_SUBSTEP_MIN_WAVES
#define FVMI_SUBSTEP_MIN_WAVES 4
#endif

// Round-weighted work split.  Workgroups are dispatched in index order, one
// per CU per round (workgroup p lands on XCD p % xcds, in round
// (p / xcds) / cus_per_xcd), and a SIMD's instruction arbiter favours its
// oldest wave, so with equal segments a SIMD's waves finish one after another
// and the last runs alone.  Here the waves of earlier rounds take longer parts
// of each row group (weights kRoundWeights).  The waves of one workgroup take
// the same rows of adjacent strips, so that each padded row is read as one
// run of waves_per_block * 240 bytes at about the same time (DRAM pages are
// opened once per row run instead of once per strip); consecutive CUs of an
// XCD take consecutive row groups of the same strips.
constexpr int kRounds = 4;
// With the banded mapping, per launch against 13:11:9:7 (same box): KP07_dimsplit
// 4096^2 113.5 / 114.1 us, HLL2 132.8 / 134.1, EE2D 8192^2 step 1.167 / 1.187 ms
// (fast) and 2.125 / 2.156 (exact); 12:11:10:9 and 10:10:10:10 were slower.
#ifndef FVMI_ROUND_WEIGHTS
#define FVMI_ROUND_WEIGHTS 14, 11, 9, 6
#endif
constexpr int kRoundWeights[kRounds] = {FVMI_ROUND_WEIGHTS};
constexpr int round_weight_sum() {
    int sum = 0;
    for (int k = 0; k < kRounds; ++k) sum += kRoundWeights[k];
    return sum;
}
constexpr int kRoundWeightSum = round_weight_sum();

// rows [lo, hi) of part k of a group of n rows
__host__ __device__ inline void round_part(int n, int k, int& lo, int& hi) {
    int c[kRounds + 1];
    c[0] = 0;
    for (int j = 0; j < kRounds - 1; ++j) c[j + 1] = c[j] + (n * kRoundWeights[j]) / kRoundWeightSum;
    c[kRounds] = n;
    lo = c[k];
    hi = c[k + 1];
}

// The segment of physical wave `wave` of workgroup `block` in the
// round-weighted split of `strips` strips of `rows` rows into `gps` groups of
// `grows` rows; false for an idle slot.
__host__ __device__ inline bool round_segment_of(int block, int wave, int xcds, int cus_per_xcd, int waves_per_block,
                                                 int strips, int rows, int gps, int grows, int& strip_x, int& row_in,
                                                 int& count) {
    const int x = block % xcds;
    const int q = block / xcds;
    const int k = q / cus_per_xcd;
    const int c = q - k * cus_per_xcd;
    if (k >= kRounds) return false;
    // CU slot T takes row group T % gps of the strip band T / gps (a band is
    // waves_per_block adjacent strips, one per wave)
    const int T = x * cus_per_xcd + c;
    const int bands = (strips + waves_per_block - 1) / waves_per_block;
    if (T >= bands * gps) return false;
    const int band = T / gps;
    strip_x = band * waves_per_block + wave;
    if (strip_x >= strips) return false;
    const int g0 = (T - band * gps) * grows;
    const int n = min(grows, rows - g0);
    if (n <= 0) return false;
    int lo, hi;
    round_part(n, k, lo, hi);
    row_in = g0 + lo;
    count = hi - lo;
    return count > 0;
}

// Whether the round-weighted split fits: row groups (gps per strip, grows rows)
// whose shortest part has at least `min_part` rows, and at least `min_fill` percent
// of the waves that equal segments would have.  A group is a CU's, so that the
// strips have to divide the CUs well: a whole step at 8192^2 gives 37 bands of
// strips 6 groups each, 222 of 256 CUs.
__host__ __device__ inline bool round_split_fits(int strips, int rows, int waves_per_block, int cu_count, int min_part,
                                                 int min_fill, int& gps, int& grows) {
    // one 4-wave workgroup per CU and round: a wave on every SIMD
    if (waves_per_block != 4 || cu_count <= 0 || cu_count % 8 != 0 || strips <= 0) return false;
    gps = cu_count / ((strips + waves_per_block - 1) / waves_per_block);
    if (gps <= 0) return false;
    if (100LL * gps * kRounds < (long long)min_fill * (4 * kRounds * cu_count / strips)) return false;
    grows = (rows + gps - 1) / gps;
    const int last = rows - (gps - 1) * grows;  // the shortest (last) group
    return (last * kRoundWeights[kRounds - 1]) / kRoundWeightSum >= min_part;
}

__host__ __device__ inline bool round_segment(const SubstepArgs& a, int block, int wave, int& strip_x, int& row_in,
                                              int& count) {
    return round_segment_of(block, wave, a.xcds, a.cus_per_xcd, a.waves_per_block, a.strips_x, a.rows_per_strip,
                            a.gps, a.grows, strip_x, row_in, count);
}

// The segment of physical wave `wave` of workgroup `block` (of `grid`) in the
// equal-segment plan: global wave gw takes segment gw % segs_per_strip of strip
// gw / segs_per_strip.  Hardware dispatch places workgroup i on XCD i % 8; with
// xcd_remap each XCD owns a contiguous range of logical blocks (neighbouring
// strips share L2).  (Giving a workgroup's waves adjacent strips instead, as
// the round-weighted split does, made WAF 19 % slower: 174 -> 207 us per
// 4096^2 substep.)
__host__ __device__ inline bool uniform_segment(const SubstepArgs& a, int block, int grid, int wave, int& strip_x,
                                                int& row_in, int& count) {
    int lb = block;
    if (a.xcd_remap) {
        const int per = grid >> 3;  // grid is a multiple of 8 when remapping
        lb = (block & 7) * per + (block >> 3);
    }
    const int gw = lb * a.waves_per_block + wave;
    if (lb >= a.num_blocks || gw >= a.num_waves) return false;
    strip_x = gw / a.segs_per_strip;
    row_in = (gw - strip_x * a.segs_per_strip) * a.seg_rows;
    count = min(a.seg_rows, a.rows_per_strip - row_in);
    return true;
}

// the segment of a physical wave in either plan
__host__ __device__ inline bool wave_segment(const SubstepArgs& a, int block, int grid, int wave, int& strip_x,
                                             int& row_in, int& count) {
    return a.round_plan ? round_segment(a, block, wave, strip_x, row_in, count)
                        : uniform_segment(a, block, grid, wave, strip_x, row_in, count);
}

template <class S, class M>
__global__ void __launch_bounds__(256, FVMI_SUBSTEP_MIN_WAVES) substep_kernel(SubstepArgs a) {
    const int lane = threadIdx.x & (kLanes - 1);
    // wave index made scalar so that every row address is computed in SGPRs
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (a.cfl != nullptr && blockIdx.x == 0 && threadIdx.x == 0) a.cfl[1 - (a.step & 1)] = __builtin_inff();
    const bool shared = block_cfl(a.round_plan, a.step == 1 ? a.cfl : nullptr);
    begin_cfl(shared);
    int strip_x, row_in, count;
    float acc = no_cfl<M>();
    if (wave_segment(a, blockIdx.x, gridDim.x, wave, strip_x, row_in, count)) {
        strip_x = __builtin_amdgcn_readfirstlane(strip_x);
        row_in = __builtin_amdgcn_readfirstlane(row_in);
        count = __builtin_amdgcn_readfirstlane(count);
        Strip<S::kC> st;
        setup_strip<S, M>(a, st, lane, strip_x, row_in, count);
        acc = march<S, M>(a, st);
    }
    if (a.cfl != nullptr && a.step == 1) reduce_cfl<M>(shared, a.cfl + 1, acc, lane);
}

}  // namespace fvmi
