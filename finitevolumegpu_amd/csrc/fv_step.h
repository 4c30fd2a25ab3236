// A whole dimensionally split step in one launch: substep 0 (x then y) and
// substep 1 (y then x) of a slope scheme, the state between them kept in
// registers.  Reads and writes the state once where the two substep launches
// read and write it twice.
//
// Work decomposition: the march of fv_substep.h with a halo of 4 cells instead
// of 2, so 56 output columns per strip of one column per lane.  A wave reads raw
// rows r = 0 .. count+7 of its segment; row r is swept in x, the y sweep then
// finishes row r-2 of the state between the substeps (the middle state), whose
// own y sweep finishes row r-4, which is swept in x and stored.  Every cell's
// arithmetic is that of the two substep kernels, so the fields and the CFL
// minimum are theirs bit for bit.
//
// What bounds it: VALU issue.  The substep launches are bound by their memory
// streams and the tail of their waves (110 us each at 4096^2, 79 us for a copy of
// their bytes); one launch moves half the bytes and executes 7 % more
// instructions (the wider halo).  With the runs of cross-lane operations and
// transcendentals (fv_substep.h, fv_fast.h), a step of three simulators in turn:
// KP07_dimsplit 4096^2 224 -> 172-179 us, HLL2 246 -> 218, 2047^2 64 -> 57, Euler
// 3001x4032 235 -> 200; one simulator alone, KP07_dimsplit 4096^2 218 -> 190 us,
// 128^2 13.4 -> 9.9.
//
// The ghost cells of the middle state follow its own interior, by the boundary
// rule of each edge:
//   * periodic: the images of the raw cells are marched along, two more of
//     them a side (the Deep maps of fv_substep.h), and give the images of the
//     middle cells;
//   * reflective, outflow: a ghost middle cell is a copy of an interior middle
//     cell of the same wave: another lane's for ghost columns, another row of
//     the window for ghost rows (the mirrored momentum changes sign).  Only
//     waves at such an edge run the march that does this.
// Dirichlet edges read the memory of the buffer between the substeps, which
// this launch does not have, and the images beyond a periodic edge are only
// right if the opposite edge is periodic too: other steps take the two substep
// launches (step_is_fused in fv_launch.h).
#pragma once

#include "fv_substep.h"

namespace fvmi {

constexpr int kStepHalo = 4;
// rows loaded ahead: with three slots (row r in slot r % 3) the raw rows share
// the unrolling of the two y windows
constexpr int kStepPrefetch = 2;
// smallest grid side and segment of a fused step: ghost cells mirror within
// the first rows of the first segment and within one wave's columns
constexpr int kStepMinSide = 8;
constexpr int kStepMinSegRows = 4;

// What a wave at a reflective or outflow edge needs to fill the middle
// state's ghost cells.
struct StepEdge {
    bool fix_x;            // wave holds ghost columns of such an edge
    int src_addr;          // bpermute address of the lane this lane's column copies (its own if none)
    unsigned xsign;        // sign mask of the copied x momentum
    bool fix_lo;           // the segment starts at such a low edge
    int lo_kind, hi_kind;  // boundary codes in y
    int hi_row;            // padded row of the first ghost row of a high edge to fill, else past every row
};

constexpr int kNoRow = 0x7fffffff;

__device__ __forceinline__ void setup_edge(const SubstepArgs& a, const Strip<1>& st, int row_in, int count,
                                           StepEdge& e) {
    const int bw = a.bc & 0xF, be = (a.bc >> 8) & 0xF, bs = (a.bc >> 16) & 0xF, bn = (a.bc >> 24) & 0xF;
    const int k = st.col[0];
    int src = k;
    bool mirrored = false;
    if (k >= 0 && k < 2 && bw != BC_PERIODIC) {
        mirrored = bw == BC_REFLECTIVE;
        src = mirrored ? 3 - k : 2;
    } else if ((k == a.nx + 2 || k == a.nx + 3) && be != BC_PERIODIC) {
        mirrored = be == BC_REFLECTIVE;
        src = mirrored ? 2 * (a.nx + 2) - 1 - k : a.nx + 1;
    }
    const int from = st.lane + src - k;  // lane of the source column
    const bool inside = src != k && from >= 0 && from < kLanes;
    e.src_addr = 4 * (inside ? from : st.lane);
    e.xsign = inside && mirrored ? 0x80000000u : 0u;
    e.fix_x = __builtin_amdgcn_ballot_w64(inside) != 0;
    e.lo_kind = bs;
    e.hi_kind = bn;
    e.fix_lo = row_in == 0 && bs != BC_PERIODIC;
    // the march reads middle rows up to padded row row_in + count + 3
    e.hi_row = (bn != BC_PERIODIC && row_in + count + 3 >= a.ny + 2) ? a.ny + 2 : kNoRow;
}

__device__ __forceinline__ bool needs_edge(const StepEdge& e) { return e.fix_x || e.fix_lo || e.hi_row != kNoRow; }

// Ghost columns of a middle row: each takes its source column's values.
template <int NV>
__device__ __forceinline__ void fill_ghost_columns(const StepEdge& e, float (&q)[1][NV]) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        int w = __builtin_amdgcn_ds_bpermute(e.src_addr, __float_as_int(q[0][k]));
        if (k == 1) w ^= (int)e.xsign;
        q[0][k] = __int_as_float(w);
    }
}

// A ghost row from an interior row: a mirroring edge flips the y momentum.
template <int NV>
__device__ __forceinline__ void copy_ghost_row(int kind, const float (&src)[1][NV], float (&q)[1][NV]) {
    const unsigned sign = kind == BC_REFLECTIVE ? 0x80000000u : 0u;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const unsigned w = __float_as_uint(src[0][k]);
        q[0][k] = __uint_as_float(k == 2 ? w ^ sign : w);
    }
}

// Middle row `row` (padded) if it is a ghost row of a filled high edge, from
// the rows one, two and three before it.
template <int NV>
__device__ __forceinline__ void fill_ghost_row(const StepEdge& e, int row, const float (&back1)[1][NV],
                                               const float (&back2)[1][NV], const float (&back3)[1][NV],
                                               float (&q)[1][NV]) {
    const int ghost = __builtin_amdgcn_readfirstlane(row - e.hi_row);
    if (ghost < 0) return;
    if (ghost == 0)  // from the last interior row, both kinds
        copy_ghost_row<NV>(e.hi_kind, back1, q);
    else if (e.hi_kind == BC_REFLECTIVE)  // from the interior row before it
        copy_ghost_row<NV>(e.hi_kind, back3, q);
    else  // outflow: the last interior row again
        copy_ghost_row<NV>(e.hi_kind, back2, q);
}

// Edge waves (and segments of one row): the four sweeps of an iteration one
// after the other.
template <class S, class M>
__device__ __forceinline__ float march_step_edge(const SubstepArgs& a, const Strip<1>& st, const StepEdge& e) {
    constexpr int NV = S::NV;
    constexpr int PF = kStepPrefetch;
    static_assert(S::kC == 1 && PF == 2, "one column per lane, raw rows in slot r % 3");
    const float kky = M::exact ? M::div(a.dt, 2.0f * a.dy) : 0.5f * a.dtdy;
    float acc = M::exact ? __builtin_inff() : 0.0f;
    const int last = st.r_end - 1;  // r_end >= 9
    float raw[3][1][NV];            // rows in flight
    unsigned ys[3];
    float w[3][1][NV], P[1][NV], G[1][NV], dq[1][NV];     // x-swept rows and y state of substep 0
    float m[3][1][NV], P2[1][NV], G2[1][NV], dq2[1][NV];  // middle rows and y state of substep 1
    auto load = [&](int slot, int r) {
        ys[slot] = load_row_raw<1, NV, S::kPinRows>(a, st, min(r, last), raw[slot]);
    };
    auto copy = [](const float (&from)[1][NV], float (&to)[1][NV]) {
#pragma unroll
        for (int k = 0; k < NV; ++k) to[0][k] = from[0][k];
    };
    // loads row r+2, sweeps row r (slot u = r % 3) in x into the window
    auto sweep_x = [&](int u, int r) {
        load((u + PF) % 3, r + PF);
        use_row<1, NV, S::kPinRows>(st, ys[u], raw[u]);
        copy(raw[u], w[u]);
        x_sweep_row<S, M>(w[u], a);
    };
    // middle row r-2 into its slot
    auto middle = [&](int u, int r) {
        float q[1][NV];
        y_sweep_step<S, M>(a, kky, w[(u + 1) % 3], w[(u + 2) % 3], w[u], P, G, dq, true, q);
        gravity_source<S>(a, q);
        if (e.fix_x) fill_ghost_columns<NV>(e, q);
        const int s = (u + 1) % 3;  // slot of row r-2; row r-3 is in slot u, row r-4 in (u + 2) % 3, row r-5 still in s
        fill_ghost_row<NV>(e, st.row0 + r - 2, m[u], m[(u + 2) % 3], m[s], q);
        copy(q, m[s]);
    };
    // y sweep of the middle rows r-4 .. r-2, x sweep and store of row r-4
    auto finish = [&](int u, int r, bool emit) {
        float q[1][NV];
        y_sweep_step<S, M>(a, kky, m[(u + 2) % 3], m[u], m[(u + 1) % 3], P2, G2, dq2, emit, q);
        if (emit) {
            x_sweep_row<S, M>(q, a);
            gravity_source<S>(a, q);
            store_row<1, NV>(a, st, r - 4, q);
            accumulate_cfl<S, M>(q, a, st, acc);
        }
    };
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int k = 0; k < NV; ++k) m[j][0][k] = 0.0f;
    load(0, 0);
    load(1, 1);
    sweep_x(0, 0);
    sweep_x(1, 1);
    sweep_x(2, 2);
    y_sweep_begin<S, M>(a, kky, w[0], w[1], w[2], P, G, dq);
    sweep_x(0, 3);
    {
        float q[1][NV];
        y_sweep_step<S, M>(a, kky, w[1], w[2], w[0], P, G, dq, false, q);  // flux (1, 2)
    }
    sweep_x(1, 4);
    middle(1, 4);
    sweep_x(2, 5);
    middle(2, 5);
    sweep_x(0, 6);
    middle(0, 6);
    y_sweep_begin<S, M>(a, kky, m[2], m[0], m[1], P2, G2, dq2);  // middle rows 2, 3, 4
    sweep_x(1, 7);
    middle(1, 7);
    // rows 2 and 3 are the ghost rows of a low edge: from rows 4 and 5
    if (e.fix_lo) {
        float g0[1][NV];
        copy_ghost_row<NV>(e.lo_kind, m[1], m[0]);
        if (e.lo_kind == BC_REFLECTIVE)
            copy_ghost_row<NV>(e.lo_kind, m[2], g0);
        else
            copy_ghost_row<NV>(e.lo_kind, m[1], g0);
        y_sweep_begin<S, M>(a, kky, g0, m[0], m[1], P2, G2, dq2);
    }
    finish(1, 7, false);  // flux (3, 4) of the middle rows
    auto row = [&](int u, int r) {
        sweep_x(u, r);
        middle(u, r);
        finish(u, r, true);
    };
    int r = 8;
    for (; r + 3 <= st.r_end; r += 3) {
        row(2, r);
        row(0, r + 1);
        row(1, r + 2);
    }
    if (r < st.r_end) row(2, r);
    if (r + 1 < st.r_end) row(0, r + 1);
    return acc;
}

// Waves away from filled edges, for segments of at least two rows.  The same rows in the same
// arithmetic, but the two x sweeps of an iteration, and then its two y sweeps,
// run side by side on different rows, so that their cross-lane operations and
// transcendentals come in runs twice as long: in iteration r the x sweeps take
// raw row r and the output row r-6 that the last iteration's y sweep finished,
// the y sweeps finish middle row r-2 and output row r-5 (from middle rows
// r-5 .. r-3).
template <class S, class M>
__device__ __forceinline__ float march_step_paired(const SubstepArgs& a, const Strip<1>& st) {
    using S2 = typename S::Pair;
    constexpr int NV = S::NV;
    constexpr int PF = kStepPrefetch;
    static_assert(S::kC == 1 && PF == 2, "one column per lane, raw rows in slot r % 3");
    const float kky = M::exact ? M::div(a.dt, 2.0f * a.dy) : 0.5f * a.dtdy;
    float acc = M::exact ? __builtin_inff() : 0.0f;
    const int last = st.r_end - 1;  // r_end >= 10
    float raw[3][1][NV];
    unsigned ys[3];
    float w[3][1][NV], m[3][1][NV];    // x-swept raw rows and middle rows, row j in slot j % 3
    float P1[1][NV], G1[1][NV], dq1[1][NV], P2[1][NV], G2[1][NV], dq2[1][NV];  // y state of the two substeps
    float P[2][NV], G[2][NV], dq[2][NV];                                       // the same, side by side
    float out[1][NV];                  // the output row whose x sweep is next
    auto load = [&](int slot, int r) {
        ys[slot] = load_row_raw<1, NV, S::kPinRows>(a, st, min(r, last), raw[slot]);
    };
    auto copy = [](const float (&from)[NV], float (&to)[NV]) {
#pragma unroll
        for (int k = 0; k < NV; ++k) to[k] = from[k];
    };
    auto store = [&](int r, float (&q)[1][NV]) {
        gravity_source<S>(a, q);
        store_row<1, NV>(a, st, r, q);
        accumulate_cfl<S, M>(q, a, st, acc);
    };
    auto sweep_x = [&](int u, int r) {  // row r alone
        load((u + PF) % 3, r + PF);
        use_row<1, NV, S::kPinRows>(st, ys[u], raw[u]);
        copy(raw[u][0], w[u][0]);
        x_sweep_row<S, M>(w[u], a);
    };
    auto sweep_x_pair = [&](int u, int r) {  // row r and output row r-6, which is stored
        load((u + PF) % 3, r + PF);
        use_row<1, NV, S::kPinRows>(st, ys[u], raw[u]);
        float q[2][NV];
        copy(raw[u][0], q[0]);
        copy(out[0], q[1]);
        x_sweep_row<S2, M, true>(q, a);
        copy(q[0], w[u][0]);
        copy(q[1], out[0]);
        store(r - 6, out);
    };
    auto middle = [&](int u, int r) {  // middle row r-2 alone
        y_sweep_step<S, M>(a, kky, w[(u + 1) % 3], w[(u + 2) % 3], w[u], P1, G1, dq1, true, m[(u + 1) % 3]);
        gravity_source<S>(a, m[(u + 1) % 3]);
    };
    auto sweep_y_pair = [&](int u) {  // middle row r-2 and output row r-5
        // middle rows r-5, r-4, r-3 in slots u+1, u+2, u; row r-2 takes the slot of row r-5
        float w0[2][NV], w1[2][NV], w2[2][NV], q[2][NV], mid[1][NV];
        copy(w[(u + 1) % 3][0], w0[0]), copy(m[(u + 1) % 3][0], w0[1]);
        copy(w[(u + 2) % 3][0], w1[0]), copy(m[(u + 2) % 3][0], w1[1]);
        copy(w[u][0], w2[0]), copy(m[u][0], w2[1]);
        y_sweep_step<S2, M>(a, kky, w0, w1, w2, P, G, dq, true, q);
        copy(q[0], mid[0]);
        gravity_source<S>(a, mid);
        copy(mid[0], m[(u + 1) % 3][0]);
        copy(q[1], out[0]);
    };
    auto drain = [&](int u, int r) {  // r = r_end: the last two output rows
        x_sweep_row<S, M>(out, a);
        store(r - 6, out);
        copy(P[1], P2[0]), copy(G[1], G2[0]), copy(dq[1], dq2[0]);
        y_sweep_step<S, M>(a, kky, m[(u + 1) % 3], m[(u + 2) % 3], m[u], P2, G2, dq2, true, out);
        x_sweep_row<S, M>(out, a);
        store(r - 5, out);
    };
    load(0, 0);
    load(1, 1);
    sweep_x(0, 0);
    sweep_x(1, 1);
    sweep_x(2, 2);
    y_sweep_begin<S, M>(a, kky, w[0], w[1], w[2], P1, G1, dq1);
    sweep_x(0, 3);
    y_sweep_step<S, M>(a, kky, w[1], w[2], w[0], P1, G1, dq1, false, out);  // flux (1, 2)
    sweep_x(1, 4);
    middle(1, 4);
    sweep_x(2, 5);
    middle(2, 5);
    sweep_x(0, 6);
    middle(0, 6);
    y_sweep_begin<S, M>(a, kky, m[2], m[0], m[1], P2, G2, dq2);  // middle rows 2, 3, 4
    sweep_x(1, 7);
    middle(1, 7);
    copy(P1[0], P[0]), copy(G1[0], G[0]), copy(dq1[0], dq[0]);
    copy(P2[0], P[1]), copy(G2[0], G[1]), copy(dq2[0], dq[1]);
    sweep_x(2, 8);
    sweep_y_pair(2);  // flux (3, 4) of the middle rows; no output row yet
    sweep_x(0, 9);
    sweep_y_pair(0);  // output row 4
    auto row = [&](int u, int r) {
        sweep_x_pair(u, r);
        sweep_y_pair(u);
    };
    int r = 10;
    for (; r + 3 <= st.r_end; r += 3) {
        row(1, r);
        row(2, r + 1);
        row(0, r + 2);
    }
    const int left = st.r_end - r;
    if (left == 0) {
        drain(1, r);
    } else {
        row(1, r);
        if (left == 1) {
            drain(2, r + 1);
        } else {
            row(2, r + 1);
            drain(0, r + 2);
        }
    }
    return acc;
}

// The march of one segment; returns the CFL accumulator.
template <class S, class M>
__device__ __forceinline__ float march_step(const SubstepArgs& a, const Strip<1>& st, int row_in, int count) {
    StepEdge e;
    setup_edge(a, st, row_in, count, e);
    return needs_edge(e) || count < 2 ? march_step_edge<S, M>(a, st, e) : march_step_paired<S, M>(a, st);
}

// Four waves fit on a SIMD: 112 VGPRs for KP07_dimsplit and 123 for HLL2, no
// scratch; for Euler 128 and 64 bytes of scratch a lane (ensemble kernel: 128 bytes),
// where the edge march keeps its middle rows: fill_ghost_row takes one of three by
// branch, which becomes a load through a selected address.  The kernels are large (60
// and 72 KB against 38 and 46 for a substep, two marches with their prologues), which
// the first launch of a program pays for.  Measured per 4096^2 step with two columns per lane
// (fewer halo lanes, 168 VGPRs with spills or 247): KP07_dimsplit 327 and 248
// us against 182; five and six waves (96 and 80 VGPRs): 178 and 176 against 172.
template <class S, class M>
__global__ void __launch_bounds__(256, 4) step_kernel(SubstepArgs a) {
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (a.cfl != nullptr && blockIdx.x == 0 && threadIdx.x == 0) a.cfl[1 - a.cfl_slot] = __builtin_inff();
    const bool shared = block_cfl(a.round_plan, a.cfl);
    begin_cfl(shared);
    int strip_x, row_in, count;
    float acc = no_cfl<M>();
    if (wave_segment(a, blockIdx.x, gridDim.x, wave, strip_x, row_in, count)) {
        strip_x = __builtin_amdgcn_readfirstlane(strip_x);
        row_in = __builtin_amdgcn_readfirstlane(row_in);
        count = __builtin_amdgcn_readfirstlane(count);
        Strip<1> st;
        setup_strip<S, M, kStepHalo>(a, st, lane, strip_x, row_in, count);
        acc = march_step<S, M>(a, st, row_in, count);
    }
    if (a.cfl != nullptr) reduce_cfl<M>(shared, a.cfl + a.cfl_slot, acc, lane);
}

}  // namespace fvmi
