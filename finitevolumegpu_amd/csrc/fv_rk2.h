// Both Runge-Kutta stages of a step of the unsplit KP07 scheme in one launch
// (SWE2D_KP07.cu:120-230, order 2): Q1 = Q + dt L(Q), then 0.5 (Q + Q1 + dt
// L(Q1)), Q1 kept in registers.  The stage launches move 60 bytes per cell (the
// second one reads Q again for the average); this one moves 24.
//
// Geometry, prefetch and the treatment of the ghost cells between the stages are
// those of the whole dimensionally split step (fv_step.h): strips of 56 columns,
// 4 halo rows a side, a march of its own for waves at reflective and outflow
// edges.  A stage needs a window of three rows, the y flux through the bottom of
// its oldest row and that row's top face.  The arithmetic of a cell is the stage
// kernel's, so the fields and the CFL minimum are the two launches' bit for bit.
//
// What bounds it: VALU issue (345 instructions a row); the stage launches were
// bound by memory.  A step of three simulators in turn: 4096^2 262 -> 148 us,
// 2048x1500 41 -> 27; of one alone 278 -> 162 and 90 -> 59.
#pragma once

#include "fv_step.h"
#include "fv_unsplit.h"

namespace fvmi {

// y state of a stage: top face of the window's oldest row, flux through its bottom
struct Rk2State {
    float top[3], g[3];
};

// top face of row 1 of the window w0, w1, w2
template <class M>
__device__ __forceinline__ void rk2_begin(const SubstepArgs& a, const float (&w0)[3], const float (&w1)[3],
                                          const float (&w2)[3], Rk2State& s) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        s.top[k] = w1[k] + half_slope<M>(w0[k], w1[k], w2[k], a);
        s.g[k] = 0.0f;
    }
}

// y faces between rows w0 and w1 of a window (sweep order), as the flux takes
// them; the state's top face moves up to w1's
template <class M>
__device__ __forceinline__ void rk2_y_faces(const SubstepArgs& a, const float (&w0)[3], const float (&w1)[3],
                                            const float (&w2)[3], Rk2State& s, float (&lo)[3], float (&hi)[3]) {
    float bot[3];
    swap_tn(s.top, lo);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float hs = half_slope<M>(w0[k], w1[k], w2[k], a);
        s.top[k] = w1[k] + hs;
        bot[k] = w1[k] - hs;
    }
    swap_tn(bot, hi);
}

// One row of K stages side by side: window rows w0, w1, w2 of each give q, the
// stage's update of w0.  The neighbour exchanges come in runs, and the K x and
// K y fluxes are taken together.
template <class M, int K>
__device__ __forceinline__ void rk2_rows(const SubstepArgs& a, const float (&w0)[K][3], const float (&w1)[K][3],
                                         const float (&w2)[K][3], Rk2State (&s)[K], float (&q)[K][3]) {
    constexpr int N = 3 * K;
    float c[N], l[N], r[N], left[N], right[N], lo[2 * K][3], hi[2 * K][3], F[2 * K][3];
#pragma unroll
    for (int i = 0; i < N; ++i) c[i] = w0[i / 3][i % 3];
    all_from_left<N>(c, l);
    all_from_right<N>(c, r);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float hs = half_slope<M>(l[i], c[i], r[i], a);
        lo[i / 3][i % 3] = c[i] + hs;  // right face of the cell
        left[i] = c[i] - hs;
    }
    all_from_right<N>(left, right);
#pragma unroll
    for (int i = 0; i < N; ++i) hi[i / 3][i % 3] = right[i];
#pragma unroll
    for (int j = 0; j < K; ++j) rk2_y_faces<M>(a, w0[j], w1[j], w2[j], s[j], lo[K + j], hi[K + j]);
    fast::swe_cu_flux<2 * K>(lo, hi, a.hg, a.sqrt_g, F);
    float fx[N], df[N];
#pragma unroll
    for (int i = 0; i < N; ++i) fx[i] = F[i / 3][i % 3];
    left_minus_all<N>(fx, fx, df);
#pragma unroll
    for (int j = 0; j < K; ++j) {
        float G[3];
        swap_tn(F[K + j], G);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            q[j][k] = u_update<M>(w0[j][k], df[3 * j + k], s[j].g[k] - G[k], a);
            s[j].g[k] = G[k];
        }
    }
}

// The march; Edge: waves at filled edges and segments of one row, whose stages
// follow each other within an iteration (middle row r-2, output row r-4).
// Otherwise iteration r takes stage 1 of row r-2 and stage 2 of row r-5 side by
// side.
template <class M, bool Edge>
__device__ __forceinline__ float march_rk2(const SubstepArgs& a, const Strip<1>& st, const StepEdge& e) {
    constexpr int PF = kStepPrefetch;
    static_assert(!M::exact && PF == 2, "fast arithmetic, raw rows in slot r % 3");
    float acc = 0.0f;
    const int last = st.r_end - 1;
    // row j in slot j % 3: rows in flight, window of stage 1, the rows before it
    // (for the average), middle rows
    float raw[3][1][3], w[3][3], old[3][3], m[3][1][3];
    unsigned ys[3];
    Rk2State s1, s2;
    auto copy = [](const float (&from)[3], float (&to)[3]) {
#pragma unroll
        for (int k = 0; k < 3; ++k) to[k] = from[k];
    };
    auto load = [&](int slot, int r) { ys[slot] = load_row_raw<1, 3, true>(a, st, min(r, last), raw[slot]); };
    auto take = [&](int u, int r) {
        load((u + PF) % 3, r + PF);
        use_row<1, 3, true>(st, ys[u], raw[u]);
        copy(raw[u][0], w[u]);
    };
    auto store = [&](int r, const float (&q)[3], const float (&before)[3]) {
        float v[1][3], cfl_q[1][3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            v[0][k] = 0.5f * (before[k] + q[k]);
            cfl_q[0][k] = q[k];
        }
        store_row<1, 3>(a, st, r, v);
        // of the stage's state before the average, as writeCfl reads the tile
        const float rate = fast::swe_cell_rate(cfl_q[0], a.sqrt_g, a.inv_dx, a.inv_dy);
        acc = st.lane_out[0] ? fmaxf(acc, rate) : acc;
    };
    // one stage alone: rows w0, w1, w2 give the update of w0
    auto stage = [&](const float (&w0)[3], const float (&w1)[3], const float (&w2)[3], Rk2State& s, float (&q)[3]) {
        float a0[1][3], a1[1][3], a2[1][3], o[1][3];
        Rk2State t[1] = {s};
        copy(w0, a0[0]), copy(w1, a1[0]), copy(w2, a2[0]);
        rk2_rows<M, 1>(a, a0, a1, a2, t, o);
        s = t[0];
        copy(o[0], q);
    };
    // stage 1 of row r-2 (u = r % 3); row r-2 moves to the rows kept for the average
    auto middle = [&](int u, int r) {
        const int v = (u + 1) % 3;  // slot of row r-2 (and of row r-5 until here)
        float q[1][3];
        stage(w[v], w[(u + 2) % 3], w[u], s1, q[0]);
        if constexpr (Edge) {
            if (e.fix_x) fill_ghost_columns<3>(e, q);
            fill_ghost_row<3>(e, st.row0 + r - 2, m[u], m[(u + 2) % 3], m[v], q);
        }
        copy(q[0], m[v][0]);
        copy(w[v], old[v]);
    };
    load(0, 0);
    load(1, 1);
    take(0, 0);
    take(1, 1);
    take(2, 2);
    rk2_begin<M>(a, w[0], w[1], w[2], s1);
    take(0, 3);
    {
        float q[3];
        stage(w[1], w[2], w[0], s1, q);  // flux (1, 2)
    }
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int k = 0; k < 3; ++k) m[j][0][k] = old[j][k] = 0.0f;
    take(1, 4);
    middle(1, 4);
    take(2, 5);
    middle(2, 5);
    take(0, 6);
    middle(0, 6);
    rk2_begin<M>(a, m[2][0], m[0][0], m[1][0], s2);  // middle rows 2, 3, 4
    if constexpr (Edge) {
        take(1, 7);
        middle(1, 7);
        if (e.fix_lo) {  // rows 2 and 3 are the ghost rows of a low edge
            float g0[1][3];
            copy_ghost_row<3>(e.lo_kind, m[1], m[0]);
            if (e.lo_kind == BC_REFLECTIVE)
                copy_ghost_row<3>(e.lo_kind, m[2], g0);
            else
                copy_ghost_row<3>(e.lo_kind, m[1], g0);
            rk2_begin<M>(a, g0[0], m[0][0], m[1][0], s2);
        }
        float q[3];
        stage(m[0][0], m[1][0], m[2][0], s2, q);  // flux (3, 4) of the middle rows
        auto row = [&](int u, int r) {
            take(u, r);
            // row r-4 (slot u + 2) before stage 1 overwrites nothing of it
            middle(u, r);
            stage(m[(u + 2) % 3][0], m[u][0], m[(u + 1) % 3][0], s2, q);
            store(r - 4, q, old[(u + 2) % 3]);
        };
        int r = 8;
        for (; r + 3 <= st.r_end; r += 3) {
            row(2, r);
            row(0, r + 1);
            row(1, r + 2);
        }
        if (r < st.r_end) row(2, r);
        if (r + 1 < st.r_end) row(0, r + 1);
    } else {
        // both stages of iteration r: middle row r-2, and q = stage 2 of row r-5
        auto both = [&](int u, float (&q)[3]) {
            const int v = (u + 1) % 3, x = (u + 2) % 3;
            float w0[2][3], w1[2][3], w2[2][3], o[2][3];
            Rk2State t[2] = {s1, s2};
            copy(w[v], w0[0]), copy(m[v][0], w0[1]);
            copy(w[x], w1[0]), copy(m[x][0], w1[1]);
            copy(w[u], w2[0]), copy(m[u][0], w2[1]);
            rk2_rows<M, 2>(a, w0, w1, w2, t, o);
            s1 = t[0];
            s2 = t[1];
            copy(o[0], m[v][0]);
            copy(o[1], q);
        };
        float q[3];
        take(1, 7);
        middle(1, 7);
        take(2, 8);
        both(2, q);  // flux (3, 4) of the middle rows
        copy(w[0], old[0]);
        auto row = [&](int u, int r) {
            take(u, r);
            both(u, q);
            store(r - 5, q, old[(u + 1) % 3]);
            copy(w[(u + 1) % 3], old[(u + 1) % 3]);
        };
        auto drain = [&](int u, int r) {  // r = r_end: the last output row
            stage(m[(u + 1) % 3][0], m[(u + 2) % 3][0], m[u][0], s2, q);
            store(r - 5, q, old[(u + 1) % 3]);
        };
        int r = 9;
        for (; r + 3 <= st.r_end; r += 3) {
            row(0, r);
            row(1, r + 1);
            row(2, r + 2);
        }
        const int left = st.r_end - r;
        if (left == 0) {
            drain(0, r);
        } else {
            row(0, r);
            if (left == 1) {
                drain(1, r + 1);
            } else {
                row(1, r + 1);
                drain(2, r + 2);
            }
        }
    }
    return acc;
}

template <class M>
__global__ void __launch_bounds__(256, 4) rk2_kernel(SubstepArgs a) {
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
        setup_strip<SweKP07<M, 1>, M, kStepHalo>(a, st, lane, strip_x, row_in, count);
        StepEdge e;
        setup_edge(a, st, row_in, count, e);
        acc = needs_edge(e) ? march_rk2<M, true>(a, st, e) : march_rk2<M, false>(a, st, e);
    }
    if (a.cfl != nullptr) reduce_cfl<M>(shared, a.cfl + a.cfl_slot, acc, lane);
}

}  // namespace fvmi
