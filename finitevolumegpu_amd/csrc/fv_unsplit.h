// The reference's other shallow-water schemes: Lax-Friedrichs, FORCE and
// first-order HLL (one ghost cell) and the unsplit second-order
// Kurganov-Petrova scheme with TVD RK2 (two ghost cells).
//
//   LxF   GPUSimulators/cuda/SWE2D_LxF.cu:93-166   x and y fluxes of the same
//         state (LxF_2D_flux, SWECommon.h:421-427), one update
//   HLL   SWE2D_HLL.cu:100-160, FORCE  SWE2D_FORCE.cu:88-140   first order,
//         x sweep of every row (halo rows included, evolveF common.h:443-456)
//         then y sweep of that state (evolveG :464-475), in one launch
//   KP07  SWE2D_KP07.cu:120-230   minmod slopes in x and y of the same state,
//         face values without predictor, central-upwind fluxes, one update;
//         the second stage of RK2 writes 0.5 (out_old + Q) (:205-214)
//
// Work split and addressing as the dimensionally split kernel (fv_substep.h):
// a wavefront owns a strip of 64 - 2*GC columns (lane c = padded column
// 62*s + c for GC = 1, 60*s + c for GC = 2; the GC lanes at each edge are the
// x halo), or for GC = 1 on large grids of 124 columns, two per lane, and marches
// down a segment of rows; x neighbours come through DPP row moves, y neighbours
// from a register ring of rows.
#pragma once

#include "fv_substep.h"

namespace fvmi {

enum UnsplitKind : int { KIND_LXF = 0, KIND_SPLIT1 = 1, KIND_KP07U = 2 };

struct UnsplitArgs {
    int nx, ny;
    float dx, dy, dt, g, theta;
    int bc;
    int stage2;    // KP07 with order 2, second stage: out = 0.5 (out_old + Q)
    int cfl_slot;  // this launch minimises cfl[cfl_slot] and resets the other slot
    const float* in[3];
    int in_pitch[3];
    float* out[3];
    int out_pitch[3];
    float* cfl;  // two floats, may be null
    int cols;  // columns per lane: two for the one-ghost-cell schemes on 8-byte aligned fields, else one
    int seg_rows;
    int segs_per_strip;
    int strips_x;
    int num_waves;
    int waves_per_block;
    int num_blocks;
    int xcd_remap;
    // round-weighted split (round_plan = 1; round_segment_of in fv_substep.h)
    int round_plan;
    int xcds, cus_per_xcd;
    int gps, grows;
    // fast-policy constants (host): 0.5 g, sqrt(g), dt/dx, dt/dy and the
    // centred fluxes' coefficients dx/(4dt), dy/(4dt) (LxF), dx/(2dt),
    // dy/(2dt), dt/(2dx), dt/(2dy) (FORCE)
    float hg, sqrt_g, inv_dx, inv_dy, dtdx, dtdy;
    float lxf_kx, lxf_ky, lf_kx, lf_ky, lw_kx, lw_ky;
    float half_theta, inv_2theta;  // theta/2 and 1/(2 theta) (0 for theta <= 0), KP07
};

// Half the limited slope, s/2, of a cell with neighbours l and r.  Fast form:
// minmod(theta b, (b + f)/2, theta f) = theta minmod(b, (b + f)/(2 theta), f)
// for theta > 0 (b, f the backward and forward differences).
template <class M, class Args>
__device__ __forceinline__ float half_slope(float l, float c, float r, const Args& a) {
    if constexpr (M::exact) {
        return 0.5f * minmod_slope((c - l) * a.theta, 0.5f * (r - l), (r - c) * a.theta);
    } else {
        const float b = c - l, f = r - c;
        return a.half_theta *
               __builtin_amdgcn_fmed3f(__builtin_amdgcn_fmed3f(b, f, 0.0f), (b + f) * a.inv_2theta, 0.0f);
    }
}

// ---------------------------------------------------------------------------
// Centred fluxes (SWECommon.h:404-473), in sweep order (h, normal, tangential)
// ---------------------------------------------------------------------------

// LxF_2D_flux, SWECommon.h:421-427: 0.5 (F_l + F_r) + dx/(4 dt) (Q_l - Q_r);
// k = dx/(4 dt) (exact: computed here in the reference's order)
template <class M>
__device__ __forceinline__ void lxf_2d_flux(const float ql[3], const float qr[3], float g, float d, float dt, float k,
                                            float out[3]) {
    float Fl[3], Fr[3];
    swe_F<M>(ql, g, Fl);
    swe_F<M>(qr, g, Fr);
    if constexpr (M::exact) k = M::quot(d, 4.0f * dt);
#pragma unroll
    for (int i = 0; i < 3; ++i) out[i] = 0.5f * (Fl[i] + Fr[i]) + k * (ql[i] - qr[i]);
}

// FORCE_1D_flux, SWECommon.h:466-470: mean of LxF_1D_flux (:404-410) and the
// Richtmyer flux LxW2_1D_flux (:443-450).  klf = dx/(2dt), klw = dt/(2dx).
template <class M>
__device__ __forceinline__ void force_1d_flux(const float ql[3], const float qr[3], float g, float d, float dt,
                                              float klf, float klw, float out[3]) {
    float Fl[3], Fr[3], q[3], Flw[3];
    swe_F<M>(ql, g, Fl);
    swe_F<M>(qr, g, Fr);
    if constexpr (M::exact) {
        klf = M::quot(d, 2.0f * dt);
        klw = M::quot(dt, 2.0f * d);
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) q[i] = 0.5f * (ql[i] + qr[i]) + klw * (Fl[i] - Fr[i]);
    swe_F<M>(q, g, Flw);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float lf = 0.5f * (Fl[i] + Fr[i]) + klf * (ql[i] - qr[i]);
        out[i] = 0.5f * (lf + Flw[i]);
    }
}

// ---------------------------------------------------------------------------
// Scheme policies
// ---------------------------------------------------------------------------

// a state as the array of one column that the fast fluxes take
__device__ __forceinline__ const float (&one_column(const float* q))[1][3] {
    return *reinterpret_cast<const float(*)[1][3]>(q);
}
__device__ __forceinline__ float (&one_column(float* q))[1][3] { return *reinterpret_cast<float(*)[1][3]>(q); }

template <class M>
struct UnsplitBase {
    __device__ static float cell_dt(const float q[3], const UnsplitArgs& a) {
        return swe_cell_dt<M>(q, a.dx, a.dy, a.g);
    }
    __device__ static float cell_rate(const float q[3], const UnsplitArgs& a) {
        return fast::swe_cell_rate(q, a.sqrt_g, a.inv_dx, a.inv_dy);
    }
};

// flux_x / flux_y take the interfaces of a lane's C columns at once.
template <class M>
struct SweLxF : UnsplitBase<M> {
    static constexpr int GC = 1;
    static constexpr int kind = KIND_LXF;
    template <int C>
    __device__ static void flux_x(const float (&l)[C][3], const float (&r)[C][3], const UnsplitArgs& a,
                                  float (&o)[C][3]) {
#pragma unroll
        for (int c = 0; c < C; ++c) lxf_2d_flux<M>(l[c], r[c], a.g, a.dx, a.dt, a.lxf_kx, o[c]);
    }
    template <int C>
    __device__ static void flux_y(const float (&l)[C][3], const float (&r)[C][3], const UnsplitArgs& a,
                                  float (&o)[C][3]) {
#pragma unroll
        for (int c = 0; c < C; ++c) lxf_2d_flux<M>(l[c], r[c], a.g, a.dy, a.dt, a.lxf_ky, o[c]);
    }
};

template <class M>
struct SweHLL1 : UnsplitBase<M> {
    static constexpr int GC = 1;
    static constexpr int kind = KIND_SPLIT1;
    template <int C>
    __device__ static void flux_x(const float (&l)[C][3], const float (&r)[C][3], const UnsplitArgs& a,
                                  float (&o)[C][3]) {
        if constexpr (M::exact) {
#pragma unroll
            for (int c = 0; c < C; ++c) swe_hll_flux(l[c], r[c], a.g, o[c]);
        } else {
            fast::swe_hll_flux<C>(l, r, a.hg, a.sqrt_g, o);
        }
    }
    template <int C>
    __device__ static void flux_y(const float (&l)[C][3], const float (&r)[C][3], const UnsplitArgs& a,
                                  float (&o)[C][3]) {
        flux_x<C>(l, r, a, o);
    }
};

template <class M>
struct SweFORCE : UnsplitBase<M> {
    static constexpr int GC = 1;
    static constexpr int kind = KIND_SPLIT1;
    template <int C>
    __device__ static void flux_x(const float (&l)[C][3], const float (&r)[C][3], const UnsplitArgs& a,
                                  float (&o)[C][3]) {
#pragma unroll
        for (int c = 0; c < C; ++c) force_1d_flux<M>(l[c], r[c], a.g, a.dx, a.dt, a.lf_kx, a.lw_kx, o[c]);
    }
    template <int C>
    __device__ static void flux_y(const float (&l)[C][3], const float (&r)[C][3], const UnsplitArgs& a,
                                  float (&o)[C][3]) {
#pragma unroll
        for (int c = 0; c < C; ++c) force_1d_flux<M>(l[c], r[c], a.g, a.dy, a.dt, a.lf_ky, a.lw_ky, o[c]);
    }
};

template <class M>
struct SweKP07U : UnsplitBase<M> {
    static constexpr int GC = 2;
    static constexpr int kind = KIND_KP07U;
    __device__ static void flux(const float l[3], const float r[3], const UnsplitArgs& a, float o[3]) {
        if constexpr (M::exact)
            swe_cu_flux(l, r, a.g, o);
        else
            fast::swe_cu_flux<1>(one_column(l), one_column(r), a.hg, a.sqrt_g, one_column(o));
    }
};

// ---------------------------------------------------------------------------
// Strip addressing (Strip, load_row_raw, use_row, store_row of fv_substep.h)
// ---------------------------------------------------------------------------

// Columns of a strip of C columns per lane.  One ghost cell: 62 with one column
// (lane 1 of strip 0 holds padded column 1), 124 with two (lane 1 holds columns
// 0 and 1, so that pairs sit at 8-byte offsets; column 0 is not written).
template <int GC, int C>
__host__ __device__ constexpr int u_strip_cols() {
    return strip_cols<C, GC>();
}
// first padded column in the output lanes of strip 0
template <int GC, int C>
__host__ __device__ constexpr int u_first_col() {
    return GC == 1 && C == 2 ? 0 : GC;
}

template <int GC, int C>
__device__ __forceinline__ void u_setup(const UnsplitArgs& a, Strip<C>& st, int lane, int strip_x, int row_in,
                                        int count) {
    constexpr int H = halo_lanes<C, GC>();
    st.row0 = __builtin_amdgcn_readfirstlane(row_in);  // padded row of the first row read
    st.r_end = __builtin_amdgcn_readfirstlane(count + 2 * GC);
    st.ymap = make_row_map<GC>(a.ny, (a.bc >> 16) & 0xF, (a.bc >> 24) & 0xF);
    const int first = u_first_col<GC, C>() + u_strip_cols<GC, C>() * strip_x;
    setup_columns<C, GC, false>(st, lane, first - H * C, H, a.nx, a.bc, GC, a.nx + GC);
    setup_fields<3>(a, st, a.ny + 2 * GC);
}

// Values first used here: an empty volatile statement hands them on, so the
// scheduler keeps their consumers behind the loads issued before this point
// and the prefetch distance holds (see use_row in fv_substep.h).  Measured at
// 4096^2 against the same code without it: LxF 9 %, FORCE 7 %, HLL 4 % faster.
__device__ __forceinline__ void u_pin(float (&v)[3]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) asm volatile("" : "+v"(v[k]));
}

// Output row `prow` (padded) of the second RK2 stage, 0.5 (old + q) with `old`
// the output buffer's value (SWE2D_KP07.cu:205-209), read ahead by u_load_old.
// Every lane stores; the halo lanes' offset is out of range (kMaskedOffset), so
// the hardware drops their writes (and returns 0 for their reads).
__device__ __forceinline__ void u_load_old(const UnsplitArgs& a, const Strip<1>& st, int prow, float (&old)[3]) {
    const int row = __builtin_amdgcn_readfirstlane(prow);
#pragma unroll
    for (int k = 0; k < 3; ++k)
        old[k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(st.rout[k], st.store_off, row * a.out_pitch[k], 0));
}

template <class S, class M>
__device__ __forceinline__ void u_cfl(const float (&q)[3], const UnsplitArgs& a, bool take, float& acc) {
    if constexpr (M::exact) {
        const float cd = S::cell_dt(q, a);
        acc = take ? fminf(acc, cd) : acc;
    } else {
        const float rate = S::cell_rate(q, a);
        acc = take ? fmaxf(acc, rate) : acc;
    }
}

__device__ __forceinline__ void swap_tn(const float (&q)[3], float (&o)[3]) {
    o[0] = q[0];
    o[1] = q[2];
    o[2] = q[1];
}

// q + (df dt / dx + dg dt / dy) with the flux differences df = fl - fr, dg = gs
// - gn: the unsplit update of SWE2D_LxF.cu:147-152 and SWE2D_KP07.cu:190-195
template <class M, class Args>
__device__ __forceinline__ float u_update(float q, float df, float dg, const Args& a) {
    if constexpr (M::exact)
        return q + (M::quot(df * a.dt, a.dx) + M::quot(dg * a.dt, a.dy));
    else
        return q + (df * a.dtdx + dg * a.dtdy);
}

// ---------------------------------------------------------------------------
// Row steps
// ---------------------------------------------------------------------------

// x fluxes of one row held across the lanes, C columns each: F[c] through the
// right interface of column c; dF[c] = left flux minus right flux of column c.
template <class S, int C>
__device__ __forceinline__ void x_flux_differences(const float (&q)[C][3], const UnsplitArgs& a, float (&dF)[C][3]) {
    float right[C][3], F[C][3];
    all_from_right<3>(q[0], right[C - 1]);
#pragma unroll
    for (int c = 0; c < C - 1; ++c)
#pragma unroll
        for (int k = 0; k < 3; ++k) right[c][k] = q[c + 1][k];
    S::template flux_x<C>(q, right, a, F);
    left_minus_all<3>(F[C - 1], F[0], dF[0]);
#pragma unroll
    for (int c = 1; c < C; ++c)
#pragma unroll
        for (int k = 0; k < 3; ++k) dF[c][k] = F[c - 1][k] - F[c][k];
}

// x sweep of a row of a split first-order scheme
template <class S, class M, int C>
__device__ __forceinline__ void x_sweep_first_order(float (&q)[C][3], const UnsplitArgs& a) {
    float dF[C][3];
    x_flux_differences<S, C>(q, a, dF);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < 3; ++k) q[c][k] = evolve<M>(q[c][k], dF[c][k], a.dt, a.dx, a.dtdx);
}

// x fluxes of KP07: minmod slope along the row, face values Q -+ slope/2,
// central-upwind flux at (c, c+1) (SWE2D_KP07.cu:30-56, 103-115)
template <class S, class M>
__device__ __forceinline__ void x_fluxes_kp07(const float (&q)[3], const UnsplitArgs& a, float (&F)[3]) {
    float l[3], r[3], qm[3], bot[3], qp[3];
    all_from_left<3>(q, l);
    all_from_right<3>(q, r);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float hs = half_slope<M>(l[k], q[k], r[k], a);
        qm[k] = q[k] + hs;   // right face of cell c
        bot[k] = q[k] - hs;  // left face of cell c
    }
    all_from_right<3>(bot, qp);  // of cell c + 1
    S::flux(qm, qp, a, F);
}

// y fluxes between two rows (lower = row r, upper = row r+1): the flux
// functions see (h, hv, hu) and the result is swapped back
template <class S, int C>
__device__ __forceinline__ void y_fluxes(const float (&lo)[C][3], const float (&hi)[C][3], const UnsplitArgs& a,
                                         float (&G)[C][3]) {
    float l[C][3], h[C][3], o[C][3];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        swap_tn(lo[c], l[c]);
        swap_tn(hi[c], h[c]);
    }
    S::template flux_y<C>(l, h, a, o);
#pragma unroll
    for (int c = 0; c < C; ++c) swap_tn(o[c], G[c]);
}

// One step of the one-ghost-cell march: w0 = row r-1 (x-evolved for the split
// schemes), w1 = raw row r on entry (x-evolved here for the split schemes);
// g = flux (r-2, r-1) on entry, (r-1, r) on return; emits row r-1.
template <class S, class M, int C, bool Edge>
__device__ __forceinline__ void gc1_row(const UnsplitArgs& a, const Strip<C>& st, const float (&w0)[C][3],
                                        float (&w1)[C][3], float (&g)[C][3], int r, bool emit, float& acc) {
    if constexpr (S::kind == KIND_SPLIT1) x_sweep_first_order<S, M, C>(w1, a);
    float G[C][3];
    y_fluxes<S, C>(w0, w1, a, G);
    if (emit) {
        float out[C][3], dF[C][3];
        if constexpr (S::kind != KIND_SPLIT1) x_flux_differences<S, C>(w0, a, dF);
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float dG = g[c][k] - G[c][k];
                if constexpr (S::kind == KIND_SPLIT1)
                    out[c][k] = evolve<M>(w0[c][k], dG, a.dt, a.dy, a.dtdy);
                else
                    out[c][k] = u_update<M>(w0[c][k], dF[c][k], dG, a);
            }
        store_row<C, 3, Edge>(a, st, r - 1, out);
#pragma unroll
        for (int c = 0; c < C; ++c) u_cfl<S, M>(out[c], a, st.lane_out[c], acc);
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < 3; ++k) g[c][k] = G[c][k];
}

// One step of the KP07 march: w0, w1, w2 = raw rows r-2, r-1, r; top = top
// face of row r-2 on entry (of r-1 on return); g = flux (r-3, r-2) on entry,
// (r-2, r-1) on return; emits row r-2 (Stage2: averaged with `old`, the output
// buffer's row r-2).
template <class S, class M, bool Stage2>
__device__ __forceinline__ void kp07u_row(const UnsplitArgs& a, const Strip<1>& st, const float (&w0)[3],
                                          const float (&w1)[3], const float (&w2)[3], const float (&old)[3],
                                          float (&top)[3], float (&g)[3], int r, bool emit, float& acc) {
    float bot[3], top_next[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float hs = half_slope<M>(w0[k], w1[k], w2[k], a);
        top_next[k] = w1[k] + hs;
        bot[k] = w1[k] - hs;
    }
    float G[3];
    {
        float l[3], h[3], o[3];
        swap_tn(top, l);
        swap_tn(bot, h);
        S::flux(l, h, a, o);
        swap_tn(o, G);
    }
    if (emit) {
        float F[3], dF[3], out[3];
        x_fluxes_kp07<S, M>(w0, a, F);
        left_minus_all<3>(F, F, dF);
#pragma unroll
        for (int k = 0; k < 3; ++k) out[k] = u_update<M>(w0[k], dF[k], g[k] - G[k], a);
        float v[1][3];
#pragma unroll
        for (int k = 0; k < 3; ++k) v[0][k] = Stage2 ? 0.5f * (old[k] + out[k]) : out[k];
        store_row<1, 3>(a, st, r - 2, v);
        u_cfl<S, M>(out, a, st.lane_out[0], acc);  // before the RK2 average, as writeCfl reads the tile
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        top[k] = top_next[k];
        g[k] = G[k];
    }
}

// ---------------------------------------------------------------------------
// Marches (row m of a segment in ring slot m % N; see march_slopes)
// ---------------------------------------------------------------------------

template <class S, class M, int C, bool Edge>
__device__ __forceinline__ float march_gc1(const UnsplitArgs& a, const Strip<C>& st) {
    constexpr int PF = kRowPrefetch;
    constexpr int N = PF + 2;  // rows r-1, r and PF rows in flight
    float acc = M::exact ? __builtin_inff() : 0.0f;
    float ring[N][C][3], G[C][3];
    unsigned ys[N];  // y-momentum sign mask of each slot's row
    const int last = st.r_end - 1;  // r_end >= 3
    auto load = [&](int slot, int m) { ys[slot] = load_row_raw<C, 3, true, Edge, 1>(a, st, min(m, last), ring[slot]); };
    auto use = [&](int slot) { use_row<C, 3, true>(st, ys[slot], ring[slot]); };
#pragma unroll
    for (int m = 0; m < N; ++m) load(m, m);
    use(0);
    use(1);
    if constexpr (S::kind == KIND_SPLIT1) x_sweep_first_order<S, M, C>(ring[0], a);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < 3; ++k) G[c][k] = 0.0f;
    // the prologue holds rows 0 .. 1+PF, all that step 1 and its prefetch need
    gc1_row<S, M, C, Edge>(a, st, ring[0], ring[1], G, 1, false, acc);  // flux (0, 1)
    auto step = [&](int u, int rr) {
        load((2 + u + PF) % N, rr + PF);
        use((2 + u) % N);
        gc1_row<S, M, C, Edge>(a, st, ring[(1 + u) % N], ring[(2 + u) % N], G, rr, true, acc);
    };
    int r = 2;
    for (; r + N <= st.r_end; r += N) {
#pragma unroll
        for (int u = 0; u < N; ++u) step(u, r + u);
    }
#pragma unroll
    for (int u = 0; u < N - 1; ++u)
        if (r + u < st.r_end) step(u, r + u);
    return acc;
}

// Stage2: the output buffer's row of step m (padded row row0 + m - 2) is read
// with input row m, into slot m % N of its own ring, PF steps before it is
// averaged and stored.  Only steps m >= 4 emit, so only their rows are read
// (the rows of steps 0 and 1 would lie above the buffer for the first segment).
template <class S, class M, bool Stage2>
__device__ __forceinline__ float march_kp07u(const UnsplitArgs& a, const Strip<1>& st) {
    constexpr int PF = kRowPrefetch;
    constexpr int N = PF + 3;
    static_assert(3 + PF >= 4, "rows loaded in the steps belong to emitting steps");
    float acc = M::exact ? __builtin_inff() : 0.0f;
    float ring[N][1][3], old[N][3], P[3], G[3];
    unsigned ys[N];  // y-momentum sign mask of each slot's row
    const int last = st.r_end - 1;  // r_end >= 5
    auto load = [&](int m, int slot) {  // m >= 4
        ys[slot] = load_row_raw<1, 3, true>(a, st, min(m, last), ring[slot]);
        if constexpr (Stage2) u_load_old(a, st, st.row0 + min(m, last) - 2, old[slot]);
    };
#pragma unroll
    for (int m = 0; m < N; ++m) {
        if (m >= 4)
            load(m, m);
        else
            ys[m] = load_row_raw<1, 3, true>(a, st, min(m, last), ring[m]);
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) use_row<1, 3, true>(st, ys[m], ring[m]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {  // top face of row 1
        P[k] = ring[1][0][k] + half_slope<M>(ring[0][0][k], ring[1][0][k], ring[2][0][k], a);
        G[k] = 0.0f;
    }
    load(3 + PF, (3 + PF) % N);
    use_row<1, 3, true>(st, ys[3 % N], ring[3 % N]);
    kp07u_row<S, M, Stage2>(a, st, ring[1][0], ring[2][0], ring[3 % N][0], old[3 % N], P, G, 3, false, acc);  // flux (1, 2)
    auto step = [&](int u, int rr) {
        load(rr + PF, (4 + u + PF) % N);
        use_row<1, 3, true>(st, ys[(4 + u) % N], ring[(4 + u) % N]);
        if constexpr (Stage2) u_pin(old[(4 + u) % N]);
        kp07u_row<S, M, Stage2>(a, st, ring[(2 + u) % N][0], ring[(3 + u) % N][0], ring[(4 + u) % N][0],
                                old[(4 + u) % N], P, G, rr, true, acc);
    };
    int r = 4;
    for (; r + N <= st.r_end; r += N) {
#pragma unroll
        for (int u = 0; u < N; ++u) step(u, r + u);
    }
#pragma unroll
    for (int u = 0; u < N - 1; ++u)
        if (r + u < st.r_end) step(u, r + u);
    return acc;
}

// The segment of physical wave `wave` of workgroup `block` (of `grid`): the
// round-weighted split, or equal segments with the XCD remap of
// uniform_segment (fv_substep.h).
__host__ __device__ inline bool unsplit_segment(const UnsplitArgs& a, int block, int grid, int wave, int& strip_x,
                                                int& row_in, int& count) {
    if (a.round_plan)
        return round_segment_of(block, wave, a.xcds, a.cus_per_xcd, a.waves_per_block, a.strips_x, a.ny, a.gps,
                                a.grows, strip_x, row_in, count);
    int lb = block;
    if (a.xcd_remap) {
        const int per = grid >> 3;
        lb = (block & 7) * per + (block >> 3);
    }
    if (lb >= a.num_blocks) return false;
    int seg;
    if (a.cols == 2) {  // the waves of a workgroup take the same rows of adjacent strips
        const int band = lb / a.segs_per_strip;
        strip_x = band * a.waves_per_block + wave;
        seg = lb - band * a.segs_per_strip;
        if (strip_x >= a.strips_x) return false;
    } else {
        const int gw = lb * a.waves_per_block + wave;
        if (gw >= a.num_waves) return false;
        strip_x = gw / a.segs_per_strip;
        seg = gw - strip_x * a.segs_per_strip;
    }
    row_in = seg * a.seg_rows;
    count = min(a.seg_rows, a.ny - row_in);
    return true;
}

// C: columns per lane (the two-ghost-cell scheme marches one)
template <class S, class M, int C>
__global__ void __launch_bounds__(256, 4) unsplit_kernel(UnsplitArgs a) {
    constexpr int GC = S::GC;
    static_assert(GC == 1 || C == 1, "KP07 marches one column per lane");
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (a.cfl != nullptr && blockIdx.x == 0 && threadIdx.x == 0) a.cfl[1 - a.cfl_slot] = __builtin_inff();
    begin_cfl(a.cfl != nullptr);
    int strip_x, row_in, count;
    float acc = no_cfl<M>();
    if (unsplit_segment(a, blockIdx.x, gridDim.x, wave, strip_x, row_in, count)) {
        strip_x = __builtin_amdgcn_readfirstlane(strip_x);
        row_in = __builtin_amdgcn_readfirstlane(row_in);
        count = __builtin_amdgcn_readfirstlane(count);
        Strip<C> st;
        u_setup<GC, C>(a, st, lane, strip_x, row_in, count);
        if constexpr (GC == 1) {
            if (C == 2 && (st.wave_fix || st.wave_single))
                acc = march_gc1<S, M, C, C == 2>(a, st);
            else
                acc = march_gc1<S, M, C, false>(a, st);
        } else {
            acc = a.stage2 ? march_kp07u<S, M, true>(a, st) : march_kp07u<S, M, false>(a, st);
        }
    }
    if (a.cfl != nullptr) reduce_cfl<M>(true, a.cfl + a.cfl_slot, acc, lane);
}

// Strip-aligned segments (as plan_substep) for a.cols columns per lane: the
// round-weighted split where `round_ok` and it fits, else equal segments, at most
// waves_per_simd waves on every SIMD.
inline int plan_unsplit(UnsplitArgs& a, int gc, int cu_count, bool round_ok, int waves_per_simd = 4,
                        int min_part = 16) {
    if (gc == 1 && a.cols == 2) {
        constexpr int W = u_strip_cols<1, 2>();
        a.strips_x = (a.nx + 1 + W - 1) / W;  // output columns from padded column 0 on
    } else {
        const int W = kLanes - 2 * gc;
        a.strips_x = (a.nx + W - 1) / W;
    }
    a.round_plan = 0;
    a.xcds = 8;
    a.cus_per_xcd = cu_count / 8;
    a.gps = a.grows = 0;
    int gps = 0, grows = 0;
    if (round_ok && a.seg_rows <= 0 && a.xcd_remap &&
        round_split_fits(a.strips_x, a.ny, a.waves_per_block, cu_count, min_part, 0, gps, grows)) {
        a.round_plan = 1;
        a.gps = gps;
        a.grows = grows;
        a.seg_rows = grows / kRounds;  // nominal, for reporting
        a.segs_per_strip = gps * kRounds;
        a.num_waves = a.strips_x * gps * kRounds;
        a.num_blocks = kRounds * cu_count;
        return a.num_blocks;
    }
    if (a.seg_rows <= 0) {
        const SegmentCost cost = {2 * gc, 2, gc == 2 ? 0.25f : 0.15f * a.cols, 0.01f};
        const int band = a.cols == 2 ? a.waves_per_block : 1;  // strips are dealt out by workgroups
        const int strips = (a.strips_x + band - 1) / band * band;
        a.seg_rows = balanced_segment_rows(a.ny, strips, cu_count, waves_per_simd, cost);
    }
    a.segs_per_strip = (a.ny + a.seg_rows - 1) / a.seg_rows;
    a.num_waves = a.strips_x * a.segs_per_strip;
    a.num_blocks = a.cols == 2 ? ((a.strips_x + a.waves_per_block - 1) / a.waves_per_block) * a.segs_per_strip
                               : (a.num_waves + a.waves_per_block - 1) / a.waves_per_block;
    int grid = a.num_blocks;
    if (a.xcd_remap) grid = ((grid + 7) / 8) * 8;
    return grid;
}

enum UnsplitSchemeId : int { USCHEME_LXF = 0, USCHEME_HLL = 1, USCHEME_FORCE = 2, USCHEME_KP07 = 3 };

// Schemes that take the round-weighted split with one column per lane.  Measured
// at 4096^2 against equal segments: HLL 5 % and the unsplit KP07 1 % faster, LxF
// even, FORCE 3 % slower.  With two columns per lane all take it where it fits
// (adjacent strips per workgroup: 98 us at 4096^2 against 114 for equal segments
// along a strip); elsewhere the equal segments of a workgroup are banded likewise
// (2800^2: 50 -> 45 us).
inline bool unsplit_round_ok(int scheme) { return scheme == USCHEME_HLL || scheme == USCHEME_KP07; }

// Columns per lane of a launch.  Two (8-byte accesses, 124-column strips) for the
// one-ghost-cell schemes, which are bound by memory: what a wave's row access
// covers decides how near they come to a copy of their bytes (79 us at 4096^2).
// Step of three simulators in turn at 4096^2: LxF 123 -> 98 us, FORCE 123 -> 98, HLL
// 111 -> 98; 2800^2 59 -> 45, 2048^2 27.5 -> 24.  One where that leaves less than
// a wave of `min_seg` rows per SIMD (1000^2: 7.7 us with one column, 11.3 with
// two), for HLL in exact arithmetic (bound by VALU issue, 145 and 149 us), and for
// fields that are not 8-byte aligned.
inline int unsplit_cols(const UnsplitArgs& a, int scheme, bool exact, bool aligned8, int cu_count, int min_seg = 24) {
    if (scheme == USCHEME_KP07 || !aligned8 || (exact && scheme == USCHEME_HLL)) return 1;
    const long long strips = (a.nx + u_strip_cols<1, 2>()) / u_strip_cols<1, 2>();
    const int seg = a.seg_rows > 0 ? a.seg_rows : min_seg;
    return strips * ((a.ny + seg - 1) / seg) >= 4LL * cu_count ? 2 : 1;
}

template <class S, class M>
void launch_unsplit_scheme(const UnsplitArgs& a, int grid, hipStream_t stream) {
    const dim3 block(kLanes * a.waves_per_block);
    const unsigned lds = block_cfl_bytes(a.cfl != nullptr);
    if constexpr (S::GC == 1) {
        if (a.cols == 2) {
            hipLaunchKernelGGL((unsplit_kernel<S, M, 2>), dim3(grid), block, lds, stream, a);
            return;
        }
    }
    hipLaunchKernelGGL((unsplit_kernel<S, M, 1>), dim3(grid), block, lds, stream, a);
}

template <class M>
hipError_t launch_unsplit(int scheme, const UnsplitArgs& a, int grid, hipStream_t stream) {
    switch (scheme) {
        case USCHEME_LXF:
            launch_unsplit_scheme<SweLxF<M>, M>(a, grid, stream);
            break;
        case USCHEME_HLL:
            launch_unsplit_scheme<SweHLL1<M>, M>(a, grid, stream);
            break;
        case USCHEME_FORCE:
            launch_unsplit_scheme<SweFORCE<M>, M>(a, grid, stream);
            break;
        case USCHEME_KP07:
            launch_unsplit_scheme<SweKP07U<M>, M>(a, grid, stream);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Defined in fv_kernels_exact.hip / fv_kernels_fast.hip.
hipError_t launch_unsplit_exact(int scheme, const UnsplitArgs& a, int grid, hipStream_t stream);
hipError_t launch_unsplit_fast(int scheme, const UnsplitArgs& a, int grid, hipStream_t stream);

}  // namespace fvmi
