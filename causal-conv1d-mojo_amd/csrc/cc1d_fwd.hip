// cc1d_fwd.hip -- forward kernels for gfx950.
//
// Semantics (per batch b, channel c, position t; the CPU definition the
// reference tests against is src/causal_conv1d_mojo/fwd_cpu/kernel.mojo:61-119):
//   pre = bias[c]; for k in 0..W-1: pre += w[c,k] * xx(t + k - (W-1))   (fp32, in that order)
//   out = silu(pre) or pre; 0 where seq_idx[b,t] < 0
// where xx(s) = x[b,c,s] (s >= 0), initial_states[b,c,s+W-1] (s < 0, when
// given) or 0, and with seq_idx a tap is kept only if seq_idx[b,s] == seq_idx[b,t].
//
// Kernels
//   fwd_rows_vec  -- rows contiguous along t (channel-first). One wavefront
//                    owns a segment of 64*VPT*EPV positions of one row; lane l
//                    holds 16-byte vectors l, l+64, ... of the segment, so each
//                    load instruction covers 1 KB of contiguous HBM. The (W-1)
//                    halo before a vector comes from the neighbouring lane
//                    (ds_bpermute); only lane 0 of a segment reads one extra
//                    vector from global memory. No LDS, no barriers.
//                    Rows that are not whole aligned vectors (any start, any
//                    length) are walked in the aligned vectors of their own
//                    memory where out lies like x, else in unaligned ones
//                    (RowsMode in cc1d_device.hpp); a row's first and last
//                    few elements are stored in smaller pieces.
//   fwd_rows_short -- rows of at most 32 vectors: a wavefront takes as many
//                    whole rows as fit into its 64 lanes, a lane one vector.
//   fwd_cl        -- rows contiguous along channels (channel-last). A lane owns
//                    4 bytes of adjacent channels, a wavefront a tile of 16
//                    time steps (plus W-1 halo rows) of 64 lanes' channels,
//                    all loaded before any arithmetic; seq_idx is
//                    wave-uniform here.
//   fwd_generic   -- any strides / alignment; one thread per
//                    (b, c, chunk of time), lanes on adjacent channels.
#include "cc1d_internal.hpp"

namespace cc1d {

struct FwdArgs {
    cc1d_fwd_params p;
    FastDiv nseg_div;  // rows_vec: item -> row; rows_short: lane -> row of the wavefront
    FastDiv dim_div;   // rows_vec: row -> batch entry
    int64_t nseg;     // segments (rows_vec), tiles (cl) or chunks (generic) per row; rows_short: vectors per row
    int64_t n_items;  // work items: segments / tiles / threads; rows_short: rows
    int64_t chunk;    // time steps per item (cl / generic); rows_short: rows per wavefront
    int64_t ngroups;  // channel groups (cl)
};

// One wavefront-segment of one row. Positions t count from m elements before
// the row's first: the row is [m, m + L), m 0 except in kRowsAlike. FULL: the
// whole segment lies inside the row (no per-vector bounds checks). on: the
// lane has a row (kRowsShort; `lane` is then the lane's vector of its row).
template <typename T, int W, int VPT, bool SILU, bool SEQ, bool FULL, int MODE>
__device__ __forceinline__ void fwd_rows_segment(const cc1d_fwd_params& p, int lane, int64_t b, int64_t c,
                                                 int32_t t0, int32_t m, bool on) {
    constexpr int EPV = elems16<T>::value;
    constexpr int H = W - 1;
    constexpr bool SHORT = MODE == kRowsShort, ALIKE = MODE == kRowsAlike;
    constexpr bool ANY = MODE == kRowsAny || SHORT;  // unaligned vectors
    static_assert(!SHORT || (VPT == 1 && !FULL), "short rows: one vector per lane");
    const int32_t Le = (int32_t)p.seqlen + m;      // end of the row
    const int32_t L = SHORT ? (on ? Le : 0) : Le;  // a lane without a row touches nothing
    const T* __restrict__ xr = static_cast<const T*>(p.x) + b * p.x_stride[0] + c * p.x_stride[1] - m;
    T* __restrict__ orow = static_cast<T*>(p.out) + b * p.out_stride[0] + c * p.out_stride[1] - m;

    // the row's last rem elements are part of a vector, which starts at tp:
    // vector jt of the lane with `tail`
    constexpr bool EDGES = MODE != kRowsAligned && !FULL;
    const int rem = EDGES ? Le & (EPV - 1) : 0;
    const int32_t tp = Le - rem;
    const int jt = SHORT ? 0 : (tp - t0) / (64 * EPV);
    const bool tail = EDGES && rem != 0 && tp >= t0 && tp == t0 + (jt * 64 + lane) * EPV && on;
    const bool head = ALIKE && !FULL && m > 0 && t0 == 0;  // wave-uniform: lane 0's first vector starts before the row
    auto whole = [&](int32_t t) {  // the vector at t lies inside the row
        return FULL || (MODE == kRowsAligned ? t < L : ALIKE ? t >= m && t + EPV <= L : t + EPV <= L);
    };

    u32x4 v[VPT];
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int32_t t = t0 + (j * 64 + lane) * EPV;
        if constexpr (ANY) v[j] = whole(t) ? vload_any_nt(xr + t) : vzero();
        else v[j] = (FULL || t < L) ? vload_nt(xr + t) : vzero();
    }
    RowTail<T> xt;
    if constexpr (ANY) {
        xt.a = u32x2{0u, 0u};
        xt.b = xt.c = 0u;
        if (tail) xt.load(xr + tp, rem);
    }
    u32x4 h = vzero();
    if constexpr (!SHORT) {
        if (lane == 0 && t0 > 0) h = ANY ? vload_any(xr - EPV + t0) : vload(xr - EPV + t0);
    }

    int32_t id[VPT][EPV];
    int32_t hid[H];
    if constexpr (SEQ) {
        const int32_t* __restrict__ sr = p.seq_idx + b * p.seq_idx_stride[0] - m;  // unit time stride
#pragma unroll
        for (int j = 0; j < VPT; ++j) {
            const int32_t t = t0 + (j * 64 + lane) * EPV;
            if constexpr (MODE == kRowsAligned) {  // 16-byte vectors of 4 ids
#pragma unroll
                for (int q = 0; q < EPV / 4; ++q) {
                    const u32x4 s = (FULL || t < L) ? *reinterpret_cast<const u32x4*>(sr + t + 4 * q)
                                                    : u32x4{0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu};
#pragma unroll
                    for (int r = 0; r < 4; ++r) id[j][4 * q + r] = (int32_t)s[r];
                }
            } else {
#pragma unroll
                for (int e = 0; e < EPV; ++e) id[j][e] = -1;
                if (whole(t)) ids_any<EPV>(sr + t, id[j]);
                // a row's first and last few ids, each into its own register (no
                // wait here); wave-uniform tests around
                if (EDGES && j == 0 && head) {
                    if (lane == 0) ids_some<EPV>(sr, m, EPV, id[0]);
                }
                if (EDGES && j == jt && rem != 0) {
                    if (tail) ids_some<EPV>(sr + t, 0, rem, id[j]);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const int32_t pos = t0 - H + i;
            hid[i] = (!SHORT && lane == 0 && pos >= m) ? sr[pos] : -1;
        }
    }

    // weights and bias: scalar reads where the row is the wavefront's, which
    // wait for no vector load (the bias address is always valid: no branch).
    // As vector loads behind the row's they held the arithmetic back until
    // the whole row had arrived (us, then -> now: bf16 4 x 5120 x 1000 17.2 ->
    // 16.1, 1 x 1536 x 2048 4.14 -> 3.85, W 9 4 x 5120 x 2048 30.2 -> 29.3, with
    // seq_idx 31.2 -> 30.4 at W 4; fp32 4 x 5120 x 1000 32.2 -> 29.1; C2 28.5 -> 28.4)
    float w[W];
    const T* __restrict__ wr = static_cast<const T*>(p.weight) + c * p.weight_stride[0];
    const T* br = p.bias ? static_cast<const T*>(p.bias) + c * p.bias_stride : wr;
    float braw;
    if constexpr (SHORT) {
#pragma unroll
        for (int k = 0; k < W; ++k) w[k] = ld(wr, k * p.weight_stride[1]);
        braw = to_f32(*br);
    } else {
#pragma unroll
        for (int k = 0; k < W; ++k) w[k] = ld_uniform(wr + k * p.weight_stride[1]);
        braw = ld_uniform(br);
    }
    const float bias = p.bias ? braw : 0.0f;

    const bool use_init = p.initial_states != nullptr && t0 == 0 && lane == 0 && on;
    float hinit[H];
#pragma unroll
    for (int i = 0; i < H; ++i) {
        hinit[i] = 0.0f;
        if (use_init)
            hinit[i] = ld(static_cast<const T*>(p.initial_states),
                          b * p.initial_states_stride[0] + c * p.initial_states_stride[1] +
                              i * p.initial_states_stride[2]);
    }
    // the first vector's m elements before the row (the previous row's) are
    // positions -m .. -1 of this one: initial_states or zero
    if (head && lane == 0) {
        float f[EPV];
#pragma unroll
        for (int e = 0; e < EPV; ++e)  // initial_states slot e - m + H (none when negative)
            f[e] = e >= m ? vget<T>(v[0], e) : pick<H>(hinit, e - m + H);
        v[0] = vpack<T>(f);
    }
    if (ANY && EDGES && rem != 0) {  // wave-uniform
        const u32x4 tv = xt.vec(rem);  // zero in the lanes without the tail
#pragma unroll
        for (int j = 0; j < VPT; ++j)
            if (j == jt) v[j] |= tv;
    }

    constexpr int D0 = ((EPV - H) * (int)sizeof(T)) / 4;  // first dword of the needed tail
    const int wl = SHORT ? (int)(threadIdx.x & 63) : lane;  // lane of the wavefront
    const int prev_lane = (wl + 63) & 63;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        const int32_t t = t0 + (j * 64 + lane) * EPV;
        u32x4 pv = vzero();
#pragma unroll
        for (int d = D0; d < 4; ++d) {
            const uint32_t send = (!SHORT && lane == 63) ? (j > 0 ? v[j > 0 ? j - 1 : 0][d] : 0u) : v[j][d];
            pv[d] = lane_get(send, prev_lane);
        }
        if (j == 0 && lane == 0) pv = h;
        float win[H + EPV];
#pragma unroll
        for (int i = 0; i < H; ++i) {  // before the row: position i - H, initial_states slot i - m
            if constexpr (ALIKE && !FULL)
                win[i] = (j == 0 && use_init) ? pick<H>(hinit, i - m) : vget<T>(pv, EPV - H + i);
            else  // m == 0 whenever a first segment is full
                win[i] = (j == 0 && use_init) ? hinit[i] : vget<T>(pv, EPV - H + i);
        }
#pragma unroll
        for (int i = 0; i < EPV; ++i) win[H + i] = vget<T>(v[j], i);

        int32_t sw[H + EPV];
        if constexpr (SEQ) {
#pragma unroll
            for (int i = 0; i < H; ++i) {
                const int32_t send = (!SHORT && lane == 63) ? (j > 0 ? id[j > 0 ? j - 1 : 0][EPV - H + i] : -1)
                                                            : id[j][EPV - H + i];
                const int32_t r = lane_get(send, prev_lane);
                sw[i] = (j == 0 && lane == 0) ? hid[i] : r;
            }
#pragma unroll
            for (int i = 0; i < EPV; ++i) sw[H + i] = id[j][i];
        }

        float o[EPV];
#pragma unroll
        for (int i = 0; i < EPV; ++i) {
            float acc;
            if constexpr (SEQ) acc = conv_taps_gated<W>(bias, w, win + i, sw + i);
            else acc = conv_taps<W>(bias, w, win + i);
            if constexpr (SILU) acc = silu(acc);
            if constexpr (SEQ) {
                if (sw[H + i] < 0) acc = 0.0f;
            }
            o[i] = acc;
        }
        const u32x4 ov = vpack<T>(o);
        if (whole(t)) {
            if constexpr (ANY) vstore_any_nt(orow + t, ov);
            else vstore_nt(orow + t, ov);
        }
        if (EDGES && j == 0 && head) {
            if (lane == 0) store_from(orow, ov, m);
        }
        if (EDGES && j == jt && rem != 0) {  // wave-uniform
            if (tail) RowTail<T>::store(orow + t, ov, rem);
        }

        // final_states (_fn.py:31-50): the lane holding the row's last
        // position writes the last W-1 columns from its window (they are
        // positions t - H .. t + EPV - 1)
        if (p.final_states_out != nullptr && (MODE != kRowsAligned ? (t < L && L <= t + EPV) : t + EPV == L)) {
            T* fs = static_cast<T*>(p.final_states_out) + b * p.final_states_stride[0] +
                    c * p.final_states_stride[1];
#pragma unroll
            for (int i = 0; i < H; ++i) {  // position L - H + i is window slot L + i - t
                const float fv = MODE != kRowsAligned ? pick<H + EPV>(win, L + i - t) : win[EPV + i];  // t + EPV == L
                st(fs, i * p.final_states_stride[2], (L - H + i >= m) ? fv : 0.0f);
            }
        }
    }
}

// Item = (row, segment) with row = b * dim + c; four wavefronts per block take
// four consecutive items, i.e. adjacent segments of a row or adjacent rows.
// All index arithmetic is 32-bit (the launcher checks the ranges).
template <typename T, int W, int VPT, bool SILU, bool SEQ, int MODE>
__global__ void __launch_bounds__(256) fwd_rows_vec(const FwdArgs a) {
    constexpr int SEG = 64 * VPT * elems16<T>::value;
    const cc1d_fwd_params& p = a.p;
    const int lane = threadIdx.x & 63;
    const uint32_t item = uniform32(blockIdx.x * 4u + (threadIdx.x >> 6));
    if (item >= (uint32_t)a.n_items) return;
    // (row, segment) and (b, c) by the host's invariant-divisor constants
    const uint32_t row = a.nseg_div.div(item);
    const int32_t t0 = (int32_t)((item - row * (uint32_t)a.nseg) * SEG);
    const uint32_t b = a.dim_div.div(row);
    const uint32_t c = row - b * (uint32_t)p.dim;
    int32_t m = 0;  // the row starts m elements past a 16-byte boundary
    if constexpr (MODE == kRowsAlike) {
        const T* xrow = static_cast<const T*>(p.x) + (int64_t)b * p.x_stride[0] + (int64_t)c * p.x_stride[1];
        m = (int32_t)uniform32((uint32_t)(reinterpret_cast<uintptr_t>(xrow) / sizeof(T)) & (elems16<T>::value - 1));
    }
    const int32_t Le = (int32_t)p.seqlen + m;
    if (MODE == kRowsAlike && t0 >= Le) return;  // the row ends before this segment
    if ((t0 > 0 || m == 0) && t0 + SEG <= Le)
        fwd_rows_segment<T, W, VPT, SILU, SEQ, true, MODE>(p, lane, b, c, t0, m, true);
    else
        fwd_rows_segment<T, W, VPT, SILU, SEQ, false, MODE>(p, lane, b, c, t0, m, true);
}

// Rows of nseg <= 32 vectors: a wavefront takes 64 / nseg (rounded down)
// consecutive rows, lane l vector l % nseg of row l / nseg. With a wavefront
// per row instead, a row of 64 bf16 kept 8 of 64 lanes busy. The window
// before a vector comes from the previous lane as in fwd_rows_vec, nothing
// (or initial_states) before a row's first; weights and bias are per-lane
// reads here (rows differ).
template <typename T, int W, bool SILU, bool SEQ>
__global__ void __launch_bounds__(256) fwd_rows_short(const FwdArgs a) {
    const cc1d_fwd_params& p = a.p;
    const uint32_t wl = threadIdx.x & 63;
    const uint32_t nv = (uint32_t)a.nseg, per = (uint32_t)a.chunk;  // vectors per row, rows per wavefront
    const uint32_t r = a.nseg_div.div(wl);
    const uint32_t row0 = uniform32(blockIdx.x * 4u + (threadIdx.x >> 6)) * per;
    if (row0 >= (uint32_t)a.n_items) return;
    const bool on = r < per && row0 + r < (uint32_t)a.n_items;
    const uint32_t row = on ? row0 + r : row0;
    const uint32_t b = a.dim_div.div(row);
    const uint32_t c = row - b * (uint32_t)p.dim;
    fwd_rows_segment<T, W, 1, SILU, SEQ, false, kRowsShort>(p, (int)(wl - r * nv), b, c, 0, 0, on);
}

// Channel-last (unit channel stride), tiled: a lane owns CPL adjacent
// channels (one CPL-element vector per time step); a wavefront covers
// 64 * CPL channels of a tile of TS time steps and issues the loads of all
// TS + W - 1 rows of its window (the W-1 halo rows before the tile included)
// before any arithmetic. seq_idx is one value per time step, the same for
// every lane: it is read through the scalar cache, and a tile whose window
// holds one sequence id (>= 0) takes the ungated path. Item order: channel
// group fastest, then tile, then batch. Index arithmetic is 32-bit inside a
// batch (the launcher checks the ranges).
template <typename T, int W, int CPL, int TS, bool SILU, bool SEQ>
__global__ void __launch_bounds__(256) fwd_cl(const FwdArgs a) {
    constexpr int H = W - 1;
    constexpr int NR = TS + H;
    using V = Lanes<T>;
    static_assert(V::N == CPL, "a dword of channels per lane");
    const cc1d_fwd_params& p = a.p;
    const int lane = threadIdx.x & 63;
    const uint32_t item = uniform32(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (item >= (uint32_t)a.n_items) return;
    const uint32_t ngroups = (uint32_t)a.ngroups, ntiles = (uint32_t)a.nseg;
    const uint32_t g = item % ngroups;
    const uint32_t rest = item / ngroups;
    const uint32_t tile = rest % ntiles;
    const uint32_t b = rest / ntiles;
    const int32_t L = (int32_t)p.seqlen;
    const int32_t cl = (int32_t)((g * 64 + lane) * CPL);
    const bool active = cl < (int32_t)p.dim;
    // the last lane of an odd number of 16-bit channels takes the last CPL ones:
    // the channel it shares with the lane before is computed and stored twice, alike
    const int32_t c0 = cl + CPL <= (int32_t)p.dim ? cl : (int32_t)p.dim - CPL;
    const int32_t t0 = (int32_t)(tile * TS);
    const int32_t xs2 = (int32_t)p.x_stride[2], os2 = (int32_t)p.out_stride[2];
    const T* __restrict__ xb = static_cast<const T*>(p.x) + b * p.x_stride[0] + c0;
    T* __restrict__ ob = static_cast<T*>(p.out) + b * p.out_stride[0] + c0;

    // with seq_idx, and for fp32: ids, weights and bias go out before the rows
    // (raw, so that no conversion waits for them here). Loads complete in
    // order, so a row's outputs can then be computed as soon as that row has
    // arrived (us, rows first -> last: bf16 1 x 4096 x 8192 with seq_idx 30.0 ->
    // 26.8, 1536 x 2048 6.6 -> 5.6; fp32 4 x 2048 x 2000 27.0 -> 24.2). 16-bit
    // types without seq_idx are quicker with the rows first in back-to-back
    // launches of larger grids and even in single ones (first / last, bf16, W 4:
    // 1 x 4096 x 8192 22.2 / 22.7, single 27.4 / 27.2; 4 x 2048 x 2000 13.0 / 13.7,
    // 16.6 / 16.6; 1 x 4096 x 4096 12.3 / 12.9, 15.2 / 15.7), slower on small ones and
    // at W 9 (1 x 1536 x 2048 6.0 / 5.6; W 9 1 x 4096 x 8192 26.5 / 25.9)
    constexpr bool PARAMS_FIRST = SEQ || sizeof(T) == 4;
    int32_t lid = 0;
    if constexpr (SEQ) {
        // lane i < NR reads the id of position t0 - H + i (clamped address,
        // -1 outside the row); the window's ids then reach every lane through
        // readlane, with no dependent scalar reads.
        static_assert(NR <= 64, "the id window must fit in one wavefront");
        const int32_t* sr = p.seq_idx + b * p.seq_idx_stride[0];
        const int32_t s = t0 - H + lane;
        lid = sr[(s < 0 ? 0 : (s < L ? s : L - 1)) * (int32_t)p.seq_idx_stride[1]];
    }
    T wr[W][CPL], br[CPL];
    if constexpr (PARAMS_FIRST) {
#pragma unroll
        for (int e = 0; e < CPL; ++e) {
            const int64_t c = active ? c0 + e : 0;
            const T* wp = static_cast<const T*>(p.weight) + c * p.weight_stride[0];
#pragma unroll
            for (int k = 0; k < W; ++k) wr[k][e] = wp[k * p.weight_stride[1]];
            br[e] = *(p.bias ? static_cast<const T*>(p.bias) + c * p.bias_stride : wp);
        }
        __builtin_amdgcn_sched_barrier(0);
    }

    V xv[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        const int32_t s = t0 - H + i;
        xv[i].zero();
        if (active && s >= 0 && s < L) xv[i].template load<false>(xb + s * xs2);
    }
    if (p.initial_states != nullptr && t0 < H && active) {
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const int32_t s = t0 - H + i;
            if (s < 0) {
                float f[CPL];
#pragma unroll
                for (int e = 0; e < CPL; ++e)
                    f[e] = ld(static_cast<const T*>(p.initial_states),
                              b * p.initial_states_stride[0] + (c0 + e) * p.initial_states_stride[1] +
                                  (s + H) * p.initial_states_stride[2]);
                xv[i].set(f);
            }
        }
    }

    float w[W][CPL], bias[CPL];
#pragma unroll
    for (int e = 0; e < CPL; ++e) {
        if constexpr (PARAMS_FIRST) {
#pragma unroll
            for (int k = 0; k < W; ++k) w[k][e] = to_f32(wr[k][e]);
            bias[e] = p.bias ? to_f32(br[e]) : 0.0f;
        } else {
            const int64_t c = active ? c0 + e : 0;
#pragma unroll
            for (int k = 0; k < W; ++k)
                w[k][e] = ld(static_cast<const T*>(p.weight), c * p.weight_stride[0] + k * p.weight_stride[1]);
            bias[e] = p.bias ? ld(static_cast<const T*>(p.bias), c * p.bias_stride) : 0.0f;
        }
    }

    int32_t id[NR];
    bool one_id = true;
    if constexpr (SEQ) {
        const int32_t s = t0 - H + lane;
        if (s < 0 || s >= L) lid = -1;
        const int32_t id_cur = __builtin_amdgcn_readlane(lid, H);
        // rows outside [0, L) hold zeros (seq_idx excludes initial_states) or
        // feed outputs that are not stored, so they do not break a single-id window
        one_id = id_cur >= 0 && __ballot(lane < NR && s >= 0 && s < L && lid != id_cur) == 0;
#pragma unroll
        for (int i = 0; i < NR; ++i) id[i] = __builtin_amdgcn_readlane(lid, i);
    }

    auto emit = [&](auto gated) {
        constexpr bool G = decltype(gated)::value;
#pragma unroll
        for (int u = 0; u < TS; ++u) {
            const int32_t t = t0 + u;
            float o[CPL];
#pragma unroll
            for (int e = 0; e < CPL; ++e) {
                float col[W], wc[W];
#pragma unroll
                for (int k = 0; k < W; ++k) {
                    col[k] = xv[u + k].get(e);
                    wc[k] = w[k][e];
                }
                float acc;
                if constexpr (G) acc = conv_taps_gated<W>(bias[e], wc, col, id + u);
                else acc = conv_taps<W>(bias[e], wc, col);
                if constexpr (SILU) acc = silu(acc);
                if constexpr (G) {
                    if (id[u + H] < 0) acc = 0.0f;
                }
                o[e] = acc;
            }
            if (active && t < L) {
                V ov;
                ov.set(o);
                ov.template store<true>(ob + t * os2);
            }
        }
    };
    if (!SEQ || one_id) emit(std::false_type{});
    else if constexpr (SEQ) emit(std::true_type{});

    if (p.final_states_out != nullptr && active && t0 + TS >= L) {
        T* fs = static_cast<T*>(p.final_states_out) + b * p.final_states_stride[0];
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const int32_t r = L - t0 + i;  // register row of position L - H + i
            float f[CPL];
#pragma unroll
            for (int e = 0; e < CPL; ++e) f[e] = 0.0f;
#pragma unroll
            for (int q = 0; q < NR; ++q)
                if (q == r && L - H + i >= 0) {
#pragma unroll
                    for (int e = 0; e < CPL; ++e) f[e] = xv[q].get(e);
                }
#pragma unroll
            for (int e = 0; e < CPL; ++e)
                st(fs, (c0 + e) * p.final_states_stride[1] + i * p.final_states_stride[2], f[e]);
        }
    }
}

template <typename T, int W, bool SILU>
__global__ void __launch_bounds__(256) fwd_generic(const FwdArgs a) {
    constexpr int H = W - 1;
    const cc1d_fwd_params& p = a.p;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= a.n_items) return;
    const int64_t c = idx % p.dim;
    const int64_t rest = idx / p.dim;
    const int64_t ch = rest % a.nseg;
    const int64_t b = rest / a.nseg;
    const int64_t L = p.seqlen;
    const int64_t t0 = ch * a.chunk;
    const int64_t t1 = (t0 + a.chunk < L) ? t0 + a.chunk : L;
    const T* __restrict__ xr = static_cast<const T*>(p.x) + b * p.x_stride[0] + c * p.x_stride[1];
    T* __restrict__ orow = static_cast<T*>(p.out) + b * p.out_stride[0] + c * p.out_stride[1];
    const int64_t xs = p.x_stride[2];
    const int32_t* sr = p.seq_idx ? p.seq_idx + b * p.seq_idx_stride[0] : nullptr;

    float w[W];
#pragma unroll
    for (int k = 0; k < W; ++k)
        w[k] = ld(static_cast<const T*>(p.weight), c * p.weight_stride[0] + k * p.weight_stride[1]);
    const float bias = p.bias ? ld(static_cast<const T*>(p.bias), c * p.bias_stride) : 0.0f;

    float win[W];
    int32_t wid[W];
#pragma unroll
    for (int i = 0; i < H; ++i) {
        const int64_t s = t0 - H + i;
        if (s >= 0) {
            win[i] = ld(xr, s * xs);
        } else if (p.initial_states != nullptr) {
            win[i] = ld(static_cast<const T*>(p.initial_states),
                        b * p.initial_states_stride[0] + c * p.initial_states_stride[1] +
                            (s + H) * p.initial_states_stride[2]);
        } else {
            win[i] = 0.0f;
        }
        wid[i] = (sr != nullptr && s >= 0) ? sr[s * p.seq_idx_stride[1]] : -1;
    }
    for (int64_t t = t0; t < t1; ++t) {
        win[H] = ld(xr, t * xs);
        float acc;
        if (sr != nullptr) {
            wid[H] = sr[t * p.seq_idx_stride[1]];
            acc = conv_taps_gated<W>(bias, w, win, wid);
            if (SILU) acc = silu(acc);
            if (wid[H] < 0) acc = 0.0f;
        } else {
            acc = conv_taps<W>(bias, w, win);
            if (SILU) acc = silu(acc);
        }
        st(orow, t * p.out_stride[2], acc);
#pragma unroll
        for (int i = 0; i < H; ++i) {
            win[i] = win[i + 1];
            wid[i] = wid[i + 1];
        }
    }
    if (p.final_states_out != nullptr && t1 == L) {
        T* fs = static_cast<T*>(p.final_states_out) + b * p.final_states_stride[0] + c * p.final_states_stride[1];
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const int64_t s = L - H + i;
            st(fs, i * p.final_states_stride[2], (s >= 0) ? ld(xr, s * xs) : 0.0f);
        }
    }
}

// ---- launch selection ------------------------------------------------------

namespace {

// channel-last launch shape: time steps per wavefront tile
constexpr int kClTS = 16;
constexpr int kClTSSmall = 8;  // on grids of fewer than 4096 wavefronts

template <typename T>
bool rows_vec_ok(const cc1d_fwd_params& p) {
    constexpr int64_t EPV = elems16<T>::value;
    if (p.width - 1 > EPV) return false;
    if (p.x_stride[2] != 1 || p.out_stride[2] != 1) return false;
    if (p.seqlen % EPV != 0) return false;
    if (!aligned16(p.x) || !aligned16(p.out)) return false;
    if (p.x_stride[0] % EPV || p.x_stride[1] % EPV || p.out_stride[0] % EPV || p.out_stride[1] % EPV) return false;
    if (p.seq_idx != nullptr &&
        (p.seq_idx_stride[1] != 1 || p.seq_idx_stride[0] % 4 != 0 || !aligned16(p.seq_idx)))
        return false;
    // 32-bit index arithmetic: positions, rows and items (4 per block) must fit
    if (p.seqlen + 64 * 4 * EPV >= ((int64_t)1 << 31)) return false;
    if (p.batch * p.dim * ceil_div(p.seqlen, 64 * EPV) * 4 >= ((int64_t)1 << 32)) return false;
    return true;
}

// rows of any length at any element boundary: unit time stride is all they
// need (seq_idx too, as 16-byte vectors of 4 ids are read from it)
template <typename T>
bool rows_any_ok(const cc1d_fwd_params& p) {
    constexpr int64_t EPV = elems16<T>::value;
    if (p.width - 1 > EPV) return false;
    if (p.x_stride[2] != 1 || p.out_stride[2] != 1) return false;
    if ((reinterpret_cast<uintptr_t>(p.x) | reinterpret_cast<uintptr_t>(p.out)) % sizeof(T)) return false;
    if (p.seq_idx != nullptr && (p.seq_idx_stride[1] != 1 || reinterpret_cast<uintptr_t>(p.seq_idx) % 4 != 0))
        return false;
    const int64_t lim = (int64_t)1 << 31;
    if (p.seqlen + 64 * 4 * EPV + EPV >= lim) return false;
    if (p.batch * p.dim * ceil_div(p.seqlen + EPV, 64 * EPV) * 4 >= lim * 2) return false;
    return true;
}

// rows_any_ok, and out laid out like x modulo the vector: the same element
// strides modulo EPV and bases a multiple of 16 bytes apart
template <typename T>
bool rows_alike(const cc1d_fwd_params& p) {
    constexpr int64_t EPV = elems16<T>::value;
    return (p.out_stride[0] - p.x_stride[0]) % EPV == 0 && (p.out_stride[1] - p.x_stride[1]) % EPV == 0 &&
           (reinterpret_cast<intptr_t>(p.out) - reinterpret_cast<intptr_t>(p.x)) % 16 == 0;
}

// channel-last tiles: unit channel stride, at least a lane's CPL channels,
// 32-bit positions inside a batch
template <typename T, int CPL>
bool cl_ok(const cc1d_fwd_params& p) {
    if (p.x_stride[1] != 1 || p.out_stride[1] != 1) return false;
    if (p.dim < CPL) return false;
    if ((reinterpret_cast<uintptr_t>(p.x) | reinterpret_cast<uintptr_t>(p.out)) % sizeof(T)) return false;
    const int64_t span = p.seqlen + kClTS + 16;  // furthest row a tile touches
    const int64_t lim = (int64_t)1 << 31;
    if (p.dim >= lim || span * p.x_stride[2] >= lim || span * p.out_stride[2] >= lim) return false;
    if (p.seq_idx != nullptr && span * p.seq_idx_stride[1] >= lim) return false;
    if (p.batch * ceil_div(p.dim, (int64_t)(64 * CPL)) * ceil_div(p.seqlen, kClTS) >= lim * 2) return false;
    return true;
}

}  // namespace

int launch_fwd(const cc1d_fwd_params& p, hipStream_t stream) {
    return with_dtype(p.dtype, [&](auto tag) {
        using T = decltype(tag);
        constexpr int64_t EPV = elems16<T>::value;
        return with_width(p.width, [&](auto wc) {
            constexpr int W = decltype(wc)::value;
            return with_flag(p.apply_silu != 0, [&](auto sc) {
                constexpr bool SILU = decltype(sc)::value;
                FwdArgs a;
                a.p = p;
                a.chunk = 0;
                a.ngroups = 0;
                const int64_t rows = p.batch * p.dim;
                if constexpr (W - 1 <= EPV) {
                    const bool aligned = rows_vec_ok<T>(p);
                    if (aligned || rows_any_ok<T>(p)) {
                        a.dim_div = FastDiv((uint32_t)p.dim);
                        const int64_t least = ceil_div(p.seqlen, EPV);  // vectors from the row's first element on
                        if (least <= kShortVecs && rows_any_ok<T>(p)) {
                            a.nseg = least;
                            a.chunk = 64 / least;
                            a.n_items = rows;
                            a.nseg_div = FastDiv((uint32_t)least);
                            const dim3 grid((unsigned)ceil_div(ceil_div(rows, a.chunk), 4));
                            return with_flag(p.seq_idx != nullptr, [&](auto qc) {
                                return launch(fwd_rows_short<T, W, SILU, decltype(qc)::value>, grid, dim3(256), stream, a);
                            });
                        }
                        // vectors per lane of rows of nvec vectors
                        auto lanes = [&](int64_t nvec) {
                            const int64_t per = ceil_div(nvec, 64);
                            int vpt = per >= 4 ? 4 : (per >= 2 ? 2 : 1);
                            // rows off the 16-byte grid (measured at C2's batch and dim; aligned ones
                            // were faster without either): one segment of 4 vectors per
                            // lane instead of two of 2 with the same lane slots when the
                            // grid keeps 2048 wavefronts (L = 1031: 22.3 instead of
                            // 25.1 us), and 2 instead of 4 when a row a
                            // little longer than a multiple of the 4-vector segment would
                            // leave its last one mostly empty and 2 take at most 85 % of
                            // the lane slots (L = 2049: 34.2 instead of 37.6 us)
                            if (!aligned && per == 3 && rows >= 2048) vpt = 4;
                            else if (!aligned && vpt == 4 &&
                                     ceil_div(nvec, (int64_t)128) * 128 * 100 <= ceil_div(nvec, (int64_t)256) * 256 * 85)
                                vpt = 2;
                            // a grid of fewer than 2048 wavefronts (2 per SIMD): half the
                            // vectors per lane, twice the wavefronts (B = 1, D = 768,
                            // L = 2048: 3.03 instead of 3.41 us; D = 512, L = 1024:
                            // 2.40 instead of 2.53)
                            if (vpt == 4 && rows * ceil_div(nvec, (int64_t)256) < 2048) vpt = 2;
                            if (vpt == 2 && rows * ceil_div(nvec, (int64_t)128) < 2048) vpt = 1;
                            return vpt;
                        };
                        int vpt = lanes(least);
                        a.nseg = ceil_div(least, 64 * (int64_t)vpt);
                        bool alike = false;
                        if (!aligned && rows_alike<T>(p)) {
                            // a row that starts past a vector boundary may span one more
                            const int64_t nvec = ceil_div(p.seqlen + EPV - 1, EPV);
                            const int va = lanes(nvec);
                            const int64_t na = ceil_div(nvec, 64 * (int64_t)va);
                            // aligned vectors, unless that one more costs much of the lane
                            // slots (16-bit types, us at C2's batch and dim, aligned ->
                            // unaligned: L = 1023 21.9 -> 18.2, with seq_idx 35.8 -> 22.4, 511
                            // 14.9 -> 13.1; ten times the batch 177 -> 152, 106 -> 102). A third
                            // of them (L = 2047) pays only with seq_idx (50.1 -> 38.9): large
                            // calls lose as much to unaligned stores (batch 40: 316 -> 330; fp32
                            // 586 -> 646)
                            const int64_t most = p.seq_idx != nullptr ? 85 : 60;  // % of the slots
                            if (sizeof(T) == 4 || vpt * a.nseg * 100 > va * na * most) {
                                alike = true;
                                vpt = va;
                                a.nseg = na;
                            }
                        }
                        a.n_items = rows * a.nseg;
                        a.nseg_div = FastDiv((uint32_t)a.nseg);
                        const dim3 grid((unsigned)ceil_div(a.n_items, 4));
                        return with_flag(p.seq_idx != nullptr, [&](auto qc) {
                            constexpr bool SEQ = decltype(qc)::value;
                            auto go = [&](auto mc) {
                                constexpr int MODE = decltype(mc)::value;
                                if (vpt == 4) return launch(fwd_rows_vec<T, W, 4, SILU, SEQ, MODE>, grid, dim3(256), stream, a);
                                if (vpt == 2) return launch(fwd_rows_vec<T, W, 2, SILU, SEQ, MODE>, grid, dim3(256), stream, a);
                                return launch(fwd_rows_vec<T, W, 1, SILU, SEQ, MODE>, grid, dim3(256), stream, a);
                            };
                            if (aligned) return go(std::integral_constant<int, kRowsAligned>{});
                            if (alike) return go(std::integral_constant<int, kRowsAlike>{});
                            return go(std::integral_constant<int, kRowsAny>{});
                        });
                    }
                }
                constexpr int CPL = 4 / (int)sizeof(T);
                if (cl_ok<T, CPL>(p)) {
                    a.ngroups = ceil_div(p.dim, (int64_t)(64 * CPL));
                    // 8-step tiles when 16-step ones would give fewer than 4096
                    // wavefronts: a tile is one round trip to memory, so a small
                    // grid gains from twice the wavefronts (bf16, B = 1, D = 768,
                    // L = 2048: 4.3 instead of 5.1 us; C3 keeps 16: 24.1 against 24.9)
                    a.chunk = p.batch * a.ngroups * ceil_div(p.seqlen, (int64_t)kClTS) < 4096 ? kClTSSmall : kClTS;
                    a.nseg = ceil_div(p.seqlen, a.chunk);
                    a.n_items = p.batch * a.nseg * a.ngroups;
                    const dim3 grid((unsigned)ceil_div(a.n_items, 4));
                    return with_flag(p.seq_idx != nullptr, [&](auto qc) {
                        constexpr bool SEQ = decltype(qc)::value;
                        if (a.chunk == kClTSSmall)
                            return launch(fwd_cl<T, W, CPL, kClTSSmall, SILU, SEQ>, grid, dim3(256), stream, a);
                        return launch(fwd_cl<T, W, CPL, kClTS, SILU, SEQ>, grid, dim3(256), stream, a);
                    });
                }
                a.chunk = 64;
                a.nseg = ceil_div(p.seqlen, a.chunk);
                a.n_items = rows * a.nseg;
                const dim3 grid((unsigned)ceil_div(a.n_items, 256));
                return launch(fwd_generic<T, W, SILU>, grid, dim3(256), stream, a);
            });
        });
    });
}

}  // namespace cc1d
