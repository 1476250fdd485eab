// lg_aout.h — attention merge, output projection and the row work ahead of gate/up as ONE launch on ONE XCD (blocks of 1..3 rows).
//
// As separate launches these are three dependent steps of 8 to 320 workgroups, 4 us each from the predecessor's end, for 3 MB of weights.
// The 32 CUs of one XCD pull those in 2 to 3 us, and hand over among themselves for less than a launch (lg_xcd.h).  Unit u of the 32:
//   merge       64 dims of each row, a wavefront a row: what it loads comes first, the tiles' partials in registers   (lg_k_attn_merge)
//   hand-over   the q8 of the rows, tagged (lg_take), to every unit's LDS: by the merging wavefronts
//   projection  ten row groups of 8, a wavefront each, their weights in registers since the partials were requested   (lg_k_mm)
//   hand-over   the f32 rows, tagged, to the first rows x E/1024 units, which do the row work of lg_k_rows
// Sums, their order and every rounding are the separate kernels', lane for lane.
// Bound by the CU's one memory path: by the stamps of one row the q8 leaves at 2.1 us and is in every LDS at 3.6, when the 92 KB of
// weights are through as well; rows at 5.6, end at 6.7.  E4B shape, the 35 sliding layers of 42: a step of one row 1776 -> 1703 us,
// two 1880 -> 1829, three 1972 -> 1962; four 2070 -> 2080, five 2160 -> 2196, eight 2302 -> 2575 (the projection on v_dot4 by an eighth of the
// chip: those keep the separate kernels).  With 4096 inputs, 276 KB a CU at rows of 3840, one row lost as well: 12B shape 2481 -> 2728.
// Weights requested ahead of the partials: 1741 us.  Partials first, but the hand-over taken by the wavefronts that hold weights: 1712.
#pragma once
#include "lg_narrow.h"

#define LG_AOUT_TILES 40            // most tiles of a row: a wavefront holds them in registers
#define LG_AOUT_BATCH 20            // ... the first so many requested at once, the others where there are more
#define LG_AOUT_K 2048              // input of attn_output (8 tiles of a row group)
#define LG_AOUT_E 2560              // widest row
#define LG_AOUT_G (LG_AOUT_E / 8 / LG_XCD_WGS)     // row groups of a unit, a wavefront each
#define LG_AOUT_ROWS 3              // widest block
struct AttnOutSync { uint32_t gen, pad[31]; uint2 w[LG_AOUT_ROWS * LG_AOUT_K / 4]; uint4 s[LG_AOUT_ROWS * LG_AOUT_K / 32]; uint2 o[LG_AOUT_ROWS * LG_AOUT_E]; };
struct AttnOutArgs {
    MergeArgs      g;               // (xq, xf are not used)
    const uint8_t *wo;              // segment tiles
    const float   *x, *w_post, *w_pre;
    float         *x_out;
    int8_t        *q;
    int            E, tiles;        // tiles: most that a row can see
    float          eps;
    AttnOutSync   *sync;
    int            spin_limit;
    unsigned long long *stamps;
};
#define LG_AOUT_FIELDS(X, v) X(const float *, pm, g.pm, v) X(const float *, pl, g.pl, v) X(const float *, pacc, g.pacc, v) X(int, tiles_max, g.tiles_max, v) \
    X(int, H, g.H, v) X(int, hd, g.hd, v) X(int, window, g.window, v) X(int, tiles, tiles, v) X(const uint8_t *, wo, wo, v) X(AttnOutSync *, sync, sync, v) X(int, E, E, v) \
    X(const float *, x, x, v) X(const float *, w_post, w_post, v) X(const float *, w_pre, w_pre, v) \
    X(float *, x_out, x_out, v) X(int8_t *, q, q, v) X(float, eps, eps, v) X(int, spin_limit, spin_limit, v) \
    X(unsigned long long *, stamps, stamps, v)

// M: rows.  The first M wavefronts of a unit take a merge (row, 64 dims) each, the other ten a row group of 8
template <int M>
__global__ __launch_bounds__(64 * (LG_AOUT_G + M)) void lg_k_attn_out(StepCtl *ctl, LG_AOUT_FIELDS(LG_XP, _) int p_end_) {
    constexpr int qd = LG_AOUT_K, NIT = qd >> 8, W = LG_AOUT_G + M, NV = (LG_AOUT_E + 1023) / 1024;
    static_assert(qd == 64 * LG_XCD_WGS, "a merge of every row per unit");
    if (blockIdx.x & (LG_XCDS - 1)) return;
    AttnOutArgs a; LG_AOUT_FIELDS(LG_XI, a)
    __shared__ __align__(16) int8_t lq[M * qd * 5 / 4];        // [M][qd] int8, then [M][qd / 32] {scale, sum}: order of lg_act_layout
    __shared__ float red[2][W];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), c = lane & 7;
    const int u = blockIdx.x >> 3, E = a.E, nq = E >> 2, slices = (E + 1023) >> 10;
    auto stamp = [&](int i) { if (a.stamps && lane == 0 && wave == 0) a.stamps[(size_t)u * 8 + i] = wall_clock64(); };
    stamp(0);
    const uint32_t gen = a.sync->gen;
    const uint32_t tag = lg_tag(gen, lg_xcc_id());
    AttnOutSync &y = *a.sync;
    int err = 0;
    const int ge = (wave - M) * LG_XCD_WGS + u;                // this wavefront's row group
    const bool eg = wave >= M && ge < (E >> 3);
    const int jr = u % M, vr = u / M;                          // the row unit's row and its float4s (row units: u < M * slices)
    const bool rowt = u < M * slices && t < LG_WG;
    uint4 wq[NIT]; uint32_t ws[NIT];
    float4 xv[NV], w1[NV], w2[NV];
    auto request_row = [&]() {
        if (rowt) {
            #pragma unroll
            for (int v = 0; v < NV; ++v) if (t + 256 * v < nq) {
                xv[v] = ((const float4 *)(a.x + (size_t)jr * E))[t + 256 * v]; w1[v] = ((const float4 *)a.w_post)[t + 256 * v]; w2[v] = ((const float4 *)a.w_pre)[t + 256 * v];
            }
        }
    };
    // The partials are requested ahead of the CU's 92 KB of weights, which its one memory path takes 2 us for: behind them they arrive a
    // microsecond later.  (A wavefront meets the barrier in one branch or in the other.)
    if (wave < M) {
        // ---- merge: 64 dims of a (row, head) ----
        const int hd = a.g.hd, j = wave, head = u * 64 / hd;
        const size_t base = ((size_t)j * a.g.H + head) * a.g.tiles_max;
        const float *acc = a.g.pacc + base * hd + (u * 64 - head * hd) + lane;
        const int mine = lane < a.tiles ? lane : a.tiles - 1;
        const float pm1 = a.g.pm[base + mine], pl1 = a.g.pl[base + mine];
        float pv[LG_AOUT_TILES];
        #pragma unroll
        for (int n = 0; n < LG_AOUT_BATCH; ++n) pv[n] = acc[(size_t)(n < a.tiles ? n : a.tiles - 1) * hd];
        const bool more = a.tiles > LG_AOUT_BATCH;
        if (more) {
            #pragma unroll
            for (int n = LG_AOUT_BATCH; n < LG_AOUT_TILES; ++n) pv[n] = acc[(size_t)(n < a.tiles ? n : a.tiles - 1) * hd];
        }
        const int pos = ctl->pos, first = lg_win_start(pos, a.g.window) >> 5, lo = (lg_win_start(pos + j, a.g.window) >> 5) - first, hi = ((pos + j) >> 5) - first;
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const float mx = lg_max_n(lane >= lo && lane <= hi ? pm1 : -INFINITY, 64), wt = lg_expf(pm1 - mx);
        stamp(1);
        float L = 0.0f, o = 0.0f;
        auto add = [&](int n) {
            const float wn = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(wt), n)), ln = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(pl1), n));
            L = lg_fmaf(ln, wn, L); o = lg_fmaf(pv[n], wn, o);
        };
        auto add4 = [&](int n) {                               // in tile order
            if (n >= lo && n + 3 <= hi) { add(n); add(n + 1); add(n + 2); add(n + 3); }
            else {
                #pragma unroll
                for (int i = 0; i < 4; ++i) if (n + i >= lo && n + i <= hi) add(n + i);
            }
        };
        #pragma unroll
        for (int n = 0; n < LG_AOUT_BATCH; n += 4) add4(n);
        if (more) {
            #pragma unroll
            for (int n = LG_AOUT_BATCH; n < LG_AOUT_TILES; n += 4) add4(n);
        }
        float d; int sum;
        const int q = lg_quant1_32lanes(o / L, &d, &sum), e = u * 64 + lane;
        const ActLayout lay = lg_act_layout(qd);
        const uint32_t w = (uint32_t)(lg_dpp_i<0x00>(q) & 255) | (uint32_t)(lg_dpp_i<0x55>(q) & 255) << 8 | (uint32_t)(lg_dpp_i<0xAA>(q) & 255) << 16 | (uint32_t)lg_dpp_i<0xFF>(q) << 24;
        if ((e & 3) == 0) y.w[(j * qd >> 2) + lg_act_unit(lay, e >> 4) * 4 + ((e >> 2) & 3)] = make_uint2(w, tag);
        if ((e & 31) == 0) y.s[(j * qd >> 5) + lg_act_block(lay, e >> 5)] = make_uint4(__float_as_uint(d), tag, (uint32_t)sum, tag);
        stamp(2);
        // ---- hand-over: the whole row, to every unit.  (Loads return in order: a wavefront with weights on their way would wait for those first.) ----
        const LgUnits<5> r = lg_take<5>([&](int i) { return i < 4 ? (const uint4 *)y.w + j * (qd >> 3) + i * 64 + lane : y.s + j * (qd >> 5) + lane; }, true, tag, a.spin_limit, err);
        #pragma unroll
        for (int i = 0; i < 4; ++i) *(uint2 *)(lq + j * qd + 512 * i + 8 * lane) = make_uint2(r.v[i].x, r.v[i].z);
        lg_q8_ds<M>(lq, qd)[j * (qd >> 5) + lane] = make_float2(__uint_as_float(r.v[4].x), __uint_as_float(r.v[4].z));
    } else {
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (eg) {
            const uint8_t *b = a.wo + (size_t)ge * NIT * LG_TILE;
            #pragma unroll
            for (int i = 0; i < NIT; ++i) { wq[i] = lg_ldt16(b, i, lane); ws[i] = lg_ldt2(b, i, lane); }
        }
    }
    __syncthreads();
    stamp(3);
    request_row();
    // ---- this wavefront's row group of the projection ----
    if (eg) {
        float p[M];
        #pragma unroll
        for (int j = 0; j < M; ++j) p[j] = 0.0f;
        const float2 *ds = lg_q8_ds<M>((const int8_t *)lq, qd);
        #pragma unroll
        for (int i = 0; i < NIT; ++i) {
            float2 d[M]; int4 a0[M], a1[M];
            #pragma unroll
            for (int j = 0; j < M; ++j) {
                d[j] = ds[(j * qd >> 5) + i * 8 + c];
                const int8_t *au = lq + j * qd + (i * 16 + c) * 16;
                a0[j] = *(const int4 *)au; a1[j] = *(const int4 *)(au + 128);
            }
            #pragma unroll
            for (int j = 0; j < M; ++j) {
                const int dot = lg_block_dot(wq[i], a0[j], a1[j], __float_as_int(d[j].y));
                p[j] = lg_fmaf(d[j].x * lg_h2f((uint16_t)ws[i]), (float)dot, p[j]);
            }
        }
        #pragma unroll
        for (int j = 0; j < M; ++j) p[j] = lg_sum8(p[j]);
        if (c < M) lg_put(y.o + (size_t)c * E + ge * 8 + (lane >> 3), lg_pick<M>(p, c), tag);
    }
    stamp(4);
    if (err) atomicOr(&ctl->err, err);
    if (u >= M * slices) return;                               // this unit has no share of the row work
    // ---- hand-over: the projection's row; the row work, this unit storing and quantizing slice vr (lg_k_rows) ----
    float4 dv[LG_ROWV];
    err = 0;
    if (rowt) lg_take_row(dv, y.o + (size_t)jr * E, t, nq, tag, a.spin_limit, err);
    if (err) atomicOr(&ctl->err, err);
    stamp(5);
    float ss = 0.0f;
    if (rowt) {
        #pragma unroll
        for (int v = 0; v < NV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(dv[v], ss);
    }
    ss = lg_block_sum256_of512(ss, red[0]);
    float sc = 1.0f / sqrtf(ss / (float)E + a.eps);
    ss = 0.0f;
    if (rowt) {
        #pragma unroll
        for (int v = 0; v < NV; ++v) if (t + 256 * v < nq) {
            const float4 w = w1[v];
            float4 x = xv[v];
            x.x = x.x + dv[v].x * sc * w.x;  x.y = x.y + dv[v].y * sc * w.y;
            x.z = x.z + dv[v].z * sc * w.z;  x.w = x.w + dv[v].w * sc * w.w;
            xv[v] = x;
            if (v == vr) ((float4 *)(a.x_out + (size_t)jr * E))[t + 256 * v] = x;
            ss = lg_sumsq4(x, ss);
        }
    }
    ss = lg_block_sum256_of512(ss, red[1]);
    sc = 1.0f / sqrtf(ss / (float)E + a.eps);
    if (rowt) {
        #pragma unroll
        for (int v = 0; v < NV; ++v) {
            if (t + 256 * v >= nq || v != vr) continue;
            const float4 w = w2[v], h = make_float4(xv[v].x * sc * w.x, xv[v].y * sc * w.y, xv[v].z * sc * w.z, xv[v].w * sc * w.w);
            float d; int sum;
            const uint32_t packed = lg_quant4_8lanes(h, &d, &sum);
            const int quad = t + 256 * v;
            uint32_t *unit = (uint32_t *)a.q + (size_t)(quad >> 3) * 32;       // (order of lg_k_geglu_t)
            unit[jr * 8 + (quad & 7)] = packed;
            if ((t & 7) == 0) *(float2 *)(unit + 24 + 2 * jr) = make_float2(d, __int_as_float(sum));
        }
    }
    stamp(6);
    if (u == 0 && t == 0) a.sync->gen = gen + 1;
}
