// lg_narrow.h — what follows the attention tiles of a layer as ONE launch on ONE XCD, for one row of a narrow model (draft heads of
// 256 and small models of 512 values: decode steps and drafts).
//
// Such a layer is a chain of six to eight dependent launches of some dozen workgroups, each of them 3.5 to 4.5 us from its
// predecessor's end to its own, whatever it computes; its matrices (0.9 to 1.8 MB) are a microsecond's work for the 32 CUs of one
// XCD.  So one workgroup of 8 wavefronts per CU of one XCD (the workgroups i of the launch with i % 8 == 0, lg_xcd.h) requests all
// its weights of the layer up front, into registers, and the phases hand over through the XCD's L2 (0.4 us, and 0.4 for the data):
//   merge      workgroup h takes 64 dims: the wavefronts load the tiles' partials, one adds them in order, q8   (lg_k_attn_merge)
//   output     row group g of 8 rows on workgroup g % 32: attn_output . that               (lg_k_mm)
//   gate/up    every workgroup forms the residual row and its q8 by itself (2 KB of loads: less than another hand-over), then takes
//              the blocks of 32 FFN columns b % 32, a K segment per wavefront; GELU, q8     (lg_k_rows, lg_k_geglu_t)
//   down       row groups as above
//   gate, projection   (models with per-layer inputs) the same with the residual row again formed by everyone (lg_k_ple_tail)
//   q/k/v      of the NEXT layer, behind its row work; on the last layer the head's input instead
// Bound by latency: 2.8 us to the merged row (a read of what other XCDs have just written, behind it the CU's 0.1 MB of weights through
// its one memory path), 0.45 per hand-over, 0.4 to 1.7 of dependent instructions per phase.  Measured against the separate kernels: a
// step of 6 layers of 512 values at 100 positions 198 -> 140 us (54 launches -> 19), a draft of 4 blocks of 256 over 2048 positions
// 138 -> 100 us.  Sums, their order and every rounding are the separate kernels', lane for lane.  Tags carry the launch's number and the XCD id; a
// wait is bounded, and what goes wrong lands in StepCtl.err, as in lg_xtail.h.
#pragma once
#include "lg_xtail.h"

#define LG_NARROW_WGS 32            // one per CU of the XCD
#define LG_NARROW_E 512             // widest row
#define LG_NARROW_K 2048            // longest input of attn_output and ffn_down
#define LG_NARROW_TILES 128         // tiles of a round of the merge by a workgroup
#define LG_NARROW_ONE 32            // ... by one wavefront
#define LG_NARROW_LONG 256          // tiles up to which a round at a time is the faster form at every position (100 positions in a cache of 4096: 140 us, 142 in rounds of two)
// q8 rows as (4 values, tag) in the order of lg_act_layout and (scale, tag, sum, tag) a block; rows as (float, tag)
struct NarrowQ8 { uint2 w[LG_NARROW_K / 4]; uint4 s[LG_NARROW_K / 32]; };
struct NarrowSync { NarrowQ8 attn, act; uint2 o[LG_NARROW_E], d[LG_NARROW_E], pr[LG_NARROW_E], gf[256]; };
struct NarrowArgs {
    MergeArgs      g;               // (xq, xf are not used)
    const float   *x;               // [E] residual
    const uint8_t *wo, *wgu, *wdn, *winp, *wproj, *wq;          // segment tiles; wgu: row-block tiles; wq: the next layer's q/k/v, nullptr behind the last layer
    const float   *post_attn, *ffn_norm, *post_ffw, *post_norm, *w_pre, *os, *ipl;      // post_norm, ipl: with per-layer inputs; w_pre: next attn_norm or output_norm
    float         *x_out, *qkv, *h_out;       // [E]; [qm]; last layer: normed row
    int8_t        *hq;              // last layer: q8 of it
    int            E, qd, FF, qm, tiles;      // tiles: most that the row can see
    float          eps;
    NarrowSync    *sync;
    int            seq;             // number of this launch inside the step (the layer)
    int           *err, *err2;      // StepCtl.err of the model and (a draft head) of its target, or nullptr
    int            spin_limit;
};

// LONG: rows that can have more than LG_NARROW_LONG tiles, two rounds of them on their way at a time.  With the rounds of the other build, one after the
// other, rows of very many tiles were slower than with the separate merge (4 layers of 512 values, every row 100000 positions: 546 us a step, 373
// with these); one build for both cost a row of few tiles 0.25 us a launch.
template <bool PLE, bool LONG>
__global__ __launch_bounds__(512, 2) void lg_k_narrow(NarrowArgs a, const StepCtl *ctl) {
    if (blockIdx.x & (LG_XCDS - 1)) return;
    __shared__ __align__(16) float wts[LONG ? 2 : 1][LG_NARROW_TILES], pls[LONG ? 2 : 1][LG_NARROW_TILES];
    __shared__ float part[LONG ? 2 : 1][LG_NARROW_TILES][64], wmx[8], red[PLE ? 6 : 4][8], pcol[2][8][64];
    __shared__ __align__(16) int8_t lq[LG_NARROW_K * 5 / 4], lrow[LG_NARROW_E * 5 / 4], lnat[LG_NARROW_E * 5 / 4], lgate[256 * 5 / 4];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), c = lane & 7;
    const int u = blockIdx.x >> 3, E = a.E, nq = E >> 2, nitE = E >> 8, nitQ = a.qd >> 8, nitF = a.FF >> 8;
    const bool rowt = t < nq;                                  // threads of the row work: a float4 of the row each (lane order of lg_k_rows)
    const int ge = u + LG_NARROW_WGS * (7 - wave);             // this wavefront's row group of 8 in every matmul (wavefront 0 merges: it has one last)
    const bool eg = ge < (E >> 3), qg = a.wq && ge < (a.qm >> 3);
    const uint32_t tag = lg_tag(ctl->launch + (uint32_t)a.seq, lg_xcc_id());

    // every load that depends on nothing
    struct Tiles { uint4 q[8]; uint32_t s[8]; } to, td;        // output, down
    uint4 guq[2][2], inq[2], pjq, nqq[2]; uint32_t gus[2][2], ins[2], pjs, nqs[2];
    float4 xv = make_float4(0, 0, 0, 0), w1 = xv, w2 = xv, w3 = xv, w4 = xv, w5 = xv;
    float osv = 1.0f, iplv = 0.0f;
    auto request = [&]() {
        auto group = [&](Tiles &w, const uint8_t *m, int nit) {
            const uint8_t *b = m + (size_t)ge * nit * LG_TILE;
            #pragma unroll
            for (int i = 0; i < 8; ++i) { const int it = i < nit ? i : nit - 1; w.q[i] = lg_ldt16(b, it, lane); w.s[i] = lg_ldt2(b, it, lane); }
        };
        if (eg) group(to, a.wo, nitQ);
        if (rowt) {
            xv = ((const float4 *)a.x)[t]; w1 = ((const float4 *)a.post_attn)[t]; w2 = ((const float4 *)a.ffn_norm)[t];
            w3 = ((const float4 *)a.post_ffw)[t]; w5 = ((const float4 *)a.w_pre)[t];
            if (PLE) w4 = ((const float4 *)a.post_norm)[t];
        }
        if (a.os) osv = a.os[0];
        #pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int blk = u + LG_NARROW_WGS * b < (a.FF >> 5) ? u + LG_NARROW_WGS * b : (a.FF >> 5) - 1;
            const uint8_t *p = a.wgu + ((size_t)blk * (E >> 5) + wave * nitE) * LG_TILE;
            #pragma unroll
            for (int i = 0; i < 2; ++i) { const int it = i < nitE ? i : nitE - 1; guq[b][i] = lg_ldt16(p, it, lane); gus[b][i] = lg_ldt2(p, it, lane); }
        }
        if (eg) group(td, a.wdn, nitF);
        if (PLE) {
            if (wave == 0) {
                const uint8_t *p = a.winp + (size_t)u * nitE * LG_TILE;
                #pragma unroll
                for (int i = 0; i < 2; ++i) { const int it = i < nitE ? i : nitE - 1; inq[i] = lg_ldt16(p, it, lane); ins[i] = lg_ldt2(p, it, lane); }
                iplv = a.ipl[u * 8 + (lane >> 3)];
            }
            if (eg) { pjq = lg_ldt16(a.wproj + (size_t)ge * LG_TILE, 0, lane); pjs = lg_ldt2(a.wproj + (size_t)ge * LG_TILE, 0, lane); }
        }
        if (qg) {
            const uint8_t *p = a.wq + (size_t)ge * nitE * LG_TILE;
            #pragma unroll
            for (int i = 0; i < 2; ++i) { const int it = i < nitE ? i : nitE - 1; nqq[i] = lg_ldt16(p, it, lane); nqs[i] = lg_ldt2(p, it, lane); }
        }
    };
    NarrowSync &y = *a.sync;
    int err = 0;
    auto put = [&](uint2 *p, float v) { lg_put(p, v, tag); };
    // q8 of k values into LDS: two words by each thread of wavefronts 0..3, a block's scale by a lane of wavefront 4
    auto take_q8 = [&](const NarrowQ8 &q, int k) {
        const int nw = k >> 3, ns = k >> 5;                    // 16-byte units of words (at most 256), of scales (at most 64)
        if (wave < 4) {
            const bool on = t < nw;
            const LgUnits<1> r = lg_take<1>([&](int) { return (const uint4 *)q.w + (on ? t : 0); }, on, tag, a.spin_limit, err);
            if (on) *(uint2 *)(lq + 8 * t) = make_uint2(r.v[0].x, r.v[0].z);
        } else if (wave == 4) {
            const bool on = lane < ns;
            const LgUnits<1> r = lg_take<1>([&](int) { return q.s + (on ? lane : 0); }, on, tag, a.spin_limit, err);
            if (on) ((uint2 *)(lq + k))[lane] = make_uint2(r.v[0].x, r.v[0].z);
        }
        __syncthreads();
    };
    auto put_q8 = [&](NarrowQ8 &q, int k, int e, int v, float d, int sum) {      // element e of a row, by 32 adjacent lanes a block
        const ActLayout lay = lg_act_layout(k);
        const uint32_t w = (uint32_t)(lg_dpp_i<0x00>(v) & 255) | (uint32_t)(lg_dpp_i<0x55>(v) & 255) << 8 | (uint32_t)(lg_dpp_i<0xAA>(v) & 255) << 16 | (uint32_t)lg_dpp_i<0xFF>(v) << 24;
        if ((e & 3) == 0) q.w[lg_act_unit(lay, e >> 4) * 4 + ((e >> 2) & 3)] = make_uint2(w, tag);
        if ((e & 31) == 0) q.s[lg_act_block(lay, e >> 5)] = make_uint4(__float_as_uint(d), tag, (uint32_t)sum, tag);
    };
    auto dot_tile = [&](const int8_t *act, int k, int i, uint4 w, uint32_t s, float p) {       // tile i of a group against a row in LDS (lg_act_layout)
        const float2 ds = ((const float2 *)(act + k))[i * 8 + c];
        const int8_t *au = act + (i * 16 + c) * 16;
        const int dot = lg_block_dot(w, *(const int4 *)au, *(const int4 *)(au + 128), __float_as_int(ds.y));
        return lg_fmaf(ds.x * lg_h2f((uint16_t)s), (float)dot, p);
    };
    auto group_sum = [&](const Tiles &w, const int8_t *act, int k, int nit) {
        float p = 0.0f;
        #pragma unroll
        for (int i = 0; i < 8; ++i) if (i < nit) p = dot_tile(act, k, i, w.q[i], w.s[i], p);
        return lg_sum8(p);
    };
    // x += rmsnorm(d) * w (* os), every workgroup for itself
    auto add_norm = [&](const uint2 *d, float4 w, bool scale, float *r) {
        float4 v = make_float4(0, 0, 0, 0);
        if (rowt) {
            const LgUnits<2> q = lg_take<2>([&](int i) { return (const uint4 *)(d + 4 * t) + i; }, true, tag, a.spin_limit, err);
            v = lg_units_float4(q.v[0], q.v[1]);
        }
        const float ss = lg_block_sum256_of512(rowt ? lg_sumsq4(v, 0.0f) : 0.0f, r), sc = 1.0f / sqrtf(ss / (float)E + a.eps);
        xv.x = xv.x + v.x * sc * w.x; xv.y = xv.y + v.y * sc * w.y; xv.z = xv.z + v.z * sc * w.z; xv.w = xv.w + v.w * sc * w.w;
        if (scale) { xv.x = xv.x * osv; xv.y = xv.y * osv; xv.z = xv.z * osv; xv.w = xv.w * osv; }
    };
    auto norm = [&](float4 w, float *r) {
        const float ss = lg_block_sum256_of512(rowt ? lg_sumsq4(xv, 0.0f) : 0.0f, r), sc = 1.0f / sqrtf(ss / (float)E + a.eps);
        return make_float4(xv.x * sc * w.x, xv.y * sc * w.y, xv.z * sc * w.z, xv.w * sc * w.w);
    };
    auto quant_row = [&](float4 h, int8_t *q) {                // q8 of a row in the order of lg_act_layout
        float d; int sum;
        const uint32_t packed = lg_quant4_8lanes(h, &d, &sum);
        *(uint32_t *)(q + lg_q8_off<1>(E, 0, t >> 2, (t & 3) * 4)) = packed;
        if ((t & 7) == 0) lg_q8_ds<1>(q, E)[lg_q8_ds_idx<1>(E, 0, t >> 3)] = make_float2(d, __int_as_float(sum));
    };

    // ---- merge: this workgroup's 64 dims of a head.  The row's tiles are slots 0..hi of the partials: what is loaded first depends on nothing ----
    if (u * 64 < a.qd) {
        const int hd = a.g.hd, head = u * 64 / hd;
        const size_t base = (size_t)head * a.g.tiles_max;
        const float *acc = a.g.pacc + base * hd + (u * 64 - head * hd) + lane, *pm = a.g.pm + base, *pl = a.g.pl + base;
        float L = 0.0f, o = 0.0f;
        if constexpr (LONG) {
            // Rounds of 128 tiles, two of them on their way: the wavefronts request 16 each, wavefront 0 adds the values of a round from LDS and
            // wavefront 1 the sums of its weights (the same two chains of fma in tile order).
            float pv[2][LG_NARROW_TILES / 8], pmn[2], pln[2];
            auto fetch = [&](auto k_, int c0) {
                constexpr int k = decltype(k_)::value;
                #pragma unroll
                for (int i = 0; i < LG_NARROW_TILES / 8; ++i) { const int n = c0 + wave + 8 * i; pv[k][i] = acc[(size_t)(n < a.tiles ? n : a.tiles - 1) * hd]; }
                if (c0 && t < LG_NARROW_TILES) { const int n = c0 + t < a.tiles ? c0 + t : a.tiles - 1; pmn[k] = pm[n]; pln[k] = pl[n]; }
            };
            constexpr std::integral_constant<int, 0> K0{}; constexpr std::integral_constant<int, 1> K1{};
            const int mine = t < a.tiles ? t : a.tiles - 1;
            pmn[0] = pm[mine]; pln[0] = pl[mine];
            const int pos = ctl->pos + a.g.pos_off;
            fetch(K0, 0);
            __builtin_amdgcn_sched_barrier(0);
            request();
            const int hi = (pos >> 5) - (lg_win_start(pos, a.g.window) >> 5);
            if (hi >= LG_NARROW_TILES) fetch(K1, LG_NARROW_TILES);
            float mx = t <= hi ? pmn[0] : -INFINITY;
            for (int n = t + 512; n <= hi; n += 4 * 512) {
                float m4[4];
                #pragma unroll
                for (int i = 0; i < 4; ++i) m4[i] = pm[n + 512 * i <= hi ? n + 512 * i : n];
                mx = fmaxf(fmaxf(fmaxf(mx, m4[0]), fmaxf(m4[1], m4[2])), m4[3]);
            }
            mx = lg_max_n(mx, 64);
            if (lane == 0) wmx[wave] = mx;
            __syncthreads();
            mx = fmaxf(fmaxf(fmaxf(wmx[0], wmx[1]), fmaxf(wmx[2], wmx[3])), fmaxf(fmaxf(wmx[4], wmx[5]), fmaxf(wmx[6], wmx[7])));
            // sum += src[tile] * weight[tile], tiles 0..cn-1 in order; the next eight tiles' reads ahead of the fma of the present ones
            auto chain = [&](const float *src, auto stride, const float *w, int cn, float &sum) {
                constexpr int ST = decltype(stride)::value;
                float p8[2][8], w8[2][8];
                auto read = [&](int k, int n0_) {
                    const int n0 = n0_ < LG_NARROW_TILES ? n0_ : LG_NARROW_TILES - 8;
                    #pragma unroll
                    for (int i = 0; i < 8; ++i) { p8[k][i] = src[(n0 + i) * ST]; w8[k][i] = w[n0 + i]; }
                };
                auto add = [&](int k, int n0) {
                    if (n0 + 8 <= cn) {
                        #pragma unroll
                        for (int i = 0; i < 8; ++i) sum = lg_fmaf(p8[k][i], w8[k][i], sum);
                    } else {
                        #pragma unroll
                        for (int i = 0; i < 8; ++i) if (n0 + i < cn) sum = lg_fmaf(p8[k][i], w8[k][i], sum);
                    }
                };
                read(0, 0);
                for (int n0 = 0; n0 < cn; n0 += 16) { read(1, n0 + 8); add(0, n0); read(0, n0 + 16); add(1, n0 + 8); }
            };
            auto round = [&](auto k_, int c0) {                // (a round's place in LDS is written again behind the other round's barrier)
                constexpr int k = decltype(k_)::value;
                #pragma unroll
                for (int i = 0; i < LG_NARROW_TILES / 8; ++i) part[k][wave + 8 * i][lane] = pv[k][i];
                if (t < LG_NARROW_TILES && c0 + t <= hi) { wts[k][t] = lg_expf(pmn[k] - mx); pls[k][t] = pln[k]; }
                __syncthreads();
                if (c0 + 2 * LG_NARROW_TILES <= hi) fetch(k_, c0 + 2 * LG_NARROW_TILES);
                const int cn = hi - c0 + 1 < LG_NARROW_TILES ? hi - c0 + 1 : LG_NARROW_TILES;
                if (wave == 0) chain(&part[k][0][lane], std::integral_constant<int, 64>{}, wts[k], cn, o);
                else if (wave == 1) chain(pls[k], std::integral_constant<int, 1>{}, wts[k], cn, L);
            };
            for (int c0 = 0; c0 <= hi; c0 += 2 * LG_NARROW_TILES) {
                round(K0, c0);
                if (c0 + LG_NARROW_TILES <= hi) round(K1, c0 + LG_NARROW_TILES);
            }
            if (wave == 1 && lane == 0) wmx[0] = L;            // (every wavefront has read the maxima before the first round's barrier)
            __syncthreads();
            L = wmx[0];
        } else if (a.tiles <= LG_NARROW_ONE) {                        // (a sliding window of 512, say)
            // one wavefront by itself, while the others request: they are a microsecond at it, and a merge that all of them take part
            // in ends behind that (3.5 us into the launch, one wavefront's 2.8)
            if (wave == 0) {
                const int mine = lane < a.tiles ? lane : a.tiles - 1;
                const float pm1 = pm[mine], pl1 = pl[mine];
                float pv[LG_NARROW_ONE];
                #pragma unroll
                for (int n = 0; n < LG_NARROW_ONE; ++n) pv[n] = acc[(size_t)(n < a.tiles ? n : a.tiles - 1) * hd];
                const int pos = ctl->pos + a.g.pos_off, hi = (pos >> 5) - (lg_win_start(pos, a.g.window) >> 5);
                __builtin_amdgcn_sched_barrier(0);
                const float mx = lg_max_n(lane <= hi ? pm1 : -INFINITY, 64), w1 = lg_expf(pm1 - mx);
                #pragma unroll
                for (int n = 0; n < LG_NARROW_ONE; ++n)
                    if (n <= hi) {                             // in tile order
                        const float wn = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w1), n)), ln = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(pl1), n));
                        L = lg_fmaf(ln, wn, L); o = lg_fmaf(pv[n], wn, o);
                    }
            }
        } else {
            float pv[LG_NARROW_TILES / 8];
            auto fetch = [&](int c0) {
                #pragma unroll
                for (int i = 0; i < LG_NARROW_TILES / 8; ++i) { const int n = c0 + wave + 8 * i; pv[i] = acc[(size_t)(n < a.tiles ? n : a.tiles - 1) * hd]; }
            };
            const int mine = t < a.tiles ? t : a.tiles - 1;
            const float pm1 = pm[mine], pl1 = pl[mine];
            const int pos = ctl->pos + a.g.pos_off;
            fetch(0);
            __builtin_amdgcn_sched_barrier(0);
            request();
            const int hi = (pos >> 5) - (lg_win_start(pos, a.g.window) >> 5);
            float mx = t <= hi ? pm1 : -INFINITY;
            for (int n = t + 512; n <= hi; n += 512) mx = fmaxf(mx, pm[n]);
            mx = lg_max_n(mx, 64);
            if (lane == 0) wmx[wave] = mx;
            __syncthreads();
            mx = fmaxf(fmaxf(fmaxf(wmx[0], wmx[1]), fmaxf(wmx[2], wmx[3])), fmaxf(fmaxf(wmx[4], wmx[5]), fmaxf(wmx[6], wmx[7])));
            for (int c0 = 0; c0 <= hi; c0 += LG_NARROW_TILES) {
                #pragma unroll
                for (int i = 0; i < LG_NARROW_TILES / 8; ++i) part[0][wave + 8 * i][lane] = pv[i];
                if (t < LG_NARROW_TILES && c0 + t <= hi) { wts[0][t] = lg_expf((c0 ? pm[c0 + t] : pm1) - mx); pls[0][t] = c0 ? pl[c0 + t] : pl1; }
                __syncthreads();
                if (c0 + LG_NARROW_TILES <= hi) fetch(c0 + LG_NARROW_TILES);
                if (wave == 0) {
                    const int cn = hi - c0 + 1 < LG_NARROW_TILES ? hi - c0 + 1 : LG_NARROW_TILES;
                    for (int n0 = 0; n0 < cn; n0 += 8) {          // in tile order; eight tiles' reads ahead of their fma
                        float p8[8], w8[8], l8[8];
                        #pragma unroll
                        for (int i = 0; i < 8; ++i) { p8[i] = part[0][n0 + i][lane]; w8[i] = wts[0][n0 + i]; l8[i] = pls[0][n0 + i]; }
                        #pragma unroll
                        for (int i = 0; i < 8; ++i) if (n0 + i < cn) { L = lg_fmaf(l8[i], w8[i], L); o = lg_fmaf(p8[i], w8[i], o); }
                    }
                }
                if (c0 + LG_NARROW_TILES <= hi) __syncthreads();
            }
        }
        if (wave == 0) {
            float d; int sum;
            const int q = lg_quant1_32lanes(o / L, &d, &sum);
            put_q8(y.attn, a.qd, u * 64 + lane, q, d, sum);
        }
        if (!LONG && a.tiles <= LG_NARROW_ONE) request();
    } else request();
    // ---- attention output ----
    take_q8(y.attn, a.qd);
    if (eg) { const float p = group_sum(to, lq, a.qd, nitQ); if (c == 0) put(y.o + ge * 8 + (lane >> 3), p); }
    // ---- gate/up: the row in natural order, a block's 32 values by every lane of a wavefront ----
    add_norm(y.o, w1, false, red[0]);
    {
        const float4 h = norm(w2, red[1]);
        if (rowt) {
            float d; int sum;
            const uint32_t packed = lg_quant4_8lanes(h, &d, &sum);
            *(uint32_t *)(lnat + 4 * t) = packed;
            if ((t & 7) == 0) ((float2 *)(lnat + E))[t >> 3] = make_float2(d, __int_as_float(sum));
        }
    }
    __syncthreads();
    #pragma unroll
    for (int b = 0; b < 2; ++b) {
        float p = 0.0f;
        #pragma unroll
        for (int i = 0; i < 2; ++i) if (i < nitE) {
            const int kb = wave * nitE + i;
            const float2 ds = ((const float2 *)(lnat + E))[kb];
            const int dot = lg_block_dot(guq[b][i], *(const int4 *)(lnat + kb * 32), *(const int4 *)(lnat + kb * 32 + 16), __float_as_int(ds.y));
            p = lg_fmaf(ds.x * lg_h2f((uint16_t)gus[b][i]), (float)dot, p);
        }
        pcol[b][wave][lane] = p;
    }
    __syncthreads();
    if (t < 64) {                                              // half a wavefront per block, a column per lane
        const int b = t >> 5, i = t & 31, blk = u + LG_NARROW_WGS * b;
        float g[8], v[8];
        #pragma unroll
        for (int s = 0; s < 8; ++s) { g[s] = pcol[b][s][i]; v[s] = pcol[b][s][32 + i]; }
        const float gate = ((g[0] + g[1]) + (g[2] + g[3])) + ((g[4] + g[5]) + (g[6] + g[7]));
        const float up = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        float d; int sum;
        const int q = lg_quant1_32lanes(lg_gelu_d(gate) * up, &d, &sum);
        if (blk < (a.FF >> 5)) put_q8(y.act, a.FF, blk * 32 + i, q, d, sum);
    }
    // ---- down ----
    take_q8(y.act, a.FF);
    if (eg) { const float p = group_sum(td, lq, a.FF, nitF); if (c == 0) put(y.d + ge * 8 + (lane >> 3), p); }
    add_norm(y.d, w3, !PLE, red[2]);
    if constexpr (PLE) {
        // ---- per-layer gate: 8 rows of 256 on the first wavefront; then the projection ----
        if (rowt) quant_row(xv, lrow);
        __syncthreads();
        if (wave == 0) {
            float p = 0.0f;
            #pragma unroll
            for (int i = 0; i < 2; ++i) if (i < nitE) p = dot_tile(lrow, E, i, inq[i], ins[i], p);
            p = lg_sum8(p);
            if (c == 0) put(y.gf + u * 8 + (lane >> 3), lg_gelu_d(p) * iplv);
        }
        lg_take_gated<1>(y.gf, lgate, t, 512, tag, a.spin_limit, err);
        __syncthreads();
        if (eg) { const float p = lg_sum8(dot_tile(lgate, 256, 0, pjq, pjs, 0.0f)); if (c == 0) put(y.pr + ge * 8 + (lane >> 3), p); }
        add_norm(y.pr, w4, true, red[4]);
    }
    // ---- the row work ahead of the next layer's q/k/v (or of the head), and that matmul ----
    const float4 h = norm(w5, red[3]);
    if (u == 0 && rowt) {
        ((float4 *)a.x_out)[t] = xv;
        if (a.h_out) ((float4 *)a.h_out)[t] = h;
        if (!a.wq) quant_row(h, a.hq);
    }
    if (a.wq) {
        if (PLE) __syncthreads();                              // (the gate has read lrow)
        if (rowt) quant_row(h, lrow);
        __syncthreads();
        if (qg) {
            float p = 0.0f;
            #pragma unroll
            for (int i = 0; i < 2; ++i) if (i < nitE) p = dot_tile(lrow, E, i, nqq[i], nqs[i], p);
            p = lg_sum8(p);
            if (c == 0) a.qkv[ge * 8 + (lane >> 3)] = p;
        }
    }
    if (err) { atomicOr(a.err, err); if (a.err2) atomicOr(a.err2, err); }
}
