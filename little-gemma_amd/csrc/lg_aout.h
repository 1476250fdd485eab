// lg_aout.h — attention merge, output projection and the row work ahead of gate/up as ONE launch on ONE XCD (sliding layers).
//
// As separate launches these are three dependent steps of 8 to 320 workgroups, 4 us each from the predecessor's end, for 3 MB of weights.
// The 32 CUs of one XCD pull those in 2 to 3 us, and hand over among themselves for less than a launch (lg_xcd.h).  Unit u of the 32:
//   merge       64 dims of each row, a wavefront a row (two from 5 rows on: with more wavefronts than twelve the registers no longer hold the projection): what it loads comes first, the tiles' partials in
//               registers   (lg_k_attn_merge)
//   hand-over   the q8 of the rows, tagged (lg_take), to every unit's LDS: by the merging wavefronts
//   projection  up to 2 rows, 3 of more than 20 tiles (lg_k_attn_out): ten row groups of 8 on v_dot4, a wavefront each   (lg_k_mm)
//               3 to 8 rows (lg_k_attn_out_m): up to three blocks of 32 rows on the matrix cores, a K segment to a wavefront   (lg_k_attn_tail)
//               either way with the weights in registers, requested right behind the partials
//   hand-over   the f32 rows, tagged, to the first rows x E/1024 units, which do the row work of lg_k_rows
// Sums, their order and every rounding are the separate kernels', lane for lane.
// Bound by the CU's one memory path up to the projection, then by LDS (v_dot4) or the vector units (matrix cores).  By the stamps the q8 of
// one row leaves at 1.9 us and is in every LDS at 3.4, when the 92 KB of weights are through as well; rows at 5.4, end at 6.4; five rows
// 3.0, 4.8, 7.9 (the projection 2.3) and 8.9.  E4B shape, the 35 sliding layers of 42, a step: one row 1784 -> 1694 us, two 1883 -> 1812,
// three 1978 -> 1923 (on v_dot4 1935), four 2061 -> 2007, five 2162 -> 2125, six 2210 -> 2162, eight 2304 -> 2276.
// The other 224 workgroups of the launch are gate/up and the GeGLU of the rows (lg_aout_geglu), which was a launch of its own behind this one.  By the stamps (two blocks
// of columns to a workgroup) one row is done at 7.4 us (1.1 of it beside 29 MB of weights on their way), in every LDS at 8.2, multiplied at 9.9 and stored at 10.5; five
// rows 9.8, 10.9, 13.3 and 13.8, where the two launches took 6.3 + 6.4 and 8.9 + 8.6.  Steps of the E4B shape (with the q/k/v projections in
// lg_k_ple_tail_s as well): one row 1765 -> 1618 us, five 2113 -> 1946, eight at 20011 2497 -> 2327, four with bf16 per-layer matrices 2546 -> 2385.
// With 32x32x32 products one row 1664, five 1983; with the rows' scales read from LDS for each product, 16 bytes of tags to 16 of values and
// divisions in the way of a unit to its place 1658, 1966; a first pass over nothing to have the instructions in the CU's cache made the second wait for it.
// v_dot4 at 4, 5, 8 rows: 2080, 2196, 2575 (every row group reads the rows from LDS again).  4096 inputs, 276 KB a CU at rows of 3840: a
// step of the 12B shape 2481 -> 2728.  Weights requested ahead of the partials: one row 1741.  Partials first, but the hand-over
// taken by the wavefronts that hold weights: 1712.  Five to eight rows with a wavefront per merge: the projection spills, 2202 at five.
#pragma once
#include "lg_narrow.h"

#define LG_AOUT_TILES 40            // most tiles of a row: a wavefront holds them in registers
#define LG_AOUT_BATCH 20            // ... the first so many requested at once, the others where there are more; the most of lg_k_attn_out_m
#define LG_AOUT_K 2048              // input of attn_output (8 tiles of a row group)
#define LG_AOUT_E 2560              // widest row
#define LG_AOUT_G (LG_AOUT_E / 8 / LG_XCD_WGS)     // row groups of a unit, a wavefront each
#define LG_AOUT_DOT_ROWS 3          // widest block on v_dot4
#define LG_AOUT_NV ((LG_AOUT_E + 1023) / 1024)     // float4 of a row per thread of 256
struct AttnOutSync { uint2 w[LG_HIP_MAX_ROWS_DEV * LG_AOUT_K / 4]; uint4 s[LG_HIP_MAX_ROWS_DEV * LG_AOUT_K / 32]; uint2 o[LG_HIP_MAX_ROWS_DEV * LG_AOUT_E]; };
#define LG_AOUT_M_LDS ((size_t)(LG_AOUT_K / 32) * LG_MU_DWORDS * 4 + 8 * ((LG_AOUT_E / 32 + LG_XCD_WGS - 1) / LG_XCD_WGS) * 8 * 32 * 4)
static_assert(LG_AOUT_K == 64 * LG_XCD_WGS, "a merge of every row per unit");
struct AttnOutArgs {
    MergeArgs      g;               // (xq, xf are not used)
    const uint8_t *wo;              // segment tiles; lg_k_attn_out_m: the chains of lg_k_attn_tail
    const float   *x, *w_post, *w_pre;
    float         *x_out;
    int8_t        *q;
    int            E, tiles;        // tiles: most that a row can see
    float          eps;
    AttnOutSync   *sync;
    int            seq;             // number of this launch inside the step (the layer)
    int            spin_limit;
    unsigned long long *stamps;
    const uint8_t *gw;              // gate/up of the rows is part of the launch (row-block tiles), or nullptr
    int            nff, gq_units;   // GegluArgs.n_ff, .gq_units
    int8_t        *gq;
    FarRows       *rows;            // the rows that it takes
};
#define LG_AOUT_FIELDS(X, v) X(const float *, pm, g.pm, v) X(const float *, pl, g.pl, v) X(const float *, pacc, g.pacc, v) X(int, tiles_max, g.tiles_max, v) \
    X(int, H, g.H, v) X(int, hd, g.hd, v) X(int, window, g.window, v) X(int, tiles, tiles, v) X(const uint8_t *, wo, wo, v) X(AttnOutSync *, sync, sync, v) X(int, seq, seq, v) X(int, E, E, v) \
    X(const float *, x, x, v) X(const float *, w_post, w_post, v) X(const float *, w_pre, w_pre, v) \
    X(float *, x_out, x_out, v) X(int8_t *, q, q, v) X(float, eps, eps, v) X(int, spin_limit, spin_limit, v) \
    X(unsigned long long *, stamps, stamps, v) X(const uint8_t *, gw, gw, v) X(int, nff, nff, v) X(int, gq_units, gq_units, v) X(int8_t *, gq, gq, v) X(FarRows *, rows, rows, v)

// Gate/up and GeGLU of the rows by the workgroups on the other seven XCDs, for every width: a workgroup's one or two blocks of 32 FFN columns are in its
// registers and LDS when the rows are there.  Wavefront (pair of K segments, gate or up): v_mfma_i32_16x16x64_i8 with a block of 32 K values of either segment in
// its K range, rows 0..7 of its operand with the first segment's values and zeros, rows 8..15 with zeros and the second's, so that a product has
// the dots of 16 weight rows with a block of either segment apart: half the matrix time of a 32x32x32 product, which has the dots of 32 weight rows with one block.
#define LG_AOUT_NIT (LG_AOUT_E / 256)
#define LG_AOUT_GU_WGS ((LG_XCDS - 1) * LG_XCD_WGS)
#define LG_AOUT_GU_LDS ((size_t)8 * LG_AOUT_NIT * (LG_FAR_BLK + LG_TILE) + LG_AOUT_NIT * LG_FAR_BLK + 2 * 8 * 8 * 64 * 4)
// The segments' sums of one or two blocks of 32 FFN columns -> their GeGLU as q8: half-wavefront per row, one FFN column per lane
template <int M>
__device__ __forceinline__ void lg_far_geglu_out(const float (*red)[8][8][64], bool two, int b0, int b1, int t, int8_t *gq, int gq_units, int nff) {
    for (int x = t >> 5; x < (two ? 2 * M : M); x += 16) {
        const int o = x >= M, j = x - (o ? M : 0), i = t & 31, b = o ? b1 : b0;
        float g[8], u[8];
        #pragma unroll
        for (int c = 0; c < 8; ++c) { g[c] = red[o][c][j][i]; u[c] = red[o][c][j][32 + i]; }
        const float gate = ((g[0] + g[1]) + (g[2] + g[3])) + ((g[4] + g[5]) + (g[6] + g[7])), up = ((u[0] + u[1]) + (u[2] + u[3])) + ((u[4] + u[5]) + (u[6] + u[7]));
        float d; int sum;
        const int v = lg_quant1_32lanes(lg_gelu_d(gate) * up, &d, &sum);
        if (gq_units == 2) {
            int8_t *blk = gq + (size_t)b * (LG_MU_DWORDS * 4);
            const int dw = i >> 2;
            blk[(j * 8 + ((dw & 1) | ((dw & 2) << 1) | ((dw & 4) >> 1))) * 4 + (i & 3)] = (int8_t)v;
            if (i == 0) *(float2 *)(blk + 256 + 8 * j) = make_float2(d, 12582912.0f + (float)(8 * sum));
        } else {
            const ActLayout lay = lg_act_layout(nff);
            gq[(size_t)j * nff + lg_act_unit(lay, b * 2 + (i >> 4)) * 16 + (i & 15)] = (int8_t)v;
            if (i == 0) lg_q8_ds<M>(gq, nff)[(size_t)j * (nff >> 5) + lg_act_block(lay, b)] = make_float2(d, __int_as_float(sum));
        }
    }
}
template <int N, typename F, int... X> __device__ __forceinline__ void lg_unroll_(F &&f, std::integer_sequence<int, X...>) { (f(std::integral_constant<int, X>{}), ...); }
template <int N, typename F> __device__ __forceinline__ void lg_unroll(F &&f) { lg_unroll_<N>(f, std::make_integer_sequence<int, N>{}); }
template <int M>
__device__ __forceinline__ void lg_aout_geglu(const AttnOutArgs &a, int rank, unsigned char *smem, uint32_t tag, StepCtl *ctl) {
    constexpr int NIT = LG_AOUT_NIT, BLK = LG_FAR_BLK, I = (M + 1) / 2;
    const int t = threadIdx.x, lane = t & 63, c16 = lane & 15, hf = (lane >> 4) & 1, sg = lane >> 5, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int E = a.E, nb = E >> 5, nit = nb >> 3, nblk = a.nff >> 5, b1 = rank + LG_AOUT_GU_WGS;
    if (rank >= nblk || wave >= 8) return;
    const bool two = b1 < nblk;
    const int seg = (wave >> 1) * 2 + sg, up = wave & 1;
    unsigned char *zero = smem + (size_t)8 * NIT * BLK, *tiles = zero + NIT * BLK + (size_t)wave * NIT * LG_TILE;      // (tiles: of the second block, this wavefront's)
    float (*red)[8][8][64] = (float (*)[8][8][64])(zero + (size_t)NIT * BLK + (size_t)8 * NIT * LG_TILE);             // [block][segment][row][gate 32, up 32]
    uint4 q[NIT]; uint32_t sc[NIT];
    // lane: a gate (or up) row of its segment's tile.  The 16-lane rows trade bytes: lane (row of 16, hf) then has nibble bytes 8 hf .. 8 hf + 7 of rows c16 and 16 + c16
    auto fetch = [&](int b) {
        const __amdgpu_buffer_rsrc_t rw = lg_buffer_rsrc(a.gw + (size_t)b * nb * LG_TILE);
        const int at = seg * nit * LG_TILE, row = up * 32 + (lane & 31);
        #pragma unroll
        for (int i = 0; i < NIT; ++i) {
            const int it = __builtin_amdgcn_readfirstlane(i < nit ? i : nit - 1) * LG_TILE;
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(rw, at + row * 16, it, 2);
            q[i] = make_uint4(v[0], v[1], v[2], v[3]);
            sc[i] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rw, at + 1024 + row * 2, it, 2);
        }
        #pragma unroll
        for (int i = 0; i < NIT; ++i) {
            const lg_v2u s0 = __builtin_amdgcn_permlane16_swap(q[i].x, q[i].z, false, false), s1 = __builtin_amdgcn_permlane16_swap(q[i].y, q[i].w, false, false);
            const lg_v2u sd = __builtin_amdgcn_permlane16_swap(sc[i], sc[i], false, false);
            q[i] = make_uint4(s0.x ^ 0x88888888u, s1.x ^ 0x88888888u, s0.y ^ 0x88888888u, s1.y ^ 0x88888888u);
            sc[i] = (sd.x & 0xFFFF) | sd.y << 16;
        }
    };
    if (two) {
        fetch(b1);
        #pragma unroll
        for (int i = 0; i < NIT; ++i) { *(uint4 *)(tiles + i * LG_TILE + lane * 16) = q[i]; if (!hf) *(uint32_t *)(tiles + i * LG_TILE + 1024 + (sg * 16 + c16) * 4) = sc[i]; }
    }
    for (int i = t; i < NIT * BLK / 16; i += 512) ((uint4 *)zero)[i] = make_uint4(0, 0, 0, 0);
    fetch(rank);
    lg_v4i w0[NIT], w1[NIT];
    #pragma unroll
    for (int i = 0; i < NIT; ++i) {
        w0[i] = lg_far_weights(q[i].x, q[i].y); w1[i] = lg_far_weights(q[i].z, q[i].w);
        asm volatile("" : "+v"(w0[i]), "+v"(w1[i]), "+v"(sc[i]));
    }
    int err = lg_wait_soon(a.rows, tag, a.spin_limit);
    err |= lg_take_far_segment<M, NIT>(a.rows, E, nit, wave, lane, smem + (size_t)wave * NIT * BLK, tag, a.spin_limit);
    if (err) atomicOr(&ctl->err, err);
    __syncthreads();
    const unsigned char *ls = smem + (size_t)seg * NIT * BLK, *la = ((lane >> 3) & 1) == sg ? ls + (lane & 7) * 32 + hf * 16 : zero;
    lg_v4i magic = { LG_FAR_MAGIC, LG_FAR_MAGIC, LG_FAR_MAGIC, LG_FAR_MAGIC };
    asm volatile("" : "+v"(magic));
    // lane i of a row of 16: the scales of block i of the row's segment and half; a product's are broadcast from there
    float xd[I];
    static_assert(NIT <= 16, "a block to a lane");
    #pragma unroll
    for (int r = 0; r < I; ++r) xd[r] = *(const float *)(ls + (c16 < NIT ? c16 : 0) * BLK + 256 + (4 * hf + r) * 4);
    float p[2][2][I];                                          // [block][16 columns][row 2i + hf]
    #pragma unroll
    for (int i = 0; i < 4 * I; ++i) p[i / (2 * I)][i / I % 2][i % I] = 0.0f;
    auto chains = [&](auto both, auto whole) {                 // one block, or two that share the reads of the rows
        constexpr bool TWO = decltype(both)::value;
        lg_unroll<NIT>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            const lg_v4i av = *(const lg_v4i *)(la + i * BLK);
            auto join = [&](const lg_v4i &d, float dw, float (&z)[I]) {
                #pragma unroll
                for (int r = 0; r < I; ++r) {
                    const float v = lg_fmaf(lg_row_bcast<i>(xd[r]) * dw, __int_as_float(d[r]) - LG_FAR_BIAS, z[r]);
                    z[r] = decltype(whole)::value || i < nit ? v : z[r];      // (no branch on a shorter segment's end)
                }
            };
            const lg_v4i d0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, w0[i], magic, 0, 0, 0), d1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, w1[i], magic, 0, 0, 0);
            if (TWO) {
                const uint4 w = *(const uint4 *)(tiles + i * LG_TILE + lane * 16);
                const uint32_t dw = *(const uint32_t *)(tiles + i * LG_TILE + 1024 + (sg * 16 + c16) * 4);
                const lg_v4i d2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, lg_far_weights(w.x, w.y), magic, 0, 0, 0), d3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, lg_far_weights(w.z, w.w), magic, 0, 0, 0);
                join(d2, lg_h2f((uint16_t)dw), p[1][0]); join(d3, lg_h2f((uint16_t)(dw >> 16)), p[1][1]);
            }
            join(d0, lg_h2f((uint16_t)sc[i]), p[0][0]); join(d1, lg_h2f((uint16_t)(sc[i] >> 16)), p[0][1]);
        });
        #pragma unroll
        for (int o = 0; o < (TWO ? 2 : 1); ++o)
            #pragma unroll
            for (int i = 0; i < I; ++i) { red[o][seg][2 * i + hf][up * 32 + c16] = p[o][0][i]; red[o][seg][2 * i + hf][up * 32 + 16 + c16] = p[o][1][i]; }
    };
    if (nit == NIT) { if (two) chains(std::true_type{}, std::true_type{}); else chains(std::false_type{}, std::true_type{}); }
    else            { if (two) chains(std::true_type{}, std::false_type{}); else chains(std::false_type{}, std::false_type{}); }
    __syncthreads();
    lg_far_geglu_out<M>(red, two, rank, b1, t, a.gq, a.gq_units, a.nff);
}

// One wavefront's merge of 64 dims (number u of the row's) of row j, lane = dim: at most T tiles
template <int T>
struct AoutMerge {
    float pm1, pl1, pv[T];
    __device__ __forceinline__ void request(const AttnOutArgs &a, int u, int j, int lane) {
        const int hd = a.g.hd, head = u * 64 / hd;
        const size_t base = ((size_t)j * a.g.H + head) * a.g.tiles_max;
        // (buffer loads, the tile's offset in a scalar register: as flat loads each takes a dozen instructions of address arithmetic)
        const __amdgpu_buffer_rsrc_t acc = lg_buffer_rsrc(a.g.pacc + base * hd + (u * 64 - head * hd));
        const int mine = lane < a.tiles ? lane : a.tiles - 1;
        pm1 = a.g.pm[base + mine]; pl1 = a.g.pl[base + mine];
        #pragma unroll
        for (int n = 0; n < LG_AOUT_BATCH; ++n) pv[n] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(acc, lane * 4, (n < a.tiles ? n : a.tiles - 1) * hd * 4, 0));
        if (T > LG_AOUT_BATCH && a.tiles > LG_AOUT_BATCH) {
            #pragma unroll
            for (int n = LG_AOUT_BATCH; n < T; ++n) pv[n] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(acc, lane * 4, (n < a.tiles ? n : a.tiles - 1) * hd * 4, 0));
        }
    }
};
// The merged values of rows j, j + 4, .. (N of them by one wavefront: their chains side by side)
template <int T, int N>
__device__ __forceinline__ void lg_aout_merge(const AoutMerge<T> (&m)[N], const AttnOutArgs &a, int pos, int j, int lane, float (&out)[N]) {
    const int first = lg_win_start(pos, a.g.window) >> 5;
    int lo[N], hi[N], lo_all = 0, hi_all = 64;
    float wt[N], L[N], o[N];
    #pragma unroll
    for (int r = 0; r < N; ++r) {
        lo[r] = (lg_win_start(pos + j + 4 * r, a.g.window) >> 5) - first; hi[r] = ((pos + j + 4 * r) >> 5) - first;
        lo_all = lo[r] > lo_all ? lo[r] : lo_all; hi_all = hi[r] < hi_all ? hi[r] : hi_all;
        const float mx = lg_max_n(lane >= lo[r] && lane <= hi[r] ? m[r].pm1 : -INFINITY, 64);
        wt[r] = lg_expf(m[r].pm1 - mx); L[r] = o[r] = 0.0f;
    }
    auto add = [&](int r, int n) {
        const float wn = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(wt[r]), n)), ln = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(m[r].pl1), n));
        L[r] = lg_fmaf(ln, wn, L[r]); o[r] = lg_fmaf(m[r].pv[n], wn, o[r]);
    };
    auto add4 = [&](int n) {                                   // in tile order
        if (n >= lo_all && n + 3 <= hi_all) {
            #pragma unroll
            for (int i = 0; i < 4; ++i)
                #pragma unroll
                for (int r = 0; r < N; ++r) add(r, n + i);
        } else {
            #pragma unroll
            for (int i = 0; i < 4; ++i)
                #pragma unroll
                for (int r = 0; r < N; ++r) if (n + i >= lo[r] && n + i <= hi[r]) add(r, n + i);
        }
    };
    #pragma unroll
    for (int n = 0; n < LG_AOUT_BATCH; n += 4) add4(n);
    if (T > LG_AOUT_BATCH && a.tiles > LG_AOUT_BATCH) {
        #pragma unroll
        for (int n = LG_AOUT_BATCH; n < T; n += 4) add4(n);
    }
    #pragma unroll
    for (int r = 0; r < N; ++r) out[r] = o[r] / L[r];
}
// four lanes' q8 values as a word
__device__ __forceinline__ uint32_t lg_aout_word(int q) {
    return (uint32_t)(lg_dpp_i<0x00>(q) & 255) | (uint32_t)(lg_dpp_i<0x55>(q) & 255) << 8 | (uint32_t)(lg_dpp_i<0xAA>(q) & 255) << 16 | (uint32_t)lg_dpp_i<0xFF>(q) << 24;
}
// 16-byte units of row j's q8 as they are handed over: four of words a lane, one of scales
__device__ __forceinline__ LgUnits<5> lg_aout_take(const AttnOutSync &y, int j, int lane, uint32_t tag, int spin_limit, int &err) {
    return lg_take<5>([&](int i) { return i < 4 ? (const uint4 *)y.w + j * (LG_AOUT_K >> 3) + i * 64 + lane : y.s + j * (LG_AOUT_K >> 5) + lane; }, true, tag, spin_limit, err);
}
// The row work ahead of gate/up (lg_k_rows) in a row unit: row j, this unit storing and quantizing the float4s t + 256 vr; every thread
// of the workgroup calls, those with rowt (the first 256) have the row
struct AoutRow {
    float4 x[LG_AOUT_NV], w1[LG_AOUT_NV], w2[LG_AOUT_NV];
    __device__ __forceinline__ void request(const AttnOutArgs &a, int j, int t) {
        const int nq = a.E >> 2;
        #pragma unroll
        for (int v = 0; v < LG_AOUT_NV; ++v) if (t + 256 * v < nq) {
            x[v] = ((const float4 *)(a.x + (size_t)j * a.E))[t + 256 * v]; w1[v] = ((const float4 *)a.w_post)[t + 256 * v]; w2[v] = ((const float4 *)a.w_pre)[t + 256 * v];
        }
    }
    template <bool MFMA>
    __device__ __forceinline__ void work(const AttnOutArgs &a, const float4 (&dv)[LG_ROWV], int j, int vr, bool rowt, int t, float *red0, float *red1, uint32_t tag) {
        const int E = a.E, nq = E >> 2;
        float ss = 0.0f;
        if (rowt) {
            #pragma unroll
            for (int v = 0; v < LG_AOUT_NV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(dv[v], ss);
        }
        ss = lg_block_sum256_of512(ss, red0);
        float sc = 1.0f / sqrtf(ss / (float)E + a.eps);
        ss = 0.0f;
        if (rowt) {
            #pragma unroll
            for (int v = 0; v < LG_AOUT_NV; ++v) if (t + 256 * v < nq) {
                const float4 w = w1[v];
                float4 r = x[v];
                r.x = r.x + dv[v].x * sc * w.x;  r.y = r.y + dv[v].y * sc * w.y;
                r.z = r.z + dv[v].z * sc * w.z;  r.w = r.w + dv[v].w * sc * w.w;
                x[v] = r;
                if (v == vr) ((float4 *)(a.x_out + (size_t)j * E))[t + 256 * v] = r;
                ss = lg_sumsq4(r, ss);
            }
        }
        ss = lg_block_sum256_of512(ss, red1);
        sc = 1.0f / sqrtf(ss / (float)E + a.eps);
        if (!rowt) return;
        #pragma unroll
        for (int v = 0; v < LG_AOUT_NV; ++v) {
            if (t + 256 * v >= nq || v != vr) continue;
            const float4 w = w2[v], h = make_float4(x[v].x * sc * w.x, x[v].y * sc * w.y, x[v].z * sc * w.z, x[v].w * sc * w.w);
            float d; int sum;
            const uint32_t packed = lg_quant4_8lanes(h, &d, &sum);
            const int quad = t + 256 * v, dw = quad & 7;
            if (a.gw) lg_put_far_q8(a.rows, E, j, quad, packed, d, lg_far_tag(tag));
            else if (MFMA) {                                   // (order of lg_k_geglu_m)
                uint32_t *blk = (uint32_t *)a.q + (size_t)(quad >> 3) * LG_MU_DWORDS;
                blk[j * 8 + ((dw & 1) | ((dw & 2) << 1) | ((dw & 4) >> 1))] = packed;
                if ((t & 7) == 0) *(float2 *)(blk + 64 + 2 * j) = make_float2(d, 12582912.0f + (float)(8 * sum));
            } else {                                           // (order of lg_k_geglu_t)
                uint32_t *unit = (uint32_t *)a.q + (size_t)(quad >> 3) * 32;
                unit[j * 8 + dw] = packed;
                if ((t & 7) == 0) *(float2 *)(unit + 24 + 2 * j) = make_float2(d, __int_as_float(sum));
            }
        }
    }
};

// M: rows.  The first M wavefronts of a unit take a merge each, the other ten a row group of 8
template <int M>
__global__ __launch_bounds__(64 * (LG_AOUT_G + M)) void lg_k_attn_out(StepCtl *ctl, LG_AOUT_FIELDS(LG_XP, _) int p_end_) {
    constexpr int qd = LG_AOUT_K, NIT = qd >> 8, W = LG_AOUT_G + M;
    AttnOutArgs a; LG_AOUT_FIELDS(LG_XI, a)
    extern __shared__ __align__(16) unsigned char smem[];
    if (blockIdx.x & (LG_XCDS - 1)) {
        if constexpr (M < LG_AOUT_DOT_ROWS)
            if (a.gw) lg_aout_geglu<M>(a, (blockIdx.x >> 3) * (LG_XCDS - 1) + (blockIdx.x & (LG_XCDS - 1)) - 1, smem, lg_tag(ctl->launch + (uint32_t)a.seq, 0), ctl);
        return;
    }
    int8_t *lq = (int8_t *)smem;                               // [M][qd] int8, then [M][qd / 32] {scale, sum}: order of lg_act_layout
    __shared__ float red[2][W];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), c = lane & 7;
    const int u = blockIdx.x >> 3, E = a.E, nq = E >> 2, slices = (E + 1023) >> 10;
    auto stamp = [&](int i) { if (a.stamps && t == 0) a.stamps[(size_t)u * 8 + i] = wall_clock64(); };
    stamp(0);
    const uint32_t tag = lg_tag(ctl->launch + (uint32_t)a.seq, lg_xcc_id());
    AttnOutSync &y = *a.sync;
    int err = 0;
    const int ge = (wave - M) * LG_XCD_WGS + u;                // this wavefront's row group
    const bool eg = wave >= M && ge < (E >> 3);
    const int jr = u % M, vr = u / M;                          // the row unit's row and its float4s (row units: u < M * slices)
    const bool rowt = u < M * slices && t < LG_WG;
    uint4 wq[NIT]; uint32_t ws[NIT];
    // The partials are requested ahead of the CU's 92 KB of weights, which its one memory path takes 2 us for: behind them they arrive a
    // microsecond later.  (A wavefront meets the barrier in one branch or in the other.)
    if (wave < M) {
        const int j = wave;
        AoutMerge<LG_AOUT_TILES> m[1];
        m[0].request(a, u, j, lane);
        const int pos = ctl->pos;
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        float v[1], d; int sum;
        lg_aout_merge(m, a, pos, j, lane, v);
        const int q = lg_quant1_32lanes(v[0], &d, &sum), e = u * 64 + lane;
        const ActLayout lay = lg_act_layout(qd);
        const uint32_t w = lg_aout_word(q);
        if ((e & 3) == 0) y.w[(j * qd >> 2) + lg_act_unit(lay, e >> 4) * 4 + ((e >> 2) & 3)] = make_uint2(w, tag);
        if ((e & 31) == 0) y.s[(j * qd >> 5) + lg_act_block(lay, e >> 5)] = make_uint4(__float_as_uint(d), tag, (uint32_t)sum, tag);
        stamp(1);
        // ---- hand-over: the whole row, to every unit.  (Loads return in order: a wavefront with weights on their way would wait for those first.) ----
        const LgUnits<5> r = lg_aout_take(y, j, lane, tag, a.spin_limit, err);
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
    stamp(2);
    AoutRow row;
    if (rowt) row.request(a, jr, t);
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
    stamp(3);
    if (err) atomicOr(&ctl->err, err);
    if (u >= M * slices) return;                               // this unit has no share of the row work
    // ---- hand-over: the projection's row; the row work ----
    float4 dv[LG_ROWV];
    err = 0;
    if (rowt) lg_take_row(dv, y.o + (size_t)jr * E, t, nq, tag, a.spin_limit, err);
    if (err) atomicOr(&ctl->err, err);
    if (a.gw && u == 0 && t == 0) lg_put_soon(a.rows, lg_far_tag(tag));
    stamp(4);
    row.work<false>(a, dv, jr, vr, rowt, t, red[0], red[1], tag);
    stamp(5);
}

// Blocks of 3..8 rows: wavefronts 0..3 of a unit merge rows w and w + 4, the other eight run a K segment each of the row blocks u, u + 32,
// u + 64 of 32 rows (a segment's activations are read once for the three: LDS would set the time otherwise)
template <int M>
__global__ __launch_bounds__(768) void lg_k_attn_out_m(StepCtl *ctl, LG_AOUT_FIELDS(LG_XP, _) int p_end_) {
    constexpr int nb = LG_AOUT_K >> 5, NIT = nb / 8, NP = NIT / 2, RB = (LG_AOUT_E / 32 + LG_XCD_WGS - 1) / LG_XCD_WGS, W = 12;
    AttnOutArgs a; LG_AOUT_FIELDS(LG_XI, a)
    extern __shared__ __align__(16) unsigned char smem[];
    if (blockIdx.x & (LG_XCDS - 1)) {
        if (a.gw) lg_aout_geglu<M>(a, (blockIdx.x >> 3) * (LG_XCDS - 1) + (blockIdx.x & (LG_XCDS - 1)) - 1, smem, lg_tag(ctl->launch + (uint32_t)a.seq, 0), ctl);
        return;
    }
    unsigned char *la = smem;                                  // the rows as blocks of lg_k_geglu_m; slots past the block's rows hold anything
    float (*sums)[RB][8][32] = (float (*)[RB][8][32])(smem + nb * LG_MU_DWORDS * 4);        // [segment][row block][row slot][row]
    __shared__ float red[2][W];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), n = lane & 31, h = lane >> 5;
    const int u = blockIdx.x >> 3, E = a.E, nq = E >> 2, nrb = E >> 5, slices = (E + 1023) >> 10;
    auto stamp = [&](int i) { if (a.stamps && t == 0) a.stamps[(size_t)u * 8 + i] = wall_clock64(); };
    stamp(0);
    const uint32_t tag = lg_tag(ctl->launch + (uint32_t)a.seq, lg_xcc_id());
    AttnOutSync &y = *a.sync;
    int err = 0;
    const int seg = wave - 4;
    const int jr = u % M, vr = u / M;
    const bool rowt = u < M * slices && t < LG_WG;
    lg_x4u wq[RB][NP]; uint32_t ws[RB][NP];
    if (wave < 4) {
        const int e = u * 64 + lane, b = e >> 5, dw = (e >> 2) & 7;
        auto merge = [&](auto two) {                           // rows wave and, of more than four, wave + 4
            constexpr int N = decltype(two)::value ? 2 : 1;
            AoutMerge<LG_AOUT_BATCH> m[N];
            #pragma unroll
            for (int r = 0; r < N; ++r) m[r].request(a, u, wave + 4 * r, lane);
            const int pos = ctl->pos;
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            float v[N], d[N]; int q[N], sum[N];
            lg_aout_merge(m, a, pos, wave, lane, v);
            #pragma unroll
            for (int r = 0; r < N; ++r) q[r] = lg_quant1_32lanes(v[r], &d[r], &sum[r]);
            #pragma unroll
            for (int r = 0; r < N; ++r) {
                const int j = wave + 4 * r;
                const uint32_t w = lg_aout_word(q[r]);
                if ((e & 3) == 0) y.w[j * (LG_AOUT_K >> 2) + b * 8 + ((dw & 1) | ((dw & 2) << 1) | ((dw & 4) >> 1))] = make_uint2(w, tag);
                if ((e & 31) == 0) y.s[j * nb + b] = make_uint4(__float_as_uint(d[r]), tag, __float_as_uint(12582912.0f + (float)(8 * sum[r])), tag);
            }
        };
        if (wave + 4 < M) merge(std::true_type{}); else if (wave < M) merge(std::false_type{});
        else __builtin_amdgcn_s_barrier();
        stamp(1);
        // ---- hand-over ----
        for (int j = wave; j < M; j += 4) {
            const LgUnits<5> r = lg_aout_take(y, j, lane, tag, a.spin_limit, err);
            #pragma unroll
            for (int i = 0; i < 4; ++i) *(uint2 *)(la + (i * 16 + (lane >> 2)) * (LG_MU_DWORDS * 4) + j * 32 + (lane & 3) * 8) = make_uint2(r.v[i].x, r.v[i].z);
            *(uint2 *)(la + lane * (LG_MU_DWORDS * 4) + 256 + j * 8) = make_uint2(r.v[4].x, r.v[4].z);
        }
    } else {
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        #pragma unroll
        for (int k = 0; k < RB; ++k) {
            const int rb = u + LG_XCD_WGS * k;
            if (rb < nrb) {
                const uint8_t *cb = a.wo + ((size_t)rb * 8 + seg) * (NIT * 576);
                #pragma unroll
                for (int jp = 0; jp < NP; ++jp) {
                    wq[k][jp] = __builtin_nontemporal_load((const lg_x4u *)(cb + (size_t)((jp * 2 + h) * 32 + n) * 16));
                    ws[k][jp] = __builtin_nontemporal_load((const uint32_t *)(cb + (size_t)NIT * 512 + (size_t)(jp * 32 + n) * 4));
                }
            }
        }
    }
    __syncthreads();
    stamp(2);
    AoutRow row;
    // ---- segment `seg` of the unit's row blocks ----
    if (wave >= 4) {
        lg_v16i magic;
        #pragma unroll
        for (int i = 0; i < 16; ++i) magic[i] = 0x4B400000;
        asm volatile("" : "+v"(magic));
        const int arow = n < 8 ? n : 7;
        float p[RB][4];
        #pragma unroll
        for (int k = 0; k < RB; ++k)
            #pragma unroll
            for (int i = 0; i < 4; ++i) p[k][i] = 0.0f;
        const unsigned char *ls = la + seg * NIT * (LG_MU_DWORDS * 4);
        XffnAct nx = lg_xffn_act(ls, arow, h);
        #pragma unroll
        for (int s = 0; s < NIT; ++s) {
            const XffnAct ac = nx;
            if (s + 1 < NIT) nx = lg_xffn_act(ls + (s + 1) * (LG_MU_DWORDS * 4), arow, h);
            #pragma unroll
            for (int k = 0; k < RB; ++k) {
                lg_v2u q; q.x = s & 1 ? wq[k][s >> 1].z : wq[k][s >> 1].x; q.y = s & 1 ? wq[k][s >> 1].w : wq[k][s >> 1].y;
                lg_xffn_step(ac.av, ac.xd, ac.cf, q, lg_h2f((uint16_t)(s & 1 ? ws[k][s >> 1] >> 16 : ws[k][s >> 1])), magic, p[k]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        #pragma unroll
        for (int k = 0; k < RB; ++k)
            #pragma unroll
            for (int i = 0; i < 4; ++i) sums[seg][k][4 * h + i][n] = p[k][i];
    } else if (rowt) row.request(a, jr, t);                    // (in the branch without the projection's registers)
    __syncthreads();
    for (int idx = t; idx < RB * M * 32; idx += 64 * W) {      // the adjacent-pair tree over the 8 segments
        const int k = idx / (M * 32), rem = idx - k * (M * 32), j = rem >> 5, i = rem & 31, rb = u + LG_XCD_WGS * k;
        if (rb < nrb)
            lg_put(y.o + (size_t)j * E + rb * 32 + i, ((sums[0][k][j][i] + sums[1][k][j][i]) + (sums[2][k][j][i] + sums[3][k][j][i])) +
                                                      ((sums[4][k][j][i] + sums[5][k][j][i]) + (sums[6][k][j][i] + sums[7][k][j][i])), tag);
    }
    stamp(3);
    if (err) atomicOr(&ctl->err, err);
    if (u >= M * slices) return;
    float4 dv[LG_ROWV];
    err = 0;
    if (rowt) lg_take_row(dv, y.o + (size_t)jr * E, t, nq, tag, a.spin_limit, err);
    if (err) atomicOr(&ctl->err, err);
    if (a.gw && u == 0 && t == 0) lg_put_soon(a.rows, lg_far_tag(tag));
    stamp(4);
    row.work<(M > 3)>(a, dv, jr, vr, rowt, t, red[0], red[1], tag);
    stamp(5);
}
