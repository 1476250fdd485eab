// lg_wide.h — the q4_0 x q8 matmuls of wide row blocks (prompts), on the matrix cores.
//
// Same arithmetic and the same float order as the wavefront-dot kernels of lg_kernels.h (so a prompt leaves
// bit-identical cache rows): per 32-weight block an exact dot, p = fma(xd*dw, (float)dot, p) along each of the S
// contiguous K segments, then the adjacent-pair tree over the segments.  What is left to the vector units is the one
// fma per output and block that this order needs; everything else of a block runs on the matrix cores:
//
//  * the dot, as v_mfma_scale_f32_32x32x64_f8f6f4 on 6-bit floats (e2m3, whose codes 0..15 are the multiples 0..15 of 2^-3 and whose
//    bit 5 is the sign: the code of an integer is its magnitude and its sign).  A weight is one such value (its nibble - 8).  A q8
//    value q is two, the high and the low four bits of |q|, each with the sign of q: the instruction's K = 64 is the block's 32 weights
//    twice against its 32 high and its 32 low digits.  The factors 16 of the high half and 2^3 of every code are the
//    E8M0 scales.  Products and sums are integers below 2^15 (an integer times 2^-6 inside), so the result
//    is the exact dot, already a float.  On int8 (v_mfma_i32_32x32x32_i8, the same 32 cycles) every output needs a
//    subtraction to become (float)(dot - 8*sum).
//  * the products xd*dw, as the outer product v_mfma_f32_32x32x1_2b_f32 with a zero accumulator: fma(x, y, 0) is the
//    correctly rounded product (subnormals included).  One instruction serves the two 32-row halves of a weight tile,
//    and a lane loads one scale per block where the vector form loads the 16 scales of its outputs through LDS.
//
// Measured issue bound per 32x32x32 block and SIMD: 36 cycles of fma (two wavefronts: 2.25 each), 32 of the dot and 32 of half a
// scale product.  The f32 product runs on the vector unit's multipliers and keeps it from everything else, and with both
// wavefronts busy the dots do not overlap the fma either: 100 cycles, of which the loop reaches 126 (int8 with sub, mul and fma: 163).
//
// A workgroup is 4 wavefronts and owns 64 weight rows x 32*TB activation rows; wavefront w runs the K segments 2w and
// 2w+1, so the wavefronts share no operands, the main loop has no barrier and the operands come straight from L2; LDS
// only carries the partial sums (the first segment's while the second runs, and the tree over the wavefronts).
#pragma once
#include "lg_kernels.h"

typedef int lg_v8i __attribute__((ext_vector_type(8)));
typedef float lg_v16f __attribute__((ext_vector_type(16)));
typedef float lg_v32f __attribute__((ext_vector_type(32)));

#define LG_WT      64                      // weight rows of a tile
#define LG_WTILE   1664                    // bytes of (64 weight rows, one block): [64][16] + [64][8] bytes of 6-bit values, [64] f16 scales
#define LG_QTILE   3328                    // bytes of (64 activation rows, one block): 2 x ([64][16] + [64][8]) bytes of digits, [64] f32 scales
#define LG_WIDE      32                    // activation rows of one matrix-core operand
#define LG_WIDE_ROWS 512                   // rows of the widest block
#define LG_WIDE_MID  128                   // the widest block of a short cache

// 6-bit float code of an integer -15..15: its value times 8, sign and magnitude
__device__ __forceinline__ uint32_t lg_e2m3(int v) { return (uint32_t)(v < 0 ? -v : v) | (v < 0 ? 0x20u : 0u); }
// four such codes in the bytes of x -> 24 bits
__device__ __forceinline__ uint32_t lg_pack6(uint32_t x) {
    return __builtin_amdgcn_udot4(x, 0x00004001u, __builtin_amdgcn_udot4(x, 0x40010000u, 0u, false) << 12, false);
}
// Where the digits of (row j, block b) of a wide activation buffer of nb blocks per row live: dword d (0..5) of the hi
// (half = 0) or lo (half = 1) digits, and the row's scale.
__device__ __forceinline__ size_t lg_qtile(int nb, int j, int b) { return ((size_t)(j >> 6) * nb + b) * LG_QTILE; }
__device__ __forceinline__ int lg_qdigit(int j, int half, int d) {
    const int lane = half * 32 + (j & 31), t = ((j >> 5) & 1) * 1536;
    return d < 4 ? t + lane * 16 + d * 4 : t + 1024 + lane * 8 + (d - 4) * 4;
}
__device__ __forceinline__ int lg_qscale(int j) { return 3072 + (j & 63) * 4; }
// bytes of a wide activation buffer
__host__ __device__ static inline size_t lg_wide_q8_bytes(int rows, int k) { return (size_t)((rows + 63) / 64) * (size_t)(k >> 5) * LG_QTILE; }

// q8 of 32 values held as one float4 in each of 8 adjacent lanes (lane % 8 = i holds elements 4i..4i+3 of block b of row
// j), written as digits: the arithmetic of lg_quant4_8lanes.  Bound by vector issue, next to which the matmuls that end in it run:
// sign and magnitude take 26 instructions for four values where digits that are sums (e3m2 codes of q = 16*hi + lo) took 94.
// With lg_gelu_d: 1000 tokens of the E4B shape 21.87 -> 21.46 ms, 4093 of the 12B shape 184.1 -> 181.0 ms.
__device__ __forceinline__ void lg_wide_quant4(float4 h, uint8_t *q, int nb, int j, int b) {
    float amax = fmaxf(fmaxf(fabsf(h.x), fabsf(h.y)), fmaxf(fabsf(h.z), fabsf(h.w)));
    amax = lg_max_n(amax, 8);
    const float d = lg_div127(amax);
    const float id = lg_inv_scale(d);
    const float p[4] = { h.x * id, h.y * id, h.z * id, h.w * id };
    // |q| in the four bytes: a NaN becomes 0, as in the conversion to int8, and the values next to it keep their digits (an infinity
    // among the 32 makes their scale a NaN, so that the block does not pass for finite).  Signs: bit 7 of the floats' last bytes.
    uint32_t mag = 0;
    #pragma unroll
    for (int i = 0; i < 4; ++i) mag = __builtin_amdgcn_cvt_pk_u8_f32(lg_rintf(fabsf(p[i])), i, mag);
    const uint32_t sg = ((__builtin_amdgcn_perm(__float_as_uint(p[1]), __float_as_uint(p[0]), 0x0C0C0703u) |
                          __builtin_amdgcn_perm(__float_as_uint(p[3]), __float_as_uint(p[2]), 0x07030C0Cu)) >> 2) & 0x20202020u;
    const uint32_t hi = lg_pack6(((mag >> 4) & 0x0F0F0F0Fu) | sg), lo = lg_pack6((mag & 0x0F0F0F0Fu) | sg);
    // 24 bits per lane, four lanes make three dwords: lane k (k = 0..2 of the four) completes its bits with its neighbour's
    const int i = (int)threadIdx.x & 7, k = i & 3, dw = 3 * (i >> 2) + k;
    const uint32_t nh = (uint32_t)lg_dpp_i<0xF9>((int)hi), nl = (uint32_t)lg_dpp_i<0xF9>((int)lo);   // quad_perm [1,2,3,3]
    uint8_t *t = q + lg_qtile(nb, j, b);
    if (k < 3) {
        *(uint32_t *)(t + lg_qdigit(j, 0, dw)) = (hi >> (8 * k)) | (nh << (24 - 8 * k));
        *(uint32_t *)(t + lg_qdigit(j, 1, dw)) = (lo >> (8 * k)) | (nl << (24 - 8 * k));
    }
    if (i == 0) *(float *)(t + lg_qscale(j)) = d;
}

// Wide form of a tiled matrix (segment tiles, or row-block tiles when RB), built on the device when a model is
// committed: one thread per (row, block).  Rows past m (a row count that is no multiple of 64) are zero.
__global__ __launch_bounds__(LG_WG) void lg_k_wide_pack(const uint8_t *w, int k, int m, int rb, uint8_t *dst) {
    const int nb = k >> 5, mp = (m + LG_WT - 1) / LG_WT * LG_WT;
    const size_t id = (size_t)blockIdx.x * LG_WG + threadIdx.x;
    if (id >= (size_t)mp * nb) return;
    const int row = (int)(id % (size_t)mp), b = (int)(id / (size_t)mp);
    uint32_t out[6] = { 0, 0, 0, 0, 0, 0 };
    uint16_t sc = 0;
    if (row < m) {
        const uint8_t *tile; int slot;
        if (rb) { tile = w + ((size_t)(row >> 6) * nb + b) * LG_TILE; slot = row & 63; }
        else {
            const int S = lg_segments(k), nit = nb / S, rw = 64 / S, c = b / nit;
            tile = w + ((size_t)(row / rw) * nit + (b - c * nit)) * LG_TILE; slot = (row % rw) * S + c;
        }
        const uint8_t *qs = tile + slot * 16;
        sc = *(const uint16_t *)(tile + 1024 + slot * 2);
        #pragma unroll
        for (int e = 0; e < 32; ++e) {
            const int nib = e < 16 ? (qs[e] & 15) : (qs[e - 16] >> 4);
            const uint64_t c = (uint64_t)lg_e2m3(nib - 8) << ((6 * e) & 31);
            out[(6 * e) >> 5] |= (uint32_t)c;
            if (((6 * e) & 31) > 26) out[((6 * e) >> 5) + 1] |= (uint32_t)(c >> 32);
        }
    }
    uint8_t *t = dst + ((size_t)(row >> 6) * nb + b) * LG_WTILE;
    const int n = row & 63;
    *(uint4 *)(t + n * 16) = make_uint4(out[0], out[1], out[2], out[3]);
    *(uint2 *)(t + 1024 + n * 8) = make_uint2(out[4], out[5]);
    *(uint16_t *)(t + 1536 + n * 2) = sc;
}
static inline size_t lg_wide_bytes(int k, int m) { return (size_t)((m + LG_WT - 1) / LG_WT) * (size_t)(k >> 5) * LG_WTILE; }

struct WideMm {
    const uint8_t *w;        // wide form of the weights
    const uint8_t *q;        // wide activation buffer
    int k, m, rows;          // row length, weight rows, activation rows of the block
    int nb_tiles;            // activation tiles of 32*TB rows
    int parts;               // 1: 8 K segments; 4: 32 segments, cut by quarter
};
// Workgroup -> (weight tile, activation tile, K quarter).  Consecutive workgroups are dealt to the 8 XCDs in turn; an
// XCD walks the activation tiles of one weight tile before the next, so a weight tile is fetched from HBM by one XCD
// once and the activations (2 MB of digits per 512 rows and 2560 inputs) stay in its 4 MB L2; with four K quarters an
// XCD keeps to one quarter's activations.
__device__ __forceinline__ bool lg_wide_map(const WideMm &a, int id, int &at, int &bt, int &part) {
    const int x = id & 7, s = id >> 3, per = 8 / a.parts, an = s / a.nb_tiles;
    bt = s - an * a.nb_tiles;
    part = x % a.parts;
    at = x / a.parts + per * an;
    return at * LG_WT < a.m;
}
static inline int lg_wide_grid(int m, int nb_tiles, int parts) {
    const int nt = (m + LG_WT - 1) / LG_WT, per = 8 / parts;
    return 8 * ((nt + per - 1) / per) * nb_tiles;
}

// The tile's sums.  WV wavefronts: wavefront w runs the 8/WV segments from 8*part + w*8/WV of the K range (WV = 2: segment 2*part + w) and leaves their
// sum in lds[w][(ta*TB + tb)*4 + g][lane] as float4 (weight rows 32*ta + 8*g + 4*h + 0..3 of the tile, activation row
// 32*tb + n, lane = 32*h + n).  Synchronised on return.
template <int TB, int WV, bool DUMP>
__device__ __forceinline__ void lg_wide_tile(const WideMm &a, int at, int bt, int part, float4 *lds, int32_t *dots) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 31;
    constexpr int SEG = WV == 2 ? 2 : 8;                      // segments of a workgroup (two: a matrix of 8 cut by K quarter)
    const int nb = a.k >> 5, nit = nb / (SEG * a.parts);
    const int kb0 = (SEG * part + SEG / WV * __builtin_amdgcn_readfirstlane(wave)) * nit;
    const __amdgpu_buffer_rsrc_t rw = lg_buffer_rsrc(a.w + ((size_t)at * nb + kb0) * LG_WTILE);
    const int sub = TB == 1 ? (bt & 1) : 0;
    const __amdgpu_buffer_rsrc_t rq = lg_buffer_rsrc(a.q + ((size_t)(TB == 1 ? bt >> 1 : bt) * nb + kb0) * LG_QTILE);
    const int vq16 = sub * 1536 + lane * 16, vq8 = sub * 1536 + 1024 + lane * 8, vxs = 3072 + (TB == 1 ? sub * 32 + n : lane) * 4;
    // The operands of a block, as loaded (a lane holds weight row `lane` of the tile and its digits of each activation tile).
    struct Ops { lg_v8i b[TB]; uint32_t a[6]; float xs; uint32_t ws; };
    auto fetch = [&](Ops &o, int kb_) {
        const int kb = __builtin_amdgcn_readfirstlane(kb_), wo = kb * LG_WTILE, qo = kb * LG_QTILE;
        const auto a16 = __builtin_amdgcn_raw_buffer_load_b128(rw, lane * 16, wo, 0);
        const auto a8 = __builtin_amdgcn_raw_buffer_load_b64(rw, 1024 + lane * 8, wo, 0);
        o.a[0] = a16[0]; o.a[1] = a16[1]; o.a[2] = a16[2]; o.a[3] = a16[3]; o.a[4] = a8[0]; o.a[5] = a8[1];
        o.ws = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rw, 1536 + lane * 2, wo, 0);
        #pragma unroll
        for (int t = 0; t < TB; ++t) {
            const auto b16 = __builtin_amdgcn_raw_buffer_load_b128(rq, vq16 + t * 1536, qo, 0);
            const auto b8 = __builtin_amdgcn_raw_buffer_load_b64(rq, vq8 + t * 1536, qo, 0);
            o.b[t] = (lg_v8i){ (int)b16[0], (int)b16[1], (int)b16[2], (int)b16[3], (int)b8[0], (int)b8[1], 0, 0 };
        }
        o.xs = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rq, vxs, qo, 0));
    };
    const int sb = lane < 32 ? 134 : 130;                     // E8M0 scales of the K halves: 2^3 of the codes, 2^4 more for the high digits
    const lg_v16f z16 = {};
    const lg_v32f z32 = {};
    float p[2][TB][16];
    auto clear = [&]() {
        #pragma unroll
        for (int t = 0; t < 2 * TB; ++t)
            #pragma unroll
            for (int i = 0; i < 16; ++i) p[t & 1][t >> 1][i] = 0.0f;
    };
    float4 *mine = lds + (size_t)wave * (2 * TB * 4 * 64);
    auto segment_end = [&]() {                                // the first segment's sums wait in LDS
        #pragma unroll
        for (int t = 0; t < 2 * TB; ++t)
            #pragma unroll
            for (int g = 0; g < 4; ++g)
                mine[(t * 4 + g) * 64 + lane] = make_float4(p[t / TB][t % TB][4 * g], p[t / TB][t % TB][4 * g + 1], p[t / TB][t % TB][4 * g + 2], p[t / TB][t % TB][4 * g + 3]);
        clear();
    };
    // A step is (block, activation tile): its two dots D0 and D1, its scale products S, and the 32 fma that use them.  S keeps the
    // vector unit from everything else while it runs, so it has one set of registers; the dots of the next step are issued
    // behind the fma that read this step's.  (With S of the next step issued ahead of this step's fma, 30 registers more: prompts
    // 0.5 to 1.2% slower.)  The last blocks run apart from the loop, which always requests.
    constexpr int NS = TB == 2 ? 2 : 4;                       // blocks in flight (32-row tiles with 6 or 8: a prompt of 23 tokens 5980 -> 6100, 6260 us)
    Ops o[NS];
    lg_v32f S;
    lg_v16f D0, D1;
    lg_v8i a0, a1;
    float dw, xd[2];
    const int nblk = SEG / WV * nit, last = nblk - 1;
    auto take = [&](const Ops &q) {                           // a block's weight operands: each 32-row half in both K halves
        #pragma unroll
        for (int i = 0; i < 6; ++i) { const lg_u2 r = lg_pair32(q.a[i]); a0[i] = (int)r.x; a1[i] = (int)r.y; }
        a0[6] = a0[7] = a1[6] = a1[7] = 0;
        dw = lg_h2f((uint16_t)q.ws);
        if (TB == 1) xd[0] = q.xs;
        else { const lg_u2 r = lg_pair32(__float_as_uint(q.xs)); xd[0] = __uint_as_float(r.x); xd[1] = __uint_as_float(r.y); }
    };
    #pragma unroll
    for (int i = 0; i < NS; ++i) fetch(o[i], i < last ? i : last);
    clear();
    take(o[0]);
    D0 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a0, o[0].b[0], z16, 2, 2, 0, 130, 0, sb);
    D1 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a1, o[0].b[0], z16, 2, 2, 0, 130, 0, sb);
    auto block = [&](int it, int u, bool more) {              // block it + u; `more`: its registers receive block it + u + NS
        if (WV == 4 && it + u == nit) segment_end();
        #pragma unroll
        for (int t = 0; t < TB; ++t) {
            const Ops &on = t + 1 < TB ? o[u] : o[(u + 1) % NS];
            const int tn = t + 1 < TB ? t + 1 : 0;
            S = __builtin_amdgcn_mfma_f32_32x32x1f32(dw, xd[t], z32, 0, 0, 0);
            if (tn == 0) take(on);
            __builtin_amdgcn_sched_barrier(0);
            if (DUMP) {
                const int an = (bt * TB + t) * 32 + n;
                if (an < a.rows)
                    for (int i = 0; i < 16; ++i) {
                        const int row = at * LG_WT + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                        if (row < a.m) dots[((size_t)an * a.m + row) * nb + kb0 + it + u] = (int)D0[i];
                        if (row + 32 < a.m) dots[((size_t)an * a.m + row + 32) * nb + kb0 + it + u] = (int)D1[i];
                    }
            }
            #pragma unroll
            for (int i = 0; i < 16; ++i) p[0][t][i] = lg_fmaf(S[i], D0[i], p[0][t][i]);
            __builtin_amdgcn_sched_barrier(0);
            D0 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a0, on.b[tn], z16, 2, 2, 0, 130, 0, sb);
            __builtin_amdgcn_sched_barrier(0);
            #pragma unroll
            for (int i = 0; i < 16; ++i) p[1][t][i] = lg_fmaf(S[16 + i], D1[i], p[1][t][i]);
            __builtin_amdgcn_sched_barrier(0);
            D1 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a1, on.b[tn], z16, 2, 2, 0, 130, 0, sb);
            if (more && t == (TB == 2 ? 0 : TB - 1)) { const int nx = it + u + NS; fetch(o[u], nx < last ? nx : last); }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int it = 0;
    for (; it + NS < nblk; it += NS) {
        #pragma unroll
        for (int u = 0; u < NS; ++u) block(it, u, true);
    }
    #pragma unroll
    for (int u = 0; u < NS; ++u) {                            // the last NS blocks at most: nothing left to request
        if (it + u < nblk) block(it, u, false);             // (a guard, not a break: the operands stay in registers)
    }
    #pragma unroll
    for (int t = 0; t < 2 * TB; ++t)
        #pragma unroll
        for (int g = 0; g < 4; ++g) {
            float4 *s = &mine[(t * 4 + g) * 64 + lane];
            const float4 v = WV == 4 ? *s : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            *s = make_float4(v.x + p[t / TB][t % TB][4 * g], v.y + p[t / TB][t % TB][4 * g + 1], v.z + p[t / TB][t % TB][4 * g + 2], v.w + p[t / TB][t % TB][4 * g + 3]);
        }
    __syncthreads();
}
// finished sums of float4 `u` (= (ta*TB + tb)*4 + g) of this lane: the tree over the wavefronts
template <int TB, int WV>
__device__ __forceinline__ float4 lg_wide_sum(const float4 *lds, int u) {
    const int lane = threadIdx.x & 63, st = 2 * TB * 4 * 64;
    if constexpr (WV == 2) {
        const float4 a = lds[u * 64 + lane], b = lds[st + u * 64 + lane];
        return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
    }
    auto quad = [&](int w) {
        const float4 *l = lds + (size_t)w * st + u * 64 + lane;
        const float4 a = l[0], b = l[st], c = l[2 * st], d = l[3 * st];
        return make_float4((a.x + b.x) + (c.x + d.x), (a.y + b.y) + (c.y + d.y), (a.z + b.z) + (c.z + d.z), (a.w + b.w) + (c.w + d.w));
    };
    const float4 r = quad(0);
    if (WV == 4) return r;
    const float4 s = quad(4);
    return make_float4(r.x + s.x, r.y + s.y, r.z + s.z, r.w + s.w);
}

// Plain matmul: out[part][row][m] f32 (four slabs when the K range is cut by quarter: the consumer adds them as
// (p0 + p1) + (p2 + p3), the top of the segment tree).
template <int TB, int WV, bool DUMP>
__global__ __launch_bounds__(64 * WV, 2) void lg_k_wide_mm(WideMm a, float *out, int32_t *dots) {
    extern __shared__ __align__(16) unsigned char smem[];
    float4 *lds = (float4 *)smem;
    int at, bt, part;
    if (!lg_wide_map(a, (int)blockIdx.x, at, bt, part)) return;
    lg_wide_tile<TB, WV, DUMP>(a, at, bt, part, lds, dots);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 31, h = lane >> 5;
    #pragma unroll
    for (int v = 0; v < 8 * TB / WV; ++v) {
        const int u = wave * (8 * TB / WV) + v, t = u >> 2, ta = t / TB, tb = t % TB, g = u & 3;
        const float4 r = lg_wide_sum<TB, WV>(lds, u);
        const int an = (bt * TB + tb) * 32 + n, col = at * LG_WT + 32 * ta + 8 * g + 4 * h;
        if (an < a.rows && col < a.m) *(float4 *)(out + ((size_t)part * a.rows + an) * a.m + col) = r;
    }
}

// Gate/up with the GeGLU and the q8 of its result: a weight tile is the 32 gate rows and the 32 up rows of 32 FFN columns.
template <int TB, int WV>
__global__ __launch_bounds__(64 * WV, 2) void lg_k_wide_geglu(WideMm a, uint8_t *gq) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ __align__(16) float vbuf[32 * TB * 36];
    float4 *lds = (float4 *)smem;
    int at, bt, part;
    if (!lg_wide_map(a, (int)blockIdx.x, at, bt, part)) return;
    lg_wide_tile<TB, WV, false>(a, at, bt, part, lds, nullptr);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 31, h = lane >> 5;
    for (int u = wave; u < 4 * TB; u += WV) {
        const int tb = u >> 2, g = u & 3;
        const float4 gv = lg_wide_sum<TB, WV>(lds, tb * 4 + g), uv = lg_wide_sum<TB, WV>(lds, (TB + tb) * 4 + g);
        *(float4 *)(vbuf + (32 * tb + n) * 36 + 8 * g + 4 * h) =
            make_float4(lg_gelu_d(gv.x) * uv.x, lg_gelu_d(gv.y) * uv.y, lg_gelu_d(gv.z) * uv.z, lg_gelu_d(gv.w) * uv.w);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 32 * TB * 8; i += 64 * WV) {
        const int row = i >> 3;
        lg_wide_quant4(*(const float4 *)(vbuf + row * 36 + (i & 7) * 4), gq, a.m >> 6, bt * 32 * TB + row, at);
    }
}

// Per-layer gate: gelu(inp_gate . x) * ipl of this layer, and the q8 of it.
template <int TB, int WV>
__global__ __launch_bounds__(64 * WV, 2) void lg_k_wide_plegate(WideMm a, const float *ipl, int layer, int n_layer, uint8_t *pq) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ __align__(16) float vbuf[2 * 32 * TB * 36];
    float4 *lds = (float4 *)smem;
    int at, bt, part;
    if (!lg_wide_map(a, (int)blockIdx.x, at, bt, part)) return;
    lg_wide_tile<TB, WV, false>(a, at, bt, part, lds, nullptr);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 31, h = lane >> 5;
    for (int u = wave; u < 8 * TB; u += WV) {
        const int t = u >> 2, g = u & 3, ta = t / TB, tb = t % TB, an = (bt * TB + tb) * 32 + n;
        const float4 v = lg_wide_sum<TB, WV>(lds, u);
        const int col = at * LG_WT + 32 * ta + 8 * g + 4 * h;
        const float4 p = *(const float4 *)(ipl + ((size_t)(an < a.rows ? an : a.rows - 1) * n_layer + layer) * a.m + col);
        *(float4 *)(vbuf + (ta * 32 * TB + 32 * tb + n) * 36 + 8 * g + 4 * h) =
            make_float4(lg_gelu_d(v.x) * p.x, lg_gelu_d(v.y) * p.y, lg_gelu_d(v.z) * p.z, lg_gelu_d(v.w) * p.w);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * 32 * TB * 8; i += 64 * WV) {
        const int row = i >> 3, ta = row / (32 * TB);
        lg_wide_quant4(*(const float4 *)(vbuf + row * 36 + (i & 7) * 4), pq, a.m >> 5, bt * 32 * TB + row - ta * 32 * TB, at * 2 + ta);
    }
}

// Per-layer gate of a block of few rows, the residual update ahead of it inside: lg_k_rows_plegate of verify blocks with the result as wide
// digits, a workgroup per (32 gate rows, block row).  On 64 x 32 tiles 256 gate rows are four workgroups, whose CUs pull a quarter of
// the matrix and all of the block's digits each: 22 rows at the E4B width 5.0 us for the rows and 9.4 for the gate -> 7.5.
__global__ __launch_bounds__(LG_WG) void lg_k_wide_rows_plegate(RowsPleGateArgs a, int rows) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ __align__(16) float gbuf[32];
    __shared__ float red[4];
    const int gb = blockIdx.x, j = blockIdx.y;
    float4 xnew[LG_ROWV];
    lg_rows_plegate_body(a, rows, gb, j, smem, gbuf, red, xnew, gb == 0, [] {}, [&](const float *v) {
        if (threadIdx.x < 8) lg_wide_quant4(((const float4 *)v)[threadIdx.x], (uint8_t *)a.g.pq, a.g.ple >> 5, j, gb);
    });
}

// Row kernel of a wide block (lg_k_rows of verify blocks, the result as wide digits): residual
// update, norm, q8.  dparts = 4: dout is four [rows][E] slabs.  A workgroup per row, or (blocks of few rows) one per slice of it:
// each forms the row's sums, stores and quantizes the float4s t + 256 * blockIdx.y of its lanes.
__global__ __launch_bounds__(LG_WG) void lg_k_wide_rows(RowArgs s, int rows) {
    __shared__ float red[2][4];
    const int t = threadIdx.x, j = blockIdx.x, E = s.E, nq = E >> 2, vs = s.slices > 1 ? (int)blockIdx.y : -1;
    float4 xv[LG_ROWV], dv[LG_ROWV], wpost[LG_ROWV], wpre[LG_ROWV];
    if (!s.x) {
        const int tok = s.toks[j];
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
            const float4 e = lg_tiled_deq4(s.emb, s.emb_nit, s.emb_seg, tok, 4 * (t + 256 * v));
            xv[v] = make_float4(e.x * s.emb_scale, e.y * s.emb_scale, e.z * s.emb_scale, e.w * s.emb_scale);
        }
    } else {
        const float4 *xr = (const float4 *)(s.x + (size_t)j * E);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) xv[v] = xr[t + 256 * v];
    }
    const bool has_os = s.dout != nullptr && s.os != nullptr;
    const float osv = has_os ? s.os[0] : 1.0f;
    if (s.dout) {
        const float4 *dr = (const float4 *)(s.dout + (size_t)j * E), *wr = (const float4 *)s.w_post;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) { dv[v] = dr[t + 256 * v]; wpost[v] = wr[t + 256 * v]; }
    }
    if (s.w_pre) {
        const float4 *wr = (const float4 *)s.w_pre;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) wpre[v] = wr[t + 256 * v];
    }
    if (s.dout && s.dparts == 4) lg_add_slabs(dv, (const float4 *)(s.dout + (size_t)j * E), (size_t)rows * nq, t, nq);
    if (s.dout) {
        float ss = 0.0f;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(dv[v], ss);
        ss = lg_block_sum256(ss, red[0]);
        const float sc = 1.0f / sqrtf(ss / (float)E + s.eps);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
            const float4 w = wpost[v];
            float4 r;
            r.x = xv[v].x + dv[v].x * sc * w.x;  r.y = xv[v].y + dv[v].y * sc * w.y;
            r.z = xv[v].z + dv[v].z * sc * w.z;  r.w = xv[v].w + dv[v].w * sc * w.w;
            if (has_os) { r.x = r.x * osv; r.y = r.y * osv; r.z = r.z * osv; r.w = r.w * osv; }
            xv[v] = r;
        }
    }
    if (s.x_out) {
        float4 *xo = (float4 *)(s.x_out + (size_t)j * E);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq && (vs < 0 || v == vs)) xo[t + 256 * v] = xv[v];
    }
    if (s.w_pre) {
        float ss = 0.0f;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(xv[v], ss);
        ss = lg_block_sum256(ss, red[1]);
        const float sc = 1.0f / sqrtf(ss / (float)E + s.eps);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
            const float4 w = wpre[v];
            xv[v] = make_float4(xv[v].x * sc * w.x, xv[v].y * sc * w.y, xv[v].z * sc * w.z, xv[v].w * sc * w.w);
        }
    }
    if (!s.q) return;
    #pragma unroll
    for (int v = 0; v < LG_ROWV; ++v) {
        if (t + 256 * v >= nq) break;                        // nq is a multiple of 64: whole wavefronts
        if (vs >= 0 && v != vs) continue;
        lg_wide_quant4(xv[v], (uint8_t *)s.q, E >> 5, j, (t + 256 * v) >> 3);
    }
}

// Plain q8 of rows x k floats as wide digits (isolated matmul).
__global__ __launch_bounds__(LG_WG) void lg_k_wide_quant(const float *x, int rows, int k, uint8_t *q) {
    const int g = (blockIdx.x * LG_WG + threadIdx.x) >> 3, l = threadIdx.x & 7, nb = k >> 5;
    if (g >= rows * nb) return;                              // (groups of 8 lanes leave together)
    lg_wide_quant4(((const float4 *)x)[(size_t)g * 8 + l], q, nb, g / nb, g - g / nb * nb);
}

// ---------------------------------------------------------------------------------------------------------
// Attention of a wide block.  A workgroup is 8 wavefronts on 16 units = (rows, query heads) of one kv head.  Both products
// run on f32 matrix instructions whose accumulation is the defined chain:
//  * scores: the four blocks of v_mfma_f32_16x16x1_4b_f32 (one fma per output and step, subnormals included) are the four
//    chains c of a score (dims 4g + c), a step per g ascending; a lane ends up with all four chains of its outputs and adds
//    (a0+a1)+(a2+a3).  Queries wait in LDS chain by chain; K rows come straight from the cache, 64 bytes of a row by four
//    lanes, and are dealt to the chains by a 4 x 4 exchange over the four 16-lane rows.  The wavefronts take key tiles in
//    turn, the next tile's rows in flight.  (v_mfma_f32_16x16x4_f32, k = four steps of a chain, adds in the same order and
//    needs no exchange, but its operands come as 8-byte pieces of a row, twice the cache accesses: 47 -> 54 us.)
//  * values: the same instruction, its four blocks are four consecutive tiles, a step per key slot (masked slots have
//    weight 0; results that are not finite are computed again without them), the columns 16 dims; a wavefront takes 32 dims
//    as two such products, so that one 4-byte load per lane feeds two steps, and adds the tiles' results to the running sum
//    in tile order with the weights exp(m_tile - M).
// The weights e of a row's tiles, their maxima and sums wait in LDS between the two (EL: up to LG_WA_TILES tiles; more: in
// the cache's scratch).  Bound by the matrix cores (8 to 9 thousand cycles per 16 units and tile) and the exponentials.
// Eight wavefronts rather than four: one workgroup is all the LDS holds on a CU, and with two wavefronts on a SIMD one
// loads, deals and exponentiates while the other multiplies.  500 rows of a 512-wide window of 256-wide heads (8 over 2):
// 65 -> 43 us; 512 rows of a 1024-wide one (16 over 8): 232 -> 137 us; all of 4093 positions (16 over 1): 584 -> 400 us.
// Pieces and runs converted ahead of their products: the 1024-wide window 132 -> 119 us; the first value runs requested ahead of
// the synchronisations: 332 rows at 3001 11.73 -> 11.70 ms a prompt.
// In memory the weights are requested with the value rows, runs ahead (512 rows at 3500, 16 heads over 8: 474 -> 450 us).
//
// PHASE 1 and 2 are the two halves as kernels of their own, for blocks whose groups do not fill the chip: the time of a
// workgroup is a matter of its tiles (22 rows at position 3000 take 40 us on 12 workgroups, 487 rows 45 on 244).  PHASE 1 deals the
// tiles of a group to gridDim.z workgroups of four wavefronts, PHASE 2 the dims, 128 to a workgroup: each wavefront has a
// matrix core of its own.  22 rows at 3000: 512-wide window 40 -> 29 us, all positions 171 -> 74 us; at 20000 1083 -> 355 us.
#define LG_WA_TILES 44
#define LG_WA_WG 512
#define LG_WA_SPLIT_WG 256
#define LG_WA_SPLIT_MAX 1024             // tiles whose weights PHASE 2 keeps in LDS
#define LG_WA_SPLIT_GROUPS 128           // groups of units (x kv heads) up to which the two kernels are launched for any number of tiles (more: launch_wide_attn)
struct WideAttn {
    const float *q;              // [rows][H*hd] normed + rotated
    const uint16_t *kc, *vc;     // cache of the layer this one reads
    int H, nkv, seq, kv_dim, window, rows;
    float *scratch;              // !EL: per group tiles * 16 * 34 floats
    int tiles;                   // tiles a group can touch, rounded up to a multiple of four
    uint8_t *xq;                 // wide digits of the result, width H*hd
};
static inline int lg_wide_attn_rows(int G) { return 16 / G; }
static inline size_t lg_wide_attn_lds(int tiles) { return (size_t)tiles * 16 * 38 * 4; }
__device__ __forceinline__ float lg_max16(float v) {
    v = lg_max8(v);
    return fmaxf(v, lg_dpp_f<LG_DPP_MIRROR16>(v));
}
// 4 x 4 exchange over the four 16-lane rows of a wavefront: lane row c holds x0..x3 and receives element c of the rows
// 0..3 in o[0..3].
__device__ __forceinline__ void lg_deal4(uint32_t x0, uint32_t x1, uint32_t x2, uint32_t x3, uint32_t (&o)[4]) {
    const lg_u2 p = __builtin_amdgcn_permlane32_swap(x0, x2, false, false), q = __builtin_amdgcn_permlane32_swap(x1, x3, false, false);
    const lg_u2 x = __builtin_amdgcn_permlane16_swap(p.x, q.x, false, false), y = __builtin_amdgcn_permlane16_swap(p.y, q.y, false, false);
    o[0] = x.x; o[1] = x.y; o[2] = y.x; o[3] = y.y;
}
template <int HD, bool EL, int PHASE = 0, bool FAR = false>
__global__ __launch_bounds__(PHASE ? LG_WA_SPLIT_WG : LG_WA_WG, 2) void lg_k_wide_attn(WideAttn a, const StepCtl *ctl) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int WG = PHASE ? LG_WA_SPLIT_WG : LG_WA_WG, NW = WG / 64;
    static_assert(PHASE == 0 || !EL, "the two kernels hand the weights over in memory");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), n = lane & 15, c = lane >> 4;
    const int G = a.H / a.nkv, RG = 16 / G, U = RG * G, kvh = blockIdx.y, row0 = blockIdx.x * RG;
    const int gi = 256 / G + 1;                               // u / G = u * gi >> 8 for u < 16
    int rlast = row0 + RG - 1;
    if (rlast >= a.rows) rlast = a.rows - 1;
    // the units' query rows are requested first: neither the position nor the K rows are needed for them, and loads return in order
    // (behind the first tile's rows they were in LDS 4.0 us into a launch of few workgroups: 22 rows of 8 heads of 256 16.0 -> 14.7 us)
    constexpr int QL = 16 * (HD / 4) / WG;                    // float4 of query per thread (64-wide heads: every second thread)
    float4 qf[QL < 1 ? 1 : QL];
    if constexpr (PHASE != 2) {
        #pragma unroll
        for (int k = 0; k < (QL < 1 ? 1 : QL); ++k) {
            const int i = threadIdx.x + k * WG, u = (i / (HD / 4)) & 15, j = i % (HD / 4), ur = u * gi >> 8;
            int qr = row0 + ur;
            if (u >= U || qr > rlast) qr = rlast;
            qf[k] = *(const float4 *)(a.q + (size_t)qr * a.H * HD + (size_t)(kvh * G + (u < U ? u - ur * G : 0)) * HD + 4 * j);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    const int pos = ctl->pos;
    const int kfirst = lg_win_start(pos + row0, a.window), klast = pos + rlast;       // positions any row of the group sees
    const int tfirst = kfirst >> 5, tlast = klast >> 5;
    const int nt = (tlast - tfirst + 4) & ~3;                 // tiles past the last one are masked throughout
    // e: [tile][16 units][ES] (36: off the bank period), weights m and sums l: [tile][16]
    constexpr int ES = EL ? 36 : 32;
    float *eb = EL ? (float *)smem : a.scratch + ((size_t)blockIdx.x * a.nkv + kvh) * a.tiles * (16 * 34);
    float *mb = eb + (size_t)a.tiles * 16 * ES, *lb = mb + (size_t)a.tiles * 16;
    float *wb = PHASE == 2 ? (float *)smem : mb;              // the tiles' weights exp(m - M): several workgroups of values read the maxima
    __shared__ float mx[16][WG / 16 + 1];
    __shared__ __align__(16) float ob[16][HD + 4];
    if constexpr (PHASE != 2) {
        // validity of this lane's outputs: units 4c + i
        int us[4], up[4];
        #pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int u = 4 * c + i, r = row0 + (u * gi >> 8);
            const bool on = u < U && r <= rlast;
            up[i] = on ? pos + r : -1;
            us[i] = on ? lg_win_start(pos + r, a.window) : 0;
        }
        // pieces of a tile's K rows are requested as soon as the ones CH ahead of them have been dealt
        constexpr int NS = HD / 32, CH = NS < 8 ? NS : 8;     // 64-byte pieces of a K row; in flight
        uint4 w0[CH], w1[CH];
        auto rows_of = [&](int t, const uint16_t *&k0, const uint16_t *&k1) {
            const int ring0 = (t << 5) % a.seq;
            int r0 = ring0 + n, r1 = ring0 + 16 + n;          // ring rows of this lane's two keys (a ring is a multiple of 32 rows, or as long as the positions go)
            if (r0 >= a.seq) r0 = a.seq - 1;
            if (r1 >= a.seq) r1 = a.seq - 1;
            k0 = a.kc + (size_t)r0 * a.kv_dim + (size_t)kvh * HD + c * 8; k1 = a.kc + (size_t)r1 * a.kv_dim + (size_t)kvh * HD + c * 8;
        };
        const int t1 = tfirst + (PHASE ? blockIdx.z * NW : 0) + wave, step = PHASE ? gridDim.z * NW : NW;
        const uint16_t *k0, *k1, *n0, *n1;                    // of this tile, of the next one
        rows_of(t1, n0, n1);
        #pragma unroll
        for (int s = 0; s < CH; ++s) { w0[s] = *(const uint4 *)(n0 + s * 32); w1[s] = *(const uint4 *)(n1 + s * 32); }
        // the query rows into LDS, chain by chain: [unit][i % 4][i / 4] (in registers a wave's copy of them spilled)
        #pragma unroll
        for (int k = 0; k < (QL < 1 ? 1 : QL); ++k) {
            const int i = threadIdx.x + k * WG;
            if (QL < 1 && i >= 16 * (HD / 4)) break;
            const float4 f = qf[k];
            float *qd = &ob[i / (HD / 4)][i % (HD / 4)];
            qd[0] = f.x; qd[HD / 4] = f.y; qd[2 * (HD / 4)] = f.z; qd[3 * (HD / 4)] = f.w;
        }
        __syncthreads();
        const float *qs = &ob[n][c * (HD / 4)];               // this lane's query elements: unit n, chain c
        for (int t = t1; t < tfirst + nt; t += step) {
            const int t0 = t << 5;
            if (t > tlast) {                                  // a tile that only fills up the last four
                float *et = eb + (size_t)(t - tfirst) * 16 * ES;
                for (int i = lane; i < 16 * 32; i += 64) et[(i >> 5) * ES + (i & 31)] = 0.0f;
                if (lane < 16) { mb[(t - tfirst) * 16 + lane] = -INFINITY; lb[(t - tfirst) * 16 + lane] = 0.0f; }
                continue;
            }
            lg_v16f d0 = {}, d1 = {};
            k0 = n0; k1 = n1;
            rows_of(t + step, n0, n1);
            // dims 32s + 8c + 0..7 of a key -> the same key's dims 32s + 4g + c, g = 0..7.  A product that waits for the conversion in front
            // of it takes 52 cycles instead of 32, so a piece is dealt and converted ahead of the products of the one before it.
            float f0[2][8], f1[2][8];
            float4 qv[2][2];
            auto piece = [&](int s) {
                auto deal = [](uint4 w, float (&f)[8]) {
                    uint32_t o[4];
                    lg_deal4(__builtin_amdgcn_perm(w.z, w.x, 0x05040100u), __builtin_amdgcn_perm(w.z, w.x, 0x07060302u),
                             __builtin_amdgcn_perm(w.w, w.y, 0x05040100u), __builtin_amdgcn_perm(w.w, w.y, 0x07060302u), o);
                    #pragma unroll
                    for (int g = 0; g < 8; ++g) f[g] = lg_h2f((uint16_t)(o[g >> 1] >> (16 * (g & 1))));
                };
                deal(w0[s % CH], f0[s & 1]); deal(w1[s % CH], f1[s & 1]);
                const int i = s + CH;
                w0[s % CH] = *(const uint4 *)(i < NS ? k0 + i * 32 : n0 + (i - NS) * 32); w1[s % CH] = *(const uint4 *)(i < NS ? k1 + i * 32 : n1 + (i - NS) * 32);
                qv[s & 1][0] = *(const float4 *)(qs + 8 * s); qv[s & 1][1] = *(const float4 *)(qs + 8 * s + 4);
            };
            piece(0);
            #pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (s + 1 < NS) piece(s + 1);
                __builtin_amdgcn_sched_barrier(0);
                const float4 qa = qv[s & 1][0], qb = qv[s & 1][1];
                const float qe[8] = { qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w };
                #pragma unroll
                for (int g = 0; g < 8; ++g) {
                    d0 = __builtin_amdgcn_mfma_f32_16x16x1f32(qe[g], f0[s & 1][g], d0, 0, 0, 0);
                    d1 = __builtin_amdgcn_mfma_f32_16x16x1f32(qe[g], f1[s & 1][g], d1, 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            float *et = eb + (size_t)(t - tfirst) * 16 * ES, *mt = mb + (t - tfirst) * 16, *lt = lb + (t - tfirst) * 16;
            const int p0 = t0 + n, p1 = p0 + 16;
            #pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool v0 = p0 >= us[i] && p0 <= up[i], v1 = p1 >= us[i] && p1 <= up[i];
                const float s0 = (d0[i] + d0[4 + i]) + (d0[8 + i] + d0[12 + i]), s1 = (d1[i] + d1[4 + i]) + (d1[8 + i] + d1[12 + i]);
                const float m = lg_max16(fmaxf(v0 ? s0 : -INFINITY, v1 ? s1 : -INFINITY));
                const float e0 = v0 ? lg_expf(s0 - m) : 0.0f, e1 = v1 ? lg_expf(s1 - m) : 0.0f;
                const float l = lg_sum16(e0) + lg_sum16(e1);
                et[(4 * c + i) * ES + n] = e0;
                et[(4 * c + i) * ES + 16 + n] = e1;
                if (n == 0) { mt[4 * c + i] = m; lt[4 * c + i] = l; }
            }
        }
    }
    if constexpr (PHASE == 1) return;
    // Value rows.  A run is 8 slots of this lane's tile 4g + c (dims dg*32 + 2n and 2n + 1; !EL: the weights as well, which
    // come from memory too): requested AHEAD runs ahead, a group of four tiles is four runs.  The first runs do not wait for the
    // weights: they are requested here, ahead of the synchronisations.
    // Buffer loads: the tile's place in the lane offset, the slot's in a scalar register (as flat loads their 64-bit
    // addresses cost more vector instructions than the conversions); the buffer ends with the ring, slots past it read 0.
    // FAR: flat loads, for blocks that reach 2 GiB and more into a layer's value rows.
    constexpr int RUN = 8, NB = PHASE == 2 ? 8 : 4, AHEAD = NB - 1;
    uint32_t v[NB][RUN];
    float4 ev[EL ? 1 : NB][2];
    const int ng = nt >> 2, vrow = a.kv_dim * 2;
    const uint64_t vbytes = (uint64_t)a.seq * a.kv_dim * 2;
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void *)a.vc, 0, (uint32_t)(vbytes < 0x7FFFFFFFu ? vbytes : 0x7FFFFFFFu), 0x00020000);
    auto fetch_v = [&](int vcol, int buf, int g, int i) {
        g = g < ng ? g : ng - 1;
        const int ring0 = ((tfirst + 4 * g + c) << 5) % a.seq;
        if constexpr (FAR) {
            #pragma unroll
            for (int k = 0; k < RUN; ++k) {
                const int r = ring0 + RUN * i + k < a.seq ? ring0 + RUN * i + k : a.seq - 1;       // (a slot past the ring is no position of the group: zeroed below)
                v[buf][k] = *(const uint32_t *)((const uint8_t *)a.vc + (size_t)r * vrow + vcol);
            }
        } else {
            const int off = ring0 * vrow + vcol;
            #pragma unroll
            for (int k = 0; k < RUN; ++k) v[buf][k] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rv, off, (RUN * i + k) * vrow, 0);
        }
    };
    auto fetch_e = [&](int buf, int g, int i) {
        if constexpr (!EL) {
            g = g < ng ? g : ng - 1;
            const float *et = eb + ((size_t)(4 * g + c) * 16 + n) * ES + RUN * i;
            ev[buf][0] = *(const float4 *)et; ev[buf][1] = *(const float4 *)(et + 4);
        }
    };
    const int ndg = PHASE == 2 ? HD / 32 / gridDim.z : HD / 32, dg0 = PHASE == 2 ? blockIdx.z * ndg : 0;      // runs of 32 dims of this workgroup
    auto first_runs = [&](int dg) {
        #pragma unroll
        for (int i = 0; i < AHEAD; ++i) fetch_v((kvh * HD + dg * 32 + 2 * n) * 2, i, i >> 2, i & 3);
    };
    if (wave < ndg) first_runs(dg0 + wave);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    {   // the units' maxima over their tiles, then m -> the tile's weight exp(m - M)
        const int u = threadIdx.x & 15, k = threadIdx.x >> 4;
        float m = -INFINITY;
        for (int t = k; t < nt; t += WG / 16) m = fmaxf(m, mb[t * 16 + u]);
        mx[u][k] = m;
        __syncthreads();
        for (int i = 0; i < WG / 16; ++i) m = fmaxf(m, mx[u][i]);
        for (int t = k; t < nt; t += WG / 16) { const float v = mb[t * 16 + u]; wb[t * 16 + u] = v == -INFINITY ? 0.0f : lg_expf(v - m); }
    }
    __syncthreads();
    for (int dg = dg0 + wave; dg < dg0 + ndg; dg += NW) {
        float o[2][4], L[4];
        #pragma unroll
        for (int i = 0; i < 4; ++i) { o[0][i] = o[1][i] = 0.0f; L[i] = 0.0f; }
        const int vcol = (kvh * HD + dg * 32 + 2 * n) * 2;
        if (dg != dg0 + wave) first_runs(dg);
        #pragma unroll
        for (int i = 0; i < AHEAD; ++i) fetch_e(i, i >> 2, i & 3);
        for (int g0 = 0; g0 < ng; g0 += NB / 4) {
            #pragma unroll
            for (int h = 0; h < NB / 4; ++h) {
                const int g = g0 + h, t = 4 * g;
                if (g >= ng) break;
                float4 w4[4], l4[4];
                auto tile_weights = [&]() {
                    #pragma unroll
                    for (int b = 0; b < 4; ++b) { w4[b] = *(const float4 *)(wb + (t + b) * 16 + 4 * c); l4[b] = *(const float4 *)(lb + (t + b) * 16 + 4 * c); }
                };
                if constexpr (!EL) tile_weights();
                lg_v16f acc0 = {}, acc1 = {};
                #pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int cur = 4 * h + i;
                    fetch_v(vcol, (cur + AHEAD) % NB, g + ((i + AHEAD) >> 2), (i + AHEAD) & 3);
                    fetch_e((cur + AHEAD) % NB, g + ((i + AHEAD) >> 2), (i + AHEAD) & 3);
                    const float *et = eb + ((size_t)(t + c) * 16 + n) * ES + RUN * i;
                    const float4 ea = EL ? *(const float4 *)et : ev[EL ? 0 : cur][0], ec = EL ? *(const float4 *)(et + 4) : ev[EL ? 0 : cur][1];
                    const float e[8] = { ea.x, ea.y, ea.z, ea.w, ec.x, ec.y, ec.z, ec.w };
                    if (g == 0 || g + 1 == ng) {              // rows that no row of the group sees may hold anything (infinities too)
                        const int p = ((tfirst + t + c) << 5) + RUN * i;
                        #pragma unroll
                        for (int k = 0; k < RUN; ++k) if (p + k < kfirst || p + k > klast) v[cur][k] = 0;
                    }
                    float vl[RUN], vh[RUN];                   // (converted ahead of the run's products, as above)
                    #pragma unroll
                    for (int k = 0; k < RUN; ++k) { vl[k] = lg_h2f((uint16_t)(v[cur][k] & 0xFFFF)); vh[k] = lg_h2f((uint16_t)(v[cur][k] >> 16)); }
                    __builtin_amdgcn_sched_barrier(0);
                    #pragma unroll
                    for (int k = 0; k < RUN; ++k) {
                        acc0 = __builtin_amdgcn_mfma_f32_16x16x1f32(e[k], vl[k], acc0, 0, 0, 0);
                        acc1 = __builtin_amdgcn_mfma_f32_16x16x1f32(e[k], vh[k], acc1, 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (EL) tile_weights();
                #pragma unroll
                for (int b = 0; b < 4; ++b) {                 // tiles in order
                    const float wv[4] = { w4[b].x, w4[b].y, w4[b].z, w4[b].w }, lv[4] = { l4[b].x, l4[b].y, l4[b].z, l4[b].w };
                    #pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        L[i] = lg_fmaf(lv[i], wv[i], L[i]);
                        o[0][i] = lg_fmaf(acc0[4 * b + i], wv[i], o[0][i]);
                        o[1][i] = lg_fmaf(acc1[4 * b + i], wv[i], o[1][i]);
                    }
                }
            }
        }
        // A value that is not finite and that some row of the group does not see was a product with weight 0 for that row: a NaN.
        // So where a result of this wavefront is not finite, all of them are computed again, each from the slots its row sees.
        float odd = 0.0f;
        #pragma unroll
        for (int i = 0; i < 4; ++i) odd = lg_fmaf(o[0][i], 0.0f, lg_fmaf(o[1][i], 0.0f, odd));
        if (__builtin_amdgcn_ballot_w64(odd != 0.0f)) {
            int u0 = 4 * c;
            asm("" : "+v"(u0));                               // (else what the scores know of these units is kept in registers for here, and spills)
            int us[4], up[4];
            #pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = row0 + (u0 + i) / G;
                us[i] = lg_win_start(pos + r, a.window); up[i] = u0 + i < U && r <= rlast ? pos + r : -1;
                o[0][i] = o[1][i] = 0.0f;
            }
            for (int t = 0; t <= tlast - tfirst; ++t) {
                float acc[2][4] = {};
                const int t0 = (tfirst + t) << 5;
                for (int s = t0 < kfirst ? kfirst - t0 : 0; s < 32 && t0 + s <= klast; ++s) {
                    const uint32_t x = *(const uint32_t *)((const uint8_t *)a.vc + (size_t)((t0 + s) % a.seq) * vrow + vcol);
                    #pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (t0 + s < us[i] || t0 + s > up[i]) continue;
                        const float e = eb[((size_t)t * 16 + u0 + i) * ES + s];
                        acc[0][i] = lg_fmaf(e, lg_h2f((uint16_t)(x & 0xFFFF)), acc[0][i]);
                        acc[1][i] = lg_fmaf(e, lg_h2f((uint16_t)(x >> 16)), acc[1][i]);
                    }
                }
                #pragma unroll
                for (int i = 0; i < 4; ++i) {
                    o[0][i] = lg_fmaf(acc[0][i], wb[t * 16 + u0 + i], o[0][i]);
                    o[1][i] = lg_fmaf(acc[1][i], wb[t * 16 + u0 + i], o[1][i]);
                }
            }
        }
        #pragma unroll
        for (int i = 0; i < 4; ++i) *(float2 *)(&ob[4 * c + i][dg * 32 + 2 * n]) = make_float2(o[0][i] / L[i], o[1][i] / L[i]);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 16 * 8 * ndg; i += WG) {
        const int u = i / (8 * ndg), qd = 8 * dg0 + i - u * (8 * ndg), ur = u * gi >> 8, r = row0 + ur;
        if (u >= U || r > rlast) continue;                   // (whole groups of 8 lanes)
        lg_wide_quant4(*(const float4 *)(&ob[u][qd * 4]), a.xq, a.H * HD >> 5, r, (kvh * G + u - ur * G) * (HD / 32) + (qd >> 3));
    }
}
