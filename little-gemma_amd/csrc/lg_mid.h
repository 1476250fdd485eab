// lg_mid.h — a matrix product, the row work behind it and the product that follows as ONE launch (blocks of up to 8 rows).
//
// Between two large products of a layer lies work on a handful of rows: the residual's update, two norms, the q8 of the result.  As launches of their own the
// three are each 4 to 5 us behind the other before they move a byte of weights, and the second product's weights (17 to 66 MB at the 12B shape) wait for
// all of that.  Here 256 workgroups, one to a CU, each
//   take an equal share of the first product and hand its f32 values, 8 bytes a value and the launch's tag, through memory to the row units;
//   the last rows x E/1024 workgroups are the row units (lg_k_rows, a slice of a row each) and hand the q8 rows on (FarRows, lg_xtail.h);
//   take a share of the second product, whose weights have been on their way to registers and LDS since the first one's had arrived.
// Sums, their order and every rounding are those of the separate kernels.  Waits are bounded and reported as in lg_xtail.h.
// Bound by memory once the first product's weights are there: 12B shape, 75 MB in lg_k_o_geglu and 51 in lg_k_down_qkv, which take 18.8 and 14.0 us at one row in the
// trace, 21.7 and 17.6 at five, where the launches they replace took 4.3 + 4.3 + 11.4 and 6.5 + 7.5 (with the row work inside), 5.1 + 4.3 + 12.2 and 9.2 + 4.3 + 6.6 and their
// gaps: a step 2480 -> 2365 us, 3333 -> 3042.  Narrow models gain nothing or lose (mid_o_faster, mid_down_faster, mid_proj_faster).  What it takes for that (12B decode and five rows, us a step): a wavefront's second product's weights requested
// behind the arrival of the first one's (2578, 3131 with them ahead); without a condition around loads in flight, where the compiler waits for all of them
// (2436, 3111; 2390, 3078); three tiles at most ahead of attn_output's products, or the wavefront stands at the CU's address unit (2365, 3052); the
// second column block's tiles in LDS, so that its products run while the first one's last tiles arrive.
// With the per-layer projection of a float type in ffn_down's place (E4B shape, bf16 per-layer matrices, four rows): 2372 -> 2277.
#pragma once
#include "lg_aout.h"

#define LG_MID_E 3840               // widest row
#define LG_MID_K 4096               // widest input of attn_output
#define LG_MID_MERGE_ROWS 3         // widest block whose merge is part of lg_k_o_geglu
// Chains of pairs of K segments (host: pack_pairs): block of 16 rows, pair of segments, pairs of blocks of 32: 64 lanes x (8 + 8) nibble bytes of two blocks, signed (lane:
// row c16, half hf of its 16 bytes, segment sg of the pair), then 32 (segment, row) x two f16 scales
__host__ __device__ static inline size_t lg_pairs_bytes(int k, int m) { const int nit = k / 256, nitp = (nit + 1) & ~1; return (size_t)m / 16 * 4 * nitp * 576; }

// ---- ffn_down as the first part of a launch: 256 workgroups with an equal share of it each --------------------------------
struct DownHere {
    const uint8_t *w;               // up to 3 rows segment tiles of 32 segments, else the streams of lg_k_down_m
    const void    *act;             // q8 rows in the order of lg_act_layout, or 80-dword blocks
    int            FF, E;
    uint2         *slabs;           // [3][M][E] lg_k_down_m's quarters 1..3, tagged
    uint2         *out;             // [M][E] tagged, written through to memory
    int            spin_limit;
};
__device__ __forceinline__ void lg_put_far(uint2 *p, float v, uint32_t tag) {
    __hip_atomic_store((unsigned long long *)p, (unsigned long long)tag << 32 | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Up to 3 rows: lg_k_mm<M, 32, 1, false, 4>, two output rows to a wavefront, the same number of wavefronts in every workgroup
template <int M>
struct DownDot {
    static constexpr bool HERE = true;
    const DownHere &d; StepCtl *ctl; uint32_t number; unsigned char *smem;
    CopyBatch rows; WChunk<1, 4> first; const uint8_t *wg[1]; int row[1]; bool live;
    __device__ __forceinline__ void request() {
        const int E = d.E, groups = E >> 1, nw = (groups + 255) >> 8, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nit = d.FF >> 10, g0 = blockIdx.x * nw + wave;
        live = wave < nw && g0 < groups;
        const int gi = live ? g0 : groups - 1;
        wg[0] = d.w + (size_t)gi * nit * LG_TILE;
        row[0] = gi * 2 + (lane >> 5);
        rows = lg_load_q8_issue<M>((const int8_t *)d.act, d.FF, 512);
        if (live) lg_mm_fetch<1, 4>(first, wg, 0, nit, lane);
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void commit() {
        lg_load_q8_commit<M>(rows, (const int8_t *)d.act, d.FF, (int8_t *)smem, 512);
        __syncthreads();
    }
    __device__ __forceinline__ void finish(uint32_t tag) {
        const int E = d.E, lane = threadIdx.x & 63, c = lane & 31;
        const int8_t *lq = (const int8_t *)smem;
        if (!live) return;
        float acc[1][M];
        lg_mm_groups<M, 32, 1, false, 4>(wg, first, d.FF >> 10, lq, lg_q8_ds<M>(lq, d.FF), d.FF, acc, lane, nullptr, E, row);
        if (c < M) lg_put_far(d.out + (size_t)c * E + row[0], lg_pick<M>(acc[0], c), tag);
    }
};
// 4 to 8 rows: lg_k_down_m<M, 2, NDP>, its quarters 1..3 handing theirs to quarter 0 in one trip
template <int M, int NDP>
struct DownMfma {
    static constexpr bool HERE = true;
    static constexpr int OPS = 2;
    const DownHere &d; StepCtl *ctl; uint32_t number; unsigned char *smem;
    uint4 t0, t1, t2, t3, t4;
    struct Pair { lg_x4u q; uint32_t sw; };
    Pair w[OPS][NDP];
    __device__ __forceinline__ void request() {
        const DownMGeo g = lg_down_m_geo(d.E, d.FF);
        const int wgi = blockIdx.x, r = wgi & 63, q = wgi >> 6, lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5, s = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const uint4 *src = (const uint4 *)((const uint32_t *)d.act + (size_t)(8 * q + s) * g.nitd * LG_MU_DWORDS);
        const int nu = g.nitd * (LG_MU_DWORDS / 4);
        t0 = src[min(lane, nu - 1)]; t1 = src[min(lane + 64, nu - 1)]; t2 = src[min(lane + 128, nu - 1)]; t3 = src[min(lane + 192, nu - 1)]; t4 = src[min(lane + 256, nu - 1)];
        __builtin_amdgcn_sched_barrier(0);
        const uint8_t *sb = d.w + (size_t)(4 * r + q) * g.wg_bytes + (size_t)s * g.seg_bytes;
        #pragma unroll
        for (int o = 0; o < OPS; ++o) {
            const int vr = g.RW - 32 * o < 32 ? g.RW - 32 * o : 32, nn = n < vr ? n : vr - 1;
            const uint8_t *ob = sb + (size_t)32 * o * g.nitdp * 18;
            #pragma unroll
            for (int jp = 0; jp < NDP; ++jp) {
                const int jc = jp < g.npairs ? jp : g.npairs - 1;
                w[o][jp].q = __builtin_nontemporal_load((const lg_x4u *)(ob + (size_t)((jc * 2 + h) * vr + nn) * 16));
                w[o][jp].sw = __builtin_nontemporal_load((const uint32_t *)(ob + (size_t)g.nitdp * vr * 16 + (size_t)(jc * vr + nn) * 4));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void commit() {
        const DownMGeo g = lg_down_m_geo(d.E, d.FF);
        const int lane = threadIdx.x & 63, s = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), nu = g.nitd * (LG_MU_DWORDS / 4);
        unsigned char *la = smem + (size_t)s * (2 * NDP) * (LG_MU_DWORDS * 4);
        ((uint4 *)la)[min(lane, nu - 1)] = t0; ((uint4 *)la)[min(lane + 64, nu - 1)] = t1; ((uint4 *)la)[min(lane + 128, nu - 1)] = t2;
        ((uint4 *)la)[min(lane + 192, nu - 1)] = t3; ((uint4 *)la)[min(lane + 256, nu - 1)] = t4;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __device__ __forceinline__ void finish(uint32_t tag) {
        const DownMGeo g = lg_down_m_geo(d.E, d.FF);
        const int E = d.E, wgi = blockIdx.x, r = wgi & 63, q = wgi >> 6, t = threadIdx.x, lane = t & 63, n = lane & 31, h = lane >> 5, s = __builtin_amdgcn_readfirstlane(t >> 6);
        unsigned char *la = smem + (size_t)s * (2 * NDP) * (LG_MU_DWORDS * 4);
        float *red = (float *)(smem + (size_t)8 * (2 * NDP) * (LG_MU_DWORDS * 4));               // [8 segments][OPS][8 row slots][32]
        lg_v16i magic;
        #pragma unroll
        for (int i = 0; i < 16; ++i) magic[i] = 0x4B400000;
        asm volatile("" : "+v"(magic));
        const int arow = n < 8 ? n : 7;
        float p[OPS][4];
        #pragma unroll
        for (int o = 0; o < OPS; ++o)
            #pragma unroll
            for (int i = 0; i < 4; ++i) p[o][i] = 0.0f;
        #pragma unroll
        for (int jp = 0; jp < NDP; ++jp) {
            #pragma unroll
            for (int e = 0; e < 2; ++e) {
                if (2 * jp + e < g.nitd) {
                    const XffnAct ac = lg_xffn_act(la + (size_t)(2 * jp + e) * (LG_MU_DWORDS * 4), arow, h);
                    #pragma unroll
                    for (int o = 0; o < OPS; ++o) {
                        lg_v2u qq; qq.x = e ? w[o][jp].q.z : w[o][jp].q.x; qq.y = e ? w[o][jp].q.w : w[o][jp].q.y;
                        lg_xffn_step(ac.av, ac.xd, ac.cf, qq, lg_h2f((uint16_t)(e ? w[o][jp].sw >> 16 : w[o][jp].sw)), magic, p[o]);
                    }
                }
            }
        }
        #pragma unroll
        for (int o = 0; o < OPS; ++o)
            #pragma unroll
            for (int i = 0; i < 4; ++i) red[((size_t)(s * OPS + o) * 8 + 4 * h + i) * 32 + n] = p[o][i];
        __syncthreads();
        // the quarter's three levels of the segment tree: one output per thread (M * RW <= 8 * 64); then the top two
        if (t >= ((M * g.RW + 63) & ~63)) return;              // (whole wavefronts: lg_take)
        const bool on = t < M * g.RW;
        const int at = on ? t : M * g.RW - 1, j = at / g.RW, rr = at - j * g.RW;
        const float *b = red + ((size_t)(rr >> 5) * 8 + j) * 32 + (rr & 31);
        const size_t sg = (size_t)OPS * 8 * 32;
        const float mine = ((b[0] + b[sg]) + (b[2 * sg] + b[3 * sg])) + ((b[4 * sg] + b[5 * sg]) + (b[6 * sg] + b[7 * sg]));
        const uint32_t here = lg_tag(number, lg_xcc_id());
        uint2 *p0 = d.slabs + ((size_t)j * E + (size_t)r * g.RW + rr);
        const size_t slab = (size_t)M * E;
        if (q) { if (on) lg_put(p0 + (q - 1) * slab, mine, here); return; }
        float v[3];
        int err = 0;
        for (int spins = 0;; ++spins) {
            uint32_t diff = 0;
            #pragma unroll
            for (int i = 0; i < 3; ++i) {
                const unsigned long long x = lg_ld_l2_u64(p0 + i * slab);
                v[i] = __uint_as_float((uint32_t)x); diff |= (uint32_t)(x >> 32) ^ here;
            }
            if (__all((diff >> 4) == 0)) { if (diff) err = LG_XFFN_ERR_PLACE; break; }
            if (spins >= d.spin_limit) { err = LG_XFFN_ERR_WAIT; break; }
        }
        if (err) atomicOr(&ctl->err, err);
        if (on) lg_put_far(d.out + (size_t)j * E + (size_t)r * g.RW + rr, (mine + v[0]) + (v[1] + v[2]), tag);
    }
};

// The per-layer projection of a model that keeps its per-layer matrices in a float type (lg_k_mmf of K = 256), as the first part of such a launch: the
// same number of rows in every workgroup, up to two to a wavefront
template <int M>
struct MmfHere {
    static constexpr bool HERE = true;
    const DownHere &d; StepCtl *ctl; uint32_t number; unsigned char *smem;      // (d.w: f32 [E][256], d.act: f32 [M][256])
    float4 x[M], w[2];
    __device__ __forceinline__ int row(int i) const { const int n = (d.E + 255) >> 8, r = (int)(threadIdx.x >> 6) + 8 * i; return r < n && (int)blockIdx.x * n + r < d.E ? (int)blockIdx.x * n + r : -1; }
    __device__ __forceinline__ void request() {
        const int lane = threadIdx.x & 63;
        #pragma unroll
        for (int j = 0; j < M; ++j) x[j] = ((const float4 *)d.act)[j * 64 + lane];
        #pragma unroll
        for (int i = 0; i < 2; ++i) w[i] = ((const float4 *)d.w)[(size_t)max(row(i), 0) * 64 + lane];
    }
    __device__ __forceinline__ void commit() {}
    __device__ __forceinline__ void finish(uint32_t tag) {
        const int lane = threadIdx.x & 63;
        #pragma unroll
        for (int i = 0; i < 2; ++i) {
            float acc[M];
            #pragma unroll
            for (int j = 0; j < M; ++j) {
                acc[j] = lg_fmaf(w[i].x, x[j].x, 0.0f); acc[j] = lg_fmaf(w[i].y, x[j].y, acc[j]);
                acc[j] = lg_fmaf(w[i].z, x[j].z, acc[j]); acc[j] = lg_fmaf(w[i].w, x[j].w, acc[j]);
            }
            #pragma unroll
            for (int j = 0; j < M; ++j) acc[j] = lg_wave_sum64(acc[j]);
            if (lane < M && row(i) >= 0) lg_put_far(d.out + (size_t)lane * d.E + row(i), lg_pick<M>(acc, lane), tag);
        }
    }
};

// ---- the row work (lg_k_rows): row j of the first product's values, this unit storing and quantizing the float4s t + 256 vr --------
struct MidRowArgs {
    const float *x, *w_post, *os, *w_pre;
    float       *x_out;
    const uint2 *in;                // [M][E] tagged
    FarRows     *rows;
    int          E, spin_limit;
    float        eps;
};
struct MidRow {
    float4 x[LG_ROWV], w1[LG_ROWV], w2[LG_ROWV];
    float os;
    __device__ __forceinline__ void request(const MidRowArgs &a, int j, int t) {
        const int nq = a.E >> 2;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) {                    // (clamped: under a condition each the loads are waited for one by one)
            const int at = min(t + 256 * v, nq - 1);
            x[v] = ((const float4 *)(a.x + (size_t)j * a.E))[at]; w1[v] = ((const float4 *)a.w_post)[at]; w2[v] = ((const float4 *)a.w_pre)[at];
        }
        os = a.os ? a.os[0] : 1.0f;
    }
    float4 dv[LG_ROWV];
    // (loads that the compiler knows of: behind the weights that are on their way it waits for its own and no others)
    __device__ __forceinline__ void take(const MidRowArgs &a, StepCtl *ctl, int j, bool first, bool rowt, int t, uint32_t tag) {
        const int E = a.E, nq = E >> 2;
        if (rowt) {
            const __amdgpu_buffer_rsrc_t r = lg_buffer_rsrc(a.in);
            lg_x4u v[2 * LG_ROWV];
            int err = 0;
            for (int spins = 0;; ++spins) {
                #pragma unroll
                for (int i = 0; i < 2 * LG_ROWV; ++i) v[i] = __builtin_bit_cast(lg_x4u, __builtin_amdgcn_raw_buffer_load_b128(r, (j * E + 4 * min(t + 256 * (i >> 1), nq - 1)) * 8 + (i & 1) * 16, 0, 16));
                uint32_t diff = 0;
                #pragma unroll
                for (int i = 0; i < 2 * LG_ROWV; ++i) diff |= (v[i].y ^ tag) | (v[i].w ^ tag);
                if (__all(diff == 0)) break;
                if (spins >= a.spin_limit) { err = LG_XFFN_ERR_WAIT; break; }
                asm volatile("" ::: "memory");
            }
            #pragma unroll
            for (int i = 0; i < LG_ROWV; ++i) dv[i] = lg_units_float4(v[2 * i], v[2 * i + 1]);
            if (err) atomicOr(&ctl->err, err);
        }
        if (first && t == 0) lg_put_soon(a.rows, tag);
    }
    __device__ __forceinline__ void work(const MidRowArgs &a, int j, int vr, bool rowt, int t, float *red0, float *red1, uint32_t tag) {
        const int E = a.E, nq = E >> 2;
        float ss = 0.0f;
        if (rowt) {
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(dv[v], ss);
        }
        ss = lg_block_sum256_of512(ss, red0);
        float sc = 1.0f / sqrtf(ss / (float)E + a.eps);
        ss = 0.0f;
        if (rowt) {
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
                const float4 w = w1[v];
                float4 r;
                r.x = x[v].x + dv[v].x * sc * w.x;  r.y = x[v].y + dv[v].y * sc * w.y;
                r.z = x[v].z + dv[v].z * sc * w.z;  r.w = x[v].w + dv[v].w * sc * w.w;
                if (a.os) { r.x = r.x * os; r.y = r.y * os; r.z = r.z * os; r.w = r.w * os; }
                x[v] = r;
                if (v == vr) ((float4 *)(a.x_out + (size_t)j * E))[t + 256 * v] = r;
                ss = lg_sumsq4(r, ss);
            }
        }
        ss = lg_block_sum256_of512(ss, red1);
        sc = 1.0f / sqrtf(ss / (float)E + a.eps);
        if (!rowt) return;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) {
            if (t + 256 * v >= nq || v != vr) continue;
            const float4 w = w2[v], h = make_float4(x[v].x * sc * w.x, x[v].y * sc * w.y, x[v].z * sc * w.z, x[v].w * sc * w.w);
            float d; int sum;
            const uint32_t packed = lg_quant4_8lanes(h, &d, &sum);
            lg_put_far_q8(a.rows, E, j, t + 256 * v, packed, d, tag);
        }
    }
};

// ---- ffn_down, the row work behind it and the next layer's q/k/v projections ----------------------------------------------
struct DownQkvArgs {
    DownHere      d;
    MidRowArgs    r;
    const uint8_t *qw;              // pack_pairs
    float         *qout;            // [M][qm]
    int            qm, seq;
};
#define LG_DOWNQKV_FIELDS(X, v) X(const uint8_t *, dw, d.w, v) X(const void *, dact, d.act, v) X(int, dFF, d.FF, v) X(int, E, d.E, v) X(uint2 *, dslabs, d.slabs, v) X(uint2 *, dout, d.out, v) \
    X(int, seq, seq, v) X(int, spin_limit, d.spin_limit, v) X(const float *, x, r.x, v) X(const float *, w_post, r.w_post, v) X(const float *, os, r.os, v) X(const float *, w_pre, r.w_pre, v) \
    X(float *, x_out, r.x_out, v) X(FarRows *, rows, r.rows, v) X(float, eps, r.eps, v) X(const uint8_t *, qw, qw, v) X(float *, qout, qout, v) X(int, qm, qm, v)
#define LG_MID_NIT 15               // most blocks of a segment of a row: LG_MID_E / 256, and of ffn_down: FF <= 15360
#define LG_MID_NDP 8
// LDS: the rows of the second product, a block of zeros to each of theirs, sums; then ffn_down's
#define LG_DOWNQKV_ACT ((size_t)8 * LG_MID_NIT * LG_FAR_BLK + LG_MID_NIT * LG_FAR_BLK + 8 * 8 * 32 * 4)
static inline size_t lg_downqkv_lds(int M, int FF) { return LG_DOWNQKV_ACT + (M >= 4 ? (size_t)8 * 2 * LG_MID_NDP * LG_MU_DWORDS * 4 + 8 * 2 * 8 * 32 * 4 : (size_t)M * FF * 5 / 4); }
template <int M, bool MMF>           // MMF: the first product is the per-layer projection of a float type
__global__ __launch_bounds__(512) void lg_k_down_qkv(StepCtl *ctl, LG_DOWNQKV_FIELDS(LG_XP, _) int p_end_) {
    constexpr int NIT = LG_MID_NIT, NP = (NIT + 1) / 2, BLK = LG_FAR_BLK, I = (M + 1) / 2;
    DownQkvArgs a; LG_DOWNQKV_FIELDS(LG_XI, a)
    a.r.E = a.d.E; a.r.spin_limit = a.d.spin_limit; a.r.in = a.d.out;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float red[2][8];
    const int t = threadIdx.x, lane = t & 63, c16 = lane & 15, hf = (lane >> 4) & 1, sg = lane >> 5, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int E = a.d.E, nit = E >> 8, nitp = (nit + 1) & ~1, slices = (E + 1023) >> 10, u = gridDim.x - 1 - blockIdx.x;
    const uint32_t number = ctl->launch + (uint32_t)a.seq, tag = lg_tag(number, 0);
    std::conditional_t<MMF, MmfHere<M>, std::conditional_t<(M >= 4), DownMfma<M, LG_MID_NDP>, DownDot<M>>> down{ a.d, ctl, number, smem + LG_DOWNQKV_ACT };
    const bool unit = u < M * slices, rowt = unit && t < 256;
    down.request();
    down.commit();
    const int j = u % M, vr = u / M;
    MidRow row;
    if (rowt) row.request(a.r, j, t);
    unsigned char *zero = smem + (size_t)8 * NIT * BLK;
    float *xch = (float *)(zero + NIT * BLK);                  // [8 segments][8 rows][32]
    for (int i = t; i < NIT * BLK / 16; i += 512) ((uint4 *)zero)[i] = make_uint4(0, 0, 0, 0);
    const bool mine = 32 * (int)blockIdx.x < a.qm;
    lg_x4u q[NP]; uint32_t s[NP];
    __builtin_amdgcn_sched_barrier(0);
    down.finish(tag);
    // (the projections' weights, behind ffn_down's: ahead of them they keep every share late.  Without a condition: what is loaded under one is waited for where it ends)
    const uint8_t *cb = a.qw + ((size_t)(2 * min((int)blockIdx.x, (a.qm >> 5) - 1) + (wave & 1)) * 4 + (wave >> 1)) * nitp * 576;
    #pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int at = 2 * i < nit ? i : 0;
        q[i] = __builtin_nontemporal_load((const lg_x4u *)(cb + (size_t)(at * 64 + lane) * 16));
        s[i] = __builtin_nontemporal_load((const uint32_t *)(cb + (size_t)nitp * 512 + (size_t)(at * 32 + sg * 16 + c16) * 4));
    }
    if (unit) {
        row.take(a.r, ctl, j, u == 0, rowt, t, tag);
        row.work(a.r, j, vr, rowt, t, red[0], red[1], tag);
    }
    if (!mine) return;
    // ---- 32 rows of the projections: wavefront (pair of segments, 16 rows) ----
    int err = lg_wait_soon(a.r.rows, tag, a.r.spin_limit);
    err |= lg_take_far_segment<M, NIT>(a.r.rows, E, nit, wave, lane, smem + (size_t)wave * NIT * BLK, tag, a.r.spin_limit);
    if (err) atomicOr(&ctl->err, err);
    __syncthreads();
    const int seg = (wave >> 1) * 2 + sg;
    const unsigned char *ls = smem + (size_t)seg * NIT * BLK, *la = ((lane >> 3) & 1) == sg ? ls + (lane & 7) * 32 + hf * 16 : zero;
    lg_v4i magic = { LG_FAR_MAGIC, LG_FAR_MAGIC, LG_FAR_MAGIC, LG_FAR_MAGIC };
    asm volatile("" : "+v"(magic));
    float xd[I], p[I];
    #pragma unroll
    for (int r = 0; r < I; ++r) { xd[r] = *(const float *)(ls + (c16 < NIT ? c16 : 0) * BLK + 256 + (4 * hf + r) * 4); p[r] = 0.0f; }
    lg_unroll<NIT>([&](auto i_) {
        constexpr int i = decltype(i_)::value;
        const lg_v4i av = *(const lg_v4i *)(la + i * BLK);
        const lg_v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, lg_far_weights(i & 1 ? q[i >> 1].z : q[i >> 1].x, i & 1 ? q[i >> 1].w : q[i >> 1].y), magic, 0, 0, 0);
        const float dw = lg_h2f((uint16_t)(i & 1 ? s[i >> 1] >> 16 : s[i >> 1]));
        #pragma unroll
        for (int r = 0; r < I; ++r) {
            const float v = lg_fmaf(lg_row_bcast<i>(xd[r]) * dw, __int_as_float(d[r]) - LG_FAR_BIAS, p[r]);
            p[r] = i < nit ? v : p[r];
        }
    });
    #pragma unroll
    for (int i = 0; i < I; ++i) xch[(seg * 8 + 2 * i + hf) * 32 + (wave & 1) * 16 + c16] = p[i];
    __syncthreads();
    if (t < 32 * M) {                                          // the adjacent-pair tree over the 8 segments
        const float *z = xch + t;
        a.qout[(size_t)(t >> 5) * a.qm + blockIdx.x * 32 + (t & 31)] = ((z[0] + z[256]) + (z[512] + z[768])) + ((z[1024] + z[1280]) + (z[1536] + z[1792]));
    }
}

// ---- attn_output, the row work behind it, gate/up and the GeGLU --------------------------------------------------------------
struct OGegluArgs {
    const uint8_t *ow;              // pack_pairs
    const int8_t  *act;             // q8 rows of attention, order of lg_act_layout
    uint2         *out;             // [M][E] attn_output's values, tagged
    MidRowArgs    r;
    const uint8_t *gw;              // row-block tiles
    int8_t        *gq;
    int            qd, nff, gq_units, seq;
    MergeArgs      g;               // MG: attention's partials (xq, xf are not used),
    FarRows       *arows;           // the rows they become
    int            tiles;           // and the most tiles that a row can see
};
#define LG_OGEGLU_FIELDS(X, v) X(const int8_t *, act, act, v) X(const uint8_t *, ow, ow, v) X(int, qd, qd, v) X(int, E, r.E, v) X(const uint8_t *, gw, gw, v) X(int, nff, nff, v) X(int, seq, seq, v) \
    X(uint2 *, out, out, v) X(const float *, x, r.x, v) X(const float *, w_post, r.w_post, v) X(const float *, os, r.os, v) X(const float *, w_pre, r.w_pre, v) X(float *, x_out, r.x_out, v) \
    X(FarRows *, rows, r.rows, v) X(float, eps, r.eps, v) X(int, spin_limit, r.spin_limit, v) X(int8_t *, gq, gq, v) X(int, gq_units, gq_units, v) \
    X(const float *, pm, g.pm, v) X(const float *, pl, g.pl, v) X(const float *, pacc, g.pacc, v) X(int, tiles_max, g.tiles_max, v) X(int, H, g.H, v) X(int, hd, g.hd, v) \
    X(int, window, g.window, v) X(FarRows *, arows, arows, v) X(int, tiles, tiles, v)
#define LG_OG_AHEAD 3                // ... of the column block that comes first: ahead of attn_output's products
#define LG_OG_EARLY 5               // blocks of the first column block's tiles that are requested ahead of the rows
#define LG_OG_LT 12                 // blocks of a segment of the second column block that wait in LDS (the others in registers)
#define LG_OG_ACT(NIT) ((size_t)9 * 16 * LG_FAR_BLK > (size_t)9 * (NIT) * LG_FAR_BLK ? (size_t)9 * 16 * LG_FAR_BLK : (size_t)9 * (NIT) * LG_FAR_BLK)
#define LG_OG_LDS(NIT) (LG_OG_ACT(NIT) + (size_t)8 * ((NIT) < LG_OG_LT ? (NIT) : LG_OG_LT) * LG_TILE + 8192)
#define LG_OG_BLOCKS (2 * LG_XCDS * LG_XCD_WGS - 32)      // two blocks of 32 FFN columns for each workgroup, one for the row units (8 rows x 4 slices)
static_assert((size_t)9 * 16 * LG_FAR_BLK >= 2 * 8 * 8 * 64 * 4, "the sums of two column blocks take the rows' place");
// MG (up to LG_MID_MERGE_ROWS rows): the merge of attention's partials (lg_k_attn_merge) is part of the launch too, 64 dims of a row by a wavefront, a workgroup
// each; the q8 is handed over as the rows are.  12B shape at 3001, one to five rows, us a step: 2322 -> 2245, 2495 -> 2413, 2635 -> 2565, 2715 -> 2704, 2855 -> 2855
// (the launch 18.8 -> 21.4 at one row in the trace, the 4.3 of the merge and its gap gone; at five, by events, 20.6 -> 24.4, where 256 workgroups pull 31 KB of q8 each and a merge takes 4.9).
// One row: gate/up's first tiles requested ahead of the q8 2276, `soon` put behind the q8 2255.
template <int M, int NIT, bool MG>
__global__ __launch_bounds__(512) void lg_k_o_geglu(StepCtl *ctl, LG_OGEGLU_FIELDS(LG_XP, _) int p_end_) {
    constexpr int BLK = LG_FAR_BLK, I = (M + 1) / 2, LT = NIT < LG_OG_LT ? NIT : LG_OG_LT;
    OGegluArgs a; LG_OGEGLU_FIELDS(LG_XI, a)
    a.r.in = a.out;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float red2[2][8];
    const int t = threadIdx.x, lane = t & 63, c16 = lane & 15, hf = (lane >> 4) & 1, sg = lane >> 5, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int E = a.r.E, nb = E >> 5, nit = nb >> 3, nblk = a.nff >> 5, slices = (E + 1023) >> 10, u = gridDim.x - 1 - blockIdx.x;
    const uint32_t tag = lg_tag(ctl->launch + (uint32_t)a.seq, 0);
    unsigned char *tiles = smem + LG_OG_ACT(NIT) + (size_t)wave * LT * LG_TILE;
    float *hand = (float *)(smem + LG_OG_ACT(NIT) + (size_t)8 * LT * LG_TILE), *sums = hand + 1024;
    const int sp = wave >> 1, lower = wave & 1, seg = sp * 2 + sg;
    const bool unit = u < M * slices, rowt = unit && t < 256;
    const int K = a.qd, na = K >> 8, nh = na >> 1, nbk = K >> 5;          // blocks of a segment, of half of it (even)
    const int j0 = u % M, vr = u / M;
    const int mrow = K >> 6, mj = (int)blockIdx.x / mrow, mu = (int)blockIdx.x - mj * mrow;
    const bool merges = MG && wave == 0 && (int)blockIdx.x < M * mrow;
    AoutMerge<LG_AOUT_TILES> part[1];
    AttnOutArgs ma;
    ma.g = a.g; ma.tiles = a.tiles;
    if (merges) part[0].request(ma, mu, mj, lane);
    MidRow row;
    if (rowt) row.request(a.r, j0, t);
    const int rb = min((int)blockIdx.x, (E >> 4) - 1);         // (workgroups without a share take the last one once more: no conditions, see lg_k_down_qkv)
    constexpr int NU = (M * (LG_MID_K / 16) + 511) / 512, NS = (M * (LG_MID_K / 32) + 511) / 512;
    uint4 au[NU]; float as[NS];
    lg_x4u ow[4]; uint32_t os[4];
    {
        if constexpr (!MG) {
            #pragma unroll
            for (int i = 0; i < NU; ++i) au[i] = ((const uint4 *)a.act)[min(t + 512 * i, M * (K >> 4) - 1)];
            #pragma unroll
            for (int i = 0; i < NS; ++i) as[i] = lg_q8_ds<M>(a.act, K)[min(t + 512 * i, M * nbk - 1)].x;
        }
        const uint8_t *cb = a.ow + ((size_t)rb * 4 + sp) * na * 576;
        #pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int at = lower * (nh >> 1) + (2 * i < nh ? i : 0);
            ow[i] = __builtin_nontemporal_load((const lg_x4u *)(cb + (size_t)(at * 64 + lane) * 16));
            os[i] = __builtin_nontemporal_load((const uint32_t *)(cb + (size_t)na * 512 + (size_t)(at * 32 + sg * 16 + c16) * 4));
        }
    }
    // ---- request: the first column block's tiles to come (the second one's, where there are two) ----
    const int rank = blockIdx.x, b1 = rank + gridDim.x;
    const bool mine = rank < nblk, two = b1 < nblk;
    const int first = two ? b1 : mine ? rank : nblk - 1;
    uint4 q[NIT], q2[NIT - LT + 1]; uint16_t sh[NIT]; uint32_t sc[NIT], sc2[NIT - LT + 1];
    // (lg_aout_geglu.  A row unit's weights behind its row would keep the row: its loads ahead of that are of one line, and it requests its block once the row is there)
    int far = !unit;
    auto fetch = [&](int b, int i) {
        const __amdgpu_buffer_rsrc_t rw = lg_buffer_rsrc(a.gw + (size_t)b * nb * LG_TILE);
        const int at = far * seg * nit * LG_TILE, r = far * (lower * 32 + (lane & 31)), it = __builtin_amdgcn_readfirstlane(far * (i < nit ? i : nit - 1)) * LG_TILE;
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rw, at + r * 16, it, 2);
        q[i] = make_uint4(v[0], v[1], v[2], v[3]);
        sh[i] = __builtin_amdgcn_raw_buffer_load_b16(rw, at + 1024 + r * 2, it, 2);
    };
    auto trade = [&](int i) {
        const lg_v2u s0 = __builtin_amdgcn_permlane16_swap(q[i].x, q[i].z, false, false), s1 = __builtin_amdgcn_permlane16_swap(q[i].y, q[i].w, false, false);
        const lg_v2u sd = __builtin_amdgcn_permlane16_swap(sh[i], sh[i], false, false);
        q[i] = make_uint4(s0.x ^ 0x88888888u, s1.x ^ 0x88888888u, s0.y ^ 0x88888888u, s1.y ^ 0x88888888u);
        sc[i] = (sd.x & 0xFFFF) | sd.y << 16;
    };
    // ---- attn_output: wavefront (pair of segments, half of their blocks) ----
    lg_v4i magic = { LG_FAR_MAGIC, LG_FAR_MAGIC, LG_FAR_MAGIC, LG_FAR_MAGIC };
    asm volatile("" : "+v"(magic));
    {
        unsigned char *zero = smem + (size_t)8 * 16 * BLK;
        for (int i = t; i < 8 * BLK / 16; i += 512) ((uint4 *)zero)[i] = make_uint4(0, 0, 0, 0);
        if constexpr (MG) {
            if (merges) {
                float v[1], d;
                int sum;
                lg_aout_merge(part, ma, ctl->pos, mj, lane, v);
                asm volatile("" : "+v"(v[0]));
                if (blockIdx.x == 0 && lane == 0) lg_put_soon(a.arows, tag);
                lg_put_far_dims(a.arows, K, mj, mu, lane, lg_quant1_32lanes(v[0], &d, &sum), d, tag);
            }
            int err = lg_wait_soon(a.arows, tag, a.r.spin_limit);
            err |= lg_take_far_segment<M, 16>(a.arows, K, na, wave, lane, smem + (size_t)wave * 16 * BLK, tag, a.r.spin_limit);
            if (err) atomicOr(&ctl->err, err);
        } else {
            #pragma unroll
            for (int i = 0; i < NU; ++i) {                     // (what is past the rows is their last unit once more)
                const int at = min(t + 512 * i, M * (K >> 4) - 1), j = at / (K >> 4), p = at - j * (K >> 4);
                unsigned char *o = smem + (size_t)((p & 7) * 16 + (p >> 4)) * BLK + lg_far_slot(j) * 32 + ((p >> 3) & 1) * 8;
                *(uint2 *)o = make_uint2(au[i].x, au[i].y); *(uint2 *)(o + 16) = make_uint2(au[i].z, au[i].w);
            }
            #pragma unroll
            for (int i = 0; i < NS; ++i) {
                const int at = min(t + 512 * i, M * nbk - 1), j = at / nbk, p = at - j * nbk;
                *(float *)(smem + (size_t)((p & 7) * 16 + (p >> 3)) * BLK + 256 + lg_far_slot(j) * 4) = as[i];
            }
        }
        __syncthreads();
        #pragma unroll
        for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(ow[i]), "+v"(os[i]));
        __builtin_amdgcn_sched_barrier(0);
        #pragma unroll
        for (int i = 0; i < LG_OG_AHEAD; ++i) fetch(first, i); // (ahead of that the rows and attn_output's weights would wait for them; more, and the wavefront waits
                                                               // for the CU's address unit to take them)
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char *ls = smem + (size_t)(seg * 16 + lower * nh) * BLK, *la = ((lane >> 3) & 1) == sg ? ls + (lane & 7) * 32 + hf * 16 : zero;
        float xd[I], p[I], fd[8][I];
        #pragma unroll
        for (int r = 0; r < I; ++r) { xd[r] = *(const float *)(ls + (c16 < nh ? c16 : 0) * BLK + 256 + (4 * hf + r) * 4); p[r] = 0.0f; }
        #pragma unroll
        for (int i = 0; i < 8; ++i) {
            const lg_v4i av = *(const lg_v4i *)(la + (i < nh ? i : 0) * BLK);
            const lg_v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, lg_far_weights(i & 1 ? ow[i >> 1].z : ow[i >> 1].x, i & 1 ? ow[i >> 1].w : ow[i >> 1].y), magic, 0, 0, 0);
            #pragma unroll
            for (int r = 0; r < I; ++r) fd[i][r] = __int_as_float(d[r]) - LG_FAR_BIAS;
        }
        auto chain = [&]() {
            lg_unroll<8>([&](auto i_) {
                constexpr int i = decltype(i_)::value;
                const float dw = lg_h2f((uint16_t)(i & 1 ? os[i >> 1] >> 16 : os[i >> 1]));
                #pragma unroll
                for (int r = 0; r < I; ++r) { const float v = lg_fmaf(lg_row_bcast<i>(xd[r]) * dw, fd[i][r], p[r]); p[r] = i < nh ? v : p[r]; }
            });
        };
        if (!lower) {
            chain();
            #pragma unroll
            for (int r = 0; r < I; ++r) hand[(sp * 4 + r) * 64 + lane] = p[r];
        }
        __syncthreads();
        if (lower) {
            #pragma unroll
            for (int r = 0; r < I; ++r) p[r] = hand[(sp * 4 + r) * 64 + lane];
            chain();
            #pragma unroll
            for (int r = 0; r < I; ++r) sums[(seg * 8 + 2 * r + hf) * 16 + c16] = p[r];
        }
        __syncthreads();
        if (t < 16 * M && rb == (int)blockIdx.x) {              // the adjacent-pair tree over the 8 segments
            const float *z = sums + t;
            lg_put_far(a.out + (size_t)(t >> 4) * E + blockIdx.x * 16 + (t & 15), ((z[0] + z[128]) + (z[256] + z[384])) + ((z[512] + z[640]) + (z[768] + z[896])), tag);
        }
    }
    #pragma unroll
    for (int i = LG_OG_AHEAD; i < NIT; ++i) fetch(first, i);
    __builtin_amdgcn_sched_barrier(0);
    if (unit) {
        row.take(a.r, ctl, j0, u == 0, rowt, t, tag);
        far = 1;
        #pragma unroll
        for (int i = 0; i < NIT; ++i) fetch(first, i);
        row.work(a.r, j0, vr, rowt, t, red2[0], red2[1], tag);
    }
    if (!mine) return;
    if (two) {                                                 // the second block to LDS; the first tiles of the first one follow it at once
        #pragma unroll
        for (int i = 0; i < NIT; ++i) {
            trade(i);
            if (i < LT) { *(uint4 *)(tiles + i * LG_TILE + lane * 16) = q[i]; if (!hf) *(uint32_t *)(tiles + i * LG_TILE + 1024 + (sg * 16 + c16) * 4) = sc[i]; }
            else { q2[i - LT] = q[i]; sc2[i - LT] = sc[i]; }
            if (i < LG_OG_EARLY) fetch(rank, i);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();                                           // (attn_output's rows in LDS are done with)
    unsigned char *zero = smem + (size_t)8 * NIT * BLK;
    for (int i = t; i < NIT * BLK / 16; i += 512) ((uint4 *)zero)[i] = make_uint4(0, 0, 0, 0);
    int err = lg_wait_soon(a.r.rows, tag, a.r.spin_limit);
    // (loads return in order: the rows are requested ahead of the first block's other tiles, which then need not have arrived)
    err |= lg_take_far_segment<M, NIT>(a.r.rows, E, nit, wave, lane, smem + (size_t)wave * NIT * BLK, tag, a.r.spin_limit, [&] {
        if (two) {
            #pragma unroll
            for (int i = LG_OG_EARLY; i < NIT; ++i) fetch(rank, i);
        }
    });
    if (err) atomicOr(&ctl->err, err);
    __syncthreads();
    const unsigned char *ls = smem + (size_t)seg * NIT * BLK, *la = ((lane >> 3) & 1) == sg ? ls + (lane & 7) * 32 + hf * 16 : zero;
    float xd[I], p[2][2][I];                                   // [block][16 columns][row 2i + hf]
    #pragma unroll
    for (int r = 0; r < I; ++r) xd[r] = *(const float *)(ls + (c16 < NIT ? c16 : 0) * BLK + 256 + (4 * hf + r) * 4);
    #pragma unroll
    for (int i = 0; i < 4 * I; ++i) p[i / (2 * I)][i / I % 2][i % I] = 0.0f;
    auto chain = [&](auto second, auto whole) {
        lg_unroll<NIT>([&](auto i_) {
            constexpr int i = decltype(i_)::value, B = decltype(second)::value;
            const lg_v4i av = *(const lg_v4i *)(la + i * BLK);
            auto join = [&](const lg_v4i &d, float dw, float (&z)[I]) {
                #pragma unroll
                for (int r = 0; r < I; ++r) {
                    const float v = lg_fmaf(lg_row_bcast<i>(xd[r]) * dw, __int_as_float(d[r]) - LG_FAR_BIAS, z[r]);
                    z[r] = decltype(whole)::value || i < nit ? v : z[r];
                }
            };
            uint4 w; uint32_t dw;
            if constexpr (!B) { trade(i); w = q[i]; dw = sc[i]; }
            else if constexpr (i < LT) { w = *(const uint4 *)(tiles + i * LG_TILE + lane * 16); dw = *(const uint32_t *)(tiles + i * LG_TILE + 1024 + (sg * 16 + c16) * 4); }
            else { w = q2[i - LT]; dw = sc2[i - LT]; }
            const lg_v4i d0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, lg_far_weights(w.x, w.y), magic, 0, 0, 0), d1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, lg_far_weights(w.z, w.w), magic, 0, 0, 0);
            join(d0, lg_h2f((uint16_t)dw), p[B][0]); join(d1, lg_h2f((uint16_t)(dw >> 16)), p[B][1]);
        });
    };
    if (nit == NIT) { if (two) chain(std::integral_constant<int, 1>{}, std::true_type{}); chain(std::integral_constant<int, 0>{}, std::true_type{}); }
    else            { if (two) chain(std::integral_constant<int, 1>{}, std::false_type{}); chain(std::integral_constant<int, 0>{}, std::false_type{}); }
    __syncthreads();                                           // (the sums take the rows' place)
    float (*red)[8][8][64] = (float (*)[8][8][64])smem;        // [block][segment][row][gate 32, up 32]
    #pragma unroll
    for (int o = 0; o < 2; ++o)
        #pragma unroll
        for (int i = 0; i < I; ++i) { red[o][seg][2 * i + hf][lower * 32 + c16] = p[o][0][i]; red[o][seg][2 * i + hf][lower * 32 + 16 + c16] = p[o][1][i]; }
    __syncthreads();
    lg_far_geglu_out<M>(red, two, rank, b1, t, a.gq, a.gq_units, a.nff);
}
