// lg_xtail.h — the narrow end of a layer as ONE launch that runs on ONE XCD (verify blocks, models with per-layer inputs).
//
// After ffn_down a layer with per-layer inputs still has three dependent steps, each of them a handful of workgroups
// and a kernel of its own when launched separately:
//   1  rows + PLE gate   x += rmsnorm(ffn_down) * w ; q8(x) ; gelu(inp_gate . q8(x)) * per-layer input ; q8    (ple/32 x M workgroups)
//   2  PLE projection    proj . that q8 row: [E] outputs of K = ple                                              (E x ple weights: 0.37 MB)
//   3  rows              x = (x + rmsnorm(2) * w) * out_scale ; q8(rmsnorm(x) * next norm weight)               (M rows)
// None of them can use the chip: what they cost is a kernel boundary each (the gap to the predecessor's end plus the
// first trip of the predecessor's data through the memory-side cache).  The workgroups of one XCD share an L2, and a
// hand-over through it costs a fraction of a boundary (lg_xcd.h).  So the three run as the phases of one kernel on the
// U = ple/32 x M workgroups i of the launch with i % 8 == 0 (the dispatcher deals workgroups to the XCDs in turn: one
// XCD gets them all; the other 7U workgroups of the launch leave at once):
//   phase 1 is lg_k_rows_plegate's body for unit (gate block, row); the unit keeps the updated residual row in registers;
//   hand-over (the M x ple gated values, which every unit quantizes) ;
//   phase 2: the E/8 row groups of the projection dealt over the 4U wavefronts, weights requested at kernel start
//   (they depend on nothing and are in registers long before the hand-over);
//   hand-over (the [M][E] f32 outputs) ;
//   phase 3: lg_k_rows' work for row j, by the units (v, j) of the row's first E/1024 gate blocks: each forms the row's
//   sums and stores and quantizes the float4s t + 256 v of every lane (the slices of lg_k_rows).
// Sums and quantization are the ones of the separate kernels, lane for lane: the results are bit-identical.
// A hand-over is one trip: every 8 bytes are a float and the launch's tag, stored together, and the reader loads them until
// the tag is there (lg_take).  With a flag behind the acknowledged stores and the data loaded behind the flag it was four
// trips, 1.25 us a hand-over at the E4B shape of 5 rows against 1.0, and 0.45 at one row; the launch 9.2 -> 8.3 us, 7.7 -> 6.5 at one
// row (there also for the wavefronts without gate rows, which no longer request any), a step 2193 -> 2156 and 1832 -> 1776 us.
// The other 7U workgroups of lg_k_ple_tail_s are the next layer's q/k/v projections (TailQkv): their weights are in registers when the rows leave the one
// XCD (FarRows, 0.9 us from the last unit's store to the last workgroup's LDS), and what was a launch of its own behind this one is 2 us of it: by the stamps five
// rows are there at 8.3 us, taken at 9.4, multiplied at 10.5.  Steps of the E4B shape, one row 1759 -> 1731 us, four 2009 -> 1938, five 2115 -> 2058,
// eight at 20011 2502 -> 2409.  On v_dot4 from four rows on (every row group reads the rows from LDS again): 2100 and 2504; the tail on all eight XCDs at once, so
// that each has its rows in its own L2: its first phase takes 5.5 us for 4.2, 2168 and 2264 (eight at 777, for 2262).
// The tag carries the writer's XCD id; a unit that sees another id, or gives up a bounded wait, reports it in
// StepCtl.err and goes on, so the kernel always ends and the host refuses the step.
#pragma once
#include <type_traits>
#include "lg_kernels.h"
#include "lg_fused.h"
#include "lg_xcd.h"
#include "lg_xffn.h"
#include "lg_far.h"

#define LG_XTAIL_UNITS 64           // most units of a launch (lane i of a wavefront polls flag i)
struct XtailSync {
    uint32_t flags[2][LG_XTAIL_UNITS];      // lg_k_attn_tail: lg_tag of each unit's last arrival
};

// q8 rows that a launch hands from its one XCD to the workgroups on the other seven, in units of 16 bytes, three dwords and the launch's marks (lg_far.h).  Stored and
// loaded with an agent's scope: through the writer's L2 to memory, and around the reader's.  A block of 32 values is three units, its 8 dwords and its scale.  On v_dot4
// (lg_take_far) the sum of the values is added up by the reader; on the matrix cores weights are signed and none is needed.
struct FarRows {
    uint2 soon;                     // {-, tag}: the rows are on their way, from here on the waiting workgroups load them until they are there
    uint2 pad[15];
    uint4 u[LG_HIP_MAX_ROWS_DEV * LG_MAXK_FAR / 32 * 3];
};
__device__ __forceinline__ uint32_t lg_far_tag(uint32_t tag) { return tag & ~15u; }      // (the reader is on another XCD)
__device__ __forceinline__ void lg_put_soon(FarRows *f, uint32_t tag) {
    __hip_atomic_store((unsigned long long *)&f->soon, (unsigned long long)tag << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A lane's four values (quad of row j) of a block that 8 lanes hold, d: its scale
__device__ __forceinline__ void lg_put_far_q8(FarRows *f, int k, int j, int quad, uint32_t packed, float d, uint32_t tag) {
    const uint32_t b = (uint32_t)lg_dpp_i<0x101>((int)packed), c = (uint32_t)lg_dpp_i<0x102>((int)packed);      // (row_shl: of the next lane and the one behind it)
    const int dw = quad & 7;
    if (dw % 3) return;                                        // lanes 0, 3 and 6 store
    const uint32_t z = dw == 6 ? __float_as_uint(d) : c;
    const __amdgpu_buffer_rsrc_t r = lg_buffer_rsrc(f->u);
    const lg_x4u v = lg_far_unit<lg_x4u>(packed, b, z, lg_far_marks(tag));
    __builtin_amdgcn_raw_buffer_store_b128(v, r, ((j * (k >> 5) + (quad >> 3)) * 3 + dw / 3) * 16, 0, 16);      // (16: the scope bit sc1)
}
// 64 values of row j (dims 64 u + lane) as q8 q, d their block's scale
__device__ __forceinline__ void lg_put_far_dims(FarRows *f, int k, int j, int u, int lane, int q, float d, uint32_t tag) {
    const uint32_t word = (uint32_t)(lg_dpp_i<0x00>(q) & 255) | (uint32_t)(lg_dpp_i<0x55>(q) & 255) << 8 | (uint32_t)(lg_dpp_i<0xAA>(q) & 255) << 16 | (uint32_t)lg_dpp_i<0xFF>(q) << 24;
    const int l = lane < 6 ? lane : 5, b = l / 3, e = l - 3 * b, at = b * 32 + e * 12;          // lanes 0 .. 5 store a unit each
    const uint32_t x = __shfl(word, at), y = __shfl(word, at + 4), w = __shfl(word, e < 2 ? at + 8 : at), s = __float_as_uint(__shfl(d, at)), z = e < 2 ? w : s;
    const __amdgpu_buffer_rsrc_t r = lg_buffer_rsrc(f->u);
    const lg_x4u v = lg_far_unit<lg_x4u>(x, y, z, lg_far_marks(tag));
    if (lane < 6) __builtin_amdgcn_raw_buffer_store_b128(v, r, ((j * (k >> 5) + 2 * u + b) * 3 + e) * 16, 0, 16);
}
// Wait until the rows are on their way (one load per wavefront and trip: workgroups that load the rows all the time keep the memory from the ones that make them)
__device__ __forceinline__ int lg_wait_soon(const FarRows *f, uint32_t tag, int spin_limit) {
    for (int spins = 0;; ++spins) {
        if ((uint32_t)(lg_ld_l2_u64(&f->soon) >> 32) == tag) return 0;
        if (spins >= spin_limit) return LG_XFFN_ERR_WAIT;
        __builtin_amdgcn_s_sleep(1);
    }
}
// Units at(i), i = 0 .. total - 1, by nt threads, at most N of a thread; then put(i, unit)
template <int N, typename A, typename P>
__device__ __forceinline__ int lg_take_far(const FarRows *f, int total, int t, int nt, uint32_t tag, int spin_limit, A &&at, P &&put) {
    const __amdgpu_buffer_rsrc_t r = lg_buffer_rsrc(f->u);
    const uint32_t marks = lg_far_marks(tag);
    lg_x4u v[N];
    int err = 0, o[N];
    #pragma unroll
    for (int i = 0; i < N; ++i) o[i] = at(t + nt * i < total ? t + nt * i : total - 1) * 16;
    for (int spins = 0;; ++spins) {
        uint32_t diff = 0;
        #pragma unroll
        for (int i = 0; i < N; ++i) v[i] = __builtin_bit_cast(lg_x4u, __builtin_amdgcn_raw_buffer_load_b128(r, o[i], 0, 16));
        #pragma unroll
        for (int i = 0; i < N; ++i) diff |= lg_far_miss(v[i], marks);
        if (__all(diff == 0)) break;
        if (spins >= spin_limit) { err = LG_XFFN_ERR_WAIT; break; }
        asm volatile("" ::: "memory");
    }
    #pragma unroll
    for (int i = 0; i < N; ++i) if (t + nt * i < total) { v[i].y = lg_far_y(v[i]); put(t + nt * i, v[i]); }
    return err;
}
// The rows in LDS for the matrix cores: a block of 32 values of all rows is LG_FAR_BLK bytes, 8 slots of 32 bytes (dwords in the order 0 1 4 5 2 3 6 7, the K halves
// that a lane takes) and 8 scales.  Row j of 2i + h is in slot 4h + i, so that the lanes of either half h, which get slots 4h .. 4h + 3 of a product, have
// (M + 1) / 2 results of rows and not four.
#define LG_FAR_BLK 288
__host__ __device__ static inline constexpr int lg_far_slot(int j) { return (j & 1) * 4 + (j >> 1); }
// Wavefront `wave`'s K segment (nit blocks of 32, at most NIT) of M rows of k values, into the blocks at la.  A lane's units are the same of every row
// that it takes (two at a time, where a half of the wavefront holds a row's units), so that nothing is left to compute when they arrive; what is past the rows
// or the segment is its last once more.
template <int M, int NIT, typename B>
__device__ __forceinline__ int lg_take_far_segment(const FarRows *f, int k, int nit, int wave, int lane, unsigned char *la, uint32_t tag, int spin_limit, B &&behind) {
    constexpr int H = 3 * NIT <= 32 ? 2 : 1, N = (M + H - 1) / H;                // rows of a trip, trips
    const int h = H == 2 ? lane >> 5 : 0, x = H == 2 ? lane & 31 : lane, w = x < 3 * nit ? x : 3 * nit - 1, b = w / 3, e = w - 3 * b, nb = k >> 5;
    auto pos = [](int m) { return (m & 1) | ((m & 2) << 1) | ((m & 4) >> 1); };
    uint32_t *blk = (uint32_t *)(la + (size_t)b * LG_FAR_BLK), *s0 = blk + (H == 2 ? 32 * h : 0) + pos(3 * e), *s1 = blk + (H == 2 ? 32 * h : 0) + pos(3 * e + 1);
    uint32_t *s2 = e == 2 ? blk + 64 + (H == 2 ? 4 * h : 0) : blk + (H == 2 ? 32 * h : 0) + pos(3 * e + 2);
    const int st = e == 2 ? 1 : 8;                             // dwords from a slot to the next
    const __amdgpu_buffer_rsrc_t r = lg_buffer_rsrc(f->u);
    const int at = (wave * nit * 3 + w) * 16, row = nb * 48;
    const uint32_t marks = lg_far_marks(tag);
    lg_x4u v[N];
    int err = 0;
    auto load = [&] {
        #pragma unroll
        for (int i = 0; i < N; ++i) {
            const int j = H * i + h < M ? H * i + h : M - 1;   // (a lane's own only where the last trip has one row)
            v[i] = __builtin_bit_cast(lg_x4u, __builtin_amdgcn_raw_buffer_load_b128(r, at + j * row, 0, 16));
        }
    };
    load();
    behind();                                                  // (further requests, behind the first load of the rows)
    for (int spins = 0;; ++spins) {
        uint32_t diff = 0;
        #pragma unroll
        for (int i = 0; i < N; ++i) diff |= lg_far_miss(v[i], marks);
        if (__all(diff == 0)) break;
        if (spins >= spin_limit) { err = LG_XFFN_ERR_WAIT; break; }
        asm volatile("" ::: "memory");
        load();
    }
    #pragma unroll
    for (int i = 0; i < N; ++i) {                              // (row H i + h: slot 4 h + i, or lg_far_slot(i))
        const int z = H == 2 ? i : lg_far_slot(i);
        s0[z * 8] = v[i].x; s1[z * 8] = lg_far_y(v[i]); s2[z * st] = v[i].z;
    }
    return err;
}
template <int M, int NIT>
__device__ __forceinline__ int lg_take_far_segment(const FarRows *f, int k, int nit, int wave, int lane, unsigned char *la, uint32_t tag, int spin_limit) {
    return lg_take_far_segment<M, NIT>(f, k, nit, wave, lane, la, tag, spin_limit, [] {});
}
// Weights as the high nibbles of bytes, two's complement: their product with values is 16 times the dot, which the accumulators' start, the bits of 1.5 * 2^19,
// turns into 786432 + dot, exactly
#define LG_FAR_MAGIC 0x49400000
#define LG_FAR_BIAS 786432.0f
__device__ __forceinline__ lg_v4i lg_far_weights(uint32_t x, uint32_t y) {      // (nibbles of x and y: signed)
    lg_v4i b; b.x = (x << 4) & 0xF0F0F0F0; b.y = (y << 4) & 0xF0F0F0F0; b.z = x & 0xF0F0F0F0; b.w = y & 0xF0F0F0F0;
    return b;
}
template <int N> __device__ __forceinline__ float lg_row_bcast(float v) { return lg_dpp_f<0x150 + N>(v); }      // lane N of each row of 16

struct XtailArgs {
    RowsPleGateArgs r;              // phase 1 (x_out is not written: the row stays in registers)
    const uint8_t *pw;              // phase 2: tiled projection weights [E][ple]
    uint2         *pout;            // [M][E] its output, tagged (the XCD's L2 hands it from phase 2 to phase 3)
    const float   *w_post2, *os;    // phase 3: norm weight for pout, layer output scale (or nullptr)
    const float   *w_pre;           // norm weight applied before quantization
    float         *x_out, *h_out;   // [M][E] new residual; normed rows before quantization, or nullptr
    int8_t        *q;               // q8 activation buffer of the result
    int            q_units;         // 0: rows in the order of lg_act_layout; 2: the 80-dword blocks of lg_k_geglu_m
    int            seq;             // number of this launch inside the step (the layer)
    int            spin_limit;
    unsigned long long *stamps;     // nullptr, or [LG_XTAIL_UNITS][8] device wall-clock ticks at the phase boundaries of every unit (measurement runs)
    uint2         *gf;              // [M][ple] the gated values as tagged floats (handed from phase 1 to phase 2 through the XCD's L2)
    const uint8_t *qw;              // lg_k_ple_tail_s: the next layer's q/k/v projections are part of the launch (segment tiles; from LG_TAIL_MFMA rows on the chains
                                    // of lg_k_attn_tail), or nullptr
    int            qm;              // their rows
    float         *qout;            // [M][qm]
    FarRows       *rows;            // the rows that they take
};
#define LG_XTAIL_FIELDS(X, v) X(const float *, x, r.x, v) X(const float *, dout, r.dout, v) X(const float *, w_post, r.w_post, v) X(const uint8_t *, gw, r.g.w, v) \
    X(int, gk, r.g.k, v) X(int, gple, r.g.ple, v) X(int, dparts, r.dparts, v) X(int, seq, seq, v) X(const float *, gipl, r.g.ipl, v) X(int, glayer, r.g.layer, v) \
    X(int, gnl, r.g.n_layer, v) X(int8_t *, gpq, r.g.pq, v) X(const uint8_t *, pw, pw, v) X(const float *, w_post2, w_post2, v) X(const float *, w_pre, w_pre, v) \
    X(const float *, os, os, v) X(uint2 *, pout, pout, v) X(float *, x_out, x_out, v) X(float *, h_out, h_out, v) X(int8_t *, q, q, v) X(int, q_units, q_units, v) \
    X(float, eps, r.eps, v) X(int, spin_limit, spin_limit, v) X(unsigned long long *, stamps, stamps, v) X(uint2 *, gf, gf, v) \
    X(const uint8_t *, qw, qw, v) X(int, qm, qm, v) X(float *, qout, qout, v) X(FarRows *, rows, rows, v)

__device__ __forceinline__ void lg_ld4_wait1(lg_x4u &a) { asm volatile("s_waitcnt vmcnt(0)" : "+v"(a) :: "memory"); }

// Tagged hand-over.  A 16-byte unit is two (dword, tag) pairs, each stored by one 8-byte store; addr(i) is the lane's i-th unit.
// All N are loaded, around the CU's L1, until every lane that is `on` finds the launch's number in all of its tags.
template <int N> struct LgUnits { lg_x4u v[N]; };
template <int N>
__device__ __forceinline__ void lg_units_wait(LgUnits<N> &r) {
    static_assert(N == 1 || N == 2 || N == 5 || N == 6 || N == 8, "units of a lane");
    if constexpr (N == 1) asm volatile("s_waitcnt vmcnt(0)" : "+v"(r.v[0]) :: "memory");
    if constexpr (N == 2) asm volatile("s_waitcnt vmcnt(0)" : "+v"(r.v[0]), "+v"(r.v[1]) :: "memory");
    if constexpr (N == 5) asm volatile("s_waitcnt vmcnt(0)" : "+v"(r.v[0]), "+v"(r.v[1]), "+v"(r.v[2]), "+v"(r.v[3]), "+v"(r.v[4]) :: "memory");
    if constexpr (N == 6) asm volatile("s_waitcnt vmcnt(0)" : "+v"(r.v[0]), "+v"(r.v[1]), "+v"(r.v[2]), "+v"(r.v[3]), "+v"(r.v[4]), "+v"(r.v[5]) :: "memory");
    if constexpr (N == 8) asm volatile("s_waitcnt vmcnt(0)" : "+v"(r.v[0]), "+v"(r.v[1]), "+v"(r.v[2]), "+v"(r.v[3]), "+v"(r.v[4]), "+v"(r.v[5]), "+v"(r.v[6]), "+v"(r.v[7]) :: "memory");
}
template <int N, typename A>
__device__ __forceinline__ LgUnits<N> lg_take(A &&addr, bool on, uint32_t tag, int spin_limit, int &err) {
    LgUnits<N> r;
    for (int spins = 0;; ++spins) {
        #pragma unroll
        for (int i = 0; i < N; ++i) r.v[i] = lg_ld4_sc_issue<2>(addr(i));
        lg_units_wait<N>(r);
        uint32_t diff = 0;                                     // any bit of any tag that is not the launch's
        #pragma unroll
        for (int i = 0; i < N; ++i) diff |= (r.v[i].y ^ tag) | (r.v[i].w ^ tag);
        if (__all(!on || (diff >> 4) == 0)) { if (on && diff) err |= LG_XFFN_ERR_PLACE; break; }
        if (spins >= spin_limit) { err |= LG_XFFN_ERR_WAIT; break; }
    }
    return r;
}
__device__ __forceinline__ float4 lg_units_float4(lg_x4u a, lg_x4u b) { return make_float4(__uint_as_float(a.x), __uint_as_float(a.z), __uint_as_float(b.x), __uint_as_float(b.z)); }
__device__ __forceinline__ void lg_put(uint2 *p, float v, uint32_t tag) { *p = make_uint2(__float_as_uint(v), tag); }
// [M][256] gated values -> their q8 in LDS ([M][256] int8, then {scale, sum}): a float4 per lane, 8 lanes a block, 64 a row; thread t of nt
template <int M>
__device__ __forceinline__ void lg_take_gated(const uint2 *gf, int8_t *lq2, int t, int nt, uint32_t tag, int spin_limit, int &err) {
    constexpr int PLE = 256;                                   // (the launch is made for ple == 256 only: constant layout arithmetic)
    for (int i = t; i < M * 64; i += nt) {                     // (whole wavefronts)
        const LgUnits<2> q = lg_take<2>([&](int k) { return (const uint4 *)(gf + 4 * i) + k; }, true, tag, spin_limit, err);
        const int r = i >> 6, blk = (i & 63) >> 3, l8 = i & 7;
        float d; int sum;
        const uint32_t packed = lg_quant4_8lanes(lg_units_float4(q.v[0], q.v[1]), &d, &sum);
        const ActLayout lay = lg_act_layout(PLE);
        *(uint32_t *)(lq2 + (size_t)r * PLE + lg_act_unit(lay, blk * 2 + (l8 >> 2)) * 16 + (l8 & 3) * 4) = packed;
        if (l8 == 0) lg_q8_ds<M>(lq2, PLE)[(size_t)r * (PLE >> 5) + lg_act_block(lay, blk)] = make_float2(d, __int_as_float(sum));
    }
}
// a lane's float4s t + 256 v of a tagged row of nq float4s
template <int N>
__device__ __forceinline__ void lg_take_row_n(float4 (&dv)[LG_ROWV], const uint2 *row, int t, int nq, uint32_t tag, int spin_limit, int &err) {
    const LgUnits<2 * N> q = lg_take<2 * N>([&](int i) { const int v = t + 256 * (i >> 1); return (const uint4 *)(row + 4 * (v < nq ? v : nq - 1)) + (i & 1); }, true, tag, spin_limit, err);
    #pragma unroll
    for (int v = 0; v < LG_ROWV; ++v) dv[v] = lg_units_float4(q.v[v < N ? 2 * v : 0], q.v[v < N ? 2 * v + 1 : 1]);
}
__device__ __forceinline__ void lg_take_row(float4 (&dv)[LG_ROWV], const uint2 *row, int t, int nq, uint32_t tag, int spin_limit, int &err) {
    if (nq <= 256) lg_take_row_n<1>(dv, row, t, nq, tag, spin_limit, err);
    else if (nq <= 768) lg_take_row_n<3>(dv, row, t, nq, tag, spin_limit, err);
    else lg_take_row_n<4>(dv, row, t, nq, tag, spin_limit, err);
}

// G: most projection row groups per wavefront (E/8 groups over 4U wavefronts).
template <int M, int G>
__global__ __launch_bounds__(LG_WG) void lg_k_ple_tail(StepCtl *ctl, LG_XTAIL_FIELDS(LG_XP, _) int p_end_) {
    if (blockIdx.x & (LG_XCDS - 1)) return;
    XtailArgs a; LG_XTAIL_FIELDS(LG_XI, a)
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float gbuf[32], red[3][4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int E = a.r.g.k, ple = a.r.g.ple, nblk = ple >> 5, U = nblk * M, nq = E >> 2;
    const int u = blockIdx.x >> 3, gb = u % nblk, j = u / nblk;
    auto stamp = [&](int i) { if (a.stamps && t == 0) a.stamps[(size_t)u * 8 + i] = wall_clock64(); };
    stamp(0);
    const uint32_t tag = lg_tag(ctl->launch + (uint32_t)a.seq, lg_xcc_id());
    int err = 0;
    // ---- phase 1, with this kernel's later loads requested behind its own ----
    const int groups = E >> 3, waves = 4 * U, gw = u * 4 + wave;
    const uint8_t *wgp[G];
    int row[G];
    bool live[G];
    #pragma unroll
    for (int g = 0; g < G; ++g) {
        const int gi = g ? g * waves + wave * (U) + u : gw;         // (what does not come out even is spread over the units)
        live[g] = gi < groups;
        const int gc = live[g] ? gi : groups - 1;
        wgp[g] = a.pw + (size_t)gc * LG_TILE;                  // K = ple = 256: one tile per group of 8 rows
        row[g] = gc * 8 + (lane >> 3);
    }
    WChunk<G, 1> pwt;
    float4 wpost2[LG_ROWV], wpre[LG_ROWV];
    float osv = 1.0f;
    float4 xv[LG_ROWV];
    lg_rows_plegate_body(a.r, M, gb, j, smem, gbuf, red[0], xv, false, [&] {
        lg_mm_fetch<G, 1>(pwt, wgp, 0, 1, lane);
        const float4 *w2 = (const float4 *)a.w_post2, *w3 = (const float4 *)a.w_pre;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) { wpost2[v] = w2[t + 256 * v]; wpre[v] = w3[t + 256 * v]; }
        if (a.os) osv = a.os[0];
    }, [&](const float *v) { if (t < 32) lg_put(a.gf + (size_t)j * ple + gb * 32 + t, v[t], tag); });
    stamp(1);
    // ---- hand-over: every unit's 32 gated values of its row ----
    int8_t *lq2 = (int8_t *)(smem + (size_t)E * 5 / 4);       // [M][ple] int8, [M][ple/32] {scale, sum}
    lg_take_gated<M>(a.gf, lq2, t, LG_WG, tag, a.spin_limit, err);
    stamp(2);
    __syncthreads();
    stamp(3);
    // ---- phase 2: this wavefront's row groups of the projection ----
    {
        float acc[G][M];
        lg_mm_groups<M, 8, G, false, 1>(wgp, pwt, 1, lq2, lg_q8_ds<M>(lq2, ple), ple, acc, lane, nullptr, E, row);
        const int c = lane & 7;
        if (c < M) {
            #pragma unroll
            for (int g = 0; g < G; ++g) if (live[g]) lg_put(a.pout + (size_t)c * E + row[g], lg_pick<M>(acc[g], c), tag);
        }
    }
    const int slices = (E + 1023) >> 10;
    stamp(4);
    if (err) atomicOr(&ctl->err, err);
    if (gb >= slices) return;                                  // this unit has no share of the row work
    // ---- hand-over: the projection's row j; phase 3: the row work, this unit storing and quantizing slice gb ----
    float4 dv[LG_ROWV];
    err = 0;
    lg_take_row(dv, a.pout + (size_t)j * E, t, nq, tag, a.spin_limit, err);
    if (err) atomicOr(&ctl->err, err);
    stamp(5);
    stamp(6);
    {
        float ss = 0.0f;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(dv[v], ss);
        ss = lg_block_sum256(ss, red[1]);
        const float sc = 1.0f / sqrtf(ss / (float)E + a.r.eps);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
            const float4 w = wpost2[v];
            float4 r;
            r.x = xv[v].x + dv[v].x * sc * w.x;  r.y = xv[v].y + dv[v].y * sc * w.y;
            r.z = xv[v].z + dv[v].z * sc * w.z;  r.w = xv[v].w + dv[v].w * sc * w.w;
            if (a.os) { r.x = r.x * osv; r.y = r.y * osv; r.z = r.z * osv; r.w = r.w * osv; }
            xv[v] = r;
        }
    }
    {
        float4 *xo = (float4 *)(a.x_out + (size_t)j * E);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq && v == gb) xo[t + 256 * v] = xv[v];
    }
    {
        float ss = 0.0f;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(xv[v], ss);
        ss = lg_block_sum256(ss, red[2]);
        const float sc = 1.0f / sqrtf(ss / (float)E + a.r.eps);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
            const float4 w = wpre[v];
            xv[v] = make_float4(xv[v].x * sc * w.x, xv[v].y * sc * w.y, xv[v].z * sc * w.z, xv[v].w * sc * w.w);
        }
    }
    if (a.h_out) {
        float4 *ho = (float4 *)(a.h_out + (size_t)j * E);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq && v == gb) ho[t + 256 * v] = xv[v];
    }
    float2 *dsb = lg_q8_ds<M>(a.q, E);
    #pragma unroll
    for (int v = 0; v < LG_ROWV; ++v) {
        if (t + 256 * v >= nq || v != gb) continue;
        float d; int sum;
        const uint32_t packed = lg_quant4_8lanes(xv[v], &d, &sum);
        const int quad = t + 256 * v;
        if (a.q_units == 2) {
            uint32_t *blk = (uint32_t *)a.q + (size_t)(quad >> 3) * LG_MU_DWORDS;
            const int dw = quad & 7;
            blk[j * 8 + ((dw & 1) | ((dw & 2) << 1) | ((dw & 4) >> 1))] = packed;
            if ((t & 7) == 0) *(float2 *)(blk + 64 + 2 * j) = make_float2(d, 12582912.0f + (float)(8 * sum));
        } else {
            *(uint32_t *)(a.q + lg_q8_off<M>(E, j, quad >> 2, (quad & 3) * 4)) = packed;
            if ((t & 7) == 0) dsb[lg_q8_ds_idx<M>(E, j, quad >> 3)] = make_float2(d, __int_as_float(sum));
        }
    }
    stamp(7);
}

// the sum over the 256 lanes of wavefronts 0..3 (order of lg_block_sum256) in a workgroup of 8 wavefronts that all call it
__device__ __forceinline__ float lg_block_sum256_of512(float v, float *scratch8) {
    v = lg_wave_sum64(v);
    if ((threadIdx.x & 63) == 0) scratch8[threadIdx.x >> 6] = v;
    __syncthreads();
    return (scratch8[0] + scratch8[1]) + (scratch8[2] + scratch8[3]);
}

// The same tail for blocks of 5..8 rows, where ple/32 x M units no longer fit one per CU of the XCD (at 5 rows 8 CUs held
// two units, pulled twice the bytes through their one memory path and kept every other unit waiting at the first
// hand-over).  Here the launch has W = M * P units, P = 32 / M per row (30, 30, 28, 32 units at 5..8 rows), each a workgroup
// of 8 wavefronts.  Unit (row j, part p):
//   phase 1: wavefronts 0..3 do the row's update and q8 exactly as lg_k_rows_plegate does (every part of a row repeats
//   it), then wavefront w runs gate row group g0 + w (8 gate rows) of the part's share g0 .. g0 + cnt - 1 of the ple/8
//   groups (cnt = 5 or 6 at 5 rows, 8 at 8 rows); the gated values go out as floats: a part's rows do not line up
//   with the q8 blocks of 32;
//   hand-over; every unit quantizes the M x ple floats into its LDS (the blocks, scales and sums of lg_k_rows_plegate);
//   phase 2 and 3 as in lg_k_ple_tail, the projection's row groups dealt over 8 W wavefronts, the row work of row j by
//   its parts 0 .. E/1024 - 1 (wavefronts 0..3).
#define LG_TAIL_MFMA 4              // rows from which the projections are on the matrix cores
// A workgroup's share of the next layer's q/k/v projections, the weights requested, and unpacked, while the rows are being made
template <int M, int NIT, bool MFMA = (M >= LG_TAIL_MFMA)> struct TailQkv;
// ... a block of 32 rows, a K segment to a wavefront (lg_k_attn_tail), which takes its part of the rows itself
template <int M, int NIT>
struct TailQkv<M, NIT, true> {
    static constexpr int ROWS = 32, N = (NIT + 1) / 2, I = (M + 1) / 2;
    lg_v4i b[NIT]; float dw[NIT];
    __device__ __forceinline__ void request(const XtailArgs &a, int rank, int wave, int lane, int nit) {
        const uint8_t *cb = a.qw + ((size_t)rank * 8 + wave) * (nit * 576);
        lg_x4u q[N]; uint32_t s[N];
        #pragma unroll
        for (int u = 0; u < N; ++u) {
            const int at = 2 * u < nit ? u : 0;
            q[u] = __builtin_nontemporal_load((const lg_x4u *)(cb + (size_t)(at * 64 + lane) * 16));
            s[u] = __builtin_nontemporal_load((const uint32_t *)(cb + (size_t)nit * 512 + (size_t)(at * 32 + (lane & 31)) * 4));
        }
        #pragma unroll
        for (int i = 0; i < NIT; ++i) {
            b[i] = lg_far_weights((i & 1 ? q[i >> 1].z : q[i >> 1].x) ^ 0x88888888u, (i & 1 ? q[i >> 1].w : q[i >> 1].y) ^ 0x88888888u);
            dw[i] = lg_h2f((uint16_t)(i & 1 ? s[i >> 1] >> 16 : s[i >> 1]));
            asm volatile("" : "+v"(b[i]), "+v"(dw[i]));
        }
    }
    __device__ __forceinline__ int take(const XtailArgs &a, int wave, int lane, int nit, unsigned char *act, uint32_t tag) {
        return lg_take_far_segment<M, NIT>(a.rows, a.r.g.k, nit, wave, lane, act + (size_t)wave * NIT * LG_FAR_BLK, tag, a.spin_limit);
    }
    // xch: 8 KB of LDS
    __device__ __forceinline__ void finish(const XtailArgs &a, int rank, int wave, int t, int nit, const unsigned char *act, float *xch, int real) {
        const int lane = t & 63, n = lane & 31, h = lane >> 5, arow = n < 8 ? n : 7;
        lg_v16i magic;
        #pragma unroll
        for (int i = 0; i < 16; ++i) magic[i] = LG_FAR_MAGIC;
        asm volatile("" : "+v"(magic));
        float p[I];
        #pragma unroll
        for (int r = 0; r < I; ++r) p[r] = 0.0f;
        const unsigned char *ls = act + (size_t)wave * NIT * LG_FAR_BLK, *la = ls + arow * 32 + h * 16;
        lg_v16i d[2];
        d[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(*(const lg_v4i *)la, b[0], magic, 0, 0, 0);
        #pragma unroll
        for (int i = 0; i < NIT; ++i) {                        // (the next block's dots on their way while this one's join the sums)
            if (i + 1 < NIT) d[(i + 1) & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(*(const lg_v4i *)(la + (i + 1) * LG_FAR_BLK), b[i + 1 < NIT ? i + 1 : i], magic, 0, 0, 0);
            #pragma unroll
            for (int r = 0; r < I; ++r) {
                const float v = lg_fmaf(*(const float *)(ls + i * LG_FAR_BLK + 256 + (4 * h + r) * 4) * dw[i], __int_as_float(d[i & 1][r]) - LG_FAR_BIAS, p[r]);
                p[r] = i < nit ? v : p[r];                     // (no branch on a shorter segment's end: what lies behind it is not taken)
                asm volatile("" : "+v"(p[r]));
            }
        }
        #pragma unroll
        for (int i = 0; i < I; ++i) xch[(wave * 8 + 2 * i + h) * 32 + n] = p[i];
        __syncthreads();
        if (t < 32 * M && real) {                              // the adjacent-pair tree over the 8 segments
            const float *z = xch + t;
            a.qout[(size_t)(t >> 5) * a.qm + rank * 32 + (t & 31)] = ((z[0] + z[256]) + (z[512] + z[768])) + ((z[1024] + z[1280]) + (z[1536] + z[1792]));
        }
    }
};
// ... two row groups of 8, the tiles of each over four wavefronts (lg_k_mm_ks<M, 4>)
template <int M, int NIT>
struct TailQkv<M, NIT, false> {
    static constexpr int ROWS = 16, KP = 4, N = (NIT + KP - 1) / KP;
    uint4 q[N]; uint32_t s[N];
    __device__ __forceinline__ void request(const XtailArgs &a, int rank, int wave, int lane, int nit) {
        const int g0 = rank * 2 + wave / KP, gi = g0 < a.qm >> 3 ? g0 : (a.qm >> 3) - 1, lo = wave % KP * nit / KP;
        const uint8_t *wg = a.qw + (size_t)gi * nit * LG_TILE;
        #pragma unroll
        for (int u = 0; u < N; ++u) {
            const int it = lo + u < nit ? lo + u : nit - 1;
            q[u] = lg_ldt16(wg, it, lane);
            s[u] = lg_ldt2(wg, it, lane);
        }
    }
    __device__ __forceinline__ int take(const XtailArgs &a, int wave, int lane, int nit, unsigned char *act, uint32_t tag) {
        // (a block's units by three lanes in a row of four, the fourth idle: its sum is added up across them)
        const int k = a.r.g.k, nb = k >> 5;
        const ActLayout lay = lg_act_layout(k);
        const int err = lg_take_far<(32 * NIT * M + 511) / 512>(a.rows, nb * M * 4, wave * 64 + lane, 512, tag, a.spin_limit, [&](int i) { return (i >> 2) * 3 + min(i & 3, 2); }, [&](int i, const lg_x4u &v) {
            const int e = i & 3, j = (i >> 2) / nb, b = (i >> 2) - j * nb;
            int sum = e == 3 ? 0 : __builtin_amdgcn_sdot4((int)v.x, 0x01010101, __builtin_amdgcn_sdot4((int)v.y, 0x01010101, e == 2 ? 0 : __builtin_amdgcn_sdot4((int)v.z, 0x01010101, 0, false), false), false);
            sum += lg_dpp_i<LG_DPP_SWAP1>(sum); sum += lg_dpp_i<LG_DPP_SWAP2>(sum);
            auto put = [&](int m, uint32_t w) { *(uint32_t *)(act + (size_t)j * k + lg_act_unit(lay, b * 2 + (m >> 2)) * 16 + (m & 3) * 4) = w; };
            if (e < 3) { put(3 * e, v.x); put(3 * e + 1, v.y); }
            if (e < 2) put(3 * e + 2, v.z);
            if (e == 2) *(float2 *)(act + (size_t)M * k + ((size_t)j * nb + lg_act_block(lay, b)) * 8) = make_float2(__uint_as_float(v.z), __int_as_float(sum));
        });
        __syncthreads();
        return err;
    }
    __device__ __forceinline__ void finish(const XtailArgs &a, int rank, int wave, int t, int nit, const unsigned char *act, float *xch, int real) {
        const int lane = t & 63, k = a.r.g.k, gsel = wave / KP, part = wave % KP, lo = part * nit / KP, nt = (part + 1) * nit / KP - lo, g0 = rank * 2 + gsel;
        float acc[M];
        lg_mm_ks_sums<M, KP, N>(q, s, lo, nt, part, (const int8_t *)act, (const float2 *)(act + (size_t)M * k), k, lane, xch + (size_t)gsel * M * 64, acc);
        if (part != KP - 1 || g0 >= a.qm >> 3) return;
        const int c = lane & 7;
        if (c < M && real) a.qout[(size_t)c * a.qm + g0 * 8 + (lane >> 3)] = lg_pick<M>(acc, c);
    }
};
// bytes of the rows in LDS
__host__ __device__ static inline size_t lg_tail_act(int M, int E) { return M >= LG_TAIL_MFMA ? (size_t)8 * (E <= 2560 ? 10 : 16) * LG_FAR_BLK : (size_t)M * E * 5 / 4; }
// bytes of LDS of lg_k_ple_tail_s; with the projections: the rows, 8 slots wide on the matrix cores, and 8 KB for sums
static inline size_t lg_tail_s_lds(int M, int E, int ple, bool qkv) {
    const size_t units = (size_t)E * 5 / 4 + (size_t)M * ple * 5 / 4, far = qkv ? lg_tail_act(M, E) + 8192 : 0;
    return units > far ? units : far;
}
template <int M, int NIT>
__device__ __forceinline__ void lg_tail_qkv(const XtailArgs &a, int rank, unsigned char *act, uint32_t tag, StepCtl *ctl) {
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), E = a.r.g.k, nit = E >> 8;
    float *xch = (float *)(act + lg_tail_act(M, E));
    TailQkv<M, NIT> qkv;
    qkv.request(a, rank, wave, t & 63, nit);
    __builtin_amdgcn_sched_barrier(0);
    // The first time over whatever LDS holds, for nothing but the instructions: they are in the CU's cache when the rows are there (five rows 2068 -> 2061 us a step)
    #pragma unroll 1
    for (int real = 0; real < 2; ++real) {
        if (real) {
            int err = lg_wait_soon(a.rows, tag, a.spin_limit);
            err |= qkv.take(a, wave, t & 63, nit, act, tag);
            if (err) atomicOr(&ctl->err, err);
        }
        qkv.finish(a, rank, wave, t, nit, act, xch, real);
        __syncthreads();
    }
}
template <int M, int G, int NIT>
__global__ __launch_bounds__(512) void lg_k_ple_tail_s(StepCtl *ctl, LG_XTAIL_FIELDS(LG_XP, _) int p_end_) {
    XtailArgs a; LG_XTAIL_FIELDS(LG_XI, a)
    extern __shared__ __align__(16) unsigned char smem[];
    if (blockIdx.x & (LG_XCDS - 1)) {
        const int rank = (blockIdx.x >> 3) * (LG_XCDS - 1) + (blockIdx.x & (LG_XCDS - 1)) - 1;
        if (a.qw && rank * TailQkv<M, NIT>::ROWS < a.qm) lg_tail_qkv<M, NIT>(a, rank, smem, lg_tag(ctl->launch + (uint32_t)a.seq, 0), ctl);
        return;
    }
    __shared__ float red[3][8];
    constexpr int P = 32 / M;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const bool rowt = t < 256;                                 // the threads of the row work (lane order of lg_k_rows)
    const int E = a.r.g.k, ple = a.r.g.ple, W = M * P, nq = E >> 2, nit = E >> 8;
    const int u = blockIdx.x >> 3, j = u / P, p = u - j * P;
    const int ngr = ple >> 3, gbase = ngr / P, gextra = ngr - gbase * P;
    const int cnt = gbase + (p < gextra ? 1 : 0), g0 = p * gbase + (p < gextra ? p : gextra);
    const bool gatew = wave < cnt;
    const int gg = g0 + (gatew ? wave : 0);                    // this wavefront's gate row group
    auto stamp = [&](int i) { if (a.stamps && t == 0) a.stamps[(size_t)u * 8 + i] = wall_clock64(); };
    stamp(0);
    const uint32_t tag = lg_tag(ctl->launch + (uint32_t)a.seq, lg_xcc_id());
    int err = 0;
    int8_t *lq = (int8_t *)smem;                               // the row: [E] int8, then [E/32] {scale, sum}
    float2 *lds = (float2 *)(smem + (size_t)E);
    int8_t *lq2 = (int8_t *)(smem + (size_t)E * 5 / 4);        // [M][ple] int8, [M][ple/32] {scale, sum}
    // ---- every load of phase 1 up front, the row's first; then what the later phases need ----
    float4 xv[LG_ROWV], dv[LG_ROWV], wp[LG_ROWV];
    if (rowt) {
        const float4 *wr = (const float4 *)a.r.w_post, *xr = (const float4 *)(a.r.x + (size_t)j * E), *dr = (const float4 *)(a.r.dout + (size_t)j * E);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) { xv[v] = xr[t + 256 * v]; dv[v] = dr[t + 256 * v]; wp[v] = wr[t + 256 * v]; }
        if (a.r.dparts == 4) {                                 // the top two levels of the tree of an ffn_down cut by K quarter
            const size_t slab = (size_t)M * nq;
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
                const float4 p1 = dr[slab + t + 256 * v], p2 = dr[2 * slab + t + 256 * v], p3 = dr[3 * slab + t + 256 * v], p0 = dv[v];
                dv[v] = make_float4((p0.x + p1.x) + (p2.x + p3.x), (p0.y + p1.y) + (p2.y + p3.y),
                                    (p0.z + p1.z) + (p2.z + p3.z), (p0.w + p1.w) + (p2.w + p3.w));
            }
        }
        if (a.r.dparts == 8) {                                 // the top three levels of the K-segment tree of an ffn_down cut over the 8 XCDs
            const size_t slab = (size_t)M * nq;
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
                const float4 *b = dr + t + 256 * v;
                const float4 p1 = b[slab], p2 = b[2 * slab], p3 = b[3 * slab], p4 = b[4 * slab], p5 = b[5 * slab], p6 = b[6 * slab], p7 = b[7 * slab], p0 = dv[v];
                dv[v] = make_float4(((p0.x + p1.x) + (p2.x + p3.x)) + ((p4.x + p5.x) + (p6.x + p7.x)), ((p0.y + p1.y) + (p2.y + p3.y)) + ((p4.y + p5.y) + (p6.y + p7.y)),
                                    ((p0.z + p1.z) + (p2.z + p3.z)) + ((p4.z + p5.z) + (p6.z + p7.z)), ((p0.w + p1.w) + (p2.w + p3.w)) + ((p4.w + p5.w) + (p6.w + p7.w)));
            }
        }
    }
    uint4 wq[NIT]; uint32_t wsc[NIT];
    float iplv = 0.0f;                                         // of this lane's gate column
    if (gatew) {                                               // (a launch of one row has one such wavefront a unit: requested by all eight, the CU's
                                                               // address unit is busy with them for a microsecond)
        const uint8_t *wg0 = a.r.g.w + (size_t)gg * nit * LG_TILE;
        #pragma unroll
        for (int k = 0; k < NIT; ++k) {
            const int it = k < nit ? k : nit - 1;
            wq[k] = *(const uint4 *)(wg0 + (size_t)it * LG_TILE + lane * 16);
            wsc[k] = *(const uint16_t *)(wg0 + (size_t)it * LG_TILE + 1024 + lane * 2);
        }
        iplv = a.r.g.ipl[(size_t)j * a.r.g.n_layer * ple + (size_t)a.r.g.layer * ple + gg * 8 + (lane >> 3)];
    }
    const int groups = E >> 3, waves = 8 * W, gw = u * 8 + wave;
    const uint8_t *wgp[G];
    int row[G];
    bool live[G];
    #pragma unroll
    for (int g = 0; g < G; ++g) {
        const int gi = g ? g * waves + wave * (W) + u : gw;         // (what does not come out even is spread over the units)
        live[g] = gi < groups;
        const int gc = live[g] ? gi : groups - 1;
        wgp[g] = a.pw + (size_t)gc * LG_TILE;                  // K = ple = 256: one tile per group of 8 rows
        row[g] = gc * 8 + (lane >> 3);
    }
    WChunk<G, 1> pwt;
    lg_mm_fetch<G, 1>(pwt, wgp, 0, 1, lane);
    float4 wpost2[LG_ROWV], wpre[LG_ROWV];
    float osv = 1.0f;
    if (rowt) {
        const float4 *w2 = (const float4 *)a.w_post2, *w3 = (const float4 *)a.w_pre;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) { wpost2[v] = w2[t + 256 * v]; wpre[v] = w3[t + 256 * v]; }
        if (a.os) osv = a.os[0];
    }
    // ---- phase 1: the row, then this wavefront's gate rows ----
    {
        float ss = 0.0f;
        if (rowt) {
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(dv[v], ss);
        }
        ss = lg_block_sum256_of512(ss, red[0]);
        const float sc = 1.0f / sqrtf(ss / (float)E + a.r.eps);
        if (rowt) {
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) {
                if (t + 256 * v < nq) {                        // nq is a multiple of 64: whole wavefronts
                    const float4 w = wp[v], d = dv[v];
                    float4 x = xv[v];
                    x.x = x.x + d.x * sc * w.x;  x.y = x.y + d.y * sc * w.y;
                    x.z = x.z + d.z * sc * w.z;  x.w = x.w + d.w * sc * w.w;
                    xv[v] = x;
                    float dq; int sum;
                    const uint32_t packed = lg_quant4_8lanes(x, &dq, &sum);
                    const int quad = t + 256 * v;
                    *(uint32_t *)(lq + lg_q8_off<1>(E, 0, quad >> 2, (quad & 3) * 4)) = packed;
                    if ((t & 7) == 0) lds[lg_q8_ds_idx<1>(E, 0, quad >> 3)] = make_float2(dq, __int_as_float(sum));
                }
            }
        }
    }
    __syncthreads();
    if (gatew) {
        const int c = lane & 7;
        float pr = 0.0f;
        #pragma unroll
        for (int k = 0; k < NIT; ++k) {
            if (k < nit) {                                     // (a guard, not a break: the arrays stay in registers)
                const float2 ds = lds[k * 8 + c];
                const int8_t *au = lq + (size_t)(k * 16 + c) * 16;
                const int dot = lg_block_dot(wq[k], *(const int4 *)au, *(const int4 *)(au + 8 * 16), __float_as_int(ds.y));
                pr = lg_fmaf(ds.x * lg_h2f((uint16_t)wsc[k]), (float)dot, pr);
            }
        }
        pr = lg_sum_seg<8>(pr);
        if (c == 0) lg_put(a.gf + (size_t)j * ple + gg * 8 + (lane >> 3), lg_gelu_d(pr) * iplv, tag);
    }
    stamp(1);
    // ---- hand-over: every part's gated values; wavefront r quantizes row r ----
    lg_take_gated<M>(a.gf, lq2, t, 512, tag, a.spin_limit, err);
    stamp(2);
    __syncthreads();
    stamp(3);
    // ---- phase 2: this wavefront's row groups of the projection ----
    {
        float acc[G][M];
        lg_mm_groups<M, 8, G, false, 1>(wgp, pwt, 1, lq2, lg_q8_ds<M>(lq2, ple), ple, acc, lane, nullptr, E, row);
        const int c = lane & 7;
        if (c < M) {
            #pragma unroll
            for (int g = 0; g < G; ++g) if (live[g]) lg_put(a.pout + (size_t)c * E + row[g], lg_pick<M>(acc[g], c), tag);
        }
    }
    const int slices = (E + 1023) >> 10;
    stamp(4);
    if (err) atomicOr(&ctl->err, err);
    if (p >= slices) return;                    // this unit has no share of the row work
    // ---- hand-over: the projection's row j; phase 3: the row work, this unit storing and quantizing slice p (wavefronts 0..3;
    //      the others only take part in the workgroup's barriers) ----
    err = 0;
    if (rowt) lg_take_row(dv, a.pout + (size_t)j * E, t, nq, tag, a.spin_limit, err);
    if (err) atomicOr(&ctl->err, err);
    if (a.qw && u == 0 && t == 0) lg_put_soon(a.rows, lg_far_tag(tag));
    stamp(5);
    {
        float ss = 0.0f;
        if (rowt) {
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(dv[v], ss);
        }
        ss = lg_block_sum256_of512(ss, red[1]);
        const float sc = 1.0f / sqrtf(ss / (float)E + a.r.eps);
        if (rowt) {
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
                const float4 w = wpost2[v];
                float4 r;
                r.x = xv[v].x + dv[v].x * sc * w.x;  r.y = xv[v].y + dv[v].y * sc * w.y;
                r.z = xv[v].z + dv[v].z * sc * w.z;  r.w = xv[v].w + dv[v].w * sc * w.w;
                if (a.os) { r.x = r.x * osv; r.y = r.y * osv; r.z = r.z * osv; r.w = r.w * osv; }
                xv[v] = r;
            }
        }
    }
    if (rowt) {
        float4 *xo = (float4 *)(a.x_out + (size_t)j * E);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq && v == p) xo[t + 256 * v] = xv[v];
    }
    {
        float ss = 0.0f;
        if (rowt) {
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(xv[v], ss);
        }
        ss = lg_block_sum256_of512(ss, red[2]);
        const float sc = 1.0f / sqrtf(ss / (float)E + a.r.eps);
        if (rowt) {
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
                const float4 w = wpre[v];
                xv[v] = make_float4(xv[v].x * sc * w.x, xv[v].y * sc * w.y, xv[v].z * sc * w.z, xv[v].w * sc * w.w);
            }
        }
    }
    if (rowt) {
        if (a.h_out) {
            float4 *ho = (float4 *)(a.h_out + (size_t)j * E);
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq && v == p) ho[t + 256 * v] = xv[v];
        }
        float2 *dsb = lg_q8_ds<M>(a.q, E);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) {
            if (t + 256 * v >= nq || v != p) continue;
            float d; int sum;
            const uint32_t packed = lg_quant4_8lanes(xv[v], &d, &sum);
            const int quad = t + 256 * v;
            if (a.qw) lg_put_far_q8(a.rows, E, j, quad, packed, d, lg_far_tag(tag));
            else if (a.q_units == 2) {
                uint32_t *blk = (uint32_t *)a.q + (size_t)(quad >> 3) * LG_MU_DWORDS;
                const int dw = quad & 7;
                blk[j * 8 + ((dw & 1) | ((dw & 2) << 1) | ((dw & 4) >> 1))] = packed;
                if ((t & 7) == 0) *(float2 *)(blk + 64 + 2 * j) = make_float2(d, 12582912.0f + (float)(8 * sum));
            } else {
                *(uint32_t *)(a.q + lg_q8_off<M>(E, j, quad >> 2, (quad & 3) * 4)) = packed;
                if ((t & 7) == 0) dsb[lg_q8_ds_idx<M>(E, j, quad >> 3)] = make_float2(d, __int_as_float(sum));
            }
        }
    }
    stamp(7);
}

// A second form was built and measured, and is not kept: 32 units of 8 gate rows and 8 wavefronts whatever the block
// width (so that no CU holds two units from 5 rows up), the row update as a phase of its own ahead of the gate (units
// (slice, row), q8 rows handed over), the gated rows handed over as floats and quantized by every unit.  Bit-identical,
// three hand-overs instead of two, and slower at every width: E4B shape, 5 rows 11.2 against 10.6 us per launch (step
// 2.231 against 2.210 ms), 6 rows 2.326 against 2.303 ms, 8 rows 2.494 against 2.477 ms.  A hand-over costs about 1 us
// once the wait for the stores and the load of what was handed over are counted, more than the lighter phases save.


// ---------------------------------------------------------------------------------------------------------
// Measured at the E4B shape (5 rows): 12.3 us per launch against 4.3 + 4.1 + 4.5 for the three kernels it replaces, and the
// step 2.219 against 2.203 ms: not a gain, so the option is off by default.  By the stamps: merges 4.3-4.8 us (the same chain of
// round trips as the separate kernel: the partials come from other XCDs), hand-over 0.45, copy of the merged rows 0.5, the
// projection 2.1 (bound by the vector instructions around the MFMA: 640 chains x 8 steps x ~20 instructions on one XCD's
// 128 SIMDs), hand-over 0.55, row work 1.7; the three separate kernels hide their launch gaps under each other's tails, the
// phases of one launch cannot.
// The narrow end of the attention half the same way: merge -> output projection -> row work, one launch on one XCD.
//   1  merge of the tile partials of every (head, row), two of them at a time per unit (a unit is 8 wavefronts, a merge
//      takes 4); the q8 of the merged head goes to the XCD's L2 in the matrix-core block order (80 dwords per block of 32:
//      8 row slots of 32 bytes, then 8 x {scale, 12582912 + 8 * sum});
//      hand-over;
//   2  the output projection on the matrix cores: a chain = (block of 32 output rows, K segment); wavefront w of unit u
//      runs segment w of the row blocks u, u + 32, ...: per block of the segment one v_mfma_i32_32x32x32_i8 (A = the
//      block's activations in 8 row slots, B = the 32 rows' nibbles) and four fma per lane, p = fma(xd * dw, (float)dot, p),
//      the chain of lg_k_mm; the 8 segment sums of a row meet in LDS in the adjacent-pair tree.  The weights (E x K / 32
//      units = 92 KB per unit at the E4B shape) are requested at kernel start and arrive under the merge: a lone XCD pulls
//      3 MB from HBM in about 2 us.  On v_dot4 the same projection would keep the XCD's 128 SIMDs busy for 4.5 us;
//      hand-over;
//   3  the row work ahead of gate/up (residual update, ffn norm, q8 in the order the gate/up kernel reads) by units (slice, row).
// Weights: per chain the stream layout of lg_xffn.h (pairs of blocks: [pair][half h][row n] 8 + 8 nibble bytes, then
// [pair][row n] the two f16 scales), chains ordered [row block][segment].
struct XattnTailArgs {
    MergeArgs      g;            // g.xq, g.xf unused
    const uint8_t *wo;           // chains of attn_output
    uint32_t      *aq;           // [K / 32][80] the merged rows as matrix-core blocks
    float         *pout;         // [M][E]
    const float   *x, *w_post, *w_pre;
    float         *x_out;
    int8_t        *q;
    int            q_units;      // 2: blocks of lg_k_geglu_m (4..8 rows), 1: units of lg_k_geglu_t (up to 3 rows)
    int            E;
    float          eps;
    XtailSync     *sync;
    int            seq;          // number of this launch inside the step (the layer)
    int            spin_limit;
    unsigned long long *stamps;
};
#define LG_XATTN_FIELDS(X, v) X(const float *, pm, g.pm, v) X(const float *, pl, g.pl, v) X(const float *, pacc, g.pacc, v) X(int, tiles_max, g.tiles_max, v) \
    X(int, H, g.H, v) X(int, hd, g.hd, v) X(int, window, g.window, v) X(int, pos_off, g.pos_off, v) X(const uint8_t *, wo, wo, v) X(XtailSync *, sync, sync, v) \
    X(const float *, x, x, v) X(const float *, w_post, w_post, v) X(const float *, w_pre, w_pre, v) X(uint32_t *, aq, aq, v) X(float *, pout, pout, v) \
    X(float *, x_out, x_out, v) X(int8_t *, q, q, v) X(int, q_units, q_units, v) X(int, E, E, v) X(float, eps, eps, v) X(int, spin_limit, spin_limit, v) X(int, seq, seq, v) \
    X(unsigned long long *, stamps, stamps, v)

// Row blocks of a unit whose weights are requested with the merge's partials; the rest after the merge.  All of them early
// is the faster choice: requested after the merge they delay the first hand-over, whose store wait also waits for them
// (the merge phase 4.3-4.8 us either way, the whole launch 10.1 against 11.0 us).
#ifndef LG_XATTN_EARLY
#define LG_XATTN_EARLY 8
#endif
// M: rows; NP: pairs of blocks per chain (K / 32 / 8 / 2); RB: most row blocks per unit (E / 32 over 32 units).
template <int M, int NP, int RB>
__global__ __launch_bounds__(512) void lg_k_attn_tail(StepCtl *ctl, LG_XATTN_FIELDS(LG_XP, _) int p_end_) {
    if (blockIdx.x & (LG_XCDS - 1)) return;
    XattnTailArgs a; LG_XATTN_FIELDS(LG_XI, a)
    a.g.xq = nullptr; a.g.xf = nullptr;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float wts[2][512], pls[2][512], wmx[2][4], red3[2][8];
    __shared__ __align__(16) int8_t hq[2][512];
    __shared__ float2 hds[2][16];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), half = wave >> 2, tid = t & 255;
    const int n = lane & 31, h = lane >> 5;
    const int E = a.E, nq = E >> 2, hd = a.g.hd, nbh = hd >> 5, nit = 2 * NP, nb = 8 * nit;
    const int U = LG_XCD_WGS, u = blockIdx.x >> 3;
    const int slices = (E + 1023) >> 10, nrow = slices * M;
    const bool rowunit = u < nrow, rowlane = t < LG_WG;
    const int v_ = u / M, jr = u - v_ * M;
    const uint32_t tag = lg_tag(ctl->launch + (uint32_t)a.seq, lg_xcc_id());
    auto stamp = [&](int i) { if (a.stamps && t == 0) a.stamps[(size_t)u * 8 + i] = wall_clock64(); };
    stamp(0);
    lg_v16i magic;
    #pragma unroll
    for (int i = 0; i < 16; ++i) magic[i] = 0x4B400000;
    asm volatile("" : "+v"(magic));
    // ---- phase 1: the merges (tasks u and u + 32), with everything else this unit reads requested behind their partials ----
    const int ntasks = a.g.H * M, task = u + U * half;
    const bool on = task < ntasks;
    const int tk = on ? task : ntasks - 1, head = tk % a.g.H, j = tk / a.g.H;
    struct Pair { lg_x4u q; uint32_t sw; };
    Pair wq[RB][NP];
    bool live[RB];
    float4 xv[LG_ROWV], wpost[LG_ROWV], wpre[LG_ROWV];
    const int nrb = E >> 5;
    auto fetch_w = [&](int k0, int k1) {
        #pragma unroll
        for (int k = 0; k < RB; ++k) {
            if (k < k0 || k >= k1) continue;
            const int rb = u + U * k;
            live[k] = rb < nrb;
            const uint8_t *cb = a.wo + ((size_t)(live[k] ? rb : 0) * 8 + wave) * ((size_t)nit * 576);    // (no such row block: the first one's weights, never stored)
            #pragma unroll
            for (int jp = 0; jp < NP; ++jp) {
                wq[k][jp].q = __builtin_nontemporal_load((const lg_x4u *)(cb + (size_t)((jp * 2 + h) * 32 + n) * 16));
                wq[k][jp].sw = __builtin_nontemporal_load((const uint32_t *)(cb + (size_t)nit * 512 + (size_t)(jp * 32 + n) * 4));
            }
        }
    };
    lg_attn_merge_body<false>(ctl, a.g, head, j, tid, wts[half], pls[half], wmx[half], [&] { fetch_w(0, LG_XATTN_EARLY); }, [&](int d, float r, int q, float dq, int sum) {
        hq[half][d] = (int8_t)q;
        if ((d & 31) == 0) hds[half][d >> 5] = make_float2(dq, 12582912.0f + (float)(8 * sum));
    });
    fetch_w(LG_XATTN_EARLY, RB);
    __syncthreads();
    if (on && tid < (hd >> 2)) {                               // dword tid of the merged head: block tid / 8, dword tid % 8 of it
        const int b = tid >> 3, dw = tid & 7;
        uint32_t *blk = a.aq + (size_t)(head * nbh + b) * LG_MU_DWORDS;
        blk[j * 8 + ((dw & 1) | ((dw & 2) << 1) | ((dw & 4) >> 1))] = *(const uint32_t *)(hq[half] + 4 * tid);
        if (dw == 0) *(float2 *)(blk + 64 + 2 * j) = hds[half][b];
    }
    stamp(1);
    // ---- hand-over: the merged rows are in the XCD's L2 ----
    const int nmerge = ntasks < U ? ntasks : U;                 // units that ran a merge
    lg_wait_vm();
    __syncthreads();
    if (wave == 0) {
        const int err = lg_xcd_arrive_wait(a.sync->flags[0], u, u < nmerge, nmerge, tag, a.spin_limit);
        if (err && lane == 0) atomicOr(&ctl->err, err);
    }
    __syncthreads();
    stamp(2);
    unsigned char *la = smem;                                  // [nb][320]
    float *red = (float *)(smem + (size_t)nb * LG_MU_DWORDS * 4);          // [8 segments][RB][8 row slots][32]
    {
        const int n16 = nb * LG_MU_DWORDS / 4;                 // 16-byte units
        for (int i0 = t; i0 < n16; i0 += 4 * 512) {
            const int i1 = min(i0 + 512, n16 - 1), i2 = min(i0 + 1024, n16 - 1), i3 = min(i0 + 1536, n16 - 1);
            lg_x4u v0 = lg_ld4_sc_issue<2>((const unsigned char *)a.aq + (size_t)i0 * 16), v1 = lg_ld4_sc_issue<2>((const unsigned char *)a.aq + (size_t)i1 * 16);
            lg_x4u v2 = lg_ld4_sc_issue<2>((const unsigned char *)a.aq + (size_t)i2 * 16), v3 = lg_ld4_sc_issue<2>((const unsigned char *)a.aq + (size_t)i3 * 16);
            lg_ld4_wait(v0, v1, v2, v3);
            *(lg_x4u *)(la + (size_t)i0 * 16) = v0; *(lg_x4u *)(la + (size_t)i1 * 16) = v1;
            *(lg_x4u *)(la + (size_t)i2 * 16) = v2; *(lg_x4u *)(la + (size_t)i3 * 16) = v3;
        }
    }
    __syncthreads();
    stamp(3);
    // (what phase 3 needs besides the projection is requested here: behind the loads this phase waits for, with a phase's
    // time to arrive, and not occupying registers during the merge)
    if (rowunit && rowlane) {
        const float4 *xr = (const float4 *)(a.x + (size_t)jr * E), *w1 = (const float4 *)a.w_post, *w2 = (const float4 *)a.w_pre;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) { xv[v] = xr[t + 256 * v]; wpost[v] = w1[t + 256 * v]; wpre[v] = w2[t + 256 * v]; }
    }
    // ---- phase 2: segment `wave` of the unit's row blocks ----
    {
        const int arow = n < 8 ? n : 7;
        float p[RB][4];
        #pragma unroll
        for (int k = 0; k < RB; ++k)
            #pragma unroll
            for (int i = 0; i < 4; ++i) p[k][i] = 0.0f;
        #pragma unroll
        for (int jp = 0; jp < NP; ++jp) {
            #pragma unroll
            for (int e = 0; e < 2; ++e) {
                const XffnAct ac = lg_xffn_act(la + (size_t)(wave * nit + 2 * jp + e) * (LG_MU_DWORDS * 4), arow, h);
                #pragma unroll
                for (int k = 0; k < RB; ++k) {
                    lg_v2u q; q.x = e ? wq[k][jp].q.z : wq[k][jp].q.x; q.y = e ? wq[k][jp].q.w : wq[k][jp].q.y;
                    lg_xffn_step(ac.av, ac.xd, ac.cf, q, lg_h2f((uint16_t)(e ? wq[k][jp].sw >> 16 : wq[k][jp].sw)), magic, p[k]);
                }
            }
        }
        #pragma unroll
        for (int k = 0; k < RB; ++k)
            #pragma unroll
            for (int i = 0; i < 4; ++i) red[((size_t)(wave * RB + k) * 8 + 4 * h + i) * 32 + n] = p[k][i];      // (all 8 row slots: the tree reads the first M)
    }
    __syncthreads();
    for (int idx = t; idx < RB * M * 32; idx += 512) {         // the adjacent-pair tree over the 8 segments
        const int k = idx / (M * 32), rem = idx - k * (M * 32), jj = rem >> 5, nn = rem & 31, rb = u + U * k;
        if (rb < nrb) {
            const float *b = red + ((size_t)k * 8 + jj) * 32 + nn;
            const size_t sg = (size_t)RB * 8 * 32;
            a.pout[(size_t)jj * E + rb * 32 + nn] = ((b[0] + b[sg]) + (b[2 * sg] + b[3 * sg])) + ((b[4 * sg] + b[5 * sg]) + (b[6 * sg] + b[7 * sg]));
        }
    }
    stamp(4);
    // ---- hand-over: the projection's [M][E] is in the XCD's L2 ----
    lg_wait_vm();
    __syncthreads();
    if (!rowunit) {
        if (t == 0) lg_st_sc<0>(a.sync->flags[1] + u, tag);
        return;
    }
    if (wave == 0) {
        const int err = lg_xcd_arrive_wait(a.sync->flags[1], u, true, U, tag, a.spin_limit);
        if (err && lane == 0) atomicOr(&ctl->err, err);
    }
    __syncthreads();
    stamp(5);
    // ---- phase 3: the row work of row jr, this unit storing and quantizing slice v_ ----
    float4 dv[LG_ROWV];
    if (rowlane) {
        lg_x4u d0, d1, d2, d3;
        const float *pr = a.pout + (size_t)jr * E;
        const int last = nq - 1;
        d0 = lg_ld4_sc_issue<2>(pr + 4 * min(t, last));
        d1 = lg_ld4_sc_issue<2>(pr + 4 * min(t + 256, last));
        d2 = lg_ld4_sc_issue<2>(pr + 4 * min(t + 512, last));
        d3 = lg_ld4_sc_issue<2>(pr + 4 * min(t + 768, last));
        lg_ld4_wait(d0, d1, d2, d3);
        const lg_x4u d[4] = { d0, d1, d2, d3 };
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) dv[v] = make_float4(__uint_as_float(d[v].x), __uint_as_float(d[v].y), __uint_as_float(d[v].z), __uint_as_float(d[v].w));
    }
    stamp(6);
    {
        float ss = 0.0f;
        if (rowlane) {
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(dv[v], ss);
        }
        ss = lg_block_sum256_of512(ss, red3[0]);
        if (rowlane) {
            const float sc = 1.0f / sqrtf(ss / (float)E + a.eps);
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
                const float4 w = wpost[v];
                float4 r;
                r.x = xv[v].x + dv[v].x * sc * w.x;  r.y = xv[v].y + dv[v].y * sc * w.y;
                r.z = xv[v].z + dv[v].z * sc * w.z;  r.w = xv[v].w + dv[v].w * sc * w.w;
                xv[v] = r;
            }
            float4 *xo = (float4 *)(a.x_out + (size_t)jr * E);
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq && v == v_) xo[t + 256 * v] = xv[v];
        }
    }
    {
        float ss = 0.0f;
        if (rowlane) {
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(xv[v], ss);
        }
        ss = lg_block_sum256_of512(ss, red3[1]);
        if (rowlane) {
            const float sc = 1.0f / sqrtf(ss / (float)E + a.eps);
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
                const float4 w = wpre[v];
                xv[v] = make_float4(xv[v].x * sc * w.x, xv[v].y * sc * w.y, xv[v].z * sc * w.z, xv[v].w * sc * w.w);
            }
        }
    }
    if (rowlane) {
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) {
            if (t + 256 * v >= nq || v != v_) continue;
            float d; int sum;
            const uint32_t packed = lg_quant4_8lanes(xv[v], &d, &sum);
            const int quad = t + 256 * v;
            if (a.q_units == 2) {
                uint32_t *blk = (uint32_t *)a.q + (size_t)(quad >> 3) * LG_MU_DWORDS;
                const int dw = quad & 7;
                blk[jr * 8 + ((dw & 1) | ((dw & 2) << 1) | ((dw & 4) >> 1))] = packed;
                if ((t & 7) == 0) *(float2 *)(blk + 64 + 2 * jr) = make_float2(d, 12582912.0f + (float)(8 * sum));
            } else {
                uint32_t *unit = (uint32_t *)a.q + ((size_t)(quad >> 3) * ((M + 2) / 3) + jr / 3) * 32;
                unit[(jr % 3) * 8 + (quad & 7)] = packed;
                if ((t & 7) == 0) *(float2 *)(unit + 24 + 2 * (jr % 3)) = make_float2(d, __int_as_float(sum));
            }
        }
    }
    stamp(7);
}
