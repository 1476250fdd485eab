// lg_fused.h — verify-step kernels that do the row work of a layer themselves.
//
// Between two matmuls of a layer the residual rows are updated, normed and quantized (lg_k_rows).  As a kernel
// of its own that is M workgroups on a 256-CU chip and a launch boundary either side.  Here every workgroup of
// the consuming matmul repeats the row work of all M rows (same lane assignment, same summation order: the
// results are the bits lg_k_rows produces) straight into its LDS operand buffer, and one workgroup also writes
// the new residual.  The repetition costs each workgroup one round trip for 2 x M rows plus the two norm
// weights, and M x E/4 quantizations of four values (about 50 instructions each): for one or two rows that is
// less than the launch it replaces (one-row decode: 2.8 us per layer saved), for four and more rows it is more
// (a 5-row block: +0.3 ms per step, also in the gate/up kernel), so wider blocks keep lg_k_rows.
#pragma once
#include "lg_kernels.h"

struct RowWork {
    const float *x;          // [M][E] residual
    const float *dout;       // [M][E] previous sub-layer output: x += rmsnorm(dout) * w_post; nullptr: x stays as it is
    const float *w_post;     // [E]
    const float *os;         // scalar applied after the add, or nullptr
    float       *x_out;      // [M][E] new residual (written by one workgroup)
    const float *w_pre;      // [E] norm weight applied before quantization
    int          E;
    float        eps;
};

// The rows of a block on NE engines of 256 lanes: engine e (threads 256e..256e+255) takes rows e, e+NE, ...
// NV = float4 per lane and row (ceil(E/1024)).  Rows are taken BJ per engine at a time; every load of such a
// batch goes out before its first use, so a batch costs one round trip (BJ bounds the registers: 2*BJ*NV float4).
// red: [2][LG_HIP_MAX_ROWS_DEV][4] floats of LDS.  sink(j, quad, packed, d, sum) receives the q8 of row j,
// four values at a time (quad = index of the float4 in the row), in all lanes of a group of 8.
// All threads of the workgroup must call it (two barriers per batch inside).
template <int M, int NV, int NE, int BJ, typename Sink>
__device__ __forceinline__ void lg_rows_fused(const RowWork &s, bool write_x, float *red, Sink sink) {
    constexpr int JB = (M + NE - 1) / NE;
    const int t = threadIdx.x & 255, e = NE > 1 ? (int)(threadIdx.x >> 8) : 0, wave = t >> 6;
    const int E = s.E, nq = E >> 2;
    const bool has_d = s.dout != nullptr;                     // false: the rows are only normed and quantized
    float4 wpost[NV], wpre[NV];
    const float4 *wr = (const float4 *)s.w_post, *wp = (const float4 *)s.w_pre;
    const bool has_os = has_d && s.os != nullptr;
    float *red0 = red, *red1 = red + LG_HIP_MAX_ROWS_DEV * 4;
    #pragma unroll
    for (int b0 = 0; b0 < JB; b0 += BJ) {
        float4 xv[BJ][NV], dv[BJ][NV];
        #pragma unroll
        for (int jb = 0; jb < BJ; ++jb) {
            const int j = e + (b0 + jb) * NE;
            if (b0 + jb >= JB || j >= M) continue;
            const float4 *xr = (const float4 *)(s.x + (size_t)j * E), *dr = (const float4 *)(s.dout + (size_t)j * E);
            #pragma unroll
            for (int v = 0; v < NV; ++v) if (t + 256 * v < nq) {
                xv[jb][v] = xr[t + 256 * v];
                dv[jb][v] = has_d ? dr[t + 256 * v] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
        }
        if (b0 == 0) {
            #pragma unroll
            for (int v = 0; v < NV; ++v) if (t + 256 * v < nq) {
                wpost[v] = has_d ? wr[t + 256 * v] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                wpre[v] = wp[t + 256 * v];
            }
        }
        const float osv = has_os ? s.os[0] : 1.0f;
        #pragma unroll
        for (int jb = 0; jb < BJ; ++jb) {
            const int j = e + (b0 + jb) * NE;
            if (b0 + jb >= JB || j >= M || !has_d) continue;
            float ss = 0.0f;
            #pragma unroll
            for (int v = 0; v < NV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(dv[jb][v], ss);
            ss = lg_wave_sum64(ss);
            if ((t & 63) == 0) red0[j * 4 + wave] = ss;
        }
        if (has_d) __syncthreads();
        #pragma unroll
        for (int jb = 0; jb < BJ; ++jb) {
            const int j = e + (b0 + jb) * NE;
            if (b0 + jb >= JB || j >= M) continue;
            float sc = 0.0f;
            if (has_d) {
                const float ssd = (red0[j * 4] + red0[j * 4 + 1]) + (red0[j * 4 + 2] + red0[j * 4 + 3]);
                sc = 1.0f / sqrtf(ssd / (float)E + s.eps);
            }
            float ss = 0.0f;
            #pragma unroll
            for (int v = 0; v < NV; ++v) if (t + 256 * v < nq) {
                float4 r = xv[jb][v];
                if (has_d) {
                    const float4 w = wpost[v], d = dv[jb][v];
                    r.x = r.x + d.x * sc * w.x;  r.y = r.y + d.y * sc * w.y;
                    r.z = r.z + d.z * sc * w.z;  r.w = r.w + d.w * sc * w.w;
                    if (has_os) { r.x = r.x * osv; r.y = r.y * osv; r.z = r.z * osv; r.w = r.w * osv; }
                    xv[jb][v] = r;
                    if (write_x) ((float4 *)(s.x_out + (size_t)j * E))[t + 256 * v] = r;
                }
                ss = lg_sumsq4(r, ss);
            }
            ss = lg_wave_sum64(ss);
            if ((t & 63) == 0) red1[j * 4 + wave] = ss;
        }
        __syncthreads();
        #pragma unroll
        for (int jb = 0; jb < BJ; ++jb) {
            const int j = e + (b0 + jb) * NE;
            if (b0 + jb >= JB || j >= M) continue;
            const float ssx = (red1[j * 4] + red1[j * 4 + 1]) + (red1[j * 4 + 2] + red1[j * 4 + 3]);
            const float sc = 1.0f / sqrtf(ssx / (float)E + s.eps);
            #pragma unroll
            for (int v = 0; v < NV; ++v) {
                if (t + 256 * v >= nq) break;                // nq is a multiple of 64: whole wavefronts
                const float4 w = wpre[v], x = xv[jb][v];
                const float4 h = make_float4(x.x * sc * w.x, x.y * sc * w.y, x.z * sc * w.z, x.w * sc * w.w);
                float d; int sum;
                const uint32_t packed = lg_quant4_8lanes(h, &d, &sum);
                sink(j, t + 256 * v, packed, d, sum);
            }
        }
    }
}
// rows per engine and batch that keep 2*BJ*NV float4 within `budget` float4 registers
__host__ __device__ constexpr int lg_rows_batch(int jb, int nv, int budget) {
    return (budget / (2 * nv) < 1) ? 1 : (budget / (2 * nv) < jb ? budget / (2 * nv) : jb);
}

// Row work + plain matmul (k = E, 8 K segments): the q/k/v projection after the attention norm.
// 256 threads: all four wavefronts do the row work, the first NW of them then take one row group each.
struct RowsMmArgs {
    MmArgs  mm;
    RowWork rows;
};
#define LG_ROWSMM_FIELDS(X, v) X(const float *, rx, rows.x, v) X(const float *, rdout, rows.dout, v) X(const float *, rw_post, rows.w_post, v) X(const float *, rw_pre, rows.w_pre, v) X(const uint8_t *, mw, mm.w, v) X(int, rE, rows.E, v) X(int, mk, mm.k, v) X(int, mm_, mm.m, v) X(const float *, ros, rows.os, v) X(float *, rx_out, rows.x_out, v) X(float, reps, rows.eps, v) X(float *, mout, mm.out, v) X(const int8_t *, mq_in, mm.q_in, v) X(int32_t *, mdots, mm.dots, v)
template <int M, int NV, int NW>
__global__ __launch_bounds__(LG_WG) void lg_k_rows_mm(LG_ROWSMM_FIELDS(LG_XP, _) int p_end_) {
    RowsMmArgs a; LG_ROWSMM_FIELDS(LG_XI, a)
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float red[2 * LG_HIP_MAX_ROWS_DEV * 4];
    const int k = a.mm.k;
    int8_t *lq = (int8_t *)smem;
    float2 *lds = (float2 *)(smem + (size_t)M * k);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nit = (k >> 5) / 8, ngroups = a.mm.m / 8, nb = k >> 5;
    const int g0 = blockIdx.x * NW + (wave < NW ? wave : 0);
    const int gi = g0 < ngroups ? g0 : ngroups - 1;
    const uint8_t *wg[1] = { a.mm.w + (size_t)gi * nit * LG_TILE };
    const int row[1] = { gi * 8 + lane / 8 };
    // tiles in flight: what is requested here arrives under the row work (12B shape, 15 tiles, one row: two 2540 us a decode step, four 2479,
    // eight 2470, sixteen 2509)
    constexpr int RU = NV == 1 ? 2 : M == 1 ? 8 : 4;          // (rows of up to 1024 values have four tiles at most: 22047 -> 22115 us for 8 draft rounds with eight)
    WChunk<1, RU> first;
    if (wave < NW) lg_mm_fetch<1, RU>(first, wg, 0, nit, lane);
    const ActLayout lay = lg_act_layout(k);
    lg_rows_fused<M, NV, 1, lg_rows_batch(M, NV, 40)>(a.rows, blockIdx.x == 0, red, [&](int j, int quad, uint32_t packed, float d, int sum) {
        *(uint32_t *)(lq + (size_t)j * k + (size_t)lg_act_unit(lay, quad >> 2) * 16 + (quad & 3) * 4) = packed;
        if ((threadIdx.x & 7) == 0) lds[j * nb + lg_act_block(lay, quad >> 3)] = make_float2(d, __int_as_float(sum));
    });
    __syncthreads();
    if (wave >= NW || g0 >= ngroups) return;
    float acc[1][M];
    lg_mm_groups<M, 8, 1, false, RU>(wg, first, nit, lq, lds, k, acc, lane, nullptr, a.mm.m, row);
    const int c = lane & 7;
    if (c < M) a.mm.out[(size_t)c * a.mm.m + row[0]] = lg_pick<M>(acc[0], c);
}

// ---------------------------------------------------------------------------------------------
// Plain 8-segment matmul, the K range of every row group cut over KP wavefronts.
// With one row a wavefront that takes its tiles two at a time waits for memory again and again; with four or more the dot phase of lg_k_mm is bound by the instruction issue of its one wavefront per row
// group (about 125 instructions per tile at five rows, ten tiles at k = 2560) while half of the chip's SIMDs have
// nothing to do.  Here wavefront (group, part) takes the tiles [part*nit/KP, (part+1)*nit/KP) of its group: it
// requests all of them at once (and tiles of the next part or the group's last one up to TMAX, which it does not use: none there under a guard
// 1827 -> 1886 us a decode step of the E4B shape, its own last one again 2208 -> 2220 at five rows), forms the exact block dots and the scale products of its tiles, and the float
// chain p = fma(xd*dw, (float)dot, p) then runs through the parts in order (part p starts from the value part
// p-1 left in LDS), so every sum is formed in the order of lg_mm_groups and the result is the same bits.
// Tiles it_lo .. it_lo + nt - 1 of a row group (wq, ws) against the rows in LDS; acc is whole in the last part's wavefront.  xch: [M][64] floats of the group
template <int M, int KP, int TMAX>
__device__ __forceinline__ void lg_mm_ks_sums(const uint4 (&wq)[TMAX], const uint32_t (&ws)[TMAX], int it_lo, int nt, int part, const int8_t *lq, const float2 *lds, int k, int lane, float *xch, float (&acc)[M]) {
    const int c = lane & 7, nb = k >> 5;
    float sc[TMAX][M], fd[TMAX][M];
    #pragma unroll
    for (int u = 0; u < TMAX; ++u) {
        if (u >= nt) continue;                                // (a guard, not a break: the arrays stay in registers)
        const int it = it_lo + u;
        float2 ds[M]; int4 a0[M], a1[M];
        #pragma unroll
        for (int j = 0; j < M; ++j) {
            ds[j] = lds[j * nb + it * 8 + c];
            const int8_t *au = lq + (size_t)j * k + (size_t)(it * 16 + c) * 16;
            a0[j] = *(const int4 *)au; a1[j] = *(const int4 *)(au + 8 * 16);
        }
        __builtin_amdgcn_sched_barrier(0);
        const float dw = lg_h2f((uint16_t)ws[u]);
        #pragma unroll
        for (int j = 0; j < M; ++j) {
            fd[u][j] = (float)lg_block_dot(wq[u], a0[j], a1[j], __float_as_int(ds[j].y));
            sc[u][j] = ds[j].x * dw;
        }
    }
    #pragma unroll
    for (int j = 0; j < M; ++j) acc[j] = 0.0f;
    float *mine = xch + lane;
    #pragma unroll
    for (int p = 0; p < KP; ++p) {
        if (part == p) {
            if (p > 0) {
                #pragma unroll
                for (int j = 0; j < M; ++j) acc[j] = mine[j * 64];
            }
            #pragma unroll
            for (int u = 0; u < TMAX; ++u) {
                if (u >= nt) continue;
                #pragma unroll
                for (int j = 0; j < M; ++j) acc[j] = lg_fmaf(sc[u][j], fd[u][j], acc[j]);
            }
            if (p < KP - 1) {
                #pragma unroll
                for (int j = 0; j < M; ++j) mine[j * 64] = acc[j];
            }
        }
        if (p < KP - 1) __syncthreads();
    }
    if (part != KP - 1) return;
    #pragma unroll
    for (int j = 0; j < M; ++j) acc[j] = lg_sum_seg<8>(acc[j]);
}
template <int M, int KP>
__global__ __launch_bounds__(128 * KP) void lg_k_mm_ks(LG_MM_FIELDS(LG_XP, _) int p_end_) {
    MmArgs a; LG_MM_FIELDS(LG_XI, a)
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int TMAX = (16 + KP - 1) / KP;                  // k <= 4096: at most 16 tiles per group
    const int k = a.k, nb = k >> 5, nit = nb >> 3, ngroups = a.m >> 3;
    int8_t *lq = (int8_t *)smem;
    const float2 *lds = (const float2 *)(smem + (size_t)M * k);
    float *xch = (float *)(smem + (((size_t)M * k + (size_t)M * nb * 8 + 15) & ~(size_t)15));   // [2 groups][M][64 lanes]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, gsel = wave / KP, part = wave - gsel * KP;
    const int g0 = blockIdx.x * 2 + gsel, gi = g0 < ngroups ? g0 : ngroups - 1;
    const int it_lo = part * nit / KP, nt = (part + 1) * nit / KP - it_lo;
    const uint8_t *wg = a.w + (size_t)gi * nit * LG_TILE;
    const CopyBatch rows = lg_load_q8_issue<M>(a.q_in, k, 128 * KP);   // the rows first, then the tiles
    uint4 wq[TMAX]; uint32_t ws[TMAX];
    #pragma unroll
    for (int u = 0; u < TMAX; ++u) {
        const int it = it_lo + u < nit ? it_lo + u : nit - 1;
        wq[u] = lg_ldt16(wg, it, lane);
        ws[u] = lg_ldt2(wg, it, lane);
    }
    __builtin_amdgcn_sched_barrier(0);
    lg_load_q8_commit<M>(rows, a.q_in, k, lq, 128 * KP);
    __syncthreads();
    float acc[M];
    lg_mm_ks_sums<M, KP, TMAX>(wq, ws, it_lo, nt, part, lq, lds, k, lane, xch + (size_t)gsel * M * 64, acc);
    if (part != KP - 1 || g0 >= ngroups) return;
    const int c = lane & 7;
    if (c < M) a.out[(size_t)c * a.m + gi * 8 + (lane >> 3)] = lg_pick<M>(acc, c);
}

// ---------------------------------------------------------------------------------------------
// Matmul against a weight matrix kept in f32 (the per-layer-embedding matrices of QAT conversions, which the
// reference's int8 backend also multiplies unquantized: src/cuda/model-cuda-i8.cu:645-653, :846-895; f16 and bf16
// files are widened to f32 at upload, which is exact).  Activations are the f32 rows themselves.  One wavefront per
// weight row and MC block rows (blockIdx.y: which MC rows of a wider block); order: lane (e/4)%64 takes element e,
// fma in ascending e, adjacent-pair tree over the 64 lanes.  Optional epilogue of the per-layer gate:
// out = gelu(sum) * ipl[row][i].
struct MmfArgs {
    const float *w; int k, m;                                 // [m][k], k a multiple of 256
    const float *x; int ldx, rows;                            // [rows][ldx]
    float *out; int ldo;                                      // [rows][ldo]
    const float *ipl; int ipl_ld;                             // nullptr, or [rows][ipl_ld] (already at the layer's slice)
};
template <int MC>
__global__ __launch_bounds__(LG_WG) void lg_k_mmf(MmfArgs a) {
    const int lane = threadIdx.x & 63, i = blockIdx.x * (LG_WG / 64) + (threadIdx.x >> 6), j0 = blockIdx.y * MC;
    if (i >= a.m) return;
    const float4 *wr = (const float4 *)(a.w + (size_t)i * a.k);
    float acc[MC];
    #pragma unroll
    for (int j = 0; j < MC; ++j) acc[j] = 0.0f;
    for (int q = lane; q < (a.k >> 2); q += 64) {             // (k/4 is a multiple of 64: whole wavefronts)
        const float4 w4 = wr[q];
        #pragma unroll
        for (int j = 0; j < MC; ++j) {
            const int jj = j0 + j < a.rows ? j0 + j : a.rows - 1;             // past the block: the last row again, never stored
            const float4 x4 = ((const float4 *)(a.x + (size_t)jj * a.ldx))[q];
            acc[j] = lg_fmaf(w4.x, x4.x, acc[j]); acc[j] = lg_fmaf(w4.y, x4.y, acc[j]);
            acc[j] = lg_fmaf(w4.z, x4.z, acc[j]); acc[j] = lg_fmaf(w4.w, x4.w, acc[j]);
        }
    }
    #pragma unroll
    for (int j = 0; j < MC; ++j) acc[j] = lg_wave_sum64(acc[j]);
    if (lane < MC && j0 + lane < a.rows) {
        float v = lg_pick<MC>(acc, lane);
        if (a.ipl) v = lg_gelu_d(v) * a.ipl[(size_t)(j0 + lane) * a.ipl_ld + i];
        a.out[(size_t)(j0 + lane) * a.ldo + i] = v;
    }
}

// The residual update ahead of the per-layer gate and the gate itself in one launch (verify blocks of models that keep the gate
// in a float type; lg_k_rows_plegate does the same for q4_0): workgroup (i, y) forms the updated rows 4y..4y+3, x + rmsnorm(dout) * w_post,
// in LDS, repeating what lg_k_rows does, and its wavefronts run row i of the gate against one of them each in
// lg_k_mmf's order.  Workgroups 0..3 store the updated rows.  A kernel boundary and a loop of dependent loads less: the gate's 256 rows were 64
// workgroups that fetched weights and rows step by step.  E4B width, 4 rows: 4.3 + 8.2 -> 6.3 us.
struct RowsMmfArgs {
    const float *x, *dout, *w_post;    // [M][k], [M][k] (four slabs of it when dparts = 4), [k]
    int          dparts;
    float       *x_out;                // [M][k]
    float        eps;
    const float *w; int k, m;          // gate [m][k], k a multiple of 256
    const float *ipl; int ipl_ld;      // [M][ipl_ld], at the layer's slice
    float       *out;                  // [M][m]
};
#define LG_RMMF_ROWS 4                     // rows of a workgroup
template <int M>
__global__ __launch_bounds__(LG_WG) void lg_k_rows_mmf(RowsMmfArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    float4 *rl = (float4 *)smem;                              // [RB][k/4]
    constexpr int RB = M < LG_RMMF_ROWS ? M : LG_RMMF_ROWS;
    __shared__ float red[RB][4];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), i = blockIdx.x, j0 = M > RB ? (int)blockIdx.y * RB : 0, nq = a.k >> 2, nit = a.k >> 8;
    float4 wp[LG_ROWV], gw[LG_MAXV], xv[RB][LG_ROWV], dv[RB][LG_ROWV];
    #pragma unroll
    for (int r = 0; r < RB; ++r) {                            // (past the block: its last row again, never stored)
        const int j = min(j0 + r, M - 1);
        const float4 *xr = (const float4 *)(a.x + (size_t)j * a.k), *dr = (const float4 *)(a.dout + (size_t)j * a.k);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) { dv[r][v] = dr[t + 256 * v]; xv[r][v] = xr[t + 256 * v]; }
    }
    #pragma unroll
    for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) wp[v] = ((const float4 *)a.w_post)[t + 256 * v];
    #pragma unroll
    for (int v = 0; v < LG_MAXV; ++v) if (v < nit) gw[v] = ((const float4 *)(a.w + (size_t)i * a.k))[lane + 64 * v];
    const float iplv = a.ipl[(size_t)min(j0 + wave, M - 1) * a.ipl_ld + i];
    __builtin_amdgcn_sched_barrier(0);
    if (a.dparts == 4) {                                      // top of the K-segment tree of a matmul cut by K quarter
        const size_t slab = (size_t)M * nq;
        #pragma unroll
        for (int r = 0; r < RB; ++r) {
            const float4 *dr = (const float4 *)(a.dout + (size_t)min(j0 + r, M - 1) * a.k);
            #pragma unroll
            for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
                const float4 p1 = dr[slab + t + 256 * v], p2 = dr[2 * slab + t + 256 * v], p3 = dr[3 * slab + t + 256 * v], p0 = dv[r][v];
                dv[r][v] = make_float4((p0.x + p1.x) + (p2.x + p3.x), (p0.y + p1.y) + (p2.y + p3.y), (p0.z + p1.z) + (p2.z + p3.z), (p0.w + p1.w) + (p2.w + p3.w));
            }
        }
    }
    #pragma unroll
    for (int r = 0; r < RB; ++r) {
        float ss = 0.0f;
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) ss = lg_sumsq4(dv[r][v], ss);
        ss = lg_wave_sum64(ss);
        if (lane == 0) red[r][wave] = ss;
    }
    __syncthreads();
    #pragma unroll
    for (int r = 0; r < RB; ++r) {
        const float ss = (red[r][0] + red[r][1]) + (red[r][2] + red[r][3]);
        const float sc = 1.0f / sqrtf(ss / (float)a.k + a.eps);
        #pragma unroll
        for (int v = 0; v < LG_ROWV; ++v) if (t + 256 * v < nq) {
            const float4 w = wp[v], d = dv[r][v];
            float4 x = xv[r][v];
            x.x = x.x + d.x * sc * w.x;  x.y = x.y + d.y * sc * w.y;
            x.z = x.z + d.z * sc * w.z;  x.w = x.w + d.w * sc * w.w;
            rl[r * nq + t + 256 * v] = x;
            if (i == r && j0 + r < M) ((float4 *)(a.x_out + (size_t)(j0 + r) * a.k))[t + 256 * v] = x;
        }
    }
    __syncthreads();
    if (wave >= RB || j0 + wave >= M) return;
    float acc = 0.0f;
    #pragma unroll
    for (int v = 0; v < LG_MAXV; ++v) if (v < nit) {
        const float4 x = rl[wave * nq + lane + 64 * v], w = gw[v];
        acc = lg_fmaf(w.x, x.x, acc); acc = lg_fmaf(w.y, x.y, acc); acc = lg_fmaf(w.z, x.z, acc); acc = lg_fmaf(w.w, x.w, acc);
    }
    acc = lg_wave_sum64(acc);
    if (lane == 0) a.out[(size_t)(j0 + wave) * a.m + i] = lg_gelu_d(acc) * iplv;
}

// ---------------------------------------------------------------------------------------------
// lm_head for verify blocks of 4..8 rows on the matrix cores: lg_k_geglu_m's tile loop (row-block tiles of the
// vocabulary matrix, a wavefront = 64 vocabulary rows x one of the 8 K segments, two v_mfma_i32_32x32x32_i8 per
// tile whatever M is, the activations in the same 80-dword block order) with lg_k_mm_head's epilogue: the 8
// segment sums of a logit meet in the adjacent-pair tree, soft cap, optional store, running argmax per draft row
// (first maximum: the lower index wins ties).  A workgroup walks `passes` consecutive blocks of 64 rows; the
// first tiles of the next block are requested while the last of this one are multiplied, and the segment sums
// go through one of two LDS buffers in turn, so a block costs one barrier.
template <int M>
__global__ __launch_bounds__(512, 2) void lg_k_head_m(LG_HEAD_FIELDS(LG_XP, _) int p_end_) {
    HeadArgs a; LG_HEAD_FIELDS(LG_XI, a)
    extern __shared__ __align__(16) unsigned char smem[];     // [8 segments][nit][80 dwords]
    __shared__ float red[2][8][LG_HIP_MAX_ROWS_DEV][64];
    constexpr int CH = 2;
    const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
    const int s = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));      // K segment of this wavefront, and its draft row in the epilogue
    const int nb = a.k >> 5, nit = nb >> 3, nblk = a.n_vocab >> 6;
    const int t0 = blockIdx.x * a.passes, np = nblk - t0 < a.passes ? nblk - t0 : a.passes;
    uint4 wq[CH], nwq[CH]; uint32_t wd[CH], nwd[CH];
    auto fetch = [&](int p, int it0) {
        const uint8_t *wt = a.w + ((size_t)(t0 + p) * nb + (size_t)s * nit) * LG_TILE;
        #pragma unroll
        for (int u = 0; u < CH; ++u) {
            const int it = it0 + u < nit ? it0 + u : nit - 1;
            nwq[u] = lg_ldt16(wt, it, lane);
            nwd[u] = lg_ldt2(wt, it, lane);
        }
    };
    unsigned char *la = smem + (size_t)s * nit * (LG_MU_DWORDS * 4);
    {   // the wavefront's K segment of the activations, once (wave-private, no barrier); its first loads go out
        // ahead of the first weight tiles
        const uint4 *src = (const uint4 *)(a.q_in + (size_t)s * nit * (LG_MU_DWORDS * 4));
        const int nu = nit * (LG_MU_DWORDS / 4);
        {   // (every lane takes part, past the end with the last unit again: the tiles are requested in here)
            const int i0 = min(lane, nu - 1), i1 = min(lane + 64, nu - 1), i2 = min(lane + 128, nu - 1), i3 = min(lane + 192, nu - 1);
            const uint4 t0v = src[i0], t1 = src[i1], t2 = src[i2], t3 = src[i3];
            __builtin_amdgcn_sched_barrier(0);
            if (np > 0) fetch(0, 0);
            __builtin_amdgcn_sched_barrier(0);
            ((uint4 *)la)[i0] = t0v; ((uint4 *)la)[i1] = t1; ((uint4 *)la)[i2] = t2; ((uint4 *)la)[i3] = t3;
        }
        for (int i0 = lane + 256; i0 < nu; i0 += 256) {
            const int i1 = min(i0 + 64, nu - 1), i2 = min(i0 + 128, nu - 1), i3 = min(i0 + 192, nu - 1);
            const uint4 t0v = src[i0], t1 = src[i1], t2 = src[i2], t3 = src[i3];
            __builtin_amdgcn_sched_barrier(0);
            ((uint4 *)la)[i0] = t0v; ((uint4 *)la)[i1] = t1; ((uint4 *)la)[i2] = t2; ((uint4 *)la)[i3] = t3;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    lg_v16i magic;                                            // (float)(dot - 8*sum) in one subtraction: see lg_k_geglu_m
    #pragma unroll
    for (int i = 0; i < 16; ++i) magic[i] = 0x4B400000;
    const int arow = n < 8 ? n : 7;
    float best = -INFINITY;                                   // wavefront s < M tracks draft row s, one vocabulary row per lane and block
    int besti = 0x7fffffff;
    for (int p = 0; p < np; ++p) {
        float p0[4] = { 0.0f, 0.0f, 0.0f, 0.0f }, p1[4] = { 0.0f, 0.0f, 0.0f, 0.0f };
        for (int it0 = 0; it0 < nit; it0 += CH) {
            #pragma unroll
            for (int u = 0; u < CH; ++u) { wq[u] = nwq[u]; wd[u] = nwd[u]; }
            if (it0 + CH < nit) fetch(p, it0 + CH);
            else if (p + 1 < np) fetch(p + 1, 0);
            #pragma unroll
            for (int c = 0; c < CH; ++c) {
                if (it0 + c < nit) {
                    const unsigned char *lb = la + (size_t)(it0 + c) * (LG_MU_DWORDS * 4);
                    const lg_v4i av = *(const lg_v4i *)(lb + arow * 32 + h * 16);
                    const int4 sc0 = *(const int4 *)(lb + 256 + h * 32), sc1 = *(const int4 *)(lb + 256 + h * 32 + 16);
                    const uint4 q = wq[c];
                    const lg_v2u s0 = __builtin_amdgcn_permlane32_swap(q.x, q.z, false, false);
                    const lg_v2u s1 = __builtin_amdgcn_permlane32_swap(q.y, q.w, false, false);
                    const lg_v2u sd = __builtin_amdgcn_permlane32_swap(wd[c], wd[c], false, false);
                    lg_v4i b0, b1;
                    b0.x = s0.x & 0x0F0F0F0F; b0.y = s1.x & 0x0F0F0F0F; b0.z = (s0.x >> 4) & 0x0F0F0F0F; b0.w = (s1.x >> 4) & 0x0F0F0F0F;
                    b1.x = s0.y & 0x0F0F0F0F; b1.y = s1.y & 0x0F0F0F0F; b1.z = (s0.y >> 4) & 0x0F0F0F0F; b1.w = (s1.y >> 4) & 0x0F0F0F0F;
                    const float w0 = lg_h2f((uint16_t)sd.x), w1 = lg_h2f((uint16_t)sd.y);
                    const lg_v16i d0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, b0, magic, 0, 0, 0);
                    const lg_v16i d1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, b1, magic, 0, 0, 0);
                    const float xd[4] = { __int_as_float(sc0.x), __int_as_float(sc0.z), __int_as_float(sc1.x), __int_as_float(sc1.z) };
                    const float cf[4] = { __int_as_float(sc0.y), __int_as_float(sc0.w), __int_as_float(sc1.y), __int_as_float(sc1.w) };
                    #pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        p0[i] = lg_fmaf(xd[i] * w0, __int_as_float(d0[i]) - cf[i], p0[i]);
                        p1[i] = lg_fmaf(xd[i] * w1, __int_as_float(d1[i]) - cf[i], p1[i]);
                    }
                }
            }
        }
        float (*rb)[LG_HIP_MAX_ROWS_DEV][64] = red[p & 1];
        #pragma unroll
        for (int i = 0; i < 4; ++i) { rb[s][4 * h + i][n] = p0[i]; rb[s][4 * h + i][32 + n] = p1[i]; }
        __syncthreads();                                      // (the buffer written two blocks ago was read before the barrier of the last block)
        if (s < M) {
            float g[8];
            #pragma unroll
            for (int c = 0; c < 8; ++c) g[c] = rb[c][s][lane];
            float v = ((g[0] + g[1]) + (g[2] + g[3])) + ((g[4] + g[5]) + (g[6] + g[7]));
            if (a.softcap > 0.0f) v = a.softcap * lg_tanhf(v / a.softcap);
            const int row = (t0 + p) * 64 + lane;
            if (a.logits) a.logits[(size_t)s * a.n_vocab + row] = v;
            if (v > best) { best = v; besti = row; }          // (rows ascend with p: a later equal value never replaces)
        }
    }
    if (s < M) {
        #pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const float ov = __shfl_xor(best, o);
            const int oi = __shfl_xor(besti, o);
            if (ov > best || (ov == best && oi < besti)) { best = ov; besti = oi; }
        }
        if (lane == 0) { a.pval[(size_t)blockIdx.x * M + s] = best; a.pidx[(size_t)blockIdx.x * M + s] = besti; }
    }
}

// ---------------------------------------------------------------------------------------------
// Matmul of a verify block (4..8 rows) against a long-row matrix (S = 32 K segments per row, ffn_down), cut by K
// quarter: workgroup (x, q) takes 8 rows per wavefront and the segments 8q .. 8q+7 of them, so it stages a quarter
// of the activations (24 KB at 5 x 15360, where a workgroup that owns whole rows stages all 96 KB and a CU then
// holds a single workgroup of four wavefronts).  A lane is (row r8, segment sg) and walks the segment's tiles with
// the same serial fma chain as lg_k_mm; the 8 segment sums of a row meet in the same adjacent-pair tree (lg_sum8),
// which is the bottom of the 32-segment tree.  The quarter's partial sums go to slab q of `out` ([4][M][m]); the
// consumer adds the top of the tree, (p0+p1)+(p2+p3).
template <int M>
__global__ __launch_bounds__(320, 2) void lg_k_mm_kq(LG_MM_FIELDS(LG_XP, _) int p_end_) {
    MmArgs a; LG_MM_FIELDS(LG_XI, a)
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = a.nthreads >> 6;
    const int q = blockIdx.y, nb = a.k >> 5, nit = nb >> 5;
    uint4 *lq = (uint4 *)smem;                                // [M][nit][2 halves][8 segments] 16-byte units
    float2 *lds = (float2 *)(smem + (size_t)M * nit * 256);   // [M][nit][8 segments] {scale, sum}
    const int r8 = lane >> 3, sg = lane & 7, c = 8 * q + sg;
    const int row0 = (blockIdx.x * nw + wave) * 8;
    const int row = row0 + r8 < a.m ? row0 + r8 : a.m - 1;    // ragged tail: recompute the last row
    // tiles hold two rows x 32 segments: this lane's 16 nibble bytes sit at (row & 1) * 32 + c
    const uint8_t *wt = a.w + (size_t)(row >> 1) * nit * LG_TILE + ((row & 1) * 32 + c) * 16;
    const uint8_t *ws = a.w + (size_t)(row >> 1) * nit * LG_TILE + 1024 + ((row & 1) * 32 + c) * 2;
    constexpr int U = 4;
    struct Chunk { uint4 q[U]; uint32_t s[U]; } cur, nxt;
    auto fetch = [&](Chunk &w, int it0) {
        #pragma unroll
        for (int u = 0; u < U; ++u) {
            const int it = it0 + u < nit ? it0 + u : nit - 1;
            w.q[u] = lg_ldw16(wt + (size_t)it * LG_TILE);
            w.s[u] = lg_ldw2(ws + (size_t)it * LG_TILE);
        }
    };
    {   // the quarter of the activations: per (row, tile) two runs of 8 units and one run of 8 {scale, sum} = 20 x 16 bytes
        // (their first pass is requested ahead of the first weight tiles and stored after them: loads return in order)
        const int n = M * nit * 20, T = a.nthreads;
        const uint4 *gq = (const uint4 *)a.q_in, *gd = (const uint4 *)(a.q_in + (size_t)M * a.k);
        auto where = [&](int i, int &dst) -> const uint4 * {
            const int jt = i / 20, r = i - jt * 20, j = jt / nit, it = jt - j * nit;
            dst = r < 16 ? jt * 16 + r : M * nit * 16 + jt * 4 + (r - 16);
            return r < 16 ? gq + ((size_t)j * (a.k >> 4) + it * 64 + (r >> 3) * 32 + 8 * q + (r & 7))
                          : gd + ((((size_t)j * nb + it * 32 + 8 * q) >> 1) + (r - 16));
        };
        {   // four loads in flight per thread (past the end: the last unit again); every thread takes part in the first pass
            const int i0 = threadIdx.x;
            int d0, d1, d2, d3;
            const uint4 *s0 = where(min(i0, n - 1), d0), *s1 = where(min(i0 + T, n - 1), d1);
            const uint4 *s2 = where(min(i0 + 2 * T, n - 1), d2), *s3 = where(min(i0 + 3 * T, n - 1), d3);
            const uint4 v0 = *s0, v1 = *s1, v2 = *s2, v3 = *s3;
            __builtin_amdgcn_sched_barrier(0);
            fetch(nxt, 0);                                    // (weights depend on nothing)
            __builtin_amdgcn_sched_barrier(0);
            lq[d0] = v0; lq[d1] = v1; lq[d2] = v2; lq[d3] = v3;
        }
        for (int i0 = threadIdx.x + 4 * T; i0 < n; i0 += 4 * T) {
            int d0, d1, d2, d3;
            const uint4 *s0 = where(min(i0, n - 1), d0), *s1 = where(min(i0 + T, n - 1), d1);
            const uint4 *s2 = where(min(i0 + 2 * T, n - 1), d2), *s3 = where(min(i0 + 3 * T, n - 1), d3);
            const uint4 v0 = *s0, v1 = *s1, v2 = *s2, v3 = *s3;
            __builtin_amdgcn_sched_barrier(0);
            lq[d0] = v0; lq[d1] = v1; lq[d2] = v2; lq[d3] = v3;
        }
    }
    __syncthreads();
    if (row0 >= a.m) return;
    float acc[M];
    #pragma unroll
    for (int j = 0; j < M; ++j) acc[j] = 0.0f;
    for (int it0 = 0; it0 < nit; it0 += U) {
        cur = nxt;
        if (it0 + U < nit) fetch(nxt, it0 + U);
        #pragma unroll
        for (int u = 0; u < U; ++u) {
            if (it0 + u < nit) {
                const int it = it0 + u;
                float2 ds[M]; int4 a0[M], a1[M];
                #pragma unroll
                for (int j = 0; j < M; ++j) {
                    const int jt = j * nit + it;
                    ds[j] = lds[jt * 8 + sg];
                    a0[j] = *(const int4 *)(lq + jt * 16 + sg); a1[j] = *(const int4 *)(lq + jt * 16 + 8 + sg);
                }
                __builtin_amdgcn_sched_barrier(0);
                const float dw = lg_h2f((uint16_t)cur.s[u]);
                #pragma unroll
                for (int j = 0; j < M; ++j) {
                    const int dot = lg_block_dot(cur.q[u], a0[j], a1[j], __float_as_int(ds[j].y));
                    acc[j] = lg_fmaf(ds[j].x * dw, (float)dot, acc[j]);
                }
            }
        }
    }
    #pragma unroll
    for (int j = 0; j < M; ++j) acc[j] = lg_sum8(acc[j]);
    if (sg < M && row0 + r8 < a.m) a.out[((size_t)q * M + sg) * a.m + row] = lg_pick<M>(acc, sg);
}

// ---------------------------------------------------------------------------------------------
// Attention tiles of a verify block for layers with many tiles (long global contexts, wide sliding windows):
// a workgroup serves ALL rows of the block against its tiles, where lg_k_attn runs a workgroup per row and stages
// every tile once per row.  FQ = false: the queries arrive normed and rotated
// (lg_k_qkv_post has run and has written the block's K/V rows to the cache).  FQ = true: the kernel does that work
// itself from the raw projections, one launch less per layer: every workgroup norms and rotates the M*G queries of
// its kv head (a wavefront per query), and the workgroup whose tiles hold rows of
// the block builds those K/V rows into LDS and stores them to the cache (K row r by wavefront
// r % 4, V row r by wavefront 3 - r % 4; the ring has spare rows, so no row another workgroup reads is overwritten).
// Same arithmetic and order as
// lg_k_attn: score = (a0+a1)+(a2+a3) over four fma chains, tile max / exp / 32-lane tree sum, value accumulation
// over the slots ascending; the partials go to the same slots and lg_k_attn_merge finishes them.
//
// A unit is one (row, query head) pair, M*G of them, in groups of 16.  Both products run on v_mfma_f32_16x16x1_4b_f32,
// one fma per output and step as in lg_k_wide_attn: the four blocks of a score step are its four chains, those of a value
// step (one slot) are four runs of 16 dims.  A workgroup is two pairs of wavefronts.  Up to 16 units: a pair to a tile, two
// tiles to a workgroup; more: a pair to a unit group of one tile.  The wavefronts of a pair take 16 keys each, then half of
// the dims each.  K and V go from the cache straight into registers in operand order (16 bytes of a K row by four lanes,
// dealt to the chains by lg_deal4; a run of a value row, one slot after another), all requested at the start, so the tile's
// memory round trip passes under the preparation of the queries; LDS holds only queries, weights and the block's own rows.
// Bound by its products (32 cycles each, 128 to a wavefront and tile) and about 500 vector instructions beside them, which run
// one after the other; without the tile's loads and the partials' stores it takes 28 of its 33 us.  On the vector units, every K and V
// row through LDS and three units to a read, LDS reads bounded it.  8 rows of 8 heads over 2 at 20011 keys 61 -> 33 us, 5 rows of
// 16 over 8 at 8192 keys 42 -> 31, at 2048 keys of 8 over 2 15.2 -> 14.2.
// Slots outside a row's keys have weight zero and zeroed values (or ones that another row of the block sees), and
// fma(0, v, acc) is acc for every acc that a chain started at +0 can hold and every finite v; a tile that gives results that
// are not finite where the rows' keys differ is computed again without those slots (5 rows of 16 over 8 at 8192 keys: a step
// 3386 -> 3396 us for the test of the results, which is out of the way of the tiles in between).
//
// Few units on few tiles go to lg_k_attn_few below.

// What both kernels do themselves where FQ: the queries of the workgroup's kv head, and the block's K and V rows that lie in its tiles
// (`mine`: whether position t does).  The queries arrive in LDS as [unit][c][HD/4], element i at c = i % 4, i / 4, QST floats a unit.
template <int M, int HD>
struct AttnRowsPrep {
    static constexpr int QST = HD + 4;                        // floats per staged query: off the bank period
    static constexpr int JOBS = 2 * ((M + 3) / 4);            // K and V rows of the block one wavefront may have to build
    static constexpr int QBATCH = 4;                          // queries one wavefront prepares at a time
    HeadVec<1> hj[JOBS], hq[QBATCH], wk, wq;
    RopeVals<1> rv;
    // What the preparation reads is requested ahead of the tile (loads return in order): the block's projections
    // come from the cache levels, the tile from memory, so the queries are prepared while the tile is on its way.
    template <typename Mine>
    __device__ __forceinline__ void request(const AttnArgs &a, int kvh, int G, int wave, int tnew, bool any, Mine &&mine) {
        const int units = M * G;
        rv = lg_rope_load<1>(a.rope_tab, a.rope_ff, HD);
        wq = lg_head_load<1>(a.q_norm, HD);
        #pragma unroll
        for (int b = 0; b < QBATCH; ++b) {                    // unit u = (row j, head g), by wavefront u % 4
            const int u = wave + b * (LG_WG / 64) < units ? wave + b * (LG_WG / 64) : min(wave, units - 1), j = u / G, g = u - j * G;
            hq[b] = lg_head_load<1>(a.qkv + (size_t)j * a.ld + (size_t)(kvh * G + g) * HD, HD);
        }
        wk = lg_head_load<1>(any ? a.k_norm : a.q_norm, HD);  // (no K rows to build: k_norm may not exist)
        #pragma unroll
        for (int u = 0; u < JOBS; ++u) {                      // first half of the slots: K rows wave, wave+4; second half: V rows 3-wave, 7-wave
            const bool isv = u >= JOBS / 2;
            const int r = (isv ? 3 - wave : wave) + 4 * (u % (JOBS / 2)), t = tnew + r;
            if (any && r < M && mine(t)) hj[u] = lg_head_load<1>(a.qkv + (size_t)r * a.ld + (isv ? a.v_off : a.k_off) + (size_t)kvh * HD, HD);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void queries(const AttnArgs &a, const StepCtl *ctl, int kvh, int G, int wave, int lane, float *qs) {
        const int units = M * G;
        // a batch in stages, so that the sums and the rotary of its queries overlap: norms of all, each into its own
        // slot of qs in natural order; all rotary pairs read back; then the slots rewritten in the staged order
        // (a unit past the last repeats the batch's first one, a slot of this wavefront, and stores nothing)
        auto unit_of = [&](int base, int b) { return base + b * (LG_WG / 64) < units ? base + b * (LG_WG / 64) : base; };
        for (int base = wave; base < units; base += QBATCH * (LG_WG / 64)) {
            if (base != wave) {
                #pragma unroll
                for (int b = 0; b < QBATCH; ++b) {
                    const int u = unit_of(base, b), j = u / G, g = u - j * G;
                    hq[b] = lg_head_load<1>(a.qkv + (size_t)j * a.ld + (size_t)(kvh * G + g) * HD, HD);
                }
            }
            HeadVec<1> nq[QBATCH];
            #pragma unroll
            for (int b = 0; b < QBATCH; ++b) nq[b] = lg_head_norm<1>(hq[b], wq, true, HD, a.eps);
            #pragma unroll
            for (int b = 0; b < QBATCH; ++b)
                if (4 * lane < HD) *(float4 *)(qs + (size_t)unit_of(base, b) * QST + 4 * lane) = nq[b].x[0];
            lg_wave_lds_sync();
            float lo[QBATCH][2], hi[QBATCH][2];
            #pragma unroll
            for (int b = 0; b < QBATCH; ++b) {
                const int u = unit_of(base, b), j = u / G;
                const float *vec = qs + (size_t)u * QST;
                #pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int p = min(lane + 64 * i, HD / 2 - 1);
                    const float ang = (float)(ctl->pos + j) * rv.tab[i] / rv.ff[i];
                    float sn, cs;
                    lg_sincosf(ang, &sn, &cs);
                    const float x0 = vec[p], x1 = vec[p + HD / 2];
                    lo[b][i] = x0 * cs - x1 * sn; hi[b][i] = x0 * sn + x1 * cs;
                }
            }
            lg_wave_lds_sync();                               // (LDS serves a wavefront in order: every read above is ahead of the stores below)
            #pragma unroll
            for (int b = 0; b < QBATCH; ++b) {
                const int u = base + b * (LG_WG / 64);
                float *qd = qs + (size_t)unit_of(base, b) * QST;
                #pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int p = lane + 64 * i, p1 = p + HD / 2;
                    if (u >= units || p >= HD / 2) continue;
                    qd[(p & 3) * (HD / 4) + (p >> 2)] = lo[b][i];
                    qd[(p1 & 3) * (HD / 4) + (p1 >> 2)] = hi[b][i];
                }
            }
            lg_wave_lds_sync();
        }
    }
    // k_row(r, t, lo, hi per rotary pair p), v_row(r, t, the lane's four values as f16)
    template <typename Mine, typename KRow, typename VRow>
    __device__ __forceinline__ void rows(const AttnArgs &a, int wave, int lane, int tnew, float *vec, Mine &&mine, KRow &&k_row, VRow &&v_row) {
        HeadVec<1> nr[JOBS];
        bool on[JOBS];
        #pragma unroll
        for (int u = 0; u < JOBS; ++u) {                      // the norms of all of them first: their sums overlap
            const bool isv = u >= JOBS / 2;
            const int r = (isv ? 3 - wave : wave) + 4 * (u % (JOBS / 2)), t = tnew + r;
            on[u] = r < M && mine(t);
            if (on[u]) nr[u] = lg_head_norm<1>(hj[u], wk, !isv, HD, a.eps);
        }
        #pragma unroll
        for (int u = 0; u < JOBS; ++u) {
            const bool isv = u >= JOBS / 2;
            const int r = (isv ? 3 - wave : wave) + 4 * (u % (JOBS / 2)), t = tnew + r;
            if (!on[u]) continue;
            if (isv) {                                        // V: no rotary, straight from the registers
                if (4 * lane < HD) v_row(r, t, make_uint2((uint32_t)lg_f2h(nr[u].x[0].x) | ((uint32_t)lg_f2h(nr[u].x[0].y) << 16),
                                                          (uint32_t)lg_f2h(nr[u].x[0].z) | ((uint32_t)lg_f2h(nr[u].x[0].w) << 16)));
            } else lg_head_rope<1>(nr[u], HD, t, rv, vec, [&](int p, float lo, float hi) { k_row(r, t, p, lg_f2h(lo), lg_f2h(hi)); });
        }
    }
    // FQ = false: the queries as lg_k_qkv_post left them
    __device__ static __forceinline__ void copy_queries(const AttnArgs &a, int kvh, int G, float *qs) {
        const int units = M * G;
        constexpr int QB = 4;                                 // float4 of query per thread and pass
        const int nq4 = units * (HD / 4);
        for (int base = 0; base < nq4; base += QB * LG_WG) {
            float4 qreg[QB];
            #pragma unroll
            for (int i = 0; i < QB; ++i) {
                const int idx = min(base + (int)threadIdx.x + i * LG_WG, nq4 - 1);
                const int u = idx / (HD / 4), g4 = idx - u * (HD / 4), j = u / G, g = u - j * G;
                qreg[i] = *(const float4 *)(a.q + (size_t)j * a.H * HD + (size_t)(kvh * G + g) * HD + 4 * g4);
            }
            #pragma unroll
            for (int i = 0; i < QB; ++i) {
                const int idx = base + (int)threadIdx.x + i * LG_WG;
                if (idx < nq4) {
                    const int u = idx / (HD / 4), g4 = idx - u * (HD / 4);
                    float *qd = qs + (size_t)u * QST + g4;
                    qd[0] = qreg[i].x; qd[HD / 4] = qreg[i].y; qd[2 * (HD / 4)] = qreg[i].z; qd[3 * (HD / 4)] = qreg[i].w;
                }
            }
        }
    }
};
template <int HD>
struct AttnRowsGeo {
    static constexpr int QST = HD + 4;
    static constexpr int EST = 36;                            // floats per unit's weights of a tile
    static size_t bytes(int units, bool fq) {         // fq: the block's K and V rows, and a vector of staging per wavefront for the rotary
        return (size_t)((units + 15) / 16) * 16 * QST * 4 + (size_t)2 * 16 * EST * 4 + (fq ? (size_t)2 * LG_HIP_MAX_ROWS_DEV * HD * 2 + (size_t)(LG_WG / 64) * HD * 4 : 0);
    }
};
// tiles a workgroup takes at a time
__host__ __device__ static inline int lg_attn_rows_tiles(int units) { return units <= 16 ? 2 : 1; }
template <int M, int HD, bool FQ = false>
__global__ __launch_bounds__(LG_WG, 2) void lg_k_attn_rows(const StepCtl *ctl, LG_ATTN_FIELDS(LG_XP, _) int p_end_) {
    AttnArgs a; LG_ATTN_FIELDS(LG_XI, a)
    using Geo = AttnRowsGeo<HD>;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float mxs[4][16], lsum[4][16];                 // a wavefront's maxima and sums over its 16 keys
    const int G = a.H / a.nkv, units = M * G, ng = (units + 15) >> 4;
    float *qs = (float *)smem;                                // [unit][c][HD/4]: element i at c = i % 4, i / 4
    float *es = qs + (size_t)ng * 16 * Geo::QST;              // [pair][unit][EST]
    uint16_t *nk = (uint16_t *)(es + 2 * 16 * Geo::EST);      // FQ: the block's K rows, then its V rows, [M][HD] each
    uint16_t *nv = nk + (size_t)LG_HIP_MAX_ROWS_DEV * HD;
    float *hv = (float *)(nv + (size_t)LG_HIP_MAX_ROWS_DEV * HD);       // FQ: [wavefront][HD] staging of the rotary
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), pair = wave >> 1, half = wave & 1;
    const int n = lane & 15, c = lane >> 4;
    const int kvh = blockIdx.y;
    const int pos0 = ctl->pos + a.pos_off, plast = pos0 + M - 1;
    // FQ: positions tnew..plast are rows of the block itself (none when the layer reads another layer's cache)
    const int tnew = (FQ && a.kcw) ? ctl->pos : 0x7FFFFFFF;
    const int start0 = lg_win_start(pos0, a.window), first = start0 >> 5, last = plast >> 5;
    // the workgroup's tiles: tw from first + tw * b on, b = blockIdx.x, blockIdx.x + gx, ...
    const int tw = ng == 1 ? 2 : 1, gx = a.gx, b0 = blockIdx.x, nb = (last - first + tw) / tw;
    if (b0 >= nb) return;                                     // no row of the block has keys here
    auto mine = [&](int t) { return (((t >> 5) - first) / tw) % gx == b0; };      // position t lies in a tile of this workgroup

    const bool any = FQ && tnew <= plast && (mine(tnew) || mine(plast));         // this workgroup's tiles hold rows of the block (at most two tiles do)
    AttnRowsPrep<M, HD> prep;
    if constexpr (FQ) prep.request(a, kvh, G, wave, tnew, any, mine);
    // a tile: this lane's key (K row, 64-byte pieces by four lanes) and its dims of every slot's value row
    constexpr int NS = HD / 32, NK = HD >= 128 ? HD / 128 : 1;          // pieces of a K row; value products per slot and wavefront
    uint4 kw[NS];
    uint32_t vw[32];
    const int vd = (HD >= 128 ? half * (HD / 2) : 0) + NK * lane;       // this lane's first dim (64-wide heads: both wavefronts all of them)
    auto tile_of = [&](int b) { const int t = first + b * tw + (ng == 1 ? pair : 0); return t <= last ? t : last; };
    // (a tile lies within the ring in one piece: a ring is a multiple of 32 rows, or as long as the positions go.  Rows past its
    // end are no keys of any row: the last row again, and zeros.)
    auto fetch_k = [&](int b) {
        const int rr = (tile_of(b) << 5) % a.seq + 16 * half + n;
        const size_t ko = (size_t)(rr < a.seq ? rr : a.seq - 1) * a.kv_dim + (size_t)kvh * HD + c * 8;
        #pragma unroll
        for (int s = 0; s < NS; ++s) kw[s] = a.kc4(ko + 32 * s);
    };
    auto fetch_v = [&](int b) {                               // buffer loads: the slot's row in a scalar register
        const int r0 = (tile_of(b) << 5) % a.seq, vrow = a.kv_dim * 2, left = a.seq - r0;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)(a.vc + (size_t)r0 * a.kv_dim), 0, (left < 32 ? left : 32) * vrow, 0x00020000);
        const int vo = (kvh * HD + vd) * 2;
        #pragma unroll
        for (int s = 0; s < 32; ++s) {
            if constexpr (NK == 2) vw[s] = __builtin_amdgcn_raw_buffer_load_b32(rs, vo, s * vrow, 0);
            else vw[s] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, vo, s * vrow, 0);
        }
    };
    fetch_k(b0);
    fetch_v(b0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (FQ) {
        prep.queries(a, ctl, kvh, G, wave, lane, qs);
        if (any) prep.rows(a, wave, lane, tnew, hv + (size_t)wave * HD, mine,       // the rows of the block in the workgroup's tiles
            [&](int r, int t, int p, uint16_t lo, uint16_t hi) {
                uint16_t *row = nk + r * HD + p, *crow = a.kcw + (size_t)(t % a.seq) * a.kv_dim + (size_t)kvh * HD + p;
                row[0] = lo; row[HD / 2] = hi;
                crow[0] = lo; crow[HD / 2] = hi;
            },
            [&](int r, int t, uint2 h4) {
                *(uint2 *)(nv + r * HD + 4 * lane) = h4;
                *(uint2 *)(a.vcw + (size_t)(t % a.seq) * a.kv_dim + (size_t)kvh * HD + 4 * lane) = h4;
            });
    } else AttnRowsPrep<M, HD>::copy_queries(a, kvh, G, qs);      // once per workgroup
    __syncthreads();
    for (int it = 0; it < ng; it += 2) {                      // unit groups of the pair (more than two: heads of more than 4 to a kv head)
        const int ug = ng == 1 ? 0 : it + pair;
        int us[4], up[4];                                     // keys that units 4c + i see: us..up
        size_t pi[4];                                         // their partials' slots, less the tile
        #pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int u = 16 * ug + 4 * c + i, j = u / G;
            up[i] = u < units ? pos0 + j : -1;
            us[i] = u < units ? lg_win_start(pos0 + j, a.window) : 0;
            pi[i] = u < units ? ((size_t)j * a.H + kvh * G + (u - j * G)) * a.tiles_max : 0;
        }
        const float *qr = qs + (size_t)(16 * (ug < ng ? ug : 0) + n) * Geo::QST + c * (HD / 4);
        float *ep = es + (size_t)pair * 16 * Geo::EST;
        if (it > 0) { fetch_k(b0); fetch_v(b0); }
        for (int bb = b0; bb < nb; bb += gx) {
            const int tile = tile_of(bb), bx = tile - first, t0 = tile << 5;
            const bool act = ug < ng && (ng > 1 || first + bb * tw + pair <= last);      // (the others compute what nobody stores)
            if constexpr (FQ) if (any && t0 + 31 >= tnew) {           // rows of the block in this tile: from LDS, they are not in the cache yet
                const int rk = t0 + 16 * half + n - tnew;
                if (rk >= 0 && rk < M) {
                    #pragma unroll
                    for (int s = 0; s < NS; ++s) kw[s] = *(const uint4 *)(nk + rk * HD + 32 * s + 8 * c);
                }
                #pragma unroll
                for (int s = 0; s < 32; ++s) {
                    const int r = t0 + s - tnew;
                    if (r >= 0 && r < M) { if constexpr (NK == 2) vw[s] = *(const uint32_t *)(nv + r * HD + vd); else vw[s] = nv[r * HD + vd]; }
                }
            }
            // slots outside the keys of every row of the block are zeroed (their weights are zero, and zero times
            // a finite value leaves the sums as they are; stale bits that read as infinities would not)
            if (t0 < start0 || t0 + 31 > plast) {
                #pragma unroll
                for (int s = 0; s < 32; ++s) vw[s] = (t0 + s >= start0 && t0 + s <= plast) ? vw[s] : 0;
            }
            lg_v16f d = {};
            // dims 32s + 8c + 0..7 of the key -> its dims 32s + 4g + c, g = 0..7.  A product that waits for the conversion in
            // front of it takes 52 cycles instead of 32, so a piece is dealt and converted before the products of the one ahead of it.
            float kf[2][8];
            float4 qv[2][2];
            auto piece = [&](int s) {
                uint32_t o[4];
                lg_deal4(__builtin_amdgcn_perm(kw[s].z, kw[s].x, 0x05040100u), __builtin_amdgcn_perm(kw[s].z, kw[s].x, 0x07060302u),
                         __builtin_amdgcn_perm(kw[s].w, kw[s].y, 0x05040100u), __builtin_amdgcn_perm(kw[s].w, kw[s].y, 0x07060302u), o);
                #pragma unroll
                for (int g = 0; g < 8; ++g) kf[s & 1][g] = lg_h2f((uint16_t)(o[g >> 1] >> (16 * (g & 1))));
            };
            qv[0][0] = *(const float4 *)qr; qv[0][1] = *(const float4 *)(qr + 4);
            piece(0);
            #pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (s + 1 < NS) { qv[(s + 1) & 1][0] = *(const float4 *)(qr + 8 * (s + 1)); qv[(s + 1) & 1][1] = *(const float4 *)(qr + 8 * (s + 1) + 4); piece(s + 1); }
                __builtin_amdgcn_sched_barrier(0);
                const float4 qa = qv[s & 1][0], qb = qv[s & 1][1];
                const float qe[8] = { qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w };
                #pragma unroll
                for (int g = 0; g < 8; ++g) d = __builtin_amdgcn_mfma_f32_16x16x1f32(qe[g], kf[s & 1][g], d, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            fetch_k(bb + gx);                                 // the next tile's K rows (past the last tile: the last one's again)
            const int p = t0 + 16 * half + n;
            float sc[4], m[4];
            #pragma unroll
            for (int i = 0; i < 4; ++i) {
                sc[i] = p >= us[i] && p <= up[i] ? (d[i] + d[4 + i]) + (d[8 + i] + d[12 + i]) : -INFINITY;
                m[i] = lg_max16(sc[i]);
                if (n == 0) mxs[wave][4 * c + i] = m[i];
            }
            __syncthreads();
            #pragma unroll
            for (int i = 0; i < 4; ++i) {
                m[i] = fmaxf(m[i], mxs[wave ^ 1][4 * c + i]);
                const float e = p >= us[i] && p <= up[i] ? lg_expf(sc[i] - m[i]) : 0.0f;
                const float l = lg_sum16(e);
                ep[(4 * c + i) * Geo::EST + 16 * half + n] = e;
                if (n == 0) lsum[wave][4 * c + i] = l;
            }
            __syncthreads();
            lg_v16f acc[NK] = {};
            float vf[2][4][NK];                               // (four slots converted ahead, as above)
            float4 e4[2];
            auto slots = [&](int s4) {
                e4[s4 & 1] = *(const float4 *)(ep + n * Geo::EST + 4 * s4);
                #pragma unroll
                for (int q = 0; q < 4; ++q) {
                    asm volatile("" : "+v"(vw[4 * s4 + q]));  // (converted here: else ahead of the scores, which then wait for every load and store)
                    #pragma unroll
                    for (int k = 0; k < NK; ++k) vf[s4 & 1][q][k] = lg_h2f((uint16_t)(vw[4 * s4 + q] >> (16 * k)));
                }
            };
            slots(0);
            #pragma unroll
            for (int s4 = 0; s4 < 8; ++s4) {
                if (s4 + 1 < 8) slots(s4 + 1);
                __builtin_amdgcn_sched_barrier(0);
                const float ev[4] = { e4[s4 & 1].x, e4[s4 & 1].y, e4[s4 & 1].z, e4[s4 & 1].w };
                #pragma unroll
                for (int q = 0; q < 4; ++q)
                    #pragma unroll
                    for (int k = 0; k < NK; ++k) acc[k] = __builtin_amdgcn_mfma_f32_16x16x1f32(ev[q], vf[s4 & 1][q][k], acc[k], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            // Where the rows' keys may differ within the tile (its slots up to M - 1 behind the first key and M - 1 ahead of the last), a
            // value that is not finite was a product with weight 0 for the units that do not see its slot: a NaN.  So where a result of
            // this wavefront is not finite there, all of them are computed again, each from the slots its row sees (the block's own rows
            // from LDS, the others from the cache).
            if (__builtin_expect(t0 < start0 + M - 1 || t0 + 31 > plast - (M - 1), 0)) {
                float o4[4] = {};
                #pragma unroll
                for (int i = 0; i < 16; ++i)
                    #pragma unroll
                    for (int k = 0; k < NK; ++k) o4[i & 3] = lg_fmaf(acc[k][i], 0.0f, o4[i & 3]);
                const float odd = (o4[0] + o4[1]) + (o4[2] + o4[3]);
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(odd != 0.0f) != 0, 0)) {
                    int n2 = n, c2 = c;
                    asm volatile("" : "+v"(n2), "+v"(c2));            // (else the addresses of this block are computed ahead of the scores and kept in registers)
                    const int d0 = (HD >= 128 ? half * (HD / 2) : 0) + NK * n2;
                    const float *eu = ep + (size_t)(4 * c2) * Geo::EST;
                    #pragma unroll
                    for (int k = 0; k < NK; ++k) acc[k] = lg_v16f{};
                    for (int t = t0 < start0 ? start0 : t0; t <= plast && t < t0 + 32; ++t) {
                        const uint16_t *vr = (FQ && t >= tnew ? nv + (t - tnew) * HD : a.vc + (size_t)(t % a.seq) * a.kv_dim + (size_t)kvh * HD) + d0;
                        uint16_t v[4][NK];
                        #pragma unroll
                        for (int b = 0; b < 4; ++b)
                            #pragma unroll
                            for (int k = 0; k < NK; ++k) v[b][k] = vr[16 * NK * b + k];
                        #pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            if (t < us[i] || t > up[i]) continue;
                            const float e = eu[i * Geo::EST + t - t0];
                            #pragma unroll
                            for (int b = 0; b < 4; ++b)
                                #pragma unroll
                                for (int k = 0; k < NK; ++k) acc[k][4 * b + i] = lg_fmaf(e, lg_h2f(v[b][k]), acc[k][4 * b + i]);
                        }
                    }
                }
            }
            #pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (!act || tile < (us[i] >> 5) || tile > (up[i] >> 5)) continue;        // no key of the unit's row in this tile
                const size_t ti = pi[i] + bx;
                if (half == 0 && n == 0) { a.pm[ti] = m[i]; a.pl[ti] = lsum[wave][4 * c + i] + lsum[wave ^ 1][4 * c + i]; }
                if (HD < 128 && half != 0) continue;
                float *dst = a.pacc + ti * HD + (HD >= 128 ? half * (HD / 2) : 0) + NK * n;
                #pragma unroll
                for (int b = 0; b < 4; ++b) {                 // block b: dims 16b + n, NK of them each
                    if constexpr (NK == 2) *(float2 *)(dst + 32 * b) = make_float2(acc[0][4 * b + i], acc[1][4 * b + i]);
                    else dst[16 * b] = acc[0][4 * b + i];
                }
            }
            fetch_v(bb + gx);
        }
    }
}

// The same for few units (attention_rows_few in lg_hip.hip): on the vector units, a workgroup to a tile, K and V rows through LDS.
// lg_k_attn_rows pays for 16 units, leaves CUs without a workgroup where it takes two tiles at a time, and the registers of its operands
// let a CU overlap the preparation of one workgroup with the tiles of another only twice.  A wavefront takes the units wave, wave + 4 and wave + 8 (UB = 4: and wave + 12), so that one LDS read of a K (V) row serves three units
// and 6 (12) independent fma chains are in flight; bound by those fma and their LDS reads.  K is staged in reader order (the lane of key slot sl
// and chain pair hf finds its hd/4 dwords as consecutive 16-byte units).
// Tiles and merge, 256-wide heads, 32 tiles of 8 kv heads: 10 units 13.9 -> 12.4 us, 4 units 13.3 -> 11.3; 33 tiles 14.0 -> 13.7 and 13.3 -> 12.7;
// whole steps (the kernels prepare the rows themselves): 12B shape, 5 rows at 3000 keys 3266 -> 3120 us, 2 rows at 1100 2837 -> 2705.
#define LG_ATTN_FEW 12                     // units: three to a wavefront (UB = 4: 16)
// fmaf(x, (float)h, acc) with h the low (high) f16 half of a packed pair: one instruction; the conversion is exact
// and the sum rounds once, as the two-instruction form does.  The compiler picks this instruction by itself when a
// converted value feeds one fma; written out here because each key/value element feeds one fma per unit.
__device__ __forceinline__ float lg_fma_hlo(float x, uint32_t hp, float acc) {
    asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel_hi:[0,1,0]" : "+v"(acc) : "v"(x), "v"(hp));
    return acc;
}
__device__ __forceinline__ float lg_fma_hhi(float x, uint32_t hp, float acc) {
    asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "+v"(acc) : "v"(x), "v"(hp));
    return acc;
}
template <int HD>
struct AttnFewGeo {
    static constexpr int QST = HD + 4;
    static constexpr int KSD = HD / 2 + 4;                    // dwords per staged K row (16-byte reads of 8 slots cover all banks)
    static constexpr int VST = HD + 8;                        // halves per staged V row
    static constexpr size_t bytes(int units, bool fq) {       // fq: a vector of staging per wavefront for the rotary
        return (size_t)units * QST * 4 + (size_t)32 * KSD * 4 + (size_t)32 * VST * 2 + (size_t)units * 32 * 4 + (fq ? (size_t)(LG_WG / 64) * HD * 4 : 0);
    }
};
static_assert(AttnFewGeo<256>::bytes(LG_ATTN_FEW, false) <= 48 * 1024, "lg_hip_attention_noalloc raises no limit for this kernel");
template <int M, int HD, bool FQ = false, int UB = LG_ATTN_FEW / 4>
__global__ __launch_bounds__(LG_WG) void lg_k_attn_few(const StepCtl *ctl, LG_ATTN_FIELDS(LG_XP, _) int p_end_) {
    AttnArgs a; LG_ATTN_FIELDS(LG_XI, a)
    using Geo = AttnFewGeo<HD>;
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int NW = LG_WG / 64;
    const int G = a.H / a.nkv, units = M * G;
    float *qs = (float *)smem;                                // [unit][c][HD/4]
    uint32_t *kt = (uint32_t *)(qs + (size_t)units * Geo::QST);         // [32][KSD]: row sl = [hf][HD/4 dwords]
    uint16_t *vt = (uint16_t *)(kt + 32 * Geo::KSD);          // [32][VST]
    float *es = (float *)(vt + 32 * Geo::VST);                // [unit][32]
    float *hv = es + (size_t)units * 32;                      // FQ: [wavefront][HD] staging of the rotary
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int kvh = blockIdx.y;
    const int pos0 = ctl->pos + a.pos_off, plast = pos0 + M - 1;
    const int tnew = (FQ && a.kcw) ? ctl->pos : 0x7FFFFFFF;   // FQ: positions tnew..plast are rows of the block itself
    const int start0 = lg_win_start(pos0, a.window), first = start0 >> 5;
    const int bx = blockIdx.x, tile = first + bx, t0 = tile << 5;
    if (t0 > plast) return;                                   // no row of the block has keys here
    auto mine = [&](int t) { return t >> 5 == tile; };
    const bool any = FQ && tnew <= plast && t0 + 31 >= tnew;  // the tile holds rows of the block
    AttnRowsPrep<M, HD> prep;
    if constexpr (FQ) prep.request(a, kvh, G, wave, tnew, any, mine);
    constexpr int U4R = HD / 8;                               // 16-byte units per K/V row
    constexpr int KL = (32 * U4R + LG_WG - 1) / LG_WG;        // 16-byte units of K (and of V) per thread
    static_assert(32 * U4R % LG_WG == 0, "tile staging assumes whole passes");
    uint4 kq[KL], vq[KL];
    {   // (a tile lies within the ring in one piece; rows past its end are no keys of any row)
        const int r0 = t0 % a.seq;
        #pragma unroll
        for (int u = 0; u < KL; ++u) {
            const int idx = (int)threadIdx.x + u * LG_WG, row = idx / U4R, u4 = idx - row * U4R;
            const size_t go = (size_t)(r0 + row < a.seq ? r0 + row : a.seq - 1) * a.kv_dim + (size_t)kvh * HD + u4 * 8;
            kq[u] = lg_ldw16(a.kc + go); vq[u] = lg_ldw16(a.vc + go);         // (no second reader: non-temporal)
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (FQ) {
        prep.queries(a, ctl, kvh, G, wave, lane, qs);
        if (any) prep.rows(a, wave, lane, tnew, hv + (size_t)wave * HD, mine,
            [&](int r, int t, int p, uint16_t lo, uint16_t hi) {
                const int p1 = p + HD / 2;                    // dims 4g, 4g+1 in dword g of the first half, 4g+2, 4g+3 of the second
                uint16_t *row = (uint16_t *)(kt + (t - t0) * Geo::KSD), *crow = a.kcw + (size_t)(t % a.seq) * a.kv_dim + (size_t)kvh * HD;
                row[2 * (((p & 3) >> 1) * (HD / 4) + (p >> 2)) + (p & 1)] = lo;
                row[2 * (((p1 & 3) >> 1) * (HD / 4) + (p1 >> 2)) + (p1 & 1)] = hi;
                crow[p] = lo; crow[p1] = hi;
            },
            [&](int r, int t, uint2 h4) {
                *(uint2 *)(vt + (t - t0) * Geo::VST + 4 * lane) = h4;
                *(uint2 *)(a.vcw + (size_t)(t % a.seq) * a.kv_dim + (size_t)kvh * HD + 4 * lane) = h4;
            });
    } else AttnRowsPrep<M, HD>::copy_queries(a, kvh, G, qs);
    {   // the tile into LDS.  Slots outside the keys of every row of the block are zeroed (their weights are zero, and zero times a
        // finite value leaves the sums as they are; stale bits that read as infinities would not)
        const int slo = start0 - t0, shi = plast - t0;
        #pragma unroll
        for (int u = 0; u < KL; ++u) {
            const int idx = (int)threadIdx.x + u * LG_WG, row = idx / U4R, u4 = idx - row * U4R;
            if (FQ && t0 + row >= tnew && row <= shi) continue;               // a row of the block: built above, not in the cache yet
            const uint32_t mk = (row >= slo && row <= shi) ? 0xFFFFFFFFu : 0u;
            uint32_t *d = kt + row * Geo::KSD + 2 * u4;
            *(uint2 *)d = make_uint2(kq[u].x & mk, kq[u].z & mk);             // chains 0,1 of two groups of four dims
            *(uint2 *)(d + HD / 4) = make_uint2(kq[u].y & mk, kq[u].w & mk);  // chains 2,3
            *(uint4 *)(vt + row * Geo::VST + u4 * 8) = make_uint4(vq[u].x & mk, vq[u].y & mk, vq[u].z & mk, vq[u].w & mk);
        }
    }
    __syncthreads();
    // this wavefront's units, the slots that they see (a missing unit repeats the first one and stores nothing), and their partials
    const bool some = wave < units;
    int un[UB], lo[UB], hi[UB];
    bool on[UB];
    size_t pi[UB];
    #pragma unroll
    for (int b = 0; b < UB; ++b) {
        const bool there = wave + b * NW < units;
        un[b] = there ? wave + b * NW : some ? wave : 0;
        const int j = un[b] / G, pj = pos0 + j;
        lo[b] = lg_win_start(pj, a.window) - t0; hi[b] = pj - t0;
        on[b] = there && lo[b] < 32 && hi[b] >= 0;            // the row has keys in this tile
        pi[b] = ((size_t)j * a.H + kvh * G + (un[b] - j * G)) * a.tiles_max + bx;
    }
    if (some) {   // scores
        const int sl = lane & 31, hf = lane >> 5;
        const uint32_t *ks = kt + sl * Geo::KSD + hf * (HD / 4);
        const float *qr[UB];
        float ax[UB], ay[UB];
        #pragma unroll
        for (int b = 0; b < UB; ++b) { qr[b] = qs + (size_t)un[b] * Geo::QST + hf * (HD / 2); ax[b] = 0.0f; ay[b] = 0.0f; }
        #pragma unroll 2
        for (int u = 0; u < HD / 16; ++u) {
            const uint4 k4 = *(const uint4 *)(ks + 4 * u);
            #pragma unroll
            for (int b = 0; b < UB; ++b) {                    // chains 2 hf and 2 hf + 1
                const float4 p0 = *(const float4 *)(qr[b] + 4 * u), p1 = *(const float4 *)(qr[b] + HD / 4 + 4 * u);
                ax[b] = lg_fma_hlo(p0.x, k4.x, ax[b]); ay[b] = lg_fma_hhi(p1.x, k4.x, ay[b]);
                ax[b] = lg_fma_hlo(p0.y, k4.y, ax[b]); ay[b] = lg_fma_hhi(p1.y, k4.y, ay[b]);
                ax[b] = lg_fma_hlo(p0.z, k4.z, ax[b]); ay[b] = lg_fma_hhi(p1.z, k4.z, ay[b]);
                ax[b] = lg_fma_hlo(p0.w, k4.w, ax[b]); ay[b] = lg_fma_hhi(p1.w, k4.w, ay[b]);
            }
        }
        #pragma unroll
        for (int b = 0; b < UB; ++b) {
            if (!on[b]) continue;
            const bool valid = sl >= lo[b] && sl <= hi[b];
            float s = lg_add_x32(ax[b] + ay[b]);              // (a0+a1) + (a2+a3): the two halves sit 32 lanes apart
            if (!valid) s = -INFINITY;
            const float mx = lg_max_n(s, 32);
            const float e = valid ? lg_expf(s - mx) : 0.0f;
            const float l = lg_sum32(e);
            if (hf == 0) es[un[b] * 32 + sl] = e;
            if (lane == 0) { a.pm[pi[b]] = mx; a.pl[pi[b]] = l; }
        }
    }
    __syncthreads();
    if (!some) return;
    // values (lane = 4 dims).  A slot that a row does not see has weight 0 for it; where another row of the block has a value there that
    // is not finite, their product is a NaN.  So where the rows' keys may differ within the tile and a result is not finite, they are
    // computed again with zeros in those slots (always with zeros there: 0.4 to 1.1 us more for the first and the last tile, which the merge waits for).
    const uint16_t *vl = vt + (4 * lane < HD ? 4 * lane : 0);
    float4 acc[UB];
    auto values = [&](auto masked) {
        #pragma unroll
        for (int b = 0; b < UB; ++b) acc[b] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        #pragma unroll 2
        for (int u4 = 0; u4 < 8; ++u4) {
            float ev[UB][4];
            #pragma unroll
            for (int b = 0; b < UB; ++b) {                    // (a unit that has no keys here has stale weights: never stored)
                const float4 e4 = *(const float4 *)(es + un[b] * 32 + 4 * u4);
                ev[b][0] = e4.x; ev[b][1] = e4.y; ev[b][2] = e4.z; ev[b][3] = e4.w;
            }
            #pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint2 v4 = *(const uint2 *)(vl + (4 * u4 + q) * Geo::VST);
                #pragma unroll
                for (int b = 0; b < UB; ++b) {
                    uint2 v = v4;
                    if constexpr (decltype(masked)::value) if (4 * u4 + q < lo[b] || 4 * u4 + q > hi[b]) v = make_uint2(0u, 0u);
                    acc[b].x = lg_fma_hlo(ev[b][q], v.x, acc[b].x); acc[b].y = lg_fma_hhi(ev[b][q], v.x, acc[b].y);
                    acc[b].z = lg_fma_hlo(ev[b][q], v.y, acc[b].z); acc[b].w = lg_fma_hhi(ev[b][q], v.y, acc[b].w);
                }
            }
        }
    };
    values(std::false_type{});
    if (__builtin_expect(t0 < start0 + M - 1 || t0 + 31 > plast - (M - 1), 0)) {
        float odd = 0.0f;
        #pragma unroll
        for (int b = 0; b < UB; ++b) odd = lg_fmaf(acc[b].x, 0.0f, lg_fmaf(acc[b].y, 0.0f, lg_fmaf(acc[b].z, 0.0f, lg_fmaf(acc[b].w, 0.0f, odd))));
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(odd != 0.0f) != 0, 0)) values(std::true_type{});
    }
    #pragma unroll
    for (int b = 0; b < UB; ++b)
        if (on[b] && 4 * lane < HD) *(float4 *)(a.pacc + pi[b] * HD + 4 * lane) = acc[b];
}

// lg_k_attn_merge for rows with very many tiles: one workgroup of NW wavefronts per (head, row, 64 dims).  The
// merge is one fma chain over the tiles ascending, and walked by a single wavefront its time is the instruction issue
// of 2 loads + 2 fma per tile, tile after tile.  Here the tiles go in rounds of 64*NW: wavefront w requests the 64
// partials of tiles 64w..64w+63 of the round at once (all wavefronts' loads in flight together) while the
// workgroup computes the round's weights exp(m_t - M) into LDS; then the chain passes through the wavefronts in
// order, each running its 64 fma back to back from registers and handing (L, o) to the next through LDS.  Same
// order, same bits: weights exp(m_t - M), L and the output as fma chains over the tiles ascending, divide, q8.
// NW: a round is a memory round trip and then its turns, so caches that hold more tiles take more wavefronts (merge_waves in
// lg_hip.hip).  8 rows, 8 heads of 256, 626 tiles: four wavefronts in 3 rounds 21.6 us, sixteen in one 14.6; 5 rows, 16 heads, 257
// tiles (a second round for the last of them): 13.0 -> 9.5 us with eight.
template <int M, int NW>
__global__ __launch_bounds__(64 * NW, 4) void lg_k_attn_merge_split(const StepCtl *ctl, LG_MERGE_FIELDS(LG_XP, _) int p_end_) {
    MergeArgs a; LG_MERGE_FIELDS(LG_XI, a)
    constexpr int U = 64, WG = 64 * NW;
    __shared__ __align__(16) float wts[WG], pls[WG], hand[2][64], wmx[NW];
    const int head = blockIdx.x, j = blockIdx.y, hd = a.hd, qd = a.H * hd, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int d = blockIdx.z * 64 + lane;                     // hd is a multiple of 64
    const int pos = ctl->pos + a.pos_off, pj = pos + j;
    const int first = lg_win_start(pos, a.window) >> 5;
    const int lo = (lg_win_start(pj, a.window) >> 5) - first, hi = (pj >> 5) - first;
    const size_t base = ((size_t)j * a.H + head) * a.tiles_max + lo;
    const int nt = hi - lo + 1;
    float pa[U];
    // (buffer loads: the row's partials as the base in scalar registers, the lane's dim as the lane offset, the tile's
    // offset in a scalar register; a flat load each cost a dozen vector instructions of 64-bit address arithmetic)
    const __amdgpu_buffer_rsrc_t rp = lg_buffer_rsrc(a.pacc + base * hd);
    auto fetch = [&](int t0_) {                               // tiles t0 .. t0+63 of this row (past the end: the last one again)
        const int t0 = __builtin_amdgcn_readfirstlane(t0_);
        if (NW > 4 && t0 >= nt) return;                       // (a wavefront without a tile in this round)
        #pragma unroll
        for (int u = 0; u < U; ++u) {
            const int n = t0 + u < nt ? t0 + u : nt - 1;
            pa[u] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rp, d * 4, n * hd * 4, 0));
        }
    };
    fetch(wave * U);                                          // the partials do not depend on the weights
    float mx = -INFINITY;
    for (int n = threadIdx.x; n < nt; n += WG) mx = fmaxf(mx, a.pm[base + n]);
    mx = lg_max_n(mx, 64);
    if (lane == 0) wmx[wave] = mx;
    __syncthreads();
    #pragma unroll
    for (int w = 0; w < NW; ++w) mx = fmaxf(mx, wmx[w]);
    float L = 0.0f, o = 0.0f;
    for (int r0 = 0; r0 < nt; r0 += WG) {
        if (r0 > 0) fetch(r0 + wave * U);
        {   // the round's weights and sums (one tile per thread)
            const int n = r0 + (int)threadIdx.x;
            if (n < nt) { wts[threadIdx.x] = lg_expf(a.pm[base + n] - mx); pls[threadIdx.x] = a.pl[base + n]; }
        }
        __syncthreads();
        for (int turn = 0; turn < NW && r0 + turn * U < nt; ++turn) {
            if (wave == turn) {
                if (r0 + turn > 0) { L = hand[0][lane]; o = hand[1][lane]; }
                // weights and sums four tiles at a time, requested ahead of their fma (tile by tile under a guard a turn
                // was 64 trips to LDS: 2 us of its time)
                constexpr int AHEAD = 2;
                float4 w4[AHEAD], l4[AHEAD];
                #pragma unroll
                for (int g = 0; g < AHEAD; ++g) { w4[g] = *(const float4 *)(wts + turn * U + 4 * g); l4[g] = *(const float4 *)(pls + turn * U + 4 * g); }
                auto chain = [&](auto full) {
                    #pragma unroll
                    for (int g = 0; g < U / 4; ++g) {
                        const float wv[4] = { w4[g % AHEAD].x, w4[g % AHEAD].y, w4[g % AHEAD].z, w4[g % AHEAD].w };
                        const float lv[4] = { l4[g % AHEAD].x, l4[g % AHEAD].y, l4[g % AHEAD].z, l4[g % AHEAD].w };
                        if (g + AHEAD < U / 4) { w4[g % AHEAD] = *(const float4 *)(wts + turn * U + 4 * (g + AHEAD)); l4[g % AHEAD] = *(const float4 *)(pls + turn * U + 4 * (g + AHEAD)); }
                        #pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float Ln = lg_fmaf(lv[i], wv[i], L), on = lg_fmaf(pa[4 * g + i], wv[i], o);
                            const bool in = full || r0 + turn * U + 4 * g + i < nt;
                            L = in ? Ln : L; o = in ? on : o;
                        }
                    }
                };
                if (r0 + (turn + 1) * U <= nt) chain(std::true_type{}); else chain(std::false_type{});
                hand[0][lane] = L; hand[1][lane] = o;
            }
            __syncthreads();
        }
    }
    if (wave != 0) return;
    L = hand[0][lane]; o = hand[1][lane];
    const float r = o / L;
    float dq; int sum;
    const int q = lg_quant1_32lanes(r, &dq, &sum);
    const int e = head * hd + d;
    a.xq[lg_q8_off<M>(qd, j, e >> 4, e & 15)] = (int8_t)q;
    if ((d & 31) == 0) lg_q8_ds<M>(a.xq, qd)[lg_q8_ds_idx<M>(qd, j, e >> 5)] = make_float2(dq, __int_as_float(sum));
    if (a.xf) a.xf[(size_t)j * qd + e] = r;
}

// ---------------------------------------------------------------------------------------------
// Attention merge + output projection in one launch, with no hand-over between workgroups.
// With 8 query heads the 8 K segments of the output projection ARE the heads (K = n_head * head_dim, a segment =
// head_dim elements): the serial chain of segment c only reads head c of the attention output, and the row's result is
// the adjacent-pair tree over the 8 chains.  So the workgroup that merges (head, row j) can run that head's chain
// for a slice of the E output rows straight from LDS, and slab `head` of 8 receives the chain sums: the consumer (the
// row kernel, dparts = 8) adds the slabs in the tree's order, bit for bit what lg_k_mm computes from the q8 row.
// Unit = (row j, head, slice s of the output rows in chunks of 64); the merge is repeated by the slices of a (head, row),
// which costs less than the kernel boundary it replaces.  Workgroup id = j * (8 * slices) + head * slices + s: the units
// that read the same weights differ by a multiple of 8 and run on one XCD (one trip from HBM, the others hit its L2).
// Weights: the projection tiled by row blocks (tile (64-row chunk, K block): lane r = row 64 * chunk + r), where the
// tiles of a head are consecutive.  Lane r of wavefront w runs the chains of the rows r of the unit's chunks w, w + 4, ...
// NIT = head_dim / 32 blocks per chain; RPL = most chunks per wavefront.
struct MergeOArgs {
    MergeArgs      g;           // g.xq unused; g.xf optional
    const uint8_t *w;           // row-block tiles of attn_output [E][n_head * head_dim]
    float         *slabs;       // [8][M][E]
    int            E, slices, rows;
};
#define LG_MERGEO_FIELDS(X, v) X(const float *, pm, g.pm, v) X(const float *, pl, g.pl, v) X(const float *, pacc, g.pacc, v) X(int, tiles_max, g.tiles_max, v) \
    X(int, H, g.H, v) X(int, hd, g.hd, v) X(int, window, g.window, v) X(int, pos_off, g.pos_off, v) X(const uint8_t *, w, w, v) X(int, E, E, v) X(int, slices, slices, v) \
    X(int, rows, rows, v) X(float *, slabs, slabs, v) X(float *, xf, g.xf, v)
template <int NIT, int RPL>
__global__ __launch_bounds__(LG_WG) void lg_k_merge_o(const StepCtl *ctl, LG_MERGEO_FIELDS(LG_XP, _) int p_end_) {
    MergeOArgs a; LG_MERGEO_FIELDS(LG_XI, a)
    a.g.xq = nullptr;
    __shared__ float wts[512], pls[512], wmx[LG_WG / 64];
    __shared__ __align__(16) int8_t hq[NIT * 32];             // the merged head as q8, natural order
    __shared__ float2 hds[NIT];
    const int W = a.g.H * a.slices, id = blockIdx.x;
    const int j = id / W, wi = id - j * W, head = wi / a.slices, s = wi - head * a.slices;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nb = a.g.H * NIT, n64 = (a.E >> 6) / a.slices, chunk0 = s * n64;
    uint4 wq[RPL][NIT];
    uint16_t wsc[RPL][NIT];
    const int qd = a.g.H * a.g.hd;
    lg_attn_merge_body(ctl, a.g, head, j, (int)threadIdx.x, wts, pls, wmx, [&] {
        #pragma unroll
        for (int r = 0; r < RPL; ++r) {
            const int c = wave + 4 * r < n64 ? wave + 4 * r : n64 - 1;     // past the unit's chunks: its last one again, unused
            const uint8_t *tb = a.w + ((size_t)(chunk0 + c) * nb + (size_t)head * NIT) * LG_TILE;
            #pragma unroll
            for (int it = 0; it < NIT; ++it) { wq[r][it] = lg_ldt16(tb, it, lane); wsc[r][it] = lg_ldt2(tb, it, lane); }
        }
    }, [&](int d, float r, int q, float dq, int sum) {
        hq[d] = (int8_t)q;
        if ((d & 31) == 0) hds[d >> 5] = make_float2(dq, __int_as_float(sum));
        if (a.g.xf && s == 0) a.g.xf[(size_t)j * qd + head * a.g.hd + d] = r;
    });
    __syncthreads();
    #pragma unroll
    for (int r = 0; r < RPL; ++r) {
        if (wave + 4 * r >= n64) break;
        float acc = 0.0f;
        #pragma unroll
        for (int it = 0; it < NIT; ++it) {
            const float2 ds = hds[it];
            const int4 a0 = *(const int4 *)(hq + it * 32), a1 = *(const int4 *)(hq + it * 32 + 16);
            const int dot = lg_block_dot(wq[r][it], a0, a1, __float_as_int(ds.y));
            acc = lg_fmaf(ds.x * lg_h2f(wsc[r][it]), (float)dot, acc);
        }
        a.slabs[((size_t)head * a.rows + j) * a.E + (size_t)(chunk0 + wave + 4 * r) * 64 + lane] = acc;
    }
}
