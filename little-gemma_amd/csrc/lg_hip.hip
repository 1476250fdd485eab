// lg_hip.hip — C ABI of the gfx950 verify-step backend (declared in include/lg_hip.h).
//
// Host side: weight layout, scratch, the launch sequence of one step, graph capture, the
// device-resident step schedule and the measurement helpers.  Device side: lg_kernels.h.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <map>
#include <mutex>
#include <optional>
#include <string>
#include <type_traits>
#include <thread>
#include <vector>

#include "../../include/lg_hip.h"
#include "lg_kernels.h"
#include "lg_wide.h"
#include "lg_fused.h"
#include "lg_xcd.h"
#include "lg_xffn.h"
#include "lg_xtail.h"
#include "lg_xrg.h"
#include "lg_narrow.h"
#include "lg_aout.h"
#include "lg_mid.h"

static_assert(LG_HIP_MAX_ROWS == LG_HIP_MAX_ROWS_DEV, "row limits must agree");
#define LG_FUSE_ROWS_MAX 2         // widest block whose q/k/v matmul does the preceding row work itself

// ---- errors -----------------------------------------------------------------------------------
static thread_local char g_err[512] = "";
static int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return code;
}
#define HIP_TRY(expr) do { hipError_t e_ = (expr); if (e_ != hipSuccess) \
    return fail(-100 - (int)e_, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); } while (0)

// Copies and clears that are done when the call returns, on a model's own stream: the forms without a stream fail (hipErrorStreamCaptureImplicit)
// while any other thread of the process captures, a step of another model, say.
static hipError_t copy_now(hipStream_t st, void *dst, const void *src, size_t n, hipMemcpyKind kind) {
    const hipError_t e = hipMemcpyAsync(dst, src, n, kind, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
}
static hipError_t clear_now(hipStream_t st, void *dst, int value, size_t n) {
    const hipError_t e = hipMemsetAsync(dst, value, n, st);
    return e == hipSuccess ? hipStreamSynchronize(st) : e;
}

extern "C" const char *lg_hip_last_error(void) { return g_err; }
extern "C" int lg_hip_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) { (void)hipGetLastError(); return 0; }
    return n;
}
// The widest prompt block a cache of max_seq positions takes: LG_WIDE_ROWS for caches of 1024 positions and more,
// LG_WIDE_MID below (a short cache does not pay 512 spare rows per sliding ring)
static int wide_rows_for(int max_seq) { return max_seq >= 1024 ? LG_WIDE_ROWS : LG_WIDE_MID; }
extern "C" int lg_hip_ring_rows(int window, int max_seq) {
    int r = (window + wide_rows_for(max_seq) + 31) / 32 * 32;   // window + spare for the widest block written before its queries run, tile multiple
    return r < max_seq ? r : max_seq;
}

// What the attention of a cache may take beside its rings: one (max, sum, hd accumulators) slot per (row of the widest block,
// head, key tile any block can touch), the widest PROMPT block of a cache stepped down (512, 128, 32 rows, then verify-width
// blocks only) until that fits LG_PARTIALS_BUDGET: late in a long cache a block touches every tile, and the slots grow with
// rows x max_seq.  Verify blocks keep such partials; the weights that prompt blocks keep of a tile in memory take less than
// them (34 floats a unit and tile), so that this bounds both: lg_hip_kv_create asks for what they need.  Pure arithmetic.
#define LG_PARTIALS_BUDGET ((size_t)2 << 30)
extern "C" size_t lg_hip_kv_partials(int max_seq, int window, int any_global, int max_rows, int n_head, int max_hd,
                                     int *wide_rows, int *tiles_max) {
    const int steps[4] = { wide_rows_for(max_seq), LG_WIDE_MID, LG_WIDE, 0 };
    size_t bytes = 0;
    int wide = 0, tiles = 1;
    for (int i = 0; i < 4; ++i) {
        wide = steps[i];
        if (i > 0 && wide >= steps[i - 1]) continue;
        const int ring_span = window > 0 ? window + (wide > max_rows ? wide : max_rows) : max_seq;
        const int span = any_global || window <= 0 ? max_seq : ring_span;
        tiles = (span < max_seq ? span : max_seq) / 32 + 2;
        const size_t slots = (size_t)(max_rows > wide ? max_rows : wide) * n_head * tiles;
        bytes = slots * ((size_t)max_hd * 4 + 8);
        if (bytes <= LG_PARTIALS_BUDGET || wide == 0) break;
    }
    if (wide_rows) *wide_rows = wide;
    if (tiles_max) *tiles_max = tiles;
    return bytes;
}

// ---- weight layout ----------------------------------------------------------------------------
extern "C" int lg_hip_segments(int k) { return lg_segments(k); }

extern "C" size_t lg_hip_repacked_bytes(int k, int m) {
    if (k <= 0 || m <= 0 || k % 256 || m % 8) return 0;
    const int S = lg_segments(k);
    if ((k / 32) % S) return 0;
    return (size_t)(m / (64 / S)) * (size_t)(k / 32 / S) * LG_TILE;
}

// rows[i] points at virtual row i (k/32 blocks of 18 bytes each)
static void repack_rows(const uint8_t *const *rows, int k, int m, uint8_t *dst) {
    const int S = lg_segments(k), rw = 64 / S, nit = k / 32 / S, groups = m / rw;
    auto work = [&](int g0, int g1) {
        for (int g = g0; g < g1; ++g)
            for (int it = 0; it < nit; ++it) {
                uint8_t *tile = dst + ((size_t)g * nit + it) * LG_TILE;
                for (int r = 0; r < rw; ++r)
                    for (int c = 0; c < S; ++c) {
                        const uint8_t *blk = rows[g * rw + r] + (size_t)(c * nit + it) * 18;
                        memcpy(tile + (r * S + c) * 16, blk + 2, 16);
                        memcpy(tile + 1024 + (r * S + c) * 2, blk, 2);
                    }
            }
    };
    unsigned hw = std::thread::hardware_concurrency();
    int nt = (int)(hw ? (hw > 16 ? 16 : hw) : 4);
    if ((size_t)groups * nit < 4096 || nt < 2) { work(0, groups); return; }
    std::vector<std::thread> pool;
    for (int t = 0; t < nt; ++t) pool.emplace_back(work, (int)((long long)groups * t / nt), (int)((long long)groups * (t + 1) / nt));
    for (auto &th : pool) th.join();
}

// Row-block tiles (lg_k_geglu_t): tile (64-row block, kb) holds for lane r the 16 nibble bytes of block kb
// of row 64*block + r, then the 64 f16 scales; tiles ordered [block][kb].  Same size as the segment tiles.
static void repack_rowblocks(const uint8_t *const *rows, int k, int m, uint8_t *dst) {
    const int nb = k / 32, blocks = m / 64;
    auto work = [&](int b0, int b1) {
        for (int b = b0; b < b1; ++b)
            for (int kb = 0; kb < nb; ++kb) {
                uint8_t *tile = dst + ((size_t)b * nb + kb) * LG_TILE;
                for (int r = 0; r < 64; ++r) {
                    const uint8_t *blk = rows[b * 64 + r] + (size_t)kb * 18;
                    memcpy(tile + r * 16, blk + 2, 16);
                    memcpy(tile + 1024 + r * 2, blk, 2);
                }
            }
    };
    unsigned hw = std::thread::hardware_concurrency();
    int nt = (int)(hw ? (hw > 16 ? 16 : hw) : 4);
    if ((size_t)blocks * nb < 4096 || nt < 2) { work(0, blocks); return; }
    std::vector<std::thread> pool;
    for (int t = 0; t < nt; ++t) pool.emplace_back(work, (int)((long long)blocks * t / nt), (int)((long long)blocks * (t + 1) / nt));
    for (auto &th : pool) th.join();
}

extern "C" int lg_hip_repack_q4_0(const void *src, int k, int m, void *dst) {
    if (!lg_hip_repacked_bytes(k, m)) return fail(-2, "repack: k=%d must be a multiple of 256 (1024 above 4096) and m=%d of 8", k, m);
    std::vector<const uint8_t *> rows((size_t)m);
    for (int i = 0; i < m; ++i) rows[i] = (const uint8_t *)src + (size_t)i * (k / 32) * 18;
    repack_rows(rows.data(), k, m, (uint8_t *)dst);
    return 0;
}

// ---- objects ----------------------------------------------------------------------------------
struct HostTensor { uint32_t type, n_dims; uint64_t dims[4]; const void *data; };

struct Layer {
    uint8_t *wqkv = nullptr, *wo = nullptr, *wgu = nullptr, *wdown = nullptr, *winp = nullptr, *wproj = nullptr;
    float *winp_f = nullptr, *wproj_f = nullptr;   // inp_gate / proj when the file keeps them in a float type (then winp / wproj are null)
    uint8_t *wdn_m = nullptr;                      // ffn_down again as the per-workgroup streams of lg_k_down_m
    uint8_t *wqkv_pc = nullptr, *wo_pc = nullptr;  // q/k/v and attn_output again as chains of pairs of K segments (pack_pairs): lg_k_down_qkv, lg_k_o_geglu
    uint8_t *wqkv_ch = nullptr;                    // q/k/v again as such chains: lg_k_ple_tail_s of 4..8 rows
    uint8_t *wo_ch = nullptr;                      // attn_output again as matrix-core chains [row block][segment]: lg_k_attn_tail, lg_k_attn_out_m
    // the matrices once more in the form of the prompt kernels (lg_wide.h)
    uint8_t *wqkv_w = nullptr, *wo_w = nullptr, *wgu_w = nullptr, *wdown_w = nullptr, *winp_w = nullptr, *wproj_w = nullptr;
    uint8_t *wo_rb = nullptr;                      // attn_output again as row-block tiles: the chains of lg_k_merge_o
    uint8_t *xgu = nullptr, *xdn = nullptr;        // gate/up and ffn_down again as per-workgroup streams of the XCD-partitioned kernel (lg_xffn.h)
    float *attn_norm = nullptr, *q_norm = nullptr, *k_norm = nullptr, *post_attn = nullptr, *ffn_norm = nullptr,
          *post_ffw = nullptr, *post_norm = nullptr, *out_scale = nullptr;
    int is_local = 0, hd = 0, nkv = 0, nff = 0, qd = 0, kd = 0, qkv_m = 0, k_off = 0, v_off = 0, owns = 0, src = 0;
    const float *rope_tab = nullptr, *rope_ff = nullptr;
};

enum KClass { KC_ROWS, KC_PMP, KC_QKV, KC_QKVPOST, KC_ATTN, KC_MERGE, KC_O, KC_GATEUP, KC_DOWN, KC_PLEGATE, KC_PLEPROJ,
              KC_HEAD, KC_ACCEPT, KC_FFN, KC_TAIL, KC_ATAIL, KC_COUNT };
static const char *k_class_names[KC_COUNT] = { "rows_norm_quant", "ple_model_proj", "qkv", "qkv_post", "attn_tiles", "attn_merge",
    "attn_output", "gate_up_geglu", "ffn_down", "ple_gate", "ple_proj", "lm_head", "accept", "ffn_xcd", "ple_tail", "attn_tail" };

// What a captured graph was captured for: the cache's id, the options, the block width and the rest of the options.
typedef std::array<uint64_t, 4> GraphKey;
struct Profile {
    bool on = false;
    std::vector<hipEvent_t> ev;        // pairs
    std::vector<int> cls;
};

struct lg_hip_model {
    int device = 0;
    hipStream_t stream = nullptr;
    bool owns_stream = true;           // false for a draft head: it runs on its target's stream and never destroys it
    // a second stream and two events for the one branch of a step that is off the critical chain: the per-layer
    // inputs (per_layer_model_proj + lg_k_ipl), needed first by layer 0's per-layer gate, run beside layer 0's
    // attention and feed-forward (the reference forks its decode graph the same way, src/cuda/model-cuda.cuh:917-935)
    hipStream_t stream2 = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    int fork_ple = 0;                  // option: use it.  Off: replayed as a graph with a second branch the step takes 2.77 ms instead of 2.26
    // config
    int n_layer = 0, E = 0, H = 0, n_vocab = 0, window = 0, ple = 0, n_kv_start = 0, max_rows = 0;
    float eps = 0, base = 0, base_swa = 0, softcap = 0;
    std::vector<int> is_local, ffn_len, head_dim, n_head_kv;
    std::map<std::string, HostTensor> host;
    bool numbered = false;             // every layer has a launch number of its own (StepCtl.launch): kernels whose workgroups wait for one another may run
    struct Turns *turns = nullptr;                         // of its device
    hipEvent_t ev_turn = nullptr;                          // end of the steps it has launched, for another model to ask about
    bool turn_recorded = false;                            // ev_turn holds the end of its latest step already
    bool launching = false;                                // a step of it is being launched or captured: its stream is its own
    bool plain = false;                                    // the step that is being launched takes the kernels that wait for nobody
    bool prompting = false;                                // prompt blocks of it are under way (PromptTurn)
    std::vector<std::pair<void *, size_t>> marks;          // memory whose words carry launch numbers (mark_alloc)
    int marked_steps = 0;                                  // steps since it was last cleared (count_steps)
    bool committed = false, wide_built = false;    // wide_built: the matrices' wide forms exist
    // weights
    std::vector<Layer> L;
    uint8_t *emb = nullptr, *pmp = nullptr, *pte = nullptr;
    uint8_t *pmp_w = nullptr;                      // per_layer_model_proj in the form of the prompt kernels
    float *pmp_f = nullptr;                        // per_layer_model_proj kept in a float type (then pmp is null)
    float *pgf = nullptr;                          // [rows][ple] f32 gate output, input of a float-typed proj
    uint8_t *emb_rb = nullptr;                     // token_embd again as row-block tiles: the lm_head of 4..8-row blocks (lg_k_head_m)
    float *output_norm = nullptr, *rope_freqs = nullptr, *proj_norm = nullptr;
    std::vector<void *> allocs;
    std::map<std::pair<int, int>, float *> rope_tabs;      // (is_local, hd) -> table
    // scratch
    float *x[2] = { nullptr, nullptr }, *qkv = nullptr, *dout = nullptr, *pmp_raw = nullptr, *hidden_rows = nullptr,
          *g_hidden = nullptr, *logits = nullptr, *pval = nullptr, *q_rot = nullptr;
    int8_t *aq = nullptr, *gq = nullptr, *pq = nullptr, *hq = nullptr;     // q8 activation buffers (values + {scale,sum})
    int8_t *eq = nullptr;              // q8 of the block's embedding rows: input of per_layer_model_proj (kept apart from hq, which layer 0 rewrites meanwhile)
    int *pidx = nullptr;
    StepCtl *ctl = nullptr;
    int32_t *sched = nullptr, *out = nullptr, *adv = nullptr;
    int sched_cap = 0, sched_steps = 0, sched_rows = 0, sched_pos0 = 0, sched_loaded = 0;
    int32_t *pin = nullptr;            // pinned host staging
    int reports = 0;                   // steps the host has waited for: the last one's StepCtl.report
    int last_rows = 0, last_adv = 0;
    float *lstage = nullptr;           // pinned: two rows of logits on their way to a caller (lg_hip_get_logits), row j in half j % 2
    int lread = -1, lcoming = -1;      // the row of the latest step read last, and the one whose copy has been started
    int store_logits = 0, use_graph = 1, wide_prefill = 1, fuse_rows = 1, attn_rows = 1, attn_rows_fq = 1, head_mfma = 1, down_kq = 1, tail_spread = 1, rows_geglu = 0, narrow = 1, attn_out = 1, tail_qkv = 1, attn_geglu = 2, mid = 2;
    uint32_t mid_rows = 0;             // bit r: blocks of r rows have launches of lg_mid.h while mid is 2
    // the feed-forward half of a layer as one XCD-partitioned launch (lg_xffn.h): built when the shape and the chip fit
    int xcd_ffn = 0;                         // option: use it (verify blocks of 4..8 rows)
    int down_m = 1;                          // option: ffn_down of 4..8-row blocks on the matrix cores (lg_k_down_m): 1 = the row group's four workgroups add
                                             // their slabs themselves, 2 = four slabs for the consumer, 0 = the v_dot4 kernels; its streams are built
                                             // at commit unless LG_HIP_DOWN_M=0
    DownMSync *dmsync = nullptr;
    int xcd_attn_tail = 0;                   // option: attention merge, output projection and the row work after it as one launch on one XCD
                                             // (lg_k_attn_tail): 0 off (as measured it gains nothing), 1 from three rows up, 2 for every verify block;
                                             // the copy of the weights it reads is only built when LG_HIP_XCD_ATTN_TAIL is set at commit
    int merge_o = 0;                         // option: attention merge and output projection as one launch (lg_k_merge_o): 0 off (as measured it loses
                                             // as much in the row kernel that adds its 8 slabs as it gains), 1 from three rows up, 2 always; the second
                                             // copy of the weights it reads is only built when LG_HIP_MERGE_O is set at commit
    int merge_o_slices = 0;                  // option: slices of the output rows per (head, row), 0 = chosen by the launcher
    // the per-layer-input block and the next row work as one launch on one XCD (lg_xtail.h)
    int xcd_tail = 1;                        // option: 0 off, 1 for blocks that do not fold the row work into q/k/v, 2 for every verify block
    XtailSync *tsync = nullptr;
    uint2 *tgf = nullptr, *tpr = nullptr;    // [LG_HIP_MAX_ROWS][ple] and [LG_HIP_MAX_ROWS][E] its gated values and projections, tagged
    uint2 *mido = nullptr, *midd = nullptr, *mids = nullptr;   // [max rows][E] the first products of lg_k_o_geglu and lg_k_down_qkv, [3][max rows][E] slabs of the latter, tagged (option mid)
    FarRows *midro = nullptr, *midrd = nullptr, *midao = nullptr;                // their rows
    FarRows *trows = nullptr;                // rows of lg_k_ple_tail_s on their way to the next layer's projections (option tail_qkv)
    FarRows *aorows = nullptr;               // rows of lg_k_attn_out on their way to gate/up (option attn_geglu)
    AttnOutSync *aosync = nullptr;           // hand-over state of lg_k_attn_out (models it serves)
    NarrowSync *nsync = nullptr;             // hand-over state of lg_k_narrow (models it serves: narrow_shape)
    RgSync *rgsync = nullptr;                // flags of lg_k_rows_geglu
    unsigned long long *tstamps = nullptr;   // [LG_XTAIL_UNITS][8] phase stamps of the last such launch (option xcd_tail_stamps)
    int tail_stamps = 0;
    int wait_polls = 1 << 16;                // option: polls after which a kernel gives up a hand-over inside its launch
    bool xffn_built = false;                 // streams and working memory exist
    int xffn_cls = -1;                       // which instantiation serves the shape
    int xffn_delay = 0;                      // option: units of 64 clocks its compute wavefronts wait before they request their weights
    float *slabs = nullptr, *xact = nullptr; // [8][max_rows][E] partial sums of ffn_down; [8][max_rows][max FF/8] gelu(gate)*up per XCD
    uint32_t *xq8 = nullptr;                 // [8][E/32][80] q8 rows per XCD
    XcdSync *xsync = nullptr;
    std::map<GraphKey, hipGraphExec_t> graphs;           // null: launched as it is (capture_behind)
    Profile prof;
    // a draft head (src/mtp.c) is a model whose layers own no cache: they read `target`'s
    lg_hip_model *target = nullptr;
    std::vector<lg_hip_model *> drafts;      // heads attached to this (target) model
    uint8_t *w_pre = nullptr, *w_post = nullptr;         // next-token pre / post projections, tiled
    int8_t *catq = nullptr;                  // q8 of [embedding(token) * sqrt(nb), h_prev], width 2*nb
    float *hprev = nullptr;                  // post-projection of the previous draft's hidden (chained drafts)
    bool draft_chain = false;
};

struct lg_hip_kv {
    lg_hip_model *m = nullptr;
    int max_seq = 0, tiles_max = 0;                     // tiles_max: stride of the partials, tiles a block can touch
    int prompt_rows = 0;                                // widest prompt block: what the rings' spare rows and the memory that lg_hip_kv_partials grants the scratch of lg_k_wide_attn allow
    size_t scratch_bytes = 0;                           // of pacc: accumulators of verify blocks, scratch of lg_k_wide_attn
    std::vector<int> seq, kv_dim;
    std::vector<uint16_t *> k, v, px_k, px_v;
    float *pm = nullptr, *pl = nullptr, *pacc = nullptr;
    unsigned id = 0;
};
static std::atomic<unsigned> g_kv_ids{0};      // (a thread per model creates caches; a graph is kept for a cache by its id)
static int cu_count();

template <typename T>
static int dev_alloc(lg_hip_model *m, T **p, size_t n) {
    HIP_TRY(hipMalloc((void **)p, n * sizeof(T) ? n * sizeof(T) : 16));
    m->allocs.push_back((void *)*p);
    return 0;
}

// Launches whose workgroups wait for one another, of several models on a device.  Such a launch is sound when its workgroups are all resident
// at some time: a waiting one keeps its CU, up to a whole one.  Two of them at a time, on the streams of two models, could each hold a part of an
// XCD's 32 and wait for the rest until both give up.  So one model has them at a time: the one whose latest such step has not ended yet.  A step of another
// model takes the kernels that wait for nobody (same bits) and overlaps with it as streams do.  With one model at work this is an uncontended lock twice a
// step.  Two models of 12 layers, a step each at a time, us a step (alone; so; with separate kernels in both): 512 values, one row, 203; 217 and 282; 313.  2560 values, five rows, 457; 534 and
// 697; 630.  3840 values, five rows, 628; 778 and 1050; 915, one row 529; 670 and 853; 747.  3840 and 2560 values, five rows, 627 and 459; 722 and 869; 797 and 739: the more of the
// chip the launches of one take, the longer the other's steps, about as many in all.  (Three layers of 512 and of 2560 values when steps waited for one another's: 162 for 106 with separate kernels, 316 for 156.)
// A prompt's blocks wait for nobody, but their kernels run for milliseconds (of rows far into a long cache for tens of them), and their workgroups go on filling the CUs
// that a waiting launch needs whole, up to all 256, while those of it that have a place hold theirs and poll, a bounded number of times: the
// step would be refused.  So while a model has prompt blocks under way the others' steps take the separate kernels too, and the
// blocks follow, on the device, what others have launched of the waiting kind before (PromptTurn).  12 layers of the E4B shape beside prompts of
// 8176 tokens of 6 layers of the 12B shape: a decode step 2440 us and a prompt 71 ms with waiting launches in the steps, 1820 and 54 so (alone 447 and 50); 5 rows
// 2555 and 81, 2170 and 57.
struct Turns {
    std::mutex mu;                             // not held over launches: a thread that launches many steps would keep the others out
    lg_hip_model *last = nullptr;              // whose step with such launches was the latest
    int prompts = 0;                           // models with prompt blocks under way
};
static Turns *turns_of(int device) {
    static std::mutex mu;
    static auto *all = new std::map<int, Turns>();         // (kept: models may outlive the library's static objects)
    std::lock_guard<std::mutex> hold(mu);
    return &(*all)[device];
}
static lg_hip_model *stream_owner(lg_hip_model *m) { return m->target ? m->target : m; }       // (a draft head has its target's stream)
// Whether a step of m that is launched now may hold such launches
static bool may_wait(const lg_hip_model *m) { return m->numbered && !(m->target ? m->target : m)->plain; }
// For a launch of that kind outside of any model, on a stream that is waited for before the lock is given back
static int take_turn_alone(std::unique_lock<std::mutex> &turn) {
    int device = 0;
    HIP_TRY(hipGetDevice(&device));
    Turns *t = turns_of(device);
    for (;;) {
        turn = std::unique_lock<std::mutex>(t->mu);
        if (!t->prompts && (!t->last || !t->last->launching)) break;
        turn.unlock();
        std::this_thread::yield();
    }
    if (t->last) HIP_TRY(hipStreamSynchronize(t->last->stream));
    return 0;
}

// Memory that workgroups of a launch hand data over in, every word or flag with the launch's number (lg_tag): zero, which is the number of no launch
// (the last of a step's LG_STEP_LAUNCHES is not used)
template <typename T>
static int mark_alloc(lg_hip_model *m, T **p, size_t n = 1) {
    if (dev_alloc(m, p, n)) return -7;
    m->marks.emplace_back((void *)*p, n * sizeof(T));
    HIP_TRY(clear_now(m->stream, *p, 0, n * sizeof(T)));
    return 0;
}
// Called ahead of `steps` more steps of the model on its stream, never under capture.  Marks come round, a tag's 28 bits after 2^20 steps, those of a FarRows unit after 2^16 (two minutes
// of steps of 1.7 ms), and what no launch has written since (the rows of a wider block, say) would then count as the present launch's.
// Cleared every LG_MARK_STEPS it is never that old.  (2 MB at most, a few microseconds.)
static int count_steps(lg_hip_model *m, int steps) {
    if ((m->marked_steps += steps) <= LG_MARK_STEPS) return 0;
    m->marked_steps = steps;
    for (auto &p : m->marks) HIP_TRY(hipMemsetAsync(p.first, 0, p.second, m->stream));
    return 0;
}

extern "C" int lg_hip_model_create(const struct lg_hip_config *c, int device, lg_hip_model **out) {
    if (!c || !out) return fail(-1, "model_create: null argument");
    if (c->n_layer <= 0 || c->n_embd <= 0 || c->n_embd % 256 || c->n_embd > 256 * LG_MAXV || c->n_head <= 0 ||
        c->n_vocab <= 0 || c->n_vocab % 32)
        return fail(-2, "model_create: unsupported shape (n_embd %d must be a multiple of 256 and <= %d, n_vocab %d a multiple of 32)",
                    c->n_embd, 256 * LG_MAXV, c->n_vocab);
    if (c->n_embd_per_layer % 32) return fail(-2, "model_create: per-layer embedding width %d must be a multiple of 256 or 0", c->n_embd_per_layer);
    if (lg_hip_device_count() <= device) return fail(-3, "model_create: no HIP device %d (the verify step has no CPU path)", device);
    HIP_TRY(hipSetDevice(device));
    if (cu_count() <= 0) return fail(-3, "model_create: device %d does not tell its number of compute units", device);      // (launches are cut by it)
    lg_hip_model *m = new lg_hip_model();
    m->device = device;
    m->turns = turns_of(device);
    m->numbered = c->n_layer < LG_STEP_LAUNCHES;
    m->n_layer = c->n_layer; m->E = c->n_embd; m->H = c->n_head; m->n_vocab = c->n_vocab;
    m->window = c->sliding_window; m->ple = c->n_embd_per_layer; m->n_kv_start = c->n_kv_start;
    m->eps = c->rms_eps; m->base = c->rope_freq_base; m->base_swa = c->rope_freq_base_swa; m->softcap = c->logit_softcap;
    m->is_local.assign(c->is_local, c->is_local + c->n_layer);
    m->ffn_len.assign(c->ffn_len, c->ffn_len + c->n_layer);
    m->head_dim.assign(c->head_dim, c->head_dim + c->n_layer);
    m->n_head_kv.assign(c->n_head_kv, c->n_head_kv + c->n_layer);
    if (getenv("LG_HIP_NO_GRAPH")) m->use_graph = 0;       // un-captured launches (kernel tracing tools)
    if (getenv("LG_HIP_NO_FUSE")) m->fuse_rows = 0;        // row work in kernels of its own (comparison runs)
    if (getenv("LG_HIP_NO_ATTN_ROWS")) m->attn_rows = 0;   // attention tiles per row everywhere (comparison runs)
    if (const char *e = getenv("LG_HIP_ATTN_ROWS_FQ")) m->attn_rows_fq = atoi(e) != 0;
    if (const char *e = getenv("LG_HIP_ROWS_GEGLU")) m->rows_geglu = atoi(e) != 0;     // the row work ahead of gate/up inside the gate/up launch
    if (const char *e = getenv("LG_HIP_XCD_TAIL_SPREAD")) m->tail_spread = atoi(e);   // 0: the one-XCD tail as ple/32 x rows units of 4 wavefronts only; 2: as 8-wavefront units at 3 and 4 rows too
    if (const char *e = getenv("LG_HIP_WIDE_PREFILL")) m->wide_prefill = atoi(e) != 0;     // 0: prompts in verify blocks, and none of the copies that prompt blocks read
    if (getenv("LG_HIP_NO_DOWN_KQ")) m->down_kq = 0;       // ffn_down of verify blocks by whole rows everywhere (comparison runs)
    hipError_t e = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&m->stream2, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&m->ev_fork, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&m->ev_join, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&m->ev_turn, hipEventDisableTiming);
    if (e != hipSuccess) { delete m; return fail(-100 - (int)e, "hipStreamCreate: %s", hipGetErrorString(e)); }
    if (getenv("LG_HIP_FORK")) m->fork_ple = atoi(getenv("LG_HIP_FORK")) != 0;   // the per-layer inputs as a second branch (comparison runs)
    *out = m;
    return 0;
}

extern "C" int lg_hip_model_tensor(lg_hip_model *m, const char *name, uint32_t type, uint32_t n_dims,
                                   const uint64_t *dims, const void *data) {
    if (!m || !name || !dims || !data || n_dims < 1 || n_dims > 4) return fail(-1, "model_tensor: bad argument");
    if (m->committed) return fail(-4, "model_tensor: model already committed");
    static const char *top[] = { "token_embd.weight", "output_norm.weight", "rope_freqs.weight",
                                 "per_layer_token_embd.weight", "per_layer_model_proj.weight", "per_layer_proj_norm.weight",
                                 "pre_projection.weight", "post_projection.weight" };
    bool known = !strncmp(name, "blk.", 4);
    for (const char *t : top) known = known || !strcmp(name, t);
    if (!known) return 1;
    HostTensor h;
    h.type = type; h.n_dims = n_dims; h.data = data;
    for (int i = 0; i < 4; ++i) h.dims[i] = i < (int)n_dims ? dims[i] : 1;
    m->host[name] = h;
    return 0;
}

static const HostTensor *find(lg_hip_model *m, const std::string &name) {
    auto it = m->host.find(name);
    return it == m->host.end() ? nullptr : &it->second;
}
static std::string lname(int L, const char *leaf) { return "blk." + std::to_string(L) + "." + leaf; }

static int upload_vec(lg_hip_model *m, const std::string &name, size_t n, bool required, float **out) {
    const HostTensor *t = find(m, name);
    *out = nullptr;
    if (!t) return required ? fail(-5, "model_commit: tensor %s is missing", name.c_str()) : 0;
    size_t have = 1;
    for (uint32_t i = 0; i < t->n_dims; ++i) have *= t->dims[i];
    if (t->type != 0 || have != n) return fail(-6, "model_commit: %s must be f32 with %zu elements", name.c_str(), n);
    if (dev_alloc(m, out, n)) return -7;
    HIP_TRY(copy_now(m->stream, *out, t->data, n * 4, hipMemcpyHostToDevice));
    return 0;
}

struct RowSrc { const HostTensor *t; };
static int check_mat(const HostTensor *t, const std::string &name, uint64_t k, uint64_t mrows) {
    if (!t) return fail(-5, "model_commit: tensor %s is missing", name.c_str());
    if (t->type != 2) return fail(-6, "model_commit: %s has ggml type %u; the verify path takes q4_0 matrices only", name.c_str(), t->type);
    if (t->dims[0] != k || t->dims[1] != mrows) return fail(-6, "model_commit: %s is %llu x %llu, expected %llu x %llu", name.c_str(),
        (unsigned long long)t->dims[0], (unsigned long long)t->dims[1], (unsigned long long)k, (unsigned long long)mrows);
    if (k % 256 || mrows % 8) return fail(-6, "model_commit: %s needs row length %% 256 == 0 and rows %% 8 == 0", name.c_str());
    return 0;
}
// f32 / f16 / bf16 (ggml types 0 / 1 / 30): matrices a QAT conversion keeps at full precision
static bool float_typed(const HostTensor *t) { return t && (t->type == 0 || t->type == 1 || t->type == 30); }
static int upload_float_mat(lg_hip_model *m, const HostTensor *t, const std::string &name, uint64_t k, uint64_t mrows, float **out) {
    if (t->dims[0] != k || t->dims[1] != mrows) return fail(-6, "model_commit: %s is %llu x %llu, expected %llu x %llu", name.c_str(),
        (unsigned long long)t->dims[0], (unsigned long long)t->dims[1], (unsigned long long)k, (unsigned long long)mrows);
    if (k % 256) return fail(-6, "model_commit: %s needs row length %% 256 == 0", name.c_str());
    const size_t n = (size_t)k * mrows;
    std::vector<float> wide;
    const float *src = (const float *)t->data;
    if (t->type != 0) {                                       // widening f16 / bf16 to f32 is exact
        wide.resize(n);
        const uint16_t *h = (const uint16_t *)t->data;
        for (size_t i = 0; i < n; ++i) {
            if (t->type == 1) wide[i] = lg_f16_to_f32(h[i]);
            else { const uint32_t u = (uint32_t)h[i] << 16; memcpy(&wide[i], &u, 4); }
        }
        src = wide.data();
    }
    if (dev_alloc(m, out, n)) return -7;
    HIP_TRY(copy_now(m->stream, *out, src, n * 4, hipMemcpyHostToDevice));
    return 0;
}
// upload a tiled matrix whose virtual rows are given by `rows`
static int upload_tiled(lg_hip_model *m, const std::vector<const uint8_t *> &rows, int k, uint8_t **out,
                        std::vector<uint8_t> &stage, bool rowblocks = false) {
    const size_t bytes = lg_hip_repacked_bytes(k, (int)rows.size());
    if (!bytes || (rowblocks && (rows.size() % 64 || lg_segments(k) != 8))) return fail(-6, "model_commit: cannot tile a %zu x %d matrix", rows.size(), k);
    stage.resize(bytes);
    if (rowblocks) repack_rowblocks(rows.data(), k, (int)rows.size(), stage.data());
    else repack_rows(rows.data(), k, (int)rows.size(), stage.data());
    if (dev_alloc(m, out, bytes)) return -7;
    HIP_TRY(copy_now(m->stream, *out, stage.data(), bytes, hipMemcpyHostToDevice));
    return 0;
}
// the wide form of an uploaded matrix: 0.81 bytes a weight beside the 0.56 of its tiles.  Only prompt blocks read it: none for a
// draft head, nor for a model whose option wide_prefill is off when it is committed.
static int wide_form(lg_hip_model *m, const uint8_t *tiles, int k, int rows, bool rowblocks, uint8_t **out) {
    if (m->target || !m->wide_prefill) return 0;
    if (dev_alloc(m, out, lg_wide_bytes(k, rows))) return -7;
    const size_t n = (size_t)((rows + LG_WT - 1) / LG_WT * LG_WT) * (size_t)(k >> 5);
    hipLaunchKernelGGL(lg_k_wide_pack, dim3((unsigned)((n + LG_WG - 1) / LG_WG)), dim3(LG_WG), 0, nullptr, tiles, k, rows, rowblocks ? 1 : 0, *out);
    HIP_TRY(hipGetLastError());
    return 0;
}
static void push_rows(std::vector<const uint8_t *> &rows, const HostTensor *t, uint64_t r0, uint64_t n) {
    const size_t rb = (size_t)(t->dims[0] / 32) * 18;
    for (uint64_t r = r0; r < r0 + n; ++r) rows.push_back((const uint8_t *)t->data + r * rb);
}


// ---- weight streams of the XCD-partitioned feed-forward kernel (lg_xffn.h) --------------------------
// Shapes it is instantiated for: { gate/up operands per workgroup, blocks per gate/up segment (capacity), ffn_down
// chains per wavefront, blocks per ffn_down segment (capacity), q8 blocks of an XCD's activations (capacity) }.
struct XffnClass { int ops, nc, uw, ndc, cbc; };
static const XffnClass k_xffn_classes[] = { { 1, 2, 1, 8, 8 },       // E <= 512, FF <= 2048 (the small test models)
                                            { 3, 10, 2, 10, 40 },    // E4B shape: E 2560, FF 10240
                                            { 4, 15, 2, 15, 60 } };  // 12B shape: E 3840, FF 15360
static size_t xffn_lds(const XffnGeo &g, int M) { return g.lds(M); }
static int xffn_class_of(const XffnGeo &g) {
    if (!g.ok || (g.SX != 1 && g.SX != 4) || g.lds(LG_HIP_MAX_ROWS) + 256 > 160 * 1024) return -1;
    for (int c = 0; c < (int)(sizeof k_xffn_classes / sizeof k_xffn_classes[0]); ++c) {
        const XffnClass &k = k_xffn_classes[c];
        if (g.ops == k.ops && g.nit <= k.nc && (g.units + 7) / 8 <= k.uw && g.nitd <= k.ndc && g.CB <= k.cbc) return c;
    }
    return -1;
}
template <typename F>
static void for_workgroups(F work) {                  // the 256 workgroup streams, on a few host threads
    unsigned hw = std::thread::hardware_concurrency();
    const int nt = (int)(hw ? (hw > 16 ? 16 : hw) : 4);
    std::vector<std::thread> pool;
    for (int t = 0; t < nt; ++t) pool.emplace_back([=]() { for (int wg = 256 * t / nt; wg < 256 * (t + 1) / nt; ++wg) work(wg); });
    for (auto &th : pool) th.join();
}
// gate/up: workgroup (XCD x = wg % 8, rank r = wg / 8) owns the FFN columns x*C + r*CW .. + CW-1; its weight rows are
// those columns' gate rows followed by their up rows, cut into operands of 32; per K segment and operand: the nibble
// bytes as [pair of blocks][half h][row n] 8 + 8 bytes, then the f16 scales as [pair][row n] 2 + 2 bytes (an odd count
// of blocks is padded with a zero block)
static void xffn_pack_gu(const uint8_t *gate, const uint8_t *up, const XffnGeo &g, uint8_t *dst) {
    const size_t rowb = (size_t)g.nb * 18;
    memset(dst, 0, 256 * g.gu_bytes);
    for_workgroups([&](int wg) {
        const int x = wg & 7, r = wg >> 3, c0 = x * g.C + r * g.CW;
        for (int sg = 0; sg < 8; ++sg)
            for (int o = 0; o < g.ops; ++o) {
                const int vr = g.R2 - 32 * o < 32 ? g.R2 - 32 * o : 32;
                uint8_t *ob = dst + (size_t)wg * g.gu_bytes + (size_t)sg * g.gu_seg + (size_t)32 * o * g.rb;
                for (int n = 0; n < vr; ++n) {
                    const int li = 32 * o + n;
                    const uint8_t *row = li < g.CW ? gate + (size_t)(c0 + li) * rowb : up + (size_t)(c0 + li - g.CW) * rowb;
                    for (int it = 0; it < g.nit; ++it) {
                        const uint8_t *blk = row + (size_t)(sg * g.nit + it) * 18;
                        for (int h = 0; h < 2; ++h) memcpy(ob + (size_t)(((it >> 1) * 2 + h) * vr + n) * 16 + (it & 1) * 8, blk + 2 + 8 * h, 8);
                        memcpy(ob + (size_t)g.nitp * vr * 16 + (size_t)((it >> 1) * vr + n) * 4 + (it & 1) * 2, blk, 2);
                    }
                }
            }
    });
}
// ffn_down: workgroup (x, r) owns the output rows r*RW .. + RW-1 and the K segments x*SX .. + SX-1 of them; per
// (operand of 32 rows, segment): nibble bytes [pair of blocks][half][row], then scales [pair][row]
static void xffn_pack_dn(const uint8_t *down, const XffnGeo &g, uint8_t *dst) {
    const size_t rowb = (size_t)(g.FF >> 5) * 18;
    memset(dst, 0, 256 * g.dn_bytes);
    for_workgroups([&](int wg) {
        const int x = wg & 7, r = wg >> 3;
        for (int gr = 0; gr < g.groups; ++gr) {
            const int vr = g.RW - 32 * gr < 32 ? g.RW - 32 * gr : 32;
            for (int sx = 0; sx < g.SX; ++sx) {
                uint8_t *ub = dst + (size_t)wg * g.dn_bytes + (size_t)(gr * g.SX * 32 + sx * vr) * g.rbd;
                for (int n = 0; n < vr; ++n) {
                    const uint8_t *row = down + (size_t)(r * g.RW + 32 * gr + n) * rowb;
                    for (int it = 0; it < g.nitd; ++it) {
                        const uint8_t *blk = row + (size_t)((x * g.SX + sx) * g.nitd + it) * 18;
                        for (int h = 0; h < 2; ++h) memcpy(ub + (size_t)(((it >> 1) * 2 + h) * vr + n) * 16 + (it & 1) * 8, blk + 2 + 8 * h, 8);
                        memcpy(ub + (size_t)g.nitdp * vr * 16 + (size_t)((it >> 1) * vr + n) * 4 + (it & 1) * 2, blk, 2);
                    }
                }
            }
        }
    });
}

// ffn_down as the streams of lg_k_down_m: workgroup (row group r of 64, K quarter q), per segment 8q + s and operand of up to
// 32 rows the pair layout of the streams above
static void pack_down_m(const uint8_t *down, const DownMGeo &g, uint8_t *dst) {
    const size_t rowb = (size_t)(g.FF >> 5) * 18;
    memset(dst, 0, 256 * g.wg_bytes);
    for_workgroups([&](int wg) {
        const int r = wg >> 2, q = wg & 3;
        for (int s = 0; s < 8; ++s)
            for (int o = 0; o < g.ops; ++o) {
                const int vr = g.RW - 32 * o < 32 ? g.RW - 32 * o : 32;
                uint8_t *ob = dst + (size_t)wg * g.wg_bytes + (size_t)s * g.seg_bytes + (size_t)32 * o * g.nitdp * 18;
                for (int n = 0; n < vr; ++n) {
                    const uint8_t *row = down + (size_t)(r * g.RW + 32 * o + n) * rowb;
                    for (int it = 0; it < g.nitd; ++it) {
                        const uint8_t *blk = row + (size_t)((8 * q + s) * g.nitd + it) * 18;
                        for (int h = 0; h < 2; ++h) memcpy(ob + (size_t)(((it >> 1) * 2 + h) * vr + n) * 16 + (it & 1) * 8, blk + 2 + 8 * h, 8);
                        memcpy(ob + (size_t)g.nitdp * vr * 16 + (size_t)((it >> 1) * vr + n) * 4 + (it & 1) * 2, blk, 2);
                    }
                }
            }
    });
}
// shapes lg_k_down_m is instantiated for: operands per workgroup, pairs of blocks per segment
static bool down_m_shape(const DownMGeo &g) {
    return g.ok && ((g.ops == 1 && g.npairs <= 3) || (g.ops == 2 && g.npairs <= 5) || (g.ops == 2 && g.npairs <= 8));
}

// attn_output as the chains of lg_k_attn_tail: chain (row block rb of 32 rows, K segment c of 8) = the segment's nit blocks
// of the 32 rows in the pair layout of the streams above; chains ordered [rb][c], nit * 576 bytes each
static void pack_o_chains(const uint8_t *const *rows, int k, int m, uint8_t *dst) {
    const int nit = k / 32 / 8;
    const size_t cb = (size_t)nit * 576;
    for (int rb = 0; rb < m / 32; ++rb)
        for (int c = 0; c < 8; ++c) {
            uint8_t *ub = dst + ((size_t)rb * 8 + c) * cb;
            for (int n = 0; n < 32; ++n)
                for (int it = 0; it < nit; ++it) {
                    const uint8_t *blk = rows[rb * 32 + n] + (size_t)(c * nit + it) * 18;
                    for (int h = 0; h < 2; ++h) memcpy(ub + (size_t)(((it >> 1) * 2 + h) * 32 + n) * 16 + (it & 1) * 8, blk + 2 + 8 * h, 8);
                    memcpy(ub + (size_t)nit * 512 + (size_t)((it >> 1) * 32 + n) * 4 + (it & 1) * 2, blk, 2);
                }
        }
}
// Chains of pairs of segments (lg_mid.h)
static void pack_pairs(const uint8_t *const *rows, int k, int m, uint8_t *dst) {
    const int nit = k / 256, nitp = (nit + 1) & ~1;
    auto work = [&](int r0, int r1) {
        for (int rb = r0; rb < r1; ++rb)
            for (int sp = 0; sp < 4; ++sp) {
                uint8_t *ub = dst + ((size_t)rb * 4 + sp) * nitp * 576;
                for (int l = 0; l < 64; ++l)
                    for (int it = 0; it < nit; ++it) {
                        const int sg = l >> 5, hf = (l >> 4) & 1, c = l & 15;
                        const uint8_t *blk = rows[rb * 16 + c] + (size_t)((2 * sp + sg) * nit + it) * 18;
                        uint8_t *q = ub + (size_t)((it >> 1) * 64 + l) * 16 + (it & 1) * 8;
                        for (int i = 0; i < 8; ++i) q[i] = blk[2 + 8 * hf + i] ^ 0x88;
                        if (!hf) memcpy(ub + (size_t)nitp * 512 + (size_t)((it >> 1) * 32 + sg * 16 + c) * 4 + (it & 1) * 2, blk, 2);
                    }
            }
    };
    std::vector<std::thread> pool;
    const int nt = m / 16 < 16 ? 1 : 8;
    for (int t = 0; t < nt; ++t) pool.emplace_back(work, (int)((long long)(m / 16) * t / nt), (int)((long long)(m / 16) * (t + 1) / nt));
    for (auto &th : pool) th.join();
}
static int upload_pairs(lg_hip_model *m, const std::vector<const uint8_t *> &rows, int k, uint8_t **out, std::vector<uint8_t> &stage) {
    stage.assign(lg_pairs_bytes(k, (int)rows.size()), 0);
    pack_pairs(rows.data(), k, (int)rows.size(), stage.data());
    if (dev_alloc(m, out, stage.size())) return -7;
    HIP_TRY(copy_now(m->stream, *out, stage.data(), stage.size(), hipMemcpyHostToDevice));
    return 0;
}
// Models and layers that lg_k_o_geglu and lg_k_down_qkv serve: one workgroup to a CU takes an equal share of either product
static bool mid_model(const lg_hip_model *m) { return m->numbered && !m->target && cu_count() == LG_XCDS * LG_XCD_WGS && m->E > LG_NARROW_E && m->E <= LG_MID_E && m->E % 256 == 0; }
static bool mid_o_shape(const lg_hip_model *m, int qd, int nff) { return mid_model(m) && qd % 1024 == 0 && qd <= LG_MID_K && nff / 32 <= LG_OG_BLOCKS; }
static bool mid_down_shape(const lg_hip_model *m, int nff, int next_qkv) {
    return mid_model(m) && !m->ple && lg_segments(nff) == 32 && nff <= 1024 * LG_MID_NIT && next_qkv % 32 == 0 && next_qkv <= 32 * LG_XCDS * LG_XCD_WGS;
}
static bool mid_proj_shape(const lg_hip_model *m, int next_qkv) { return mid_model(m) && m->ple == 256 && m->E % 256 == 0 && next_qkv % 32 == 0 && next_qkv <= 32 * LG_XCDS * LG_XCD_WGS; }
// Where the launches of lg_mid.h are faster than the ones they replace (models of 12 layers, one to eight rows, us a layer saved; option mid = 1: everywhere).
// attn_output with gate/up pays for the hand-overs with work that the first product's rows, K values of attention, leave its 256 workgroups little of, and for
// every block of a segment that its form is cut for and the rows have not (10 up to 2560 values, else 15: the loads and products are made all the same).
//   full rows: 2560, K 2048 0.9 .. 0.3, K 4096 1.0 .. 2.6; 2304, K 3072 1.0 .. 1.4; 3840, K 4096 2.0 .. 1.0; K 1024 at four rows 0.5, 0.7, 0.3, at eight -0.4, -1.2, -2.1;
//     3840, K 2048 at four rows 1.0, at eight -0.9
//   one or two blocks short of 15: 3584 and 3328, K 4096, two rows 1.2 and 0.6, four 1.1 and 0.7, eight -0.3 and -1.0; K 1024 0.6 and 0.2, -0.8 and -1.3, -3.7 and -3.4
//   others: 3072, FFN 11776, -0.4 .. -1.5 (K 4096), -0.8 .. -4.0 (K 2048); 768 to 1536, K 1024, -0.5 .. -1.7; 768 to 2048, K 4096, -0.4 at one row, 0.7 .. 1.3 at eight
static bool mid_o_faster(int E, int K, int rows) {
    const int spare = (E <= 2560 ? 10 : LG_MID_NIT) - (E >> 8);
    if (spare == 0 || (E <= 2560 && spare == 1)) return rows <= 4 || K >= (E <= 2560 ? 2048 : 3072);
    if (E > 2560) return spare <= 2 && rows <= (K >= 3072 ? 4 : 2);
    return rows >= 4 && K >= (E >= 1280 ? 3072 : 4096);
}
// ffn_down with q/k/v: one and two rows have had the row work inside the q/k/v launch, so that there is one launch less to save.  One row: 768 to 2048 -0.4 .. -1.3,
// 2304 to 3584 +-0.2, 3840 0.8; two: 768 and 1024 -0.1 .. -0.7, 1280 to 2048 0.8 .. 0, wider 1.0 .. 3.1; three and more (from 2304 on) 0.6 .. 7.2
static bool mid_down_faster(int E, int rows) { return rows >= 3 || (rows == 2 && E >= 1280) || E > 3584; }
// the per-layer projection with q/k/v, the same: one row 768 to 2048 -0.8 .. -1.6, wider -0.1 .. -0.3; two: up to 1280 -0.4 .. -0.8, wider 0.1 .. 1.1; three and more 0.2 .. 6.7
static bool mid_proj_faster(int E, int rows) { return rows >= 3 || (rows == 2 && E >= 1536); }
// shapes lg_k_attn_tail is instantiated for: pairs of blocks per chain, row blocks per unit
static bool attn_tail_shape(int qd, int E, int *np, int *rbs) {
    if (qd % 512 || lg_segments(qd) != 8 || E % 256 || E > 4096) return false;
    const int p = qd / 512, r = (E / 32 + LG_XCD_WGS - 1) / LG_XCD_WGS;
    if (np) *np = p;
    if (rbs) *rbs = r;
    return (p == 1 && r == 1) || (p == 2 && r == 1) || (p == 4 && r == 3);
}

// Models whose layers lg_k_narrow serves: what its registers, LDS and 256 wavefronts hold, q4_0 matrices throughout
static bool narrow_shape(const lg_hip_model *m) {
    if (!m->numbered || cu_count() != LG_XCDS * LG_XCD_WGS || m->E % 256 || m->E > LG_NARROW_E || m->H > LG_NARROW_WGS || (m->ple && m->ple != 256)) return false;
    for (const Layer &y : m->L)
        if (y.hd > LG_WG || y.hd % 64 || y.qd % 256 || y.qd > LG_NARROW_K || y.nff % 256 || y.nff > LG_NARROW_K || y.qkv_m % 8 || y.qkv_m > LG_NARROW_K ||
            !y.wqkv || !y.wo || !y.wgu || !y.wdown || (m->ple && (!y.winp || !y.wproj))) return false;
    return true;
}

// Layers that lg_k_attn_out serves.  (Rows of up to 512 values: lg_k_narrow, or launches as short as this one.)
static bool attn_out_shape(const lg_hip_model *m, const Layer &y) {
    return m->numbered && m->E > LG_NARROW_E && m->E <= LG_AOUT_E && m->E % 256 == 0 && y.qd == LG_AOUT_K && y.hd % 64 == 0 && y.wo;
}

// tiles of 32 positions that a block of `rows` rows of a sliding layer can touch, wherever it starts
static int window_tiles(int window, int rows) { return (window + rows - 1 + 31) / 32 + 1; }
// Layers that it serves at every width of the model's blocks: nothing then asks for attn_output in another launch's form
static bool attn_out_always(const lg_hip_model *m, const Layer &y, int max_rows) {
    return attn_out_shape(m, y) && y.is_local && m->window > 0 && window_tiles(m->window, max_rows) <= (max_rows > LG_AOUT_DOT_ROWS ? LG_AOUT_BATCH : LG_AOUT_TILES);
}

static const float *rope_table(lg_hip_model *m, int is_local, int hd, int *rc) {
    auto key = std::make_pair(is_local, hd);
    auto it = m->rope_tabs.find(key);
    if (it != m->rope_tabs.end()) return it->second;
    std::vector<float> tab((size_t)hd / 2);
    const float base = is_local ? m->base_swa : m->base;
    for (int i = 0; i < hd / 2; ++i) tab[i] = powf(base, -2.0f * (float)i / (float)hd);   // src/cpu/model-cpu.c:90
    float *d = nullptr;
    if (hipMalloc((void **)&d, tab.size() * 4) != hipSuccess || copy_now(m->stream, d, tab.data(), tab.size() * 4, hipMemcpyHostToDevice) != hipSuccess) {
        *rc = fail(-7, "model_commit: rope table upload failed");
        return nullptr;
    }
    m->allocs.push_back(d);
    m->rope_tabs[key] = d;
    return d;
}

extern "C" int lg_hip_model_commit(lg_hip_model *m, int max_rows) {
    if (!m) return fail(-1, "model_commit: null model");
    if (m->committed) return fail(-4, "model_commit: already committed");
    if (max_rows < 1 || max_rows > LG_HIP_MAX_ROWS) return fail(-2, "model_commit: max_rows %d outside 1..%d", max_rows, LG_HIP_MAX_ROWS);
    HIP_TRY(hipSetDevice(m->device));
    m->max_rows = max_rows;
    const int E = m->E, H = m->H, nl = m->n_layer;
    std::vector<uint8_t> stage;
    int rc = 0;
    {
        const HostTensor *t = find(m, "token_embd.weight");
        if ((rc = check_mat(t, "token_embd.weight", E, m->n_vocab))) return rc;
        std::vector<const uint8_t *> rows;
        push_rows(rows, t, 0, m->n_vocab);
        if ((rc = upload_tiled(m, rows, E, &m->emb, stage))) return rc;
        // a second copy in the order the matrix-core lm_head reads (the first also serves the embedding lookup)
        if (max_rows >= 4 && m->n_vocab % 64 == 0 && lg_segments(E) == 8 && !getenv("LG_HIP_NO_HEAD_MFMA"))
            if ((rc = upload_tiled(m, rows, E, &m->emb_rb, stage, true))) return rc;
    }
    if ((rc = upload_vec(m, "output_norm.weight", E, true, &m->output_norm))) return rc;
    int hd_global = 0;
    for (int L = 0; L < nl; ++L) if (!m->is_local[L]) hd_global = m->head_dim[L];
    if (find(m, "rope_freqs.weight") && hd_global)
        if ((rc = upload_vec(m, "rope_freqs.weight", hd_global / 2, true, &m->rope_freqs))) return rc;
    if (m->ple > 0 && find(m, "per_layer_token_embd.weight")) {
        if (m->ple % 32) return fail(-2, "model_commit: per-layer width %d", m->ple);
        const HostTensor *t = find(m, "per_layer_token_embd.weight");
        const uint64_t total = (uint64_t)m->ple * nl;
        if (t->type != 2 || t->dims[0] != total || t->dims[1] != (uint64_t)m->n_vocab)
            return fail(-6, "model_commit: per_layer_token_embd.weight must be q4_0 %llu x %d", (unsigned long long)total, m->n_vocab);
        const size_t bytes = (size_t)m->n_vocab * (total / 32) * 18;
        if (dev_alloc(m, &m->pte, bytes)) return -7;
        HIP_TRY(copy_now(m->stream, m->pte, t->data, bytes, hipMemcpyHostToDevice));
        const HostTensor *p = find(m, "per_layer_model_proj.weight");
        if (float_typed(p)) {
            if ((rc = upload_float_mat(m, p, "per_layer_model_proj.weight", E, total, &m->pmp_f))) return rc;
        } else {
            if ((rc = check_mat(p, "per_layer_model_proj.weight", E, total))) return rc;
            std::vector<const uint8_t *> rows;
            push_rows(rows, p, 0, total);
            if ((rc = upload_tiled(m, rows, E, &m->pmp, stage))) return rc;
            if ((rc = wide_form(m, m->pmp, E, (int)total, false, &m->pmp_w))) return rc;
        }
        if ((rc = upload_vec(m, "per_layer_proj_norm.weight", m->ple, true, &m->proj_norm))) return rc;
    } else m->ple = 0;

    m->L.resize(nl);
    int max_qkv = 0, max_ff = 0, max_qd = 0;
    // the XCD-partitioned feed-forward kernel: one shape for all layers, a chip of 256 CUs in 8 XCDs, blocks of 4+ rows
    XffnGeo xg = lg_xffn_geo(E, m->ffn_len[0]);
    // (its weight streams are second copies of the FFN matrices: built only when the option is asked for at commit)
    bool xffn = max_rows >= 4 && !m->target && m->numbered && cu_count() == LG_XCDS * LG_XCD_WGS && xffn_class_of(xg) >= 0 &&
                getenv("LG_HIP_XCD_FFN") && atoi(getenv("LG_HIP_XCD_FFN")) != 0;
    for (int L = 1; L < nl && xffn; ++L) xffn = m->ffn_len[L] == m->ffn_len[0];
    std::vector<uint8_t> xstage;
    for (int L = 0; L < nl; ++L) {
        Layer &y = m->L[L];
        y.is_local = m->is_local[L]; y.hd = m->head_dim[L]; y.nkv = m->n_head_kv[L]; y.nff = m->ffn_len[L];
        if (y.hd != 64 && y.hd != 128 && y.hd != 256 && y.hd != 512) return fail(-2, "model_commit: layer %d head size %d (64/128/256/512 are built)", L, y.hd);
        if (y.nkv <= 0 || H % y.nkv || H / y.nkv > 8) return fail(-2, "model_commit: layer %d: %d query heads per kv head (at most 8 are built)", L, H / y.nkv);
        if (y.nff % 32) return fail(-2, "model_commit: layer %d feed-forward width %d must be a multiple of 32", L, y.nff);
        y.qd = H * y.hd; y.kd = y.nkv * y.hd;
        y.owns = !m->target && L < m->n_kv_start;
        const int kv_start = m->target ? m->target->n_kv_start : m->n_kv_start;
        y.src = y.owns ? L : kv_start - (y.is_local ? 2 : 1);               // src/cpu/model-cpu.c:175-179, src/mtp.c:173-176
        if (y.src < 0) return fail(-2, "model_commit: layer %d has no layer to share KV with", L);
        if (m->target) {
            const Layer &t = m->target->L[y.src];
            if (t.hd != y.hd || t.nkv != y.nkv || (t.is_local != 0) != (y.is_local != 0))
                return fail(-2, "model_commit: draft block %d (head size %d, %d kv heads, %s) does not match the target layer %d it reads",
                            L, y.hd, y.nkv, y.is_local ? "sliding" : "global", y.src);
        }
        const HostTensor *q = find(m, lname(L, "attn_q.weight")), *k = find(m, lname(L, "attn_k.weight")),
                         *v = find(m, lname(L, "attn_v.weight"));
        if ((rc = check_mat(q, lname(L, "attn_q.weight"), E, y.qd))) return rc;
        std::vector<const uint8_t *> rows;
        push_rows(rows, q, 0, y.qd);
        y.qkv_m = y.qd;
        if (y.owns) {
            if ((rc = check_mat(k, lname(L, "attn_k.weight"), E, y.kd))) return rc;
            push_rows(rows, k, 0, y.kd);
            y.k_off = y.qd; y.v_off = y.qd; y.qkv_m += y.kd;                // no attn_v: V = raw K projection
            if (v) {
                if ((rc = check_mat(v, lname(L, "attn_v.weight"), E, y.kd))) return rc;
                push_rows(rows, v, 0, y.kd);
                y.v_off = y.qd + y.kd; y.qkv_m += y.kd;
            }
        }
        if ((rc = upload_tiled(m, rows, E, &y.wqkv, stage))) return rc;
        if ((rc = wide_form(m, y.wqkv, E, y.qkv_m, false, &y.wqkv_w))) return rc;
        const HostTensor *ig = m->ple == 256 ? find(m, lname(L, "inp_gate.weight")) : nullptr;
        if (L > 0 && (mid_down_shape(m, m->L[L - 1].nff, y.qkv_m) || (ig && ig->type != 2 && mid_proj_shape(m, y.qkv_m))) && (rc = upload_pairs(m, rows, E, &y.wqkv_pc, stage))) return rc;
        if (ig && ig->type == 2 && !m->target && m->numbered && L > 0 && max_rows >= LG_TAIL_MFMA && E % 512 == 0 && E <= 4096 && y.qkv_m % 32 == 0 && cu_count() == LG_XCDS * LG_XCD_WGS) {
            stage.resize((size_t)y.qkv_m * (E / 32) * 18);       // (once more: the chains that lg_k_ple_tail_s takes)
            pack_o_chains(rows.data(), E, y.qkv_m, stage.data());
            if (dev_alloc(m, &y.wqkv_ch, stage.size())) return -7;
            HIP_TRY(copy_now(m->stream, y.wqkv_ch, stage.data(), stage.size(), hipMemcpyHostToDevice));
        }
        rows.clear();
        const HostTensor *o = find(m, lname(L, "attn_output.weight"));
        if ((rc = check_mat(o, lname(L, "attn_output.weight"), y.qd, E))) return rc;
        push_rows(rows, o, 0, E);
        if ((rc = upload_tiled(m, rows, y.qd, &y.wo, stage))) return rc;
        if ((rc = wide_form(m, y.wo, y.qd, E, false, &y.wo_w))) return rc;
        if (mid_o_shape(m, y.qd, y.nff) && !attn_out_always(m, y, max_rows) && (rc = upload_pairs(m, rows, y.qd, &y.wo_pc, stage))) return rc;
        // (8 query heads: the K segments of this projection are the heads, and the merge can run their chains itself)
        if (!m->target && cu_count() == LG_XCDS * LG_XCD_WGS &&
            ((getenv("LG_HIP_XCD_ATTN_TAIL") && atoi(getenv("LG_HIP_XCD_ATTN_TAIL")) > 0 && attn_tail_shape(y.qd, E, nullptr, nullptr)) ||
             (max_rows >= LG_AOUT_DOT_ROWS && attn_out_shape(m, y)))) {
            stage.resize((size_t)E * (y.qd / 32) * 18);
            pack_o_chains(rows.data(), y.qd, E, stage.data());
            if (dev_alloc(m, &y.wo_ch, stage.size())) return -7;
            HIP_TRY(copy_now(m->stream, y.wo_ch, stage.data(), stage.size(), hipMemcpyHostToDevice));
        }
        if (getenv("LG_HIP_MERGE_O") && atoi(getenv("LG_HIP_MERGE_O")) > 0 && !m->target && m->H == 8 && lg_segments(y.qd) == 8 && E % 64 == 0 && y.hd % 32 == 0 && y.hd <= 512 &&
            (rc = upload_tiled(m, rows, y.qd, &y.wo_rb, stage, true))) return rc;
        rows.clear();
        const HostTensor *g = find(m, lname(L, "ffn_gate.weight")), *u = find(m, lname(L, "ffn_up.weight")),
                         *d = find(m, lname(L, "ffn_down.weight"));
        if ((rc = check_mat(g, lname(L, "ffn_gate.weight"), E, y.nff))) return rc;
        if ((rc = check_mat(u, lname(L, "ffn_up.weight"), E, y.nff))) return rc;
        if ((rc = check_mat(d, lname(L, "ffn_down.weight"), y.nff, E))) return rc;
        for (int t = 0; t < y.nff / 32; ++t) { push_rows(rows, g, (uint64_t)t * 32, 32); push_rows(rows, u, (uint64_t)t * 32, 32); }
        if ((rc = upload_tiled(m, rows, E, &y.wgu, stage, true))) return rc;    // row-block tiles (lg_k_geglu_t)
        if ((rc = wide_form(m, y.wgu, E, 2 * y.nff, true, &y.wgu_w))) return rc;
        rows.clear();
        push_rows(rows, d, 0, E);
        if ((rc = upload_tiled(m, rows, y.nff, &y.wdown, stage))) return rc;
        if ((rc = wide_form(m, y.wdown, y.nff, E, false, &y.wdown_w))) return rc;
        rows.clear();
        if (!(getenv("LG_HIP_DOWN_M") && atoi(getenv("LG_HIP_DOWN_M")) <= 0) && !m->target && max_rows >= 4 && cu_count() == LG_XCDS * LG_XCD_WGS) {
            const DownMGeo dg = lg_down_m_geo(E, y.nff);
            if (down_m_shape(dg)) {
                xstage.resize(256 * dg.wg_bytes);
                pack_down_m((const uint8_t *)d->data, dg, xstage.data());
                if (dev_alloc(m, &y.wdn_m, 256 * dg.wg_bytes)) return -7;
                HIP_TRY(copy_now(m->stream, y.wdn_m, xstage.data(), 256 * dg.wg_bytes, hipMemcpyHostToDevice));
                if (!m->dmsync) {
                    if (mark_alloc(m, &m->dmsync)) return -7;
                }
            }
        }
        if (xffn) {                                               // (second copies)
            xstage.resize(256 * (xg.gu_bytes > xg.dn_bytes ? xg.gu_bytes : xg.dn_bytes));
            xffn_pack_gu((const uint8_t *)g->data, (const uint8_t *)u->data, xg, xstage.data());
            if (dev_alloc(m, &y.xgu, 256 * xg.gu_bytes)) return -7;
            HIP_TRY(copy_now(m->stream, y.xgu, xstage.data(), 256 * xg.gu_bytes, hipMemcpyHostToDevice));
            xffn_pack_dn((const uint8_t *)d->data, xg, xstage.data());
            if (dev_alloc(m, &y.xdn, 256 * xg.dn_bytes)) return -7;
            HIP_TRY(copy_now(m->stream, y.xdn, xstage.data(), 256 * xg.dn_bytes, hipMemcpyHostToDevice));
        }
        if (m->ple) {
            if (m->ple != 256) return fail(-2, "model_commit: per-layer width %d (256 is built)", m->ple);
            const HostTensor *ig = find(m, lname(L, "inp_gate.weight")), *pj = find(m, lname(L, "proj.weight"));
            if (float_typed(ig) != float_typed(pj))
                return fail(-6, "model_commit: blk.%d inp_gate and proj must both be q4_0 or both f32/f16/bf16", L);
            if (float_typed(ig)) {
                if ((rc = upload_float_mat(m, ig, lname(L, "inp_gate.weight"), E, m->ple, &y.winp_f))) return rc;
                if ((rc = upload_float_mat(m, pj, lname(L, "proj.weight"), m->ple, E, &y.wproj_f))) return rc;
            } else {
            if ((rc = check_mat(ig, lname(L, "inp_gate.weight"), E, m->ple))) return rc;
            if ((rc = check_mat(pj, lname(L, "proj.weight"), m->ple, E))) return rc;
            push_rows(rows, ig, 0, m->ple);
            if ((rc = upload_tiled(m, rows, E, &y.winp, stage))) return rc;
            if ((rc = wide_form(m, y.winp, E, m->ple, false, &y.winp_w))) return rc;
            rows.clear();
            push_rows(rows, pj, 0, E);
            if ((rc = upload_tiled(m, rows, m->ple, &y.wproj, stage))) return rc;
            if ((rc = wide_form(m, y.wproj, m->ple, E, false, &y.wproj_w))) return rc;
            }
            if ((rc = upload_vec(m, lname(L, "post_norm.weight"), E, true, &y.post_norm))) return rc;
        }
        if ((rc = upload_vec(m, lname(L, "attn_norm.weight"), E, true, &y.attn_norm))) return rc;
        if ((rc = upload_vec(m, lname(L, "attn_q_norm.weight"), y.hd, true, &y.q_norm))) return rc;
        if ((rc = upload_vec(m, lname(L, "attn_k_norm.weight"), y.hd, y.owns, &y.k_norm))) return rc;
        if ((rc = upload_vec(m, lname(L, "post_attention_norm.weight"), E, true, &y.post_attn))) return rc;
        if ((rc = upload_vec(m, lname(L, "ffn_norm.weight"), E, true, &y.ffn_norm))) return rc;
        if ((rc = upload_vec(m, lname(L, "post_ffw_norm.weight"), E, true, &y.post_ffw))) return rc;
        if ((rc = upload_vec(m, lname(L, "layer_output_scale.weight"), 1, false, &y.out_scale))) return rc;
        y.rope_tab = rope_table(m, y.is_local, y.hd, &rc);
        if (!y.rope_tab) return rc;
        y.rope_ff = y.is_local ? nullptr : m->rope_freqs;
        if (y.qkv_m > max_qkv) max_qkv = y.qkv_m;
        if (y.nff > max_ff) max_ff = y.nff;
        if (y.qd > max_qd) max_qd = y.qd;
    }
    if (m->target) {
        const int nb = m->target->E;
        const HostTensor *pre = find(m, "pre_projection.weight"), *post = find(m, "post_projection.weight");
        if ((rc = check_mat(pre, "pre_projection.weight", 2 * (uint64_t)nb, E))) return rc;
        std::vector<const uint8_t *> rows;
        push_rows(rows, pre, 0, E);
        if ((rc = upload_tiled(m, rows, 2 * nb, &m->w_pre, stage))) return rc;
        if (post) {                                                 // optional: without it drafts cannot chain
            if ((rc = check_mat(post, "post_projection.weight", E, nb))) return rc;
            rows.clear();
            push_rows(rows, post, 0, nb);
            if ((rc = upload_tiled(m, rows, E, &m->w_post, stage))) return rc;
        }
        if (dev_alloc(m, &m->catq, (size_t)2 * nb * 5 / 4) || dev_alloc(m, &m->hprev, (size_t)nb)) return -7;
        if (max_rows != 1) return fail(-2, "model_commit: a draft head runs one row at a time");
    }
    m->host.clear();
    // Layer scratch holds the widest block that can run: LG_WIDE_ROWS for a model that takes prompts, max_rows for a
    // draft head (it is never prefilled).  What only the head touches (final-norm rows, per-workgroup maxima, logits)
    // holds max_rows: a prompt block has no head.
    const size_t R = (size_t)(m->target || max_rows > LG_WIDE_ROWS ? max_rows : LG_WIDE_ROWS), HR = (size_t)max_rows;
    // a q8 row is 5/4 bytes per value in a verify block and 13/8 as the digits of a prompt block (tiles of 64 rows)
    auto qb = [&](int k) { return m->target ? R * k * 5 / 4 : lg_wide_q8_bytes((int)R, k) + 256; };
    if (dev_alloc(m, &m->x[0], R * E) || dev_alloc(m, &m->x[1], R * E) || dev_alloc(m, &m->qkv, R * max_qkv) ||
        dev_alloc(m, &m->dout, 4 * R * E) || dev_alloc(m, &m->q_rot, R * max_qd) || dev_alloc(m, &m->hidden_rows, HR * E) || dev_alloc(m, &m->g_hidden, (size_t)E) ||
        dev_alloc(m, &m->aq, qb(max_qd)) || dev_alloc(m, &m->gq, qb(max_ff)) || dev_alloc(m, &m->hq, qb(E) + (size_t)12 * E) ||
        dev_alloc(m, &m->pval, HR * (m->n_vocab / 32)) || dev_alloc(m, &m->pidx, HR * (m->n_vocab / 32)) ||
        dev_alloc(m, &m->logits, HR * m->n_vocab) || dev_alloc(m, &m->ctl, (size_t)1))
        return -7;
    if (m->ple && dev_alloc(m, &m->eq, qb(E) + (size_t)12 * E)) return -7;
    if (!m->target) {                        // hand-over state of the one-XCD kernels (lg_xtail.h)
        if (mark_alloc(m, &m->tsync) || mark_alloc(m, &m->rgsync) || dev_alloc(m, &m->tstamps, (size_t)2 * LG_XTAIL_UNITS * 8) ||
            (m->ple > 0 && (mark_alloc(m, &m->tgf, (size_t)LG_HIP_MAX_ROWS * m->ple) || mark_alloc(m, &m->tpr, (size_t)LG_HIP_MAX_ROWS * E) || mark_alloc(m, &m->trows)))) return -7;
        HIP_TRY(clear_now(m->stream, m->tstamps, 0, (size_t)2 * LG_XTAIL_UNITS * 8 * 8));
        HIP_TRY(clear_now(m->stream, m->aq, 0, qb(max_qd)));       // (row slots past the block are read as operand rows of the matrix cores)
        if (getenv("LG_HIP_XCD_TAIL")) m->xcd_tail = atoi(getenv("LG_HIP_XCD_TAIL"));
    }
    if (mid_model(m) && (mark_alloc(m, &m->mido, (size_t)LG_HIP_MAX_ROWS * E) || mark_alloc(m, &m->midd, (size_t)LG_HIP_MAX_ROWS * E) || mark_alloc(m, &m->mids, (size_t)3 * LG_HIP_MAX_ROWS * E) ||
                         mark_alloc(m, &m->midro) || mark_alloc(m, &m->midao) || mark_alloc(m, &m->midrd))) return -7;
    if (narrow_shape(m)) {
        if (mark_alloc(m, &m->nsync)) return -7;
    } else if (!m->target && cu_count() == LG_XCDS * LG_XCD_WGS) {
        bool any = false;
        for (const Layer &y : m->L) any = any || attn_out_shape(m, y);
        if (any && (mark_alloc(m, &m->aosync) || mark_alloc(m, &m->aorows))) return -7;
    }
    if (getenv("LG_HIP_XCD_ATTN_TAIL")) m->xcd_attn_tail = atoi(getenv("LG_HIP_XCD_ATTN_TAIL"));
    if (getenv("LG_HIP_DOWN_M")) m->down_m = atoi(getenv("LG_HIP_DOWN_M"));
    if (getenv("LG_HIP_MERGE_O")) m->merge_o = atoi(getenv("LG_HIP_MERGE_O"));
    if (getenv("LG_HIP_MERGE_O_SLICES")) m->merge_o_slices = atoi(getenv("LG_HIP_MERGE_O_SLICES"));
    if (m->ple && (dev_alloc(m, &m->pmp_raw, R * m->ple * nl) || dev_alloc(m, &m->pq, qb(m->ple)) || dev_alloc(m, &m->pgf, R * m->ple)))
        return -7;
    if (xffn) {
        if (dev_alloc(m, &m->slabs, (size_t)LG_XCDS * max_rows * E) || dev_alloc(m, &m->xact, (size_t)LG_XCDS * max_rows * xg.C) ||
            dev_alloc(m, &m->xq8, (size_t)LG_XCDS * xg.nb * LG_MU_DWORDS) || mark_alloc(m, &m->xsync)) return -7;
        HIP_TRY(clear_now(m->stream, m->xq8, 0, (size_t)LG_XCDS * xg.nb * LG_MU_DWORDS * 4));        // row slots past the block are read as operand rows
        m->xffn_built = true; m->xffn_cls = xffn_class_of(xg);
        m->xcd_ffn = getenv("LG_HIP_XCD_FFN") && atoi(getenv("LG_HIP_XCD_FFN")) != 0;     // off unless asked for: the separate kernels are faster (see lg_xffn.h)
        m->xffn_delay = 0x100;
    }
    HIP_TRY(hipHostMalloc((void **)&m->lstage, (size_t)2 * m->n_vocab * 4, hipHostMallocDefault));
    memset(m->lstage, 0, (size_t)2 * m->n_vocab * 4);       // (the host's pages of it, 0.4 ms a MB when first touched)
    HIP_TRY(clear_now(m->stream, m->ctl, 0, sizeof(StepCtl)));
    HIP_TRY(clear_now(m->stream, m->g_hidden, 0, (size_t)E * 4));
    m->sched_cap = 4096;
    if (dev_alloc(m, &m->sched, (size_t)m->sched_cap * LG_HIP_MAX_ROWS) || dev_alloc(m, &m->out, (size_t)m->sched_cap * LG_HIP_MAX_ROWS) ||
        dev_alloc(m, &m->adv, (size_t)m->sched_cap))
        return -7;
    // pinned staging: a step's state at 0, a reported step's results at 32 (LG_REPORT_*), from 64 a prompt's tokens or the results of rounds
    HIP_TRY(hipHostMalloc((void **)&m->pin, (64 + (size_t)m->sched_cap * (2 * LG_HIP_MAX_ROWS + 1)) * sizeof(int32_t), hipHostMallocDefault));
    m->pin[32 + LG_REPORT_SEQ] = 0;
    HIP_TRY(hipDeviceSynchronize());
    m->wide_built = !m->target && m->wide_prefill;
    for (int rows = 1; rows <= LG_HIP_MAX_ROWS; ++rows)
        for (const Layer &y : m->L)
            if ((y.wo_pc && mid_o_faster(E, y.qd, rows)) || (y.wqkv_pc && (m->ple ? mid_proj_faster(E, rows) : mid_down_faster(E, rows)))) m->mid_rows |= 1u << rows;
    m->committed = true;
    return 0;
}

extern "C" void lg_hip_model_destroy(lg_hip_model *m) {
    if (!m) return;
    (void)hipSetDevice(m->device);
    (void)hipDeviceSynchronize();
    {
        std::lock_guard<std::mutex> turn(m->turns->mu);
        if (m->turns->last == m) m->turns->last = nullptr;
    }
    for (auto &g : m->graphs) if (g.second) (void)hipGraphExecDestroy(g.second);
    for (void *p : m->allocs) (void)hipFree(p);
    for (hipEvent_t e : m->prof.ev) (void)hipEventDestroy(e);
    if (m->pin) (void)hipHostFree(m->pin);
    if (m->lstage) (void)hipHostFree(m->lstage);
    if (m->target) {
        auto &v = m->target->drafts;
        for (size_t i = 0; i < v.size(); ++i) if (v[i] == m) { v.erase(v.begin() + i); break; }
    }
    if (m->owns_stream && m->stream) (void)hipStreamDestroy(m->stream);
    if (m->stream2) (void)hipStreamDestroy(m->stream2);
    if (m->ev_fork) (void)hipEventDestroy(m->ev_fork);
    if (m->ev_join) (void)hipEventDestroy(m->ev_join);
    if (m->ev_turn) (void)hipEventDestroy(m->ev_turn);
    for (lg_hip_model *d : m->drafts) { d->target = nullptr; d->stream = nullptr; }        // orphaned heads refuse to run
    delete m;
}

// Key tiles that the attention of a prompt block can touch per group of rows, and the scratch it keeps their weights in
// when they are too many for LDS.
static int wide_attn_tiles(const lg_hip_model *m, const Layer &y, int rows, int pos) {
    const int rg = lg_wide_attn_rows(m->H / y.nkv), all = ((pos + rows - 1) >> 5) + 1;
    const int t = (y.is_local && m->window > 0) ? (m->window + rg - 1 + 31) / 32 + 1 : all;
    return ((t < all ? t : all) + 3) & ~3;
}
static size_t wide_attn_scratch(const lg_hip_model *m, const Layer &y, int rows, int pos) {
    const int rg = lg_wide_attn_rows(m->H / y.nkv), tiles = wide_attn_tiles(m, y, rows, pos);
    return tiles <= LG_WA_TILES ? 0 : (size_t)((rows + rg - 1) / rg) * y.nkv * tiles * (16 * 34 * 4);
}

// ---- KV cache ---------------------------------------------------------------------------------
extern "C" int lg_hip_kv_create(lg_hip_model *m, int max_seq, lg_hip_kv **out) {
    if (!m || !out || !m->committed) return fail(-1, "kv_create: model not committed");
    if (max_seq < 1) return fail(-2, "kv_create: max_seq %d", max_seq);
    HIP_TRY(hipSetDevice(m->device));
    lg_hip_kv *kv = new lg_hip_kv();
    kv->m = m; kv->max_seq = max_seq; kv->id = ++g_kv_ids;
    const int nl = m->n_layer;
    kv->seq.assign(nl, 0); kv->kv_dim.assign(nl, 0);
    kv->k.assign(nl, nullptr); kv->v.assign(nl, nullptr); kv->px_k.assign(nl, nullptr); kv->px_v.assign(nl, nullptr);
    int max_hd = 0, any_global = 0;
    for (int L = 0; L < nl; ++L) {
        const Layer &y = m->L[L];
        if (y.hd > max_hd) max_hd = y.hd;
        if (!(y.is_local && m->window > 0)) any_global = 1;
    }
    const size_t pbytes = lg_hip_kv_partials(max_seq, m->window, any_global, m->max_rows, m->H, max_hd, nullptr, &kv->tiles_max);
    for (int L = 0; L < nl; ++L) {
        const Layer &y = m->L[L];
        kv->kv_dim[L] = y.kd;
        if (!y.owns) continue;
        const bool ring = y.is_local && m->window > 0;
        kv->seq[L] = ring ? lg_hip_ring_rows(m->window, max_seq) : max_seq;
        const size_t bytes = (size_t)kv->seq[L] * y.kd * 2;
        hipError_t e1 = hipMalloc((void **)&kv->k[L], bytes), e2 = hipMalloc((void **)&kv->v[L], bytes);
        if (e1 != hipSuccess || e2 != hipSuccess) { lg_hip_kv_destroy(kv); return fail(-7, "kv_create: out of device memory at layer %d", L); }
        (void)hipMemsetAsync(kv->k[L], 0, bytes, m->stream); (void)hipMemsetAsync(kv->v[L], 0, bytes, m->stream);
    }
    const size_t slots = (size_t)m->max_rows * m->H * kv->tiles_max, grant = pbytes / ((size_t)max_hd * 4 + 8) * max_hd * 4;
    auto most = [&](auto need) { size_t n = 0; for (const Layer &y : m->L) n = std::max(n, need(y)); return n; };
    auto prompt_scratch = [&](int rows) { return most([&](const Layer &y) { return wide_attn_scratch(m, y, rows, max_seq > rows ? max_seq - rows : 0); }); };
    kv->prompt_rows = wide_rows_for(max_seq);
    while (kv->prompt_rows > LG_WIDE && prompt_scratch(kv->prompt_rows) > grant) kv->prompt_rows -= LG_WIDE;
    // partials of verify blocks of one or two rows (a long cache, a model committed for no more) are smaller than what 32 prompt rows need
    kv->scratch_bytes = std::max(slots * max_hd * 4, prompt_scratch(kv->prompt_rows));
    // and the two-launch attention of few workgroups, within the same grant
    kv->scratch_bytes = std::max(kv->scratch_bytes, std::min(grant, most([&](const Layer &y) {
        return (size_t)LG_WA_SPLIT_GROUPS * std::min(wide_attn_tiles(m, y, kv->prompt_rows, max_seq > kv->prompt_rows ? max_seq - kv->prompt_rows : 0), LG_WA_SPLIT_MAX) * (16 * 34 * 4); })));
    if (hipMalloc((void **)&kv->pm, slots * 4) != hipSuccess || hipMalloc((void **)&kv->pl, slots * 4) != hipSuccess ||
        hipMalloc((void **)&kv->pacc, kv->scratch_bytes) != hipSuccess) { lg_hip_kv_destroy(kv); return fail(-7, "kv_create: out of device memory for attention partials"); }
    HIP_TRY(hipDeviceSynchronize());
    *out = kv;
    return 0;
}

extern "C" void lg_hip_kv_destroy(lg_hip_kv *kv) {
    if (!kv) return;
    (void)hipSetDevice(kv->m->device);
    (void)hipDeviceSynchronize();
    // graphs captured for this cache hold its pointers
    std::vector<lg_hip_model *> holders(kv->m->drafts);
    holders.push_back(kv->m);
    for (lg_hip_model *h : holders)
        for (auto it = h->graphs.begin(); it != h->graphs.end();) {
            if (it->first[0] == (uint64_t)kv->id) { if (it->second) (void)hipGraphExecDestroy(it->second); it = h->graphs.erase(it); }
            else ++it;
        }
    for (size_t L = 0; L < kv->k.size(); ++L) {
        (void)hipFree(kv->k[L]); (void)hipFree(kv->v[L]); (void)hipFree(kv->px_k[L]); (void)hipFree(kv->px_v[L]);
    }
    (void)hipFree(kv->pm); (void)hipFree(kv->pl); (void)hipFree(kv->pacc);
    delete kv;
}

extern "C" int lg_hip_kv_layout(const lg_hip_kv *kv, int layer, int *rows, int *width) {
    if (!kv || layer < 0 || layer >= (int)kv->seq.size()) return fail(-1, "kv_layout: bad layer %d", layer);
    if (rows) *rows = kv->seq[layer];
    if (width) *width = kv->kv_dim[layer];
    return 0;
}
static int kv_span(const lg_hip_kv *kv, int layer, int which, int row0, int n, size_t *off, size_t *bytes, uint16_t **base) {
    if (!kv || layer < 0 || layer >= (int)kv->seq.size() || !kv->k[layer]) return fail(-1, "kv copy: layer %d owns no cache", layer);
    if (row0 < 0 || n < 0 || row0 + n > kv->seq[layer]) return fail(-2, "kv copy: rows %d..%d outside 0..%d", row0, row0 + n, kv->seq[layer]);
    *off = (size_t)row0 * kv->kv_dim[layer];
    *bytes = (size_t)n * kv->kv_dim[layer] * 2;
    *base = which ? kv->v[layer] : kv->k[layer];
    return 0;
}
extern "C" int lg_hip_kv_write(lg_hip_kv *kv, int layer, int which, int row0, int n, const uint16_t *src) {
    size_t off, bytes; uint16_t *base;
    int rc = kv_span(kv, layer, which, row0, n, &off, &bytes, &base);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(kv->m->device));
    HIP_TRY(hipStreamSynchronize(kv->m->stream));
    HIP_TRY(copy_now(kv->m->stream, base + off, src, bytes, hipMemcpyHostToDevice));
    return 0;
}
extern "C" int lg_hip_kv_read(const lg_hip_kv *kv, int layer, int which, int row0, int n, uint16_t *dst) {
    size_t off, bytes; uint16_t *base;
    int rc = kv_span(kv, layer, which, row0, n, &off, &bytes, &base);
    if (rc) return rc;
    HIP_TRY(hipSetDevice(kv->m->device));
    HIP_TRY(hipStreamSynchronize(kv->m->stream));
    HIP_TRY(copy_now(kv->m->stream, dst, base + off, bytes, hipMemcpyDeviceToHost));
    return 0;
}
extern "C" int lg_hip_kv_save_prefix(lg_hip_kv *kv, int n) {
    if (!kv || n < 0) return fail(-1, "kv_save_prefix: bad argument");
    HIP_TRY(hipSetDevice(kv->m->device));
    HIP_TRY(hipStreamSynchronize(kv->m->stream));
    for (size_t L = 0; L < kv->k.size(); ++L) {
        if (!kv->k[L]) continue;
        const int rows = n < kv->seq[L] ? n : kv->seq[L];
        const size_t bytes = (size_t)rows * kv->kv_dim[L] * 2;
        (void)hipFree(kv->px_k[L]); (void)hipFree(kv->px_v[L]);
        kv->px_k[L] = kv->px_v[L] = nullptr;
        if (!bytes) continue;
        HIP_TRY(hipMalloc((void **)&kv->px_k[L], bytes));
        HIP_TRY(hipMalloc((void **)&kv->px_v[L], bytes));
        HIP_TRY(copy_now(kv->m->stream, kv->px_k[L], kv->k[L], bytes, hipMemcpyDeviceToDevice));
        HIP_TRY(copy_now(kv->m->stream, kv->px_v[L], kv->v[L], bytes, hipMemcpyDeviceToDevice));
    }
    return 0;
}
extern "C" int lg_hip_kv_restore_prefix(lg_hip_kv *kv, int n) {
    if (!kv || n < 0) return fail(-1, "kv_restore_prefix: bad argument");
    HIP_TRY(hipSetDevice(kv->m->device));
    for (size_t L = 0; L < kv->k.size(); ++L) {
        if (!kv->px_k[L]) continue;
        const int rows = n < kv->seq[L] ? n : kv->seq[L];
        const size_t bytes = (size_t)rows * kv->kv_dim[L] * 2;
        HIP_TRY(hipMemcpyAsync(kv->k[L], kv->px_k[L], bytes, hipMemcpyDeviceToDevice, kv->m->stream));
        HIP_TRY(hipMemcpyAsync(kv->v[L], kv->px_v[L], bytes, hipMemcpyDeviceToDevice, kv->m->stream));
    }
    return 0;
}

// (first: of the call's blocks; what an earlier one reported stays)
__global__ void lg_k_set_ctl(StepCtl *ctl, int pos, bool first) { ctl->pos = pos; ctl->step = 0; ctl->report = 0; if (first) ctl->err = 0; }

// ---- launching --------------------------------------------------------------------------------
static size_t lds_mm(int M, int k) { return (size_t)M * k + (size_t)M * (k / 32) * 8; }
// lg_k_attn: queries of the G heads, K and V tiles, exponentials; with the q/k/v preparation fused in, a head
// vector of staging per wavefront (16-byte aligned)
static size_t attn_lds(int G, int hd, bool fused_post) {
    const size_t b = (size_t)G * hd * 4 + (size_t)2 * 32 * (hd + 8) * 2 + (size_t)G * 32 * 4 + (size_t)G * 4;
    return fused_post ? ((b + 15) & ~(size_t)15) + (size_t)(LG_WG / 64) * hd * 4 : b;
}

// Kernels that want more than the default dynamic LDS limit have it raised once per (device, kernel, size).  What
// has been raised is kept in a fixed table (open addressing on the kernel's address; nothing is allocated, so a
// look-up is safe on a path that promises not to allocate); a kernel that finds no free slot has its limit set on
// every call, which costs time and nothing else.
struct LdsRaised { const void *fn; int dev; size_t bytes; };
static LdsRaised g_lds_raised[1024];
static std::mutex g_lds_mu;
template <typename K>
static int set_lds(K kernel, size_t bytes) {
    if (bytes <= 48 * 1024) return 0;
    if (bytes > 160 * 1024) return fail(-8, "kernel needs %zu bytes of LDS (160 KiB per workgroup)", bytes);
    const void *fn = reinterpret_cast<const void *>(kernel);
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_lds_mu);
    const size_t n = sizeof(g_lds_raised) / sizeof(g_lds_raised[0]);
    size_t at = ((uintptr_t)fn >> 4) * 0x9E3779B97F4A7C15ull >> 54;          // 10 bits
    LdsRaised *slot = nullptr;
    for (size_t probe = 0; probe < 32; ++probe, at = (at + 1) % n) {
        LdsRaised &e = g_lds_raised[at];
        if (!e.fn || (e.fn == fn && e.dev == dev)) { slot = &e; break; }
    }
    if (slot && slot->fn && slot->bytes >= bytes) return 0;
    HIP_TRY(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    if (slot) { slot->fn = fn; slot->dev = dev; slot->bytes = bytes; }
    return 0;
}

struct Launcher {
    lg_hip_model *m;
    bool dry;              // only raise LDS limits, launch nothing (done once before a capture)
    int rc = 0;
    bool side = false;     // launches go to the model's second stream (the forked branch of a step)
    hipStream_t stream() const { return side ? m->stream2 : m->stream; }
    // per-class timing: an event pair that the launch itself fills in (begin and end of the kernel's own execution,
    // what a kernel trace reports; a pair recorded around the launch also counts the packet handling, ~1.5 us)
    bool events(int cls, hipEvent_t *a, hipEvent_t *b) {
        if (rc) return false;
        if (hipEventCreate(a) != hipSuccess || hipEventCreate(b) != hipSuccess) { rc = fail(-9, "event create failed"); return false; }
        m->prof.ev.push_back(*a); m->prof.ev.push_back(*b); m->prof.cls.push_back(cls);
        return true;
    }
    void end() {
        if (!rc) { hipError_t e = hipGetLastError(); if (e != hipSuccess) rc = fail(-100 - (int)e, "kernel launch failed: %s", hipGetErrorString(e)); }
    }
};
// (the kernel's parameter types come from the kernel, the arguments are converted to them one by one)
template <typename... P, typename... A>
static void launch_timed(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t st, hipEvent_t e0, hipEvent_t e1, A &&...a) {
    hipExtLaunchKernelGGL(kernel, grid, block, (uint32_t)lds, st, e0, e1, 0, static_cast<P>(a)...);
}

#define LAUNCH(cls, kernel, grid, block, lds, ...) do { if (!lx.rc) { lx.rc = set_lds(kernel, lds); } if (!lx.rc && !lx.dry) { \
    if (lx.m->prof.on) { hipEvent_t e0_, e1_; if (lx.events(cls, &e0_, &e1_)) launch_timed(kernel, grid, block, lds, lx.stream(), e0_, e1_, __VA_ARGS__); } \
    else hipLaunchKernelGGL(kernel, grid, block, lds, lx.stream(), __VA_ARGS__); \
    lx.end(); } } while (0)

// Compute units of the current device (asked until it answers); 0 when it does not, and then no model is created.
static int cu_count() {
    static int n = 0;
    if (n <= 0) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) v = 0;
        n = v;
    }
    return n;
}

// Plain matmul launch: picks the segment count from k and the workgroup shape from the row count
// (small matrices get one wavefront per workgroup so that every CU has work).
template <int M, bool DUMP>
static int launch_mm(Launcher &lx, int cls, const MmArgs &a_in, bool slabs_ok = false) {
    MmArgs a = a_in;                                      // (+ the workgroup size of the launch, set below)
    const int S = lg_segments(a.k), rw = 64 / S, ngroups = a.m / rw;
    const size_t lds = lds_mm(M, a.k);
    if (S == 32 && M >= 4 && slabs_ok && !DUMP) {
        // blocks of four and more rows whose consumer adds four slabs: cut by K quarter (a quarter of the activations
        // per workgroup, several workgroups per CU).  12B shape, 5 rows: ffn_down 16.9 -> 14.3 us, the rows kernel that
        // adds the slabs 6.6 -> 7.5 us, the step 3.814 -> 3.775 ms (2 and 5 wavefronts per workgroup: 3.827, 3.924)
        if constexpr (M >= 4) {
            const int oct = (a.m + 7) / 8, W = 4;
            a.nthreads = 64 * W;
            LAUNCH(cls, (lg_k_mm_kq<M>), dim3((oct + W - 1) / W, 4), dim3(64 * W), (size_t)M * (a.k / 1024) * 320, LG_MM_FIELDS(LG_XA, a) 0);
        }
        return 4;
    } else if (S == 32) {
        // 4 wavefronts (8 rows) per workgroup, or 5 when that makes exactly one workgroup per CU (2560 rows on 256 CUs):
        // with 320 workgroups a quarter of the CUs would hold two of them and the kernel would wait for those
        const int cus = cu_count();
        const int W = (ngroups % 5 == 0 && ngroups / 5 <= cus && ngroups / 4 > cus) ? 5 : 4;
        // chunks of four tiles for the longest rows (15 tiles per lane at k = 15360: 3.96 against 4.00 ms per step at
        // the 12B shape), of two otherwise (10 tiles at k = 10240: 2.602 against 2.618 ms at the E4B shape); one and two rows leave
        // registers for four (1849 -> 1832 and 1966 -> 1954 us; of eight 1851 and 1988)
        a.nthreads = 64 * W;
        if ((a.k >> 5) / 32 >= 12 || M <= 2) LAUNCH(cls, (lg_k_mm<M, 32, 1, DUMP, 4>), dim3((ngroups + W - 1) / W), dim3(64 * W), lds, LG_MM_FIELDS(LG_XA, a) 0);
        else                       LAUNCH(cls, (lg_k_mm<M, 32, 1, DUMP>), dim3((ngroups + W - 1) / W), dim3(64 * W), lds, LG_MM_FIELDS(LG_XA, a) 0);
    } else if (ngroups >= 4096) {
        const int W = 4;
        a.nthreads = 64 * W;
        LAUNCH(cls, (lg_k_mm<M, 8, 2, DUMP>), dim3((ngroups + 2 * W - 1) / (2 * W)), dim3(64 * W), lds, LG_MM_FIELDS(LG_XA, a) 0);
    } else if (a.k >= 2048 && a.k <= 4096 && !DUMP) {         // (longer rows of 8 segments, a head's pre-projection: more than the 16 tiles a group holds)
        // two row groups per workgroup, the tiles of each cut over two wavefronts, which request all of theirs at once
        // (over four was no faster at 8 and 10 tiles per group).  For one row too: a wavefront that takes its tiles two at a time
        // waits for memory five times (E4B shape, decode 1960 -> 1850 us a step, 2 rows 2050 -> 1960, 3 rows 2125 -> 2034; 12B shape
        // 2646 -> 2545, 3 rows 3216 -> 3007)
        if constexpr (!DUMP) {
            const size_t l2 = ((lds + 15) & ~(size_t)15) + (size_t)2 * M * 64 * 4;
            // (over four wavefronts from 12 tiles per group on: 12B shape, k = 3840 and 4096, 3.662 -> 3.645 ms per step)
            a.nthreads = (a.k >> 8) >= 12 ? 512 : 256;
            if ((a.k >> 8) >= 12) LAUNCH(cls, (lg_k_mm_ks<M, 4>), dim3((ngroups + 1) / 2), dim3(512), l2, LG_MM_FIELDS(LG_XA, a) 0);
            else                  LAUNCH(cls, (lg_k_mm_ks<M, 2>), dim3((ngroups + 1) / 2), dim3(256), l2, LG_MM_FIELDS(LG_XA, a) 0);
        }
    } else {
        // Two row groups per workgroup when there are very many groups, and for blocks of 4+ rows when one group per
        // workgroup would leave some CUs with two of them: their activations (16 KB at M = 5) are then staged twice
        // on the CUs that set the kernel's time.  (Short rows, k < 1024, have too little to stage for that to matter.)
        const int W = (ngroups >= 1024 || (M >= 4 && a.k >= 1024 && ngroups > cu_count())) ? 2 : 1;
        a.nthreads = 64 * W;
        LAUNCH(cls, (lg_k_mm<M, 8, 1, DUMP>), dim3((ngroups + W - 1) / W), dim3(64 * W), lds, LG_MM_FIELDS(LG_XA, a) 0);
    }
    return 1;
}

// one block of M rows through the decoder (and the head when with_head)
// f32-weight matmul of a block of M rows: one wavefront per weight row, 8 block rows per workgroup row
template <int M>
static void launch_mmf(Launcher &lx, int cls, const MmfArgs &a) {
    constexpr int MC = M < 8 ? M : 8;
    LAUNCH(cls, (lg_k_mmf<MC>), dim3((a.m + LG_WG / 64 - 1) / (LG_WG / 64), (a.rows + MC - 1) / MC), dim3(LG_WG), 0, a);
}
// `reach`: the positions that the rows go to; a ring of other than a multiple of 32 rows has tiles around its end, which only
// the kernel per row takes (this library's own rings are multiples of 32: reach 0)
static bool attention_rows_shared(int rows, int tiles, int nkv, int hd, int seq, int reach) {
    return rows > 1 && hd <= 256 && seq >= 32 && (seq % 32 == 0 || reach <= seq) && tiles * nkv >= 256;
}
// ... by lg_k_attn_few: up to 9 tiles a CU where the kernel prepares the block's rows itself (whole steps, lg_k_attn_rows against it: 12B shape,
// 4 rows, 1840 (tile, kv head) pairs 3204 -> 3136 us; E4B shape, 3 rows, 2052 pairs 2192 -> 2161; 12B, 4112 pairs, 6 rows at 14000 keys
// 3523 -> 3551, 5 at 8192 3350 -> 3295), up to three where the rows arrive prepared (768 pairs, 5 rows of 16 over 8: 256-wide heads 24.4 -> 24.6 us,
// 64-wide 16.7 -> 17.1, 2 rows 22.4 -> 20.7 and 16.2 -> 15.9; 1600 pairs, 5 rows 34.0 -> 36.9).  13 to 16 units: up to three, where it prepares
// (12B shape, 7 and 8 rows at 3000 keys 3687 -> 3604 and 3766 -> 3698 us, up to nine at 7000 keys 3816 -> 3844 and 3860 -> 3907)
static bool attention_rows_few(int tiles, int units, int nkv, bool prepares) {
    const int per_cu = units <= LG_ATTN_FEW ? (prepares ? 9 : 3) : units <= 16 && prepares ? 3 : 0;
    return tiles * nkv <= per_cu * cu_count();
}
// workgroups of lg_k_attn_rows per kv head: three to a CU at most (its registers hold no more), each walking its share of the tiles
static int attention_rows_wgs(int tiles, int units, int nkv) {
    const int steps = (tiles + lg_attn_rows_tiles(units) - 1) / lg_attn_rows_tiles(units), cap = 3 * cu_count() / nkv;
    return steps < cap ? steps : cap > 1 ? cap : 1;
}

// wavefronts of lg_k_attn_merge_split: a round of 64 tiles each covers the cache's tiles, while the CUs hold all workgroups
// at once (128 registers a wavefront: one workgroup of 16 wavefronts per CU, two of eight)
static int merge_waves(int tiles, int wgs) {
    return tiles <= 256 ? 4 : tiles <= 512 || wgs > cu_count() ? 8 : 16;
}
#define MERGE_SPLIT(M, go, H, hd, tiles) do { const dim3 grid_(H, M, (hd) / 64); const int nw_ = merge_waves(tiles, (H) * (M) * ((hd) / 64)); \
    if (nw_ == 4)      go((lg_k_attn_merge_split<M, 4>), grid_, dim3(256)); \
    else if (nw_ == 8) go((lg_k_attn_merge_split<M, 8>), grid_, dim3(512)); \
    else               go((lg_k_attn_merge_split<M, 16>), grid_, dim3(1024)); } while (0)

// the XCD-partitioned feed-forward launch: 256 workgroups of 512 threads, the instantiation of the shape's class
template <int M>
static void launch_xffn(Launcher &lx, const XffnArgs &a, int cls) {
    if constexpr (M >= 4) {
        const size_t lds = xffn_lds(lg_xffn_geo(a.E, a.FF), M);
        switch (cls) {
            case 0: LAUNCH(KC_FFN, (lg_k_ffn_xcd<M, 1, 2, 1, 8, 8>), dim3(256), dim3(LG_XFFN_THREADS), lds, LG_XFFN_FIELDS(LG_XA, a) 0); break;
            case 1: LAUNCH(KC_FFN, (lg_k_ffn_xcd<M, 3, 10, 2, 10, 40>), dim3(256), dim3(LG_XFFN_THREADS), lds, LG_XFFN_FIELDS(LG_XA, a) 0); break;
            case 2: LAUNCH(KC_FFN, (lg_k_ffn_xcd<M, 4, 15, 2, 15, 60>), dim3(256), dim3(LG_XFFN_THREADS), lds, LG_XFFN_FIELDS(LG_XA, a) 0); break;
            default: lx.rc = fail(-2, "ffn_xcd: no instantiation for this shape");
        }
    }
}

// Whether the layer tail's launch is lg_k_ple_tail_s: 5 to 8 rows (its units fit one per CU), 1 and 2 (it has enough wavefronts for the projection), and 3 and 4 where
// the next layer's projections are part of it (joins; without them it is no faster there: 12 layers of 768 values, four rows, 404 us a step and 395 with lg_k_ple_tail)
static bool tail_spreads(const lg_hip_model *m, int rows, bool joins) { return m->tail_spread && (rows >= 5 || rows <= 2 || joins || m->tail_spread == 2); }
// ... which they are while the workgroups on the other seven XCDs, one to a CU, take 16 or 32 of their rows each
static bool tail_does_qkv(const lg_hip_model *m, int rows, const Layer &next) {
    return m->tail_qkv && m->trows && m->tail_spread && next.qkv_m <= (LG_XCDS - 1) * rows * (LG_XCD_WGS / rows) * (rows >= LG_TAIL_MFMA ? 32 : 16) &&
           (rows < LG_TAIL_MFMA || next.wqkv_ch);
}
// The per-layer-input block of a verify block of `rows` rows as the one-XCD launch lg_k_ple_tail: q4_0 matrices of the
// 256-wide per-layer input, at most LG_XTAIL_UNITS (gate block, row) units, a chip whose workgroups are dealt over 8 XCDs.  joins: with the next layer's projections
static bool use_ple_tail(const lg_hip_model *m, int rows, bool joins) {
    if (!m->ple || !m->tsync || !may_wait(m) || m->xcd_tail <= 0 || m->target) return false;
    if (m->ple != 256 || (m->ple / 32) * rows > LG_XTAIL_UNITS || m->E % 256 || m->E > 4096 || (m->E + 1023) / 1024 > m->ple / 32) return false;
    const int U = (m->ple / 32) * rows;
    const bool spread = tail_spreads(m, rows, joins);        // (lg_k_ple_tail_s: 8 wavefronts per unit, enough of them at every width)
    // blocks of one and two rows: with lg_k_ple_tail_s the tail beats folding the next layer's row work into its q/k/v
    // matmul (E4B shape: 1.994 -> 1.958 ms at one row, 2.127 -> 2.032 at two); with lg_k_ple_tail alone it does not
    if (m->xcd_tail == 1 && rows <= LG_FUSE_ROWS_MAX && m->fuse_rows && !spread) return false;
    if (!spread && (m->E / 8 + 4 * U - 1) / (4 * U) > 4) return false;       // (few rows of a wide model: too few wavefronts for the projection)
    return cu_count() == LG_XCDS * LG_XCD_WGS;
}
// One row of a narrow model: a layer from the merge on, and the next layer's q/k/v, as one launch (every kernel choice left as it comes)
static bool use_narrow(const lg_hip_model *m, int rows) {
    return rows == 1 && m->narrow && m->nsync && may_wait(m) && m->fuse_rows && m->xcd_tail == 1 && m->tail_spread == 1 && !m->xcd_attn_tail && !m->merge_o && !m->fork_ple;
}
// Slices of the E output rows per (head, row) of lg_k_merge_o: a divisor of the E/64 chunks that leaves at most two
// chunks per wavefront, the largest that keeps the launch within one workgroup per CU (else the smallest)
static int merge_o_slices(const lg_hip_model *m, int rows) {
    const int chunks = m->E / 64;
    int best = 0, least = 0;
    for (int d = 1; d <= chunks; ++d) {
        if (chunks % d || (chunks / d + 3) / 4 > 2) continue;
        if (!least) least = d;
        if (8 * rows * d <= cu_count()) best = d;
    }
    const int pick = best ? best : least;
    if (m->merge_o_slices > 0 && chunks % m->merge_o_slices == 0 && (chunks / m->merge_o_slices + 3) / 4 <= 2) return m->merge_o_slices;
    return pick;
}
static bool use_merge_o(const lg_hip_model *m, const Layer &y, int rows, int tiles) {
    if (!y.wo_rb || m->merge_o <= 0 || (m->merge_o == 1 && rows < 3)) return false;
    return tiles < 128 && merge_o_slices(m, rows) > 0;
}
static void launch_merge_o(Launcher &lx, const MergeOArgs &a) {
    const int nit = a.g.hd / 32, rpl = ((a.E / 64) / a.slices + 3) / 4;
    const dim3 grid(a.rows * a.g.H * a.slices);
#define CASE(N, R) if (nit == N && rpl == R) { LAUNCH(KC_MERGE, (lg_k_merge_o<N, R>), grid, dim3(LG_WG), 0, lx.m->ctl, LG_MERGEO_FIELDS(LG_XA, a) 0); return; }
    CASE(2, 1) CASE(2, 2) CASE(4, 1) CASE(4, 2) CASE(8, 1) CASE(8, 2) CASE(16, 1) CASE(16, 2)
#undef CASE
    lx.rc = fail(-2, "merge_o: no instantiation for head_dim %d with %d chunks per wavefront", a.g.hd, rpl);
}

template <int M>
static void launch_down_m(Launcher &lx, const DownMArgs &a) {
    if constexpr (M >= 4) {
        const DownMGeo g = lg_down_m_geo(a.E, a.FF);
        const size_t lds = (size_t)8 * g.nitd * (LG_MU_DWORDS * 4) + (size_t)8 * g.ops * 8 * 32 * 4;
        if (g.ops == 1 && g.npairs <= 3) LAUNCH(KC_DOWN, (lg_k_down_m<M, 1, 3>), dim3(256), dim3(512), lds, LG_DOWNM_FIELDS(LG_XA, a) 0);
        else if (g.ops == 2 && g.npairs <= 5) LAUNCH(KC_DOWN, (lg_k_down_m<M, 2, 5>), dim3(256), dim3(512), lds, LG_DOWNM_FIELDS(LG_XA, a) 0);
        else if (g.ops == 2 && g.npairs <= 8) LAUNCH(KC_DOWN, (lg_k_down_m<M, 2, 8>), dim3(256), dim3(512), lds, LG_DOWNM_FIELDS(LG_XA, a) 0);
        else lx.rc = fail(-2, "down_m: no instantiation for this shape");
    }
}
// tiles a block of `rows` rows can touch (a sliding layer needs only its window's, not the cache's)
static int step_tiles(const lg_hip_model *m, const lg_hip_kv *kv, const Layer &y, int rows, int pos_off) {
    const int window = (y.is_local && m->window > 0) ? m->window + pos_off : 0;
    if (window <= 0) return kv->tiles_max;
    const int t = window_tiles(window, rows);
    return t < kv->tiles_max ? t : kv->tiles_max;
}
// (tiles: what one wavefront holds; more of them, a global layer in a cache of 1248 positions and more, are merged by more of the chip.  The row work
// ahead of gate/up is part of this launch: asked for in another one, by rows_geglu or xcd_ffn, it stays there)
static bool use_attn_out(const lg_hip_model *m, const Layer &y, int rows, int tiles) {
    if (rows >= 4 && ((m->rows_geglu && m->E == 2560) || (m->xcd_ffn && y.xgu))) return false;
    return m->attn_out && m->aosync && may_wait(m) && attn_out_shape(m, y) && (rows <= LG_AOUT_DOT_ROWS ? tiles <= LG_AOUT_TILES : y.wo_ch && tiles <= LG_AOUT_BATCH);
}
// ... on the matrix cores: 4 rows and more, and three of up to 20 tiles
static bool attn_out_chains(const Layer &y, int rows, int tiles) { return rows > LG_AOUT_DOT_ROWS || (rows == LG_AOUT_DOT_ROWS && y.wo_ch && tiles <= LG_AOUT_BATCH); }
// With gate/up the launch has 224 workgroups for blocks of 32 FFN columns, a launch of its own one for each of up to 256: in between, two blocks to some workgroups cost narrow models of
// five rows and more what the join gives (12 layers, us a layer saved at four, five and eight rows: 768 values, FFN 7168 1.3, 0.6, 0.7; 7424 0.1, -0.3, -1.3; 9216 0.6, -0.3, -0.3;
// 1280, 8192 0.3, -0.3, -0.7; 8960 1.3, 0.4, 0.2; 1536, 8192 0.7, -0.2, -0.5; 1792, 7424 0.8, 0.4, 0.1; 2304, 7424 1.4, 0.8, 0.9)
static bool attn_geglu_faster(int E, int blocks, int rows) { return rows <= 4 || blocks <= LG_AOUT_GU_WGS || blocks > LG_XCDS * LG_XCD_WGS || E > 1536; }
// ... with gate/up as part of the launch: two blocks of 32 FFN columns at most for a workgroup on the other seven XCDs; not beside the 13 wavefronts of lg_k_attn_out<3>
static bool attn_out_geglu(const lg_hip_model *m, const Layer &y, int rows, int tiles) {
    return m->attn_geglu && (m->attn_geglu == 1 || attn_geglu_faster(m->E, y.nff / 32, rows)) && m->aorows && y.wgu && y.nff / 32 <= 2 * LG_AOUT_GU_WGS && (rows < LG_AOUT_DOT_ROWS || attn_out_chains(y, rows, tiles));
}
static bool use_attn_tail(const lg_hip_model *m, const Layer &y, int rows, int tiles) {
    if (!y.wo_ch || !m->tsync || !may_wait(m) || !attn_tail_shape(y.qd, m->E, nullptr, nullptr) || m->xcd_attn_tail <= 0 || (m->xcd_attn_tail == 1 && rows < 3)) return false;
    const int slices = (m->E + 1023) / 1024;
    return tiles < 128 && m->H * rows <= 2 * LG_XCD_WGS && slices * rows <= LG_XCD_WGS && y.hd % 32 == 0 && y.hd <= 256;
}
// attn_output, row work and gate/up as one launch; not where one of the options does that row work elsewhere, or has attn_output as a launch of its own (attn_out = 0)
static bool use_mid_o(const lg_hip_model *m, const Layer &y, int rows) {
    return m->mid && (m->mid == 1 || mid_o_faster(m->E, y.qd, rows)) && m->attn_out && m->mido && may_wait(m) && y.wo_pc && y.wgu && !(rows >= 4 && (m->rows_geglu || (m->xcd_ffn && y.xgu)));
}
// ... and the merge of attention's partials: up to LG_MID_MERGE_ROWS rows (more: no gain, see lg_k_o_geglu) of up to LG_AOUT_TILES tiles, which a wavefront holds in
// registers.  (Rows of up to 2560 values have lg_k_attn_out where their layers have 2048 inputs; the others' merge was not tried in here.)
static bool use_mid_merge(const lg_hip_model *m, const Layer &y, int rows, int tiles) {
    return rows <= LG_MID_MERGE_ROWS && use_mid_o(m, y, rows) && m->E > 2560 && tiles <= LG_AOUT_TILES && y.hd % 64 == 0;
}
// ffn_down, row work and the next layer's q/k/v projections as one launch (1 to 3 rows: with the whole rows in LDS)
static bool use_mid_down(const lg_hip_model *m, const Layer &y, const Layer &next, int rows) {
    if (!m->mid || !(m->mid == 1 || mid_down_faster(m->E, rows)) || !m->midd || !may_wait(m) || m->ple || !next.wqkv_pc) return false;
    if (rows >= 4) return m->down_m == 1 && y.wdn_m && m->E > 2048 && lg_down_m_geo(m->E, y.nff).npairs <= LG_MID_NDP;
    return lg_downqkv_lds(rows, y.nff) <= 160 * 1024;
}
// ... with the per-layer projection of a float type in ffn_down's place
static bool use_mid_proj(const lg_hip_model *m, const Layer &next, int rows) {
    return m->mid && (m->mid == 1 || mid_proj_faster(m->E, rows)) && m->midd && may_wait(m) && m->ple && next.wqkv_pc;
}
// Whether a step has launches whose workgroups wait for one another, if it may
static bool step_waits(const lg_hip_model *m, int rows) {
    return may_wait(m) && (use_narrow(m, rows) || (m->attn_out && m->aosync) || (m->mido && (m->mid == 1 || (m->mid && m->mid_rows >> rows & 1))) || use_ple_tail(m, rows, true) || m->rows_geglu || m->xcd_attn_tail > 0 ||
                           (rows >= 4 && ((m->down_m == 1 && m->dmsync) || m->xcd_ffn)));
}
// Held while a step of m is launched (or a round of `head` and m, its target); begin() finds out whether it may have such launches
struct Turn {
    lg_hip_model *own = nullptr;
    int begin(lg_hip_model *m, int rows, const lg_hip_model *head = nullptr) {
        own = stream_owner(m);
        std::lock_guard<std::mutex> lock(own->turns->mu);
        own->launching = true;
        own->plain = false;
        return step_waits(m, rows) || (head && step_waits(head, 1)) ? claim() : 0;
    }
    ~Turn() {
        if (!own) return;
        std::lock_guard<std::mutex> lock(own->turns->mu);
        own->launching = false;
    }
    int claim() {
        lg_hip_model *&last = own->turns->last;
        if (own->turns->prompts > own->prompting) { own->plain = true; return 0; }
        if (last && last != own) {
            if (last->launching) { own->plain = true; return 0; }
            if (!last->turn_recorded) HIP_TRY(hipEventRecord(last->ev_turn, last->stream));
            last->turn_recorded = true;
            const hipError_t e = hipEventQuery(last->ev_turn);
            if (e == hipErrorNotReady) {
                (void)hipGetLastError();                   // (no error, and not to be found as one by the next launch)
                own->plain = true;
                return 0;
            }
            if (e != hipSuccess) return fail(-100 - (int)e, "hipEventQuery: %s", hipGetErrorString(e));
        }
        last = own;
        own->turn_recorded = false;
        return 0;
    }
};
// Held while prompt blocks of m are launched and run.  The caller waits for m's stream before it gives this back, and a failed call here.
struct PromptTurn {
    lg_hip_model *own = nullptr;
    bool done = false;                         // the stream has been waited for
    int begin(lg_hip_model *m) {
        Turns *t = m->turns;
        std::unique_lock<std::mutex> lock(t->mu);
        (own = m)->prompting = true;
        ++t->prompts;                          // (from here on no step of another model is launched with such launches)
        while (t->last && t->last != m && t->last->launching) {
            lock.unlock();
            std::this_thread::yield();
            lock.lock();
        }
        lg_hip_model *last = t->last;
        if (!last || last == m) return 0;
        if (!last->turn_recorded) HIP_TRY(hipEventRecord(last->ev_turn, last->stream));
        last->turn_recorded = true;
        HIP_TRY(hipStreamWaitEvent(m->stream, last->ev_turn, 0));
        return 0;
    }
    ~PromptTurn() {
        if (!own) return;
        if (!done) (void)hipStreamSynchronize(own->stream);
        std::lock_guard<std::mutex> lock(own->turns->mu);
        own->prompting = false;
        --own->turns->prompts;
    }
};
template <int M>
static void launch_attn_tail(Launcher &lx, const XattnTailArgs &a) {
    lg_hip_model *m = lx.m;
    int np = 0, rb = 0;
    if (!attn_tail_shape(a.g.H * a.g.hd, a.E, &np, &rb)) { lx.rc = fail(-2, "attn_tail: no instantiation for this shape"); return; }
    const size_t lds = (size_t)(16 * np) * LG_MU_DWORDS * 4 + (size_t)8 * rb * 8 * 32 * 4;
    const dim3 grid(LG_XCDS * LG_XCD_WGS);
    if (np == 1 && rb == 1) LAUNCH(KC_ATAIL, (lg_k_attn_tail<M, 1, 1>), grid, dim3(512), lds, m->ctl, LG_XATTN_FIELDS(LG_XA, a) 0);
    else if (np == 2 && rb == 1) LAUNCH(KC_ATAIL, (lg_k_attn_tail<M, 2, 1>), grid, dim3(512), lds, m->ctl, LG_XATTN_FIELDS(LG_XA, a) 0);
    else LAUNCH(KC_ATAIL, (lg_k_attn_tail<M, 4, 3>), grid, dim3(512), lds, m->ctl, LG_XATTN_FIELDS(LG_XA, a) 0);
}

template <int M>
static void launch_ple_tail(Launcher &lx, const XtailArgs &a) {
    lg_hip_model *m = lx.m;
    const int E = a.r.g.k;
    {
        // (row j by 32 / M workgroups of 8 wavefronts)
        constexpr int W = M * (32 / M);
        const int G = (E / 8 + 8 * W - 1) / (8 * W);
        static_assert((4096 / 8 + 8 * W - 1) / (8 * W) <= 3, "every row that use_ple_tail admits has an instantiation");
        if (tail_spreads(m, M, a.qw != nullptr) && a.gf && a.r.g.ple == 256 && G >= 1 && G <= 3) {
            const size_t lds = lg_tail_s_lds(M, E, a.r.g.ple, a.qw != nullptr);
            const dim3 grid(LG_XCDS * W);
            static int fits[2][4] = {};                       // per tiles of a gate row group (10, 16) and G: 0 unknown, 1 yes, -1 no (asked once, outside any capture)
            auto launch = [&](auto nit_) {
                constexpr int NIT = decltype(nit_)::value;
                int &ok = fits[NIT == 10][G];
                if (!ok) {
                    int per_cu = 0;
                    hipError_t e = hipErrorInvalidValue;
                    switch (G) {
                        case 1: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, lg_k_ple_tail_s<M, 1, NIT>, 512, lds); break;
                        case 2: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, lg_k_ple_tail_s<M, 2, NIT>, 512, lds); break;
                        case 3: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, lg_k_ple_tail_s<M, 3, NIT>, 512, lds); break;
                    }
                    ok = (e == hipSuccess && per_cu * LG_XCD_WGS >= W) ? 1 : -1;
                }
                if (ok < 0) return false;
                switch (G) {
                    case 1: LAUNCH(KC_TAIL, (lg_k_ple_tail_s<M, 1, NIT>), grid, dim3(512), lds, m->ctl, LG_XTAIL_FIELDS(LG_XA, a) 0); break;
                    case 2: LAUNCH(KC_TAIL, (lg_k_ple_tail_s<M, 2, NIT>), grid, dim3(512), lds, m->ctl, LG_XTAIL_FIELDS(LG_XA, a) 0); break;
                    case 3: LAUNCH(KC_TAIL, (lg_k_ple_tail_s<M, 3, NIT>), grid, dim3(512), lds, m->ctl, LG_XTAIL_FIELDS(LG_XA, a) 0); break;
                }
                return true;
            };
            if (E <= 2560 ? launch(std::integral_constant<int, 10>{}) : launch(std::integral_constant<int, 16>{})) return;
        }
        // (the caller counts on q/k/v once it has asked for them, and the form below does not know of them)
        if (a.qw) { lx.rc = fail(-2, "ple_tail: the units of %d rows of %d values do not fit one XCD with q/k/v", M, E); return; }
    }
    const int U = (a.r.g.ple / 32) * M;
    const int G = (E / 8 + 4 * U - 1) / (4 * U);
    const size_t lds = (size_t)E * 5 / 4 + (size_t)M * a.r.g.ple * 5 / 4;
    const dim3 grid(LG_XCDS * U);
    // the U units wait for each other: all of them must be resident on the 32 CUs of one XCD at once
    static int fits[5] = { 0, 0, 0, 0, 0 };              // per G: 0 unknown, 1 yes, -1 no (asked once, outside any capture)
    if (G >= 1 && G <= 4 && !fits[G]) {
        int per_cu = 0;
        hipError_t e = hipErrorInvalidValue;
        switch (G) {
            case 1: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, lg_k_ple_tail<M, 1>, LG_WG, lds); break;
            case 2: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, lg_k_ple_tail<M, 2>, LG_WG, lds); break;
            case 3: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, lg_k_ple_tail<M, 3>, LG_WG, lds); break;
            case 4: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, lg_k_ple_tail<M, 4>, LG_WG, lds); break;
        }
        fits[G] = (e == hipSuccess && per_cu * LG_XCD_WGS >= U) ? 1 : -1;
    }
    if (G < 1 || G > 4 || fits[G] < 0) { lx.rc = fail(-2, "ple_tail: %d units of %d row groups per wavefront do not fit one XCD", U, G); return; }
    switch (G) {
        case 1: LAUNCH(KC_TAIL, (lg_k_ple_tail<M, 1>), grid, dim3(LG_WG), lds, m->ctl, LG_XTAIL_FIELDS(LG_XA, a) 0); break;
        case 2: LAUNCH(KC_TAIL, (lg_k_ple_tail<M, 2>), grid, dim3(LG_WG), lds, m->ctl, LG_XTAIL_FIELDS(LG_XA, a) 0); break;
        case 3: LAUNCH(KC_TAIL, (lg_k_ple_tail<M, 3>), grid, dim3(LG_WG), lds, m->ctl, LG_XTAIL_FIELDS(LG_XA, a) 0); break;
        case 4: LAUNCH(KC_TAIL, (lg_k_ple_tail<M, 4>), grid, dim3(LG_WG), lds, m->ctl, LG_XTAIL_FIELDS(LG_XA, a) 0); break;
        default: lx.rc = fail(-2, "ple_tail: %d row groups per wavefront", G);
    }
}

template <int M>
static int enqueue_step(lg_hip_model *m, lg_hip_kv *kv, bool with_head, bool dry) {
    Launcher lx{ m, dry };
    const int E = m->E, H = m->H, nl = m->n_layer;
    int cur = 0;                                   // x[cur] holds the residual
    bool have_x = false;                           // false: rows are still token ids
    const float *pend_dout = nullptr, *pend_w = nullptr, *pend_os = nullptr;   // sub-layer output waiting to be added
    int pend_parts = 1;                            // 4 when that output is four slabs of partial sums (wide ffn_down)
    const bool draft = m->target != nullptr;
    const int pos_off = draft ? -1 : 0;            // a draft at pos sees the cache as a query at pos-1 (src/cuda/mtp-kernel.cuh:170-182)
    if (draft) {
        // x = pre . [embedding(token)*sqrt(nb), h_prev] (src/mtp.c:268-278); h_prev is the target's hidden of the
        // accepted row, or for a chained draft post . (this head's previous hidden) (src/cuda/mtp-kernel.cuh:372-389)
        const lg_hip_model *t = m->target;
        const int nb = t->E;
        if (m->draft_chain) {
            MmArgs a{ m->w_post, E, nb, m->hprev, m->hq, nullptr };
            launch_mm<M, false>(lx, KC_PMP, a);
        }
        DraftInArgs d{};
        d.emb = t->emb; d.emb_seg = lg_segments(nb); d.emb_nit = nb / 32 / d.emb_seg; d.emb_scale = sqrtf((float)nb);
        d.toks = m->sched; d.h_prev = m->draft_chain ? m->hprev : t->g_hidden; d.nb = nb; d.q = m->catq;
        LAUNCH(KC_ROWS, lg_k_draft_input, dim3((2 * nb / 4 + LG_WG - 1) / LG_WG), dim3(LG_WG), 0, d, m->ctl);
        MmArgs p{ m->w_pre, 2 * nb, E, m->x[0], m->catq, nullptr };
        launch_mm<M, false>(lx, KC_PMP, p);
        have_x = true;
    }

    // rows kernel: fold the pending sub-layer output into the residual, norm with w_pre, quantize
    auto rows = [&](const float *w_pre, float *h_out, int units = 0, int8_t *q_out = nullptr) {
        RowArgs s{};
        s.q_units = units;
        s.E = E; s.eps = m->eps; s.toks = m->sched; s.q = q_out ? q_out : m->hq;
        if (!have_x) {
            s.emb = m->emb; s.emb_seg = lg_segments(E); s.emb_nit = E / 32 / s.emb_seg; s.emb_scale = sqrtf((float)E);
            s.bump = &m->ctl->launch;                          // the step's first kernel: a new range of launch numbers
        } else s.x = m->x[cur];
        s.dout = pend_dout; s.w_post = pend_w; s.os = pend_os; s.dparts = pend_parts;
        s.w_pre = w_pre; s.h_out = h_out;
        if (pend_dout || !have_x) s.x_out = m->x[cur ^ 1];
        // verify blocks: the tail of the row work (store, norm weight, q8) cut over one workgroup per float4 of a lane
        const int slices = (E + 1023) / 1024;
        s.slices = slices;
        LAUNCH(KC_ROWS, (lg_k_rows<M>), dim3(M, slices), dim3(LG_WG), 0, m->ctl, LG_ROW_FIELDS(LG_XA, s) 0);
        if (s.x_out) cur ^= 1;
        have_x = true; pend_dout = pend_w = pend_os = nullptr; pend_parts = 1;
    };

    // The same row work done by the workgroups of the matmul that consumes it (lg_fused.h): verify-width blocks
    // whose residual is already in memory.  NV = float4 per lane of a row.
    const int NVr = (E + 1023) / 1024;
    // (blocks of one or two rows: wider ones pay more for the repeated row work than for the launch, see lg_fused.h)
    // (two rows of more than 3072 values: 12B shape, 2862 us a step inside the matmul, 2840 ahead of it)
    auto can_fuse = [&]() { return (M == 1 || (M <= LG_FUSE_ROWS_MAX && NVr <= 3)) && have_x && m->fuse_rows && pend_parts == 1; };
    auto row_work = [&](const float *w_pre) {
        RowWork r{ m->x[cur], pend_dout, pend_w, pend_os, m->x[cur ^ 1], w_pre, E, m->eps };
        return r;
    };
    auto row_work_done = [&]() {
        if (pend_dout) cur ^= 1;
        pend_dout = pend_w = pend_os = nullptr; pend_parts = 1;
    };
    auto rows_mm = [&](const float *w_pre, const MmArgs &a, int cls) {      // rows(w_pre) then an 8-segment matmul of the result
        if constexpr (M <= LG_FUSE_ROWS_MAX) {
            constexpr int NW = 4;                            // row groups per workgroup, which all repeat the row work (12B shape, 1024 groups: one 2746 us a decode step, two 2670, four 2648; 5 or 10 MB matrices: no difference)
            RowsMmArgs f{ a, row_work(w_pre) };
            const dim3 grid((a.m / 8 + NW - 1) / NW);
            const size_t lds = lds_mm(M, a.k);
            switch (NVr) {
                case 1: LAUNCH(cls, (lg_k_rows_mm<M, 1, NW>), grid, dim3(LG_WG), lds, LG_ROWSMM_FIELDS(LG_XA, f) 0); break;
                case 2: LAUNCH(cls, (lg_k_rows_mm<M, 2, NW>), grid, dim3(LG_WG), lds, LG_ROWSMM_FIELDS(LG_XA, f) 0); break;
                case 3: LAUNCH(cls, (lg_k_rows_mm<M, 3, NW>), grid, dim3(LG_WG), lds, LG_ROWSMM_FIELDS(LG_XA, f) 0); break;
                default: if constexpr (M == 1) LAUNCH(cls, (lg_k_rows_mm<M, 4, NW>), grid, dim3(LG_WG), lds, LG_ROWSMM_FIELDS(LG_XA, f) 0);      // (two such rows: can_fuse)
            }
            row_work_done();
        }
    };

    const bool narrow = use_narrow(m, M);
    bool qkv_done = false;                         // the layer's projections have been done by the launch before it (lg_k_narrow)
    bool rows_done = false;                        // the row work ahead of the next matmul has been done by the launch before it
    bool join_ple = false;                         // the forked branch has to be waited for before its result is used
    if (m->ple) {
        rows(nullptr, nullptr, 0, m->eq);
        // the per-layer inputs are not needed before layer 0's per-layer gate: they run on the second stream, beside
        // layer 0's attention and feed-forward (captured, the graph gets a second branch)
        const bool fork = m->fork_ple && !dry && !m->prof.on && m->stream2 && !lx.rc;
        if (fork) {
            hipError_t e = hipEventRecord(m->ev_fork, m->stream);
            if (e == hipSuccess) e = hipStreamWaitEvent(m->stream2, m->ev_fork, 0);
            if (e != hipSuccess) lx.rc = fail(-100 - (int)e, "fork of the per-layer input branch: %s", hipGetErrorString(e));
            lx.side = true;
        }
        if (m->pmp_f) {                                       // kept in a float type: the f32 rows themselves are the input
            MmfArgs f{ m->pmp_f, E, m->ple * nl, m->x[cur], E, M, m->pmp_raw, m->ple * nl, nullptr, 0 };
            launch_mmf<M>(lx, KC_PMP, f);
        } else {
        MmArgs a{ m->pmp, E, m->ple * nl, m->pmp_raw, m->eq, nullptr };
        launch_mm<M, false>(lx, KC_PMP, a);
        }
        IplArgs i{ m->pmp_raw, m->ple, nl, M, m->proj_norm, m->pte, m->sched,
                   1.0f / sqrtf((float)E), sqrtf((float)m->ple), 1.0f / sqrtf(2.0f), m->eps };
        LAUNCH(KC_PMP, lg_k_ipl, dim3(nl, M), dim3(64), 0, i, m->ctl);
        if (fork) {
            lx.side = false;
            hipError_t e = hipEventRecord(m->ev_join, m->stream2);
            if (e != hipSuccess && !lx.rc) lx.rc = fail(-100 - (int)e, "fork of the per-layer input branch: %s", hipGetErrorString(e));
            join_ple = true;
        }
    }
    auto join = [&]() {
        if (!join_ple) return;
        join_ple = false;
        hipError_t e = hipStreamWaitEvent(m->stream, m->ev_join, 0);
        if (e != hipSuccess && !lx.rc) lx.rc = fail(-100 - (int)e, "join of the per-layer input branch: %s", hipGetErrorString(e));
    };
    // tiles a block of layer L can touch (a sliding layer needs only its window's, not the cache's), and whether the
    // layer takes the kernel that serves all rows of a block per (tile, kv head)
    auto layer_tiles = [&](int L) { return step_tiles(m, kv, m->L[L], M, pos_off); };
    auto rows_shared = [&](int L) {
        const Layer &y = m->L[L];
        return pos_off == 0 && m->attn_rows && attention_rows_shared(M, layer_tiles(L), y.nkv, y.hd, kv->seq[y.src], 0);
    };
    for (int L = 0; L < nl && !lx.rc; ++L) {
        const Layer &y = m->L[L];
        const int window = (y.is_local && m->window > 0) ? m->window + pos_off : 0;
        bool fused_post = false, merged_o = false, ffn_rows_done = false, gate_up_done = false;
        bool mid_merge = false;                                // the merge is left to lg_k_o_geglu, with these
        MergeArgs mg{};
        int mg_tiles = 0;
        {   // q/k/v projections, then per-head norm, rotary and the K/V rows of this block
            MmArgs a{ y.wqkv, E, y.qkv_m, m->qkv, m->hq, nullptr };
            if (qkv_done) { qkv_done = rows_done = false; }
            else if (rows_done) { launch_mm<M, false>(lx, KC_QKV, a); rows_done = false; }      // (the previous layer's tail did this layer's row work)
            else if (can_fuse()) rows_mm(y.attn_norm, a, KC_QKV);
            else { rows(y.attn_norm, nullptr); launch_mm<M, false>(lx, KC_QKV, a); }
            // blocks of the model itself, up to LG_HIP_MAX_ROWS rows: the attention kernel does this part as well
            fused_post = pos_off == 0 || !y.owns;    // (a draft head's layers own no cache: queries only)
            // (so does the one for layers whose workgroups serve all rows of the block, unless more than two workgroups a CU would each
            // prepare more than 16 queries: 8 rows x 4 heads at 20011 keys 2595 -> 2580 us a step with a launch of its own, but 5 rows x
            // 2 heads at 8192 keys 3361 -> 3384)
            if (rows_shared(L) && (!m->attn_rows_fq || (M * (H / y.nkv) > 16 && attention_rows_wgs(layer_tiles(L), M * (H / y.nkv), y.nkv) * y.nkv > 2 * cu_count()))) fused_post = false;
            QkvPostArgs p{};
            p.qkv = m->qkv; p.ld = y.qkv_m; p.k_off = y.k_off; p.v_off = y.v_off;
            p.H = H; p.nkv = y.nkv; p.hd = y.hd;
            p.q_norm = y.q_norm; p.k_norm = y.k_norm; p.rope_tab = y.rope_tab; p.rope_ff = y.rope_ff;
            p.q_rot = m->q_rot;
            p.kc = y.owns ? kv->k[L] : nullptr; p.vc = y.owns ? kv->v[L] : nullptr;
            p.seq = kv->seq[y.src]; p.kv_dim = y.kd; p.eps = m->eps;
            if (!fused_post) LAUNCH(KC_QKVPOST, lg_k_qkv_post, dim3(H + (y.owns ? 2 * y.nkv : 0), M), dim3(64), 0, p, m->ctl);
        }
        {   // attention tiles + merge
            const int G = H / y.nkv;
            AttnArgs a{};
            a.q = m->q_rot; a.H = H; a.nkv = y.nkv; a.hd = y.hd;
            a.kc = kv->k[y.src]; a.vc = kv->v[y.src]; a.seq = kv->seq[y.src]; a.kv_dim = y.kd; a.window = window;
            a.pm = kv->pm; a.pl = kv->pl; a.pacc = kv->pacc; a.tiles_max = kv->tiles_max; a.pos_off = pos_off;
            const int tiles = layer_tiles(L);
            a.gx = tiles; a.gz = M;
            const bool shared = rows_shared(L);
            if (shared) {
                if constexpr (M > 1) {
                    const bool few = attention_rows_few(tiles, M * G, y.nkv, fused_post);
                    const size_t lds = few ? y.hd == 256 ? AttnFewGeo<256>::bytes(M * G, fused_post) : y.hd == 128 ? AttnFewGeo<128>::bytes(M * G, fused_post) : AttnFewGeo<64>::bytes(M * G, fused_post)
                                           : y.hd == 256 ? AttnRowsGeo<256>::bytes(M * G, fused_post) : y.hd == 128 ? AttnRowsGeo<128>::bytes(M * G, fused_post) : AttnRowsGeo<64>::bytes(M * G, fused_post);
                    const dim3 grid(few ? tiles : attention_rows_wgs(tiles, M * G, y.nkv), y.nkv);
                    a.gx = (int)grid.x;
#define ATTN_ROWS(HD, FQ) do { \
    if constexpr (FQ && 16 / M * M > LG_ATTN_FEW) if (few && M * G > LG_ATTN_FEW) { LAUNCH(KC_ATTN, (lg_k_attn_few<M, HD, FQ, 4>), grid, dim3(LG_WG), lds, m->ctl, LG_ATTN_FIELDS(LG_XA, a) 0); break; } \
    if (few) LAUNCH(KC_ATTN, (lg_k_attn_few<M, HD, FQ>), grid, dim3(LG_WG), lds, m->ctl, LG_ATTN_FIELDS(LG_XA, a) 0); \
    else     LAUNCH(KC_ATTN, (lg_k_attn_rows<M, HD, FQ>), grid, dim3(LG_WG), lds, m->ctl, LG_ATTN_FIELDS(LG_XA, a) 0); } while (0)
                    if (fused_post) {
                        a.qkv = m->qkv; a.ld = y.qkv_m; a.k_off = y.k_off; a.v_off = y.v_off;
                        a.q_norm = y.q_norm; a.k_norm = y.k_norm; a.rope_tab = y.rope_tab; a.rope_ff = y.rope_ff;
                        a.kcw = y.owns ? kv->k[L] : nullptr; a.vcw = y.owns ? kv->v[L] : nullptr; a.eps = m->eps;
                        if (y.hd == 256)      ATTN_ROWS(256, true);
                        else if (y.hd == 128) ATTN_ROWS(128, true);
                        else                  ATTN_ROWS(64, true);
                    } else
                    if (y.hd == 256)      ATTN_ROWS(256, false);
                    else if (y.hd == 128) ATTN_ROWS(128, false);
                    else                  ATTN_ROWS(64, false);
#undef ATTN_ROWS
                }
            } else
            if (fused_post) {
                a.qkv = m->qkv; a.ld = y.qkv_m; a.k_off = y.k_off; a.v_off = y.v_off;
                a.q_norm = y.q_norm; a.k_norm = y.k_norm; a.rope_tab = y.rope_tab; a.rope_ff = y.rope_ff;
                a.kcw = y.owns ? kv->k[L] : nullptr; a.vcw = y.owns ? kv->v[L] : nullptr; a.eps = m->eps;
                if (y.hd <= 256) LAUNCH(KC_ATTN, (lg_k_attn<true, 1>), dim3(tiles, y.nkv, M), dim3(LG_WG), attn_lds(G, y.hd, true), m->ctl, LG_ATTN_FIELDS(LG_XA, a) 0);
                else             LAUNCH(KC_ATTN, (lg_k_attn<true, 2>), dim3(tiles, y.nkv, M), dim3(LG_WG), attn_lds(G, y.hd, true), m->ctl, LG_ATTN_FIELDS(LG_XA, a) 0);
            } else {
                LAUNCH(KC_ATTN, (lg_k_attn<false, 1>), dim3(tiles, y.nkv, M), dim3(LG_WG), attn_lds(G, y.hd, false), m->ctl, LG_ATTN_FIELDS(LG_XA, a) 0);
            }
            MergeArgs g{ kv->pm, kv->pl, kv->pacc, kv->tiles_max, H, y.hd, window, pos_off, m->aq, nullptr };
            if constexpr (M == 1) if (narrow && (L + 1 < nl || with_head)) {
                const bool last = L + 1 == nl;
                NarrowArgs f{};
                f.g = g; f.x = m->x[cur]; f.x_out = m->x[cur ^ 1];
                f.wo = y.wo; f.wgu = y.wgu; f.wdn = y.wdown; f.winp = y.winp; f.wproj = y.wproj; f.wq = last ? nullptr : m->L[L + 1].wqkv;
                f.post_attn = y.post_attn; f.ffn_norm = y.ffn_norm; f.post_ffw = y.post_ffw; f.post_norm = y.post_norm; f.os = y.out_scale;
                f.w_pre = last ? m->output_norm : m->L[L + 1].attn_norm;
                f.ipl = m->ple ? m->pmp_raw + (size_t)L * m->ple : nullptr;
                f.qkv = m->qkv; f.h_out = last ? m->hidden_rows : nullptr; f.hq = m->hq;
                f.E = E; f.qd = y.qd; f.FF = y.nff; f.qm = last ? 0 : m->L[L + 1].qkv_m; f.tiles = tiles; f.eps = m->eps;
                f.sync = m->nsync; f.seq = L; f.err = &m->ctl->err; f.err2 = draft ? &m->target->ctl->err : nullptr; f.spin_limit = m->wait_polls;
                const dim3 grid(LG_XCDS * LG_NARROW_WGS);
                if (tiles > LG_NARROW_LONG) {
                    if (m->ple) LAUNCH(KC_TAIL, (lg_k_narrow<true, true>), grid, dim3(512), 0, f, m->ctl);
                    else        LAUNCH(KC_TAIL, (lg_k_narrow<false, true>), grid, dim3(512), 0, f, m->ctl);
                } else if (m->ple) LAUNCH(KC_TAIL, (lg_k_narrow<true, false>), grid, dim3(512), 0, f, m->ctl);
                else               LAUNCH(KC_TAIL, (lg_k_narrow<false, false>), grid, dim3(512), 0, f, m->ctl);
                cur ^= 1;
                rows_done = true; qkv_done = !last;
                continue;
            }
            merged_o = pos_off == 0 && use_merge_o(m, y, M, tiles);
            if (pos_off == 0 && have_x && use_attn_tail(m, y, M, tiles)) {
                // merge, output projection and the row work ahead of gate/up as one launch on one XCD
                XattnTailArgs f{};
                f.g = g; f.wo = y.wo_ch; f.aq = (uint32_t *)m->aq; f.pout = m->dout;
                f.x = m->x[cur]; f.w_post = y.post_attn; f.w_pre = y.ffn_norm; f.x_out = m->x[cur ^ 1];
                f.q = m->hq; f.q_units = (M >= 4) ? 2 : 1; f.E = E; f.eps = m->eps;
                f.sync = m->tsync; f.seq = L; f.spin_limit = m->wait_polls; f.stamps = m->tail_stamps ? m->tstamps + LG_XTAIL_UNITS * 8 : nullptr;
                launch_attn_tail<M>(lx, f);
                cur ^= 1;
                pend_dout = pend_w = pend_os = nullptr; pend_parts = 1;
                merged_o = true; ffn_rows_done = true;
            } else
            if (!merged_o && pos_off == 0 && have_x && use_attn_out(m, y, M, tiles)) {
                const bool chains = attn_out_chains(y, M, tiles);
                AttnOutArgs f{};
                f.g = g; f.wo = chains ? y.wo_ch : y.wo; f.x = m->x[cur]; f.w_post = y.post_attn; f.w_pre = y.ffn_norm; f.x_out = m->x[cur ^ 1];
                f.q = m->hq; f.E = E; f.tiles = tiles; f.eps = m->eps; f.sync = m->aosync; f.seq = L; f.spin_limit = m->wait_polls;
                f.stamps = m->tail_stamps ? m->tstamps + LG_XTAIL_UNITS * 8 : nullptr;
                if (attn_out_geglu(m, y, M, tiles)) {
                    f.gw = y.wgu; f.nff = y.nff; f.gq = m->gq; f.gq_units = M >= 4 && m->down_m && y.wdn_m ? 2 : 0; f.rows = m->aorows;
                    gate_up_done = true;
                }
                size_t lds = chains ? LG_AOUT_M_LDS : (size_t)M * LG_AOUT_K * 5 / 4;
                if (gate_up_done) lds = std::max(lds, LG_AOUT_GU_LDS);
                if constexpr (M >= LG_AOUT_DOT_ROWS)
                    if (chains) LAUNCH(KC_ATAIL, lg_k_attn_out_m<M>, dim3(LG_XCDS * LG_XCD_WGS), dim3(768), lds, m->ctl, LG_AOUT_FIELDS(LG_XA, f) 0);
                if constexpr (M <= LG_AOUT_DOT_ROWS)
                    if (!chains) LAUNCH(KC_ATAIL, lg_k_attn_out<M>, dim3(LG_XCDS * LG_XCD_WGS), dim3(64 * (LG_AOUT_G + M)), lds, m->ctl, LG_AOUT_FIELDS(LG_XA, f) 0);
                cur ^= 1;
                merged_o = true; ffn_rows_done = true;
            } else
            if (merged_o) {
                // the merge of (head, row) runs that head's chain of the output projection itself: eight slabs for the row kernel
                MergeOArgs f{ g, y.wo_rb, m->dout, E, merge_o_slices(m, M), M };
                launch_merge_o(lx, f);
                pend_dout = m->dout; pend_w = y.post_attn; pend_os = nullptr; pend_parts = 8;
            } else
            if ((mid_merge = pos_off == 0 && have_x && use_mid_merge(m, y, M, tiles))) {
                mg = g;
                mg_tiles = tiles;
            } else
            if (tiles >= 128 && y.hd % 64 == 0) {
#define GO(k, grid, block) LAUNCH(KC_MERGE, k, grid, block, 0, m->ctl, LG_MERGE_FIELDS(LG_XA, g) 0)
                MERGE_SPLIT(M, GO, H, y.hd, tiles);
#undef GO
            } else LAUNCH(KC_MERGE, (lg_k_attn_merge<M>), dim3(H, M), dim3(LG_WG), 0, m->ctl, LG_MERGE_FIELDS(LG_XA, g) 0);
        }
        if (!merged_o && pos_off == 0 && have_x && use_mid_o(m, y, M)) {
            OGegluArgs f{};
            f.ow = y.wo_pc; f.act = m->aq; f.out = m->mido; f.gw = y.wgu; f.gq = m->gq; f.qd = y.qd; f.nff = y.nff;
            f.gq_units = M >= 4 && m->down_m && y.wdn_m ? 2 : 0; f.seq = L;
            f.r = MidRowArgs{ m->x[cur], y.post_attn, nullptr, y.ffn_norm, m->x[cur ^ 1], nullptr, m->midro, E, m->wait_polls, m->eps };
            f.g = mg; f.tiles = mg_tiles; f.arows = m->midao;
            if constexpr (M <= LG_MID_MERGE_ROWS)
                if (mid_merge) LAUNCH(KC_O, (lg_k_o_geglu<M, 15, true>), dim3(LG_XCDS * LG_XCD_WGS), dim3(512), LG_OG_LDS(15), m->ctl, LG_OGEGLU_FIELDS(LG_XA, f) 0);
            if (E <= 2560)       LAUNCH(KC_O, (lg_k_o_geglu<M, 10, false>), dim3(LG_XCDS * LG_XCD_WGS), dim3(512), LG_OG_LDS(10), m->ctl, LG_OGEGLU_FIELDS(LG_XA, f) 0);
            else if (!mid_merge) LAUNCH(KC_O, (lg_k_o_geglu<M, 15, false>), dim3(LG_XCDS * LG_XCD_WGS), dim3(512), LG_OG_LDS(15), m->ctl, LG_OGEGLU_FIELDS(LG_XA, f) 0);
            cur ^= 1;
            merged_o = true; ffn_rows_done = true; gate_up_done = true;
        }
        if (!merged_o) {   // attention output projection
            MmArgs a{ y.wo, y.qd, E, m->dout, m->aq, nullptr };
            pend_parts = launch_mm<M, false>(lx, KC_O, a);
            pend_dout = m->dout; pend_w = y.post_attn; pend_os = nullptr;
        }
        {   // feed-forward: gate/up + GeGLU, then down
            // verify blocks: 1..3 rows through v_dot4 with scalar operands, 4..8 rows through the matrix cores
            // (its float work per tile does not grow with the row count); each has its own activation order
            constexpr bool mfma = M >= 4;
            if (mfma && m->xffn_built && m->xcd_ffn && may_wait(m) && y.xgu && have_x && pend_dout && pend_parts == 1 && !pend_os) {
                // the whole half as one launch partitioned by XCD: row work, gate/up + GeGLU and the XCD's K share of
                // ffn_down; the consumer adds the 8 slabs (the top of the segment tree)
                XffnArgs f{ y.xgu, y.xdn, m->x[cur], pend_dout, pend_w, y.ffn_norm, m->x[cur ^ 1], m->slabs, m->xq8, m->xact,
                            m->xsync, m->ctl, E, y.nff, m->eps, 4 * m->wait_polls, L, m->xffn_delay, nullptr };
                launch_xffn<M>(lx, f, m->xffn_cls);
                cur ^= 1;
                pend_dout = m->slabs; pend_parts = LG_XCDS; pend_w = y.post_ffw; pend_os = m->ple ? nullptr : y.out_scale;
            } else {
            const bool dn_m = mfma && m->down_m && y.wdn_m;       // ffn_down on the matrix cores: the activations as 80-dword blocks
            GegluArgs a{ y.wgu, E, y.nff, m->hq, m->gq, dn_m ? 2 : 0 };
            bool rows_in_geglu = false;
            if constexpr (mfma) {
                // the row work as the first workgroups of the gate/up launch, whose other workgroups request their weights
                // while it runs (lg_xrg.h); shapes whose K segment of E/256 tiles has a build
                const int slices = (E + 1023) / 1024;
                if (m->rows_geglu && m->rgsync && may_wait(m) && !ffn_rows_done && have_x && pend_dout && !pend_os && (pend_parts == 1 || pend_parts == 4) && (E == 2560 || E == 3840 || E == 512) &&
                    M * slices <= LG_RG_MAXP) {
                    RowsGegluArgs f{ m->x[cur], pend_dout, pend_w, y.ffn_norm, m->x[cur ^ 1], m->hq, E, pend_parts, slices, m->eps,
                                     y.wgu, y.nff, m->gq, dn_m ? 2 : 0, m->rgsync, L, m->wait_polls, m->tail_stamps ? m->tstamps + LG_XTAIL_UNITS * 8 : nullptr };
                    const dim3 grid(M * slices + y.nff / 32);
                    const size_t lds = (size_t)(E / 32) * LG_MU_DWORDS * 4;
                    if (E == 512)  LAUNCH(KC_GATEUP, (lg_k_rows_geglu<M, 2>), grid, dim3(512), lds, m->ctl, LG_RG_FIELDS(LG_XA, f) 0);
                    else if (E == 2560) LAUNCH(KC_GATEUP, (lg_k_rows_geglu<M, 10>), grid, dim3(512), lds, m->ctl, LG_RG_FIELDS(LG_XA, f) 0);
                    else           LAUNCH(KC_GATEUP, (lg_k_rows_geglu<M, 15>), grid, dim3(512), lds, m->ctl, LG_RG_FIELDS(LG_XA, f) 0);
                    cur ^= 1;
                    pend_dout = pend_w = pend_os = nullptr; pend_parts = 1;
                    rows_in_geglu = true;
                }
            }
            if (rows_in_geglu || gate_up_done) {
            } else {
            if (!ffn_rows_done) rows(y.ffn_norm, nullptr, mfma ? 2 : 1);
            if constexpr (mfma)
                LAUNCH(KC_GATEUP, (lg_k_geglu_m<M>), dim3(y.nff / 32), dim3(512), (size_t)(E / 32) * LG_MU_DWORDS * 4, LG_GEGLU_FIELDS(LG_XA, a) 0);
            else
                LAUNCH(KC_GATEUP, (lg_k_geglu_t<M>), dim3(y.nff / 32), dim3(512), 0, LG_GEGLU_FIELDS(LG_XA, a) 0);
            }
            MmArgs d{ y.wdown, y.nff, E, m->dout, m->gq, nullptr };
            if (pos_off == 0 && have_x && L + 1 < nl && use_mid_down(m, y, m->L[L + 1], M)) {
                DownQkvArgs f{};
                f.d = DownHere{ M >= 4 ? y.wdn_m : y.wdown, m->gq, y.nff, E, m->mids, m->midd, m->wait_polls };
                f.r = MidRowArgs{ m->x[cur], y.post_ffw, y.out_scale, m->L[L + 1].attn_norm, m->x[cur ^ 1], nullptr, m->midrd, E, m->wait_polls, m->eps };
                f.qw = m->L[L + 1].wqkv_pc; f.qout = m->qkv; f.qm = m->L[L + 1].qkv_m; f.seq = L;
                LAUNCH(KC_ROWS, (lg_k_down_qkv<M, false>), dim3(LG_XCDS * LG_XCD_WGS), dim3(512), lg_downqkv_lds(M, y.nff), m->ctl, LG_DOWNQKV_FIELDS(LG_XA, f) 0);
                cur ^= 1;
                rows_done = qkv_done = true;
                continue;
            }
            if (dn_m) {
                DownMArgs dm{ y.wdn_m, (const uint32_t *)m->gq, m->dout, E, y.nff, m->down_m == 1 && may_wait(m) ? m->dmsync : nullptr, m->ctl, m->wait_polls, L };
                launch_down_m<M>(lx, dm);
                pend_parts = dm.sync ? 1 : 4;
            } else
            // (the rows kernel adds four slabs; the fused rows + PLE gate kernel of verify blocks takes whole sums)
            pend_parts = launch_mm<M, false>(lx, KC_DOWN, d, !m->ple && m->down_kq);
            pend_dout = m->dout; pend_w = y.post_ffw; pend_os = m->ple ? nullptr : y.out_scale;
            }
        }
        if (m->ple) join();
        if (m->ple && y.winp_f) {   // per-layer embedding block, matrices kept in a float type: residual update, then the
            // gate on the f32 rows (gelu(.) * ipl in its epilogue), then the projection of the f32 gate rows
            if (have_x && pend_dout && !pend_os && (pend_parts == 1 || pend_parts == 4)) {
                RowsMmfArgs f{ m->x[cur], pend_dout, pend_w, pend_parts, m->x[cur ^ 1], m->eps, y.winp_f, E, m->ple, m->pmp_raw + (size_t)L * m->ple, m->ple * nl, m->pgf };
                LAUNCH(KC_PLEGATE, lg_k_rows_mmf<M>, dim3(m->ple, (M + LG_RMMF_ROWS - 1) / LG_RMMF_ROWS), dim3(LG_WG), (size_t)(M < LG_RMMF_ROWS ? M : LG_RMMF_ROWS) * E * 4, f);
                cur ^= 1;
                pend_dout = pend_w = pend_os = nullptr; pend_parts = 1;
            } else {
            rows(nullptr, nullptr);
            MmfArgs g{ y.winp_f, E, m->ple, m->x[cur], E, M, m->pgf, m->ple, m->pmp_raw + (size_t)L * m->ple, m->ple * nl };
            launch_mmf<M>(lx, KC_PLEGATE, g);
            }
            if (pos_off == 0 && L + 1 < nl && use_mid_proj(m, m->L[L + 1], M)) {      // the projection, the row work behind it and the next layer's projections
                DownQkvArgs f{};
                f.d = DownHere{ (const uint8_t *)y.wproj_f, m->pgf, 0, E, nullptr, m->midd, m->wait_polls };
                f.r = MidRowArgs{ m->x[cur], y.post_norm, y.out_scale, m->L[L + 1].attn_norm, m->x[cur ^ 1], nullptr, m->midrd, E, m->wait_polls, m->eps };
                f.qw = m->L[L + 1].wqkv_pc; f.qout = m->qkv; f.qm = m->L[L + 1].qkv_m; f.seq = L;
                LAUNCH(KC_ROWS, (lg_k_down_qkv<M, true>), dim3(LG_XCDS * LG_XCD_WGS), dim3(512), LG_DOWNQKV_ACT, m->ctl, LG_DOWNQKV_FIELDS(LG_XA, f) 0);
                cur ^= 1;
                rows_done = qkv_done = true;
                continue;
            }
            MmfArgs p{ y.wproj_f, m->ple, E, m->pgf, m->ple, M, m->dout, E, nullptr, 0 };
            launch_mmf<M>(lx, KC_PLEPROJ, p);
            pend_dout = m->dout; pend_w = y.post_norm; pend_os = y.out_scale;
        } else
        if (m->ple) {   // per-layer embedding block
            PleGateArgs a{ y.winp, E, m->ple, m->hq, m->pmp_raw, L, nl, m->pq };
            const bool last = L + 1 == nl, joins = !last && tail_does_qkv(m, M, m->L[L + 1]);
            if (use_ple_tail(m, M, joins) && (!last || with_head) && pend_dout && have_x && !pend_os) {
                // the whole block and the row work that follows it (the next layer's, or the head's) in one launch on one XCD
                const bool head_m = M >= 4 && m->emb_rb && m->head_mfma;
                XtailArgs f{};
                f.r = RowsPleGateArgs{ a, m->x[cur], pend_dout, pend_w, nullptr, m->eps, pend_parts };
                f.pw = y.wproj; f.pout = m->tpr; f.w_post2 = y.post_norm; f.os = y.out_scale;
                f.w_pre = last ? m->output_norm : m->L[L + 1].attn_norm;
                f.x_out = m->x[cur ^ 1]; f.h_out = last ? m->hidden_rows : nullptr;
                f.q = m->hq; f.q_units = last && head_m ? 2 : 0;
                f.seq = L; f.spin_limit = m->wait_polls; f.stamps = m->tail_stamps ? m->tstamps : nullptr;
                f.gf = m->tgf; f.rows = m->trows;
                if (joins) {
                    f.qw = M >= LG_TAIL_MFMA ? m->L[L + 1].wqkv_ch : m->L[L + 1].wqkv; f.qm = m->L[L + 1].qkv_m; f.qout = m->qkv;
                    qkv_done = true;
                }
                launch_ple_tail<M>(lx, f);
                cur ^= 1;
                pend_dout = pend_w = pend_os = nullptr; pend_parts = 1;
                rows_done = true;
                continue;
            } else {
                // the residual update after ffn_down and its q8 happen inside the gate kernel (no rows kernel here)
                RowsPleGateArgs r{ a, m->x[cur], pend_dout, pend_w, m->x[cur ^ 1], m->eps, pend_parts };
                LAUNCH(KC_PLEGATE, (lg_k_rows_plegate<M>), dim3(m->ple / 32, M), dim3(LG_WG), lds_mm(1, E), LG_RPG_FIELDS(LG_XA, r) 0);
                cur ^= 1;
                pend_dout = pend_w = pend_os = nullptr; pend_parts = 1;
            }
            MmArgs p{ y.wproj, m->ple, E, m->dout, m->pq, nullptr };
            launch_mm<M, false>(lx, KC_PLEPROJ, p);
            pend_dout = m->dout; pend_w = y.post_norm; pend_os = y.out_scale;
        }
    }
    join();
    if (with_head && !lx.rc) {
        const bool head_m = M >= 4 && m->emb_rb && m->head_mfma;
        if (!rows_done) rows(m->output_norm, m->hidden_rows, head_m ? 2 : 0);
        int grid = 512;                                  // two workgroups per CU, each walks `passes` blocks of 64 rows
        int passes = (m->n_vocab / 64 + grid - 1) / grid;
        if (passes < 1) passes = 1;
        grid = (m->n_vocab / 64 + passes - 1) / passes;
        HeadArgs h{ head_m ? m->emb_rb : m->emb, E, m->n_vocab, passes, m->hq, m->softcap, m->store_logits ? m->logits : nullptr, m->pval, m->pidx };
        if (head_m) {
            if constexpr (M >= 4)
                LAUNCH(KC_HEAD, (lg_k_head_m<M>), dim3(grid), dim3(512), (size_t)(E / 32) * LG_MU_DWORDS * 4, LG_HEAD_FIELDS(LG_XA, h) 0);
        } else
        LAUNCH(KC_HEAD, (lg_k_mm_head<M>), dim3(grid), dim3(LG_WG), lds_mm(M, E), LG_HEAD_FIELDS(LG_XA, h) 0);
        AcceptArgs c{ m->pval, m->pidx, grid, m->sched, m->out, m->adv, m->hidden_rows, m->g_hidden, E, m->pin + 32 };
        LAUNCH(KC_ACCEPT, (lg_k_accept<M>), dim3(1), dim3(LG_WG), 0, m->ctl, LG_ACCEPT_FIELDS(LG_XA, c) 0);
    } else if (!lx.rc && !dry) {
        hipLaunchKernelGGL(lg_k_advance, dim3(1), dim3(1), 0, m->stream, m->ctl, M, m->pin + 32);
    }
    return lx.rc;
}

// ---- prompt blocks ------------------------------------------------------------------------------
// A matmul of a prompt block (lg_wide.h).  The workgroup's shape: 64 weight rows x 64 activation rows by four wavefronts
// of two K segments each; 32 activation rows when the block has no more; and where 64 x 32 tiles would leave some CU
// without a workgroup, eight wavefronts of one segment on such a tile (3072 x 2560, 32 rows, 48 workgroups: 8.8 -> 7.1 us).
// `slabs`: the consumer adds four slabs, so that a matrix of 8 segments may be cut by K quarter too: workgroups of two wavefronts,
// where a quarter of the CUs would do for whole rows (a CU pulls 48 GB/s: 22 rows, 3072 x 2560 on 48 CUs 9.1 us, on 192 6.2).
// 256: the compute units of a whole device, as a constant because the per-layer gate is built for the shape that it gives.
struct WideShape { int tb, wv, parts; };
static WideShape wide_shape(int k, int m, int rows, bool slabs) {
    const int parts = lg_segments(k) / 8, tiles = ((m + LG_WT - 1) / LG_WT) * ((rows + 31) / 32);
    if (slabs && parts == 1 && tiles * 4 <= 256 && 4 * rows <= LG_WIDE_ROWS) return { 1, 2, 4 };      // (the slabs lie in a buffer of LG_WIDE_ROWS rows)
    if (tiles * parts <= 256) return { 1, 8, parts };
    return { rows <= 32 ? 1 : 2, 4, parts };
}
struct WideLaunch { WideMm a; WideShape c; dim3 grid, block; size_t lds; };
static WideLaunch wide_launch(const uint8_t *w, const int8_t *q, int k, int m, int rows, bool slabs = false) {
    const WideShape c = wide_shape(k, m, rows, slabs);
    const int parts = c.parts;
    const WideMm a{ w, (const uint8_t *)q, k, m, rows, (rows + 32 * c.tb - 1) / (32 * c.tb), parts };
    return { a, c, dim3(lg_wide_grid(m, a.nb_tiles, parts)), dim3(64 * c.wv), (size_t)c.wv * 2 * c.tb * 4096 };
}
// k18, k14, k24: the kernel's builds for 32 activation rows by eight and by four wavefronts and for 64 by four
#define LAUNCH_WIDE(cls, l, k18, k14, k24, ...) do { if (l.c.wv == 8) LAUNCH(cls, k18, l.grid, l.block, l.lds, l.a, __VA_ARGS__); \
    else if (l.c.tb == 1) LAUNCH(cls, k14, l.grid, l.block, l.lds, l.a, __VA_ARGS__); \
    else LAUNCH(cls, k24, l.grid, l.block, l.lds, l.a, __VA_ARGS__); } while (0)
template <bool DUMP>
static int launch_wide_mm(Launcher &lx, int cls, const uint8_t *w, const int8_t *q, int k, int m, int rows, float *out, int32_t *dots, bool slabs = false) {
    const WideLaunch l = wide_launch(w, q, k, m, rows, slabs);
    if (l.c.wv == 2) LAUNCH(cls, (lg_k_wide_mm<1, 2, DUMP>), l.grid, l.block, l.lds, l.a, out, dots);
    else LAUNCH_WIDE(cls, l, (lg_k_wide_mm<1, 8, DUMP>), (lg_k_wide_mm<1, 4, DUMP>), (lg_k_wide_mm<2, 4, DUMP>), out, dots);
    return l.a.parts;
}
// Whether a prompt block reaches value rows 2 GiB and more behind a layer's first one (524288 positions at the 12B shape), where
// lg_k_wide_attn's 32-bit addresses end.  (It fetches value rows four tiles at a time.)
static bool far_block(const lg_hip_kv *kv, const Layer &y, int rows, int pos) {
    const long long reach = (long long)pos + rows + 127;
    return (size_t)(reach < kv->seq[y.src] ? reach : kv->seq[y.src]) * y.kd * 2 >= (size_t)1 << 31;
}
// Such a block runs as verify blocks when it has heads of up to 256 there: their attention serves a tile to all rows (96 rows at
// 524288 positions, 16 heads of 256 over 8: 34 ms against 104; 512-wide heads have no such kernel: 376 against 142, 16 over 2).
static bool far_in_narrow_heads(const lg_hip_model *m, const lg_hip_kv *kv, int rows, int pos) {
    for (const Layer &y : m->L) if (y.hd < 512 && far_block(kv, y, rows, pos)) return true;
    return false;
}
// Up to LG_WA_SPLIT_GROUPS workgroups (half of the chip) with 12 tiles and more: scores and values as two launches over more workgroups (200
// rows, 100 workgroups: 41 -> 39 us in a 512-wide window, 175 -> 113 us over 100 tiles; with 130 workgroups 42 -> 55 us, with 8
// tiles 23 us both ways).  Where the weights wait in memory anyway, also wherever the last round of workgroups would leave a fifth of
// the CU time unused (332 rows at 3001, 166 workgroups: a prompt's 11.68 -> 11.55 ms; 300 rows at 3001, 304 workgroups: 22.18 -> 21.41 ms; with 256 or 512
// of them 0.5% slower).  Score workgroups take 4 tiles, or up to 16 while there are more than 512 of them.
// `far`: the block reaches value rows 2 GiB and more behind a layer's first one and takes 64-bit addresses (96 rows, 16 heads of 512
// over 2, a million positions: 140.9 -> 141.7 ms).  Built for heads of 512; narrower ones go to verify blocks there (far_in_narrow_heads).
template <int HD>
static void launch_wide_attn(Launcher &lx, const WideAttn &a, int groups, bool far, size_t scratch_bytes) {
    const dim3 grid(groups, a.nkv);
    const int wgs = groups * a.nkv;
    if constexpr (HD == 512)
        if (far) { LAUNCH(KC_ATTN, (lg_k_wide_attn<HD, false, 0, true>), grid, dim3(LG_WA_WG), 0, a, lx.m->ctl); return; }
    const int round = cu_count(), rounds = (wgs + round - 1) / round;       // one such workgroup of eight wavefronts to a CU
    const bool split = wgs <= LG_WA_SPLIT_GROUPS || (a.tiles > LG_WA_TILES && 5 * wgs < 4 * rounds * round);
    if (split && a.tiles >= 12 && a.tiles <= LG_WA_SPLIT_MAX && (size_t)wgs * a.tiles * (16 * 34 * 4) <= scratch_bytes) {
        int chunk = 4;
        while (chunk < 16 && wgs * (a.tiles / chunk) > 512) chunk *= 2;
        LAUNCH(KC_ATTN, (lg_k_wide_attn<HD, false, 1>), dim3(groups, a.nkv, (a.tiles + chunk - 1) / chunk), dim3(LG_WA_SPLIT_WG), 0, a, lx.m->ctl);
        LAUNCH(KC_ATTN, (lg_k_wide_attn<HD, false, 2>), dim3(groups, a.nkv, HD > 128 ? HD / 128 : 1), dim3(LG_WA_SPLIT_WG), (size_t)a.tiles * 64, a, lx.m->ctl);
    } else if (a.tiles <= LG_WA_TILES) LAUNCH(KC_ATTN, (lg_k_wide_attn<HD, true>), grid, dim3(LG_WA_WG), lg_wide_attn_lds(a.tiles), a, lx.m->ctl);
    else                               LAUNCH(KC_ATTN, (lg_k_wide_attn<HD, false>), grid, dim3(LG_WA_WG), 0, a, lx.m->ctl);
}

// Rows of a prompt block up to which a row's work is cut over its slices, and up to which the per-layer gate does the row work ahead of it.
// Prompts of 33 to 256 tokens with either always and never (never -> always, us): slices, E4B shape, 32 rows 5394 -> 5334, 64 5970 -> 5902,
// 79 6590 -> 6548, 96 6637 -> 6589, 111 6737 -> 6775, 127 6779 -> 6841, 255 8544 -> 8716; 12B shape, 32 rows 6780 -> 6668, 96 8972 -> 8906,
// 111 9040 -> 9076, 127 9110 -> 9183.  Gate, 32 rows 5570 -> 5343, 64 6045 -> 5916, 96 6724 -> 6657, 111 6746 -> 6800, 255 8558 -> 9011.
#define WIDE_SLICE_ROWS 96
#define WIDE_GATE_ROWS 96
// One block of `rows` prompt positions from pos on (tokens in device memory): the launch sequence of a verify step with
// the kernels of lg_wide.h.  Launched as it is, not captured: a prompt's blocks differ in width and tile counts, and the
// host stays ahead of launches of this size.
static int enqueue_prompt(lg_hip_model *m, lg_hip_kv *kv, const int32_t *toks, int rows, int pos, bool first) {
    Launcher lx{ m, false };
    const int E = m->E, H = m->H, nl = m->n_layer;
    int cur = 0;
    bool have_x = false;
    const float *pend_dout = nullptr, *pend_w = nullptr, *pend_os = nullptr;
    int pend_parts = 1;
    hipLaunchKernelGGL(lg_k_set_ctl, dim3(1), dim3(1), 0, m->stream, m->ctl, pos, first);
    auto row_work = [&](const float *w_pre, int8_t *q) {
        RowArgs s{};
        s.E = E; s.eps = m->eps; s.toks = toks; s.q = q;
        if (!have_x) { s.emb = m->emb; s.emb_seg = lg_segments(E); s.emb_nit = E / 32 / s.emb_seg; s.emb_scale = sqrtf((float)E); }
        else s.x = m->x[cur];
        s.dout = pend_dout; s.w_post = pend_w; s.os = pend_os; s.dparts = pend_parts;
        s.w_pre = w_pre;
        if (pend_dout || !have_x) s.x_out = m->x[cur ^ 1];
        s.slices = rows <= WIDE_SLICE_ROWS ? (E + 1023) / 1024 : 1;
        LAUNCH(KC_ROWS, lg_k_wide_rows, dim3(rows, s.slices), dim3(LG_WG), 0, s, rows);
        if (s.x_out) cur ^= 1;
        have_x = true; pend_dout = pend_w = pend_os = nullptr; pend_parts = 1;
    };
    if (m->ple) {
        row_work(nullptr, m->eq);
        if (m->pmp_f) {
            MmfArgs f{ m->pmp_f, E, m->ple * nl, m->x[cur], E, rows, m->pmp_raw, m->ple * nl, nullptr, 0 };
            launch_mmf<LG_HIP_MAX_ROWS>(lx, KC_PMP, f);
        } else launch_wide_mm<false>(lx, KC_PMP, m->pmp_w, m->eq, E, m->ple * nl, rows, m->pmp_raw, nullptr);
        IplArgs i{ m->pmp_raw, m->ple, nl, rows, m->proj_norm, m->pte, toks,
                   1.0f / sqrtf((float)E), sqrtf((float)m->ple), 1.0f / sqrtf(2.0f), m->eps };
        LAUNCH(KC_PMP, lg_k_ipl, dim3(nl, rows), dim3(64), 0, i, m->ctl);
    }
    for (int L = 0; L < nl && !lx.rc; ++L) {
        const Layer &y = m->L[L];
        const int window = (y.is_local && m->window > 0) ? m->window : 0;
        row_work(y.attn_norm, m->hq);
        QkvPostArgs p{};
        p.parts = launch_wide_mm<false>(lx, KC_QKV, y.wqkv_w, m->hq, E, y.qkv_m, rows, m->qkv, nullptr, true);
        p.slab = (size_t)rows * y.qkv_m;
        p.qkv = m->qkv; p.ld = y.qkv_m; p.k_off = y.k_off; p.v_off = y.v_off;
        p.H = H; p.nkv = y.nkv; p.hd = y.hd;
        p.q_norm = y.q_norm; p.k_norm = y.k_norm; p.rope_tab = y.rope_tab; p.rope_ff = y.rope_ff;
        p.q_rot = m->q_rot;
        p.kc = y.owns ? kv->k[L] : nullptr; p.vc = y.owns ? kv->v[L] : nullptr;
        p.seq = kv->seq[y.src]; p.kv_dim = y.kd; p.eps = m->eps;
        LAUNCH(KC_QKVPOST, lg_k_qkv_post, dim3(H + (y.owns ? 2 * y.nkv : 0), rows), dim3(64), 0, p, m->ctl);
        const int rg = lg_wide_attn_rows(H / y.nkv), groups = (rows + rg - 1) / rg;
        const WideAttn a{ m->q_rot, kv->k[y.src], kv->v[y.src], H, y.nkv, kv->seq[y.src], y.kd, window, rows, kv->pacc,
                          wide_attn_tiles(m, y, rows, pos), (uint8_t *)m->aq };
        const bool far = far_block(kv, y, rows, pos);
        switch (y.hd) {
            case 512: launch_wide_attn<512>(lx, a, groups, far, kv->scratch_bytes); break;
            case 256: launch_wide_attn<256>(lx, a, groups, far, kv->scratch_bytes); break;
            case 128: launch_wide_attn<128>(lx, a, groups, far, kv->scratch_bytes); break;
            default:  launch_wide_attn<64>(lx, a, groups, far, kv->scratch_bytes);
        }
        pend_parts = launch_wide_mm<false>(lx, KC_O, y.wo_w, m->aq, y.qd, E, rows, m->dout, nullptr, true);
        pend_dout = m->dout; pend_w = y.post_attn;
        row_work(y.ffn_norm, m->hq);
        const WideLaunch gu = wide_launch(y.wgu_w, m->hq, E, 2 * y.nff, rows);
        LAUNCH_WIDE(KC_GATEUP, gu, (lg_k_wide_geglu<1, 8>), (lg_k_wide_geglu<1, 4>), (lg_k_wide_geglu<2, 4>), (uint8_t *)m->gq);
        pend_parts = launch_wide_mm<false>(lx, KC_DOWN, y.wdown_w, m->gq, y.nff, E, rows, m->dout, nullptr);
        pend_dout = m->dout; pend_w = y.post_ffw; pend_os = m->ple ? nullptr : y.out_scale;
        if (!m->ple) continue;
        const bool rows_in_gate = !y.winp_f && rows <= WIDE_GATE_ROWS;
        if (!rows_in_gate) row_work(nullptr, y.winp_f ? nullptr : m->hq);
        if (y.winp_f) {
            MmfArgs g{ y.winp_f, E, m->ple, m->x[cur], E, rows, m->pgf, m->ple, m->pmp_raw + (size_t)L * m->ple, m->ple * nl };
            launch_mmf<LG_HIP_MAX_ROWS>(lx, KC_PLEGATE, g);
            MmfArgs pr{ y.wproj_f, m->ple, E, m->pgf, m->ple, rows, m->dout, E, nullptr, 0 };
            launch_mmf<LG_HIP_MAX_ROWS>(lx, KC_PLEPROJ, pr);
            pend_parts = 1;
        } else {
            // (256 gate rows: at most 4 weight tiles x 16 activation tiles, always eight wavefronts)
            static_assert((256 / LG_WT) * (LG_WIDE_ROWS / 32) <= 256, "lg_k_wide_plegate is built for tiles of 64 x 32 by eight wavefronts");
            if (rows_in_gate) {
                RowsPleGateArgs r{ PleGateArgs{ y.winp, E, m->ple, nullptr, m->pmp_raw, L, nl, m->pq }, m->x[cur], pend_dout, pend_w, m->x[cur ^ 1], m->eps, pend_parts };
                LAUNCH(KC_PLEGATE, lg_k_wide_rows_plegate, dim3(m->ple / 32, rows), dim3(LG_WG), (size_t)E * 5 / 4, r, rows);
                cur ^= 1;
                pend_os = nullptr;
            } else {
                const WideLaunch g = wide_launch(y.winp_w, m->hq, E, m->ple, rows);
                LAUNCH(KC_PLEGATE, (lg_k_wide_plegate<1, 8>), g.grid, g.block, g.lds, g.a, m->pmp_raw, L, nl, (uint8_t *)m->pq);
            }
            pend_parts = launch_wide_mm<false>(lx, KC_PLEPROJ, y.wproj_w, m->pq, m->ple, E, rows, m->dout, nullptr);
        }
        pend_dout = m->dout; pend_w = y.post_norm; pend_os = y.out_scale;
    }
    return lx.rc;
}

static int enqueue_step_rows(lg_hip_model *m, lg_hip_kv *kv, int rows, bool with_head, bool dry = false) {
    switch (rows) {
        case 1: return enqueue_step<1>(m, kv, with_head, dry);
        case 2: return enqueue_step<2>(m, kv, with_head, dry);
        case 3: return enqueue_step<3>(m, kv, with_head, dry);
        case 4: return enqueue_step<4>(m, kv, with_head, dry);
        case 5: return enqueue_step<5>(m, kv, with_head, dry);
        case 6: return enqueue_step<6>(m, kv, with_head, dry);
        case 7: return enqueue_step<7>(m, kv, with_head, dry);
        case 8: return enqueue_step<8>(m, kv, with_head, dry);
    }
    return fail(-2, "rows %d outside 1..%d", rows, LG_HIP_MAX_ROWS);
}

// what: 0 a block without its head, 1 a step, 2 a speculative round
static GraphKey graph_key(const lg_hip_model *m, const lg_hip_kv *kv, int rows, int what) {
    uint64_t o = 0;
    auto put = [&](unsigned v, int bits) { o = o << bits | (v & ((1u << bits) - 1u)); };
    put(what, 2); put(rows, 4); put(m->store_logits != 0, 1); put(m->draft_chain, 1); put(m->fuse_rows, 1); put(m->attn_rows, 1); put(m->attn_rows_fq, 1);
    put(m->head_mfma, 1); put(m->down_kq, 1); put(m->xcd_ffn, 1); put(m->fork_ple, 1); put(m->rows_geglu, 1); put(m->tail_stamps != 0, 1);
    put(m->tail_spread == 1 ? 1 : m->tail_spread ? 2 : 0, 2); put(m->xcd_tail, 2); put(m->down_m, 2); put(m->xcd_attn_tail, 2); put(m->merge_o, 2);
    put(m->xffn_delay, 10); put(m->narrow, 1); put(m->attn_out, 1); put(m->tail_qkv, 1); put(m->attn_geglu, 2); put(m->mid, 2); put(m->wait_polls, 17); put(may_wait(m), 1);
    return { (uint64_t)kv->id, o, (uint64_t)m->merge_o_slices, 0 };
}

// What `enqueue` launches on the stream, as a graph for the calls to come.  The caller has just launched the same thing: it
// ran, whether a graph of it can be made or not, so a failure here (no memory for the graph, say) is none of the call's.
// Null then, and the calls to come launch it as it is.
template <typename F>
static hipGraphExec_t capture_behind(hipStream_t st, F enqueue) {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    if (hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal) == hipSuccess) {
        const int rc = enqueue();
        const hipError_t e = hipStreamEndCapture(st, &graph);
        if (rc || e != hipSuccess || hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess) exec = nullptr;
        if (graph) (void)hipGraphDestroy(graph);
    }
    if (!exec) (void)hipGetLastError();                       // (else the next launch would report it)
    return exec;
}

// Launch one step, through a captured graph when enabled.  The first step of a (cache, width, options) runs as plain
// launches, and its graph is captured behind them, while the device works on the step and the host would only wait
// (a first decode step on a new cache, E4B shape: 3.95 -> 2.28 ms; capturing and instantiating 341 launches takes 1.5).
static int launch_step(lg_hip_model *m, lg_hip_kv *kv, int rows, bool with_head) {
    m->lread = m->lcoming = -1;
    Turn turn;
    int rc = turn.begin(m, rows);
    if (rc || (rc = count_steps(m, 1))) return rc;
    if (!m->use_graph || m->prof.on) return enqueue_step_rows(m, kv, rows, with_head);
    const GraphKey key = graph_key(m, kv, rows, with_head ? 1 : 0);
    auto it = m->graphs.find(key);
    if (it != m->graphs.end()) {
        if (!it->second) return enqueue_step_rows(m, kv, rows, with_head);
        HIP_TRY(hipGraphLaunch(it->second, m->stream));
        return 0;
    }
    rc = enqueue_step_rows(m, kv, rows, with_head, true);
    if (!rc) rc = enqueue_step_rows(m, kv, rows, with_head);
    if (!rc) m->graphs.emplace(key, capture_behind(m->stream, [&]() { return enqueue_step_rows(m, kv, rows, with_head); }));
    return rc;
}

static int check_block(lg_hip_model *m, lg_hip_kv *kv, const int32_t *toks, int n, int rows, int pos) {
    if (!m || !kv || !toks || kv->m != m) return fail(-1, "bad model / cache / token pointer");
    if (rows < 1 || rows > m->max_rows) return fail(-2, "block of %d rows; the model was committed for 1..%d", rows, m->max_rows);
    if (pos < 0 || pos + rows > kv->max_seq) return fail(-2, "positions %d..%d do not fit a cache of %d", pos, pos + rows - 1, kv->max_seq);
    for (int i = 0; i < n; ++i) if (toks[i] < 0 || toks[i] >= m->n_vocab) return fail(-2, "token id %d outside the vocabulary of %d", toks[i], m->n_vocab);
    return 0;
}

extern "C" int lg_hip_set_option(lg_hip_model *m, const char *name, int value) {
    if (!m || !name) return fail(-1, "set_option: null argument");
    if (!strcmp(name, "store_logits")) m->store_logits = value != 0;
    else if (!strcmp(name, "head_mfma")) m->head_mfma = value != 0;
    else if (!strcmp(name, "use_graph")) m->use_graph = value != 0;
    else if (!strcmp(name, "wide_prefill")) m->wide_prefill = value != 0 && (!m->committed || m->wide_built);
    else if (!strcmp(name, "fuse_rows")) m->fuse_rows = value != 0;
    else if (!strcmp(name, "attn_rows")) m->attn_rows = value != 0;
    else if (!strcmp(name, "attn_rows_fq")) m->attn_rows_fq = value != 0;
    else if (!strcmp(name, "xcd_tail_spread")) m->tail_spread = value;
    else if (!strcmp(name, "rows_geglu")) m->rows_geglu = value != 0;
    else if (!strcmp(name, "narrow")) m->narrow = value != 0;
    else if (!strcmp(name, "attn_out")) m->attn_out = value != 0;
    else if (!strcmp(name, "mid")) m->mid = value == 1 ? 1 : value ? 2 : 0;
    else if (!strcmp(name, "tail_qkv")) m->tail_qkv = value != 0;
    else if (!strcmp(name, "attn_geglu")) m->attn_geglu = value == 1 ? 1 : value ? 2 : 0;
    else if (!strcmp(name, "down_kq")) m->down_kq = value != 0;
    else if (!strcmp(name, "xcd_ffn")) m->xcd_ffn = value != 0 && m->xffn_built;
    else if (!strcmp(name, "fork_ple")) m->fork_ple = value != 0;
    else if (!strcmp(name, "down_m")) m->down_m = value < 0 ? 0 : value > 2 ? 2 : value;
    else if (!strcmp(name, "xcd_attn_tail")) m->xcd_attn_tail = value < 0 ? 0 : value > 2 ? 2 : value;
    else if (!strcmp(name, "merge_o")) m->merge_o = value < 0 ? 0 : value > 2 ? 2 : value;
    else if (!strcmp(name, "merge_o_slices")) m->merge_o_slices = value < 0 ? 0 : value;
    else if (!strcmp(name, "xcd_tail")) m->xcd_tail = value < 0 ? 0 : value > 2 ? 2 : value;
    else if (!strcmp(name, "wait_polls")) m->wait_polls = value < 0 ? 0 : value > 1 << 16 ? 1 << 16 : value;
    else if (!strcmp(name, "xcd_tail_stamps")) m->tail_stamps = value != 0;
    else if (!strcmp(name, "xcd_ffn_delay")) m->xffn_delay = value < 0 ? 0 : value > 0x3FF ? 0x3FF : value;
    else return fail(-2, "set_option: unknown option %s", name);
    return 0;
}

// What a kernel of a step left in StepCtl.err (a hand-over inside an XCD that was given up, or whose workgroups were not
// on one XCD): the step's results are not to be used.
static int step_err(const char *who, int err) {
    if (!err) return 0;
    return fail(-9, "%s: a kernel of the step reported %s%s(err 0x%x); its results are void", who,
                (err & LG_XFFN_ERR_PLACE) ? "workgroups of one group on different XCDs " : "",
                (err & LG_XFFN_ERR_WAIT) ? "a hand-over that was given up " : "", err);
}

// The step's state and tokens.  `report`: its accept kernel also writes its results to the host, who waits for them with
// wait_report: two copies in front of a step and three behind it cost 20 to 30 us of it.
static int load_block(lg_hip_model *m, const int32_t *toks, int rows, int pos, bool report) {
    LoadArgs a{};
    memcpy(a.tok, toks, (size_t)rows * 4);
    if (report && ++m->reports == INT32_MAX) m->reports = 1;
    hipLaunchKernelGGL(lg_k_load, dim3(1), dim3(1), 0, m->stream, m->ctl, m->sched, pos, rows, report ? m->reports : 0, a);
    HIP_TRY(hipGetLastError());
    return 0;
}
// A process that asked the runtime to give the processor away while it waits (hipSetDeviceFlags: yield, blocking) waits for the
// stream, which does so.  Every other one polls, as the runtime's own wait does, for up to 50 ms: far longer than a step takes.
static int wait_report(lg_hip_model *m, const char *who, int rows, int32_t *out, int32_t *adv) {
    const int32_t *r = m->pin + 32;
    auto there = [&]() { return __atomic_load_n(r + LG_REPORT_SEQ, __ATOMIC_ACQUIRE) == m->reports; };
    unsigned flags = 0;
    if (hipGetDeviceFlags(&flags) != hipSuccess) { (void)hipGetLastError(); flags = 0; }
    const bool poll = !(flags & (hipDeviceScheduleYield | hipDeviceScheduleBlockingSync));
    const auto t0 = std::chrono::steady_clock::now();
    for (int spins = 0; poll && !there(); ++spins) {
        if ((spins & 1023) == 1023 && std::chrono::steady_clock::now() - t0 >= std::chrono::milliseconds(50)) break;
        __builtin_ia32_pause();
    }
    if (!there()) {                                          // (also a slow device, or an error that this returns)
        HIP_TRY(hipStreamSynchronize(m->stream));
        if (!there()) return fail(-9, "%s: the step ended without its results", who);
    }
    const int rc = step_err(who, r[LG_REPORT_ERR]);
    if (rc) return rc;
    memcpy(out, r + LG_REPORT_OUT, (size_t)rows * 4);
    *adv = r[LG_REPORT_ADV];
    return 0;
}

extern "C" int lg_hip_forward_spec(lg_hip_model *m, lg_hip_kv *kv, const int32_t *toks, int rows, int pos,
                                   int32_t *out, int32_t *adv) {
    int rc = check_block(m, kv, toks, rows, rows, pos);
    if (rc) return rc;
    if (!out || !adv) return fail(-1, "forward_spec: null output");
    HIP_TRY(hipSetDevice(m->device));
    if ((rc = load_block(m, toks, rows, pos, true))) return rc;
    if ((rc = launch_step(m, kv, rows, true))) return rc;
    if ((rc = wait_report(m, "forward_spec", rows, out, adv))) return rc;
    m->last_rows = rows; m->last_adv = *adv;
    return 0;
}

// ---- draft head ---------------------------------------------------------------------------------
extern "C" int lg_hip_draft_create(lg_hip_model *target, const struct lg_hip_config *c, lg_hip_model **out) {
    if (!target || !c || !out || !target->committed) return fail(-1, "draft_create: the target model must be committed first");
    if (target->target) return fail(-2, "draft_create: the target is itself a draft head");
    if (target->n_kv_start < 2) return fail(-2, "draft_create: the target needs a sliding and a global cache layer to read");
    if (c->n_embd_per_layer) return fail(-2, "draft_create: a draft head has no per-layer embedding");
    // the rounds kept on the device copy the head's tokens straight into the target's blocks: same vocabulary or none
    if (c->n_vocab != target->n_vocab) return fail(-2, "draft_create: the head's vocabulary (%d) is not the target's (%d)", c->n_vocab, target->n_vocab);
    lg_hip_model *m = nullptr;
    int rc = lg_hip_model_create(c, target->device, &m);
    if (rc) return rc;
    (void)hipStreamDestroy(m->stream);
    m->stream = target->stream;                    // same queue: a draft reads what the last verify step wrote
    m->owns_stream = false;
    m->target = target;
    m->window = target->window;
    m->n_kv_start = 0;
    target->drafts.push_back(m);
    *out = m;
    return 0;
}

extern "C" int lg_hip_draft_step(lg_hip_model *d, lg_hip_kv *kv, int token, int pos, int chain, int32_t *tok_out) {
    if (!d || !kv || !tok_out || !d->target || !d->committed || kv->m != d->target) return fail(-1, "draft_step: bad draft / cache pointer");
    const lg_hip_model *t = d->target;
    if (token < 0 || token >= t->n_vocab) return fail(-2, "draft_step: token id %d outside the target vocabulary of %d", token, t->n_vocab);
    if (pos < 1 || pos > kv->max_seq) return fail(-2, "draft_step: position %d (the cache must hold 1..%d positions before it)", pos, kv->max_seq);
    if (chain && !d->w_post) return fail(-4, "draft_step: this head has no post-projection, drafts cannot chain");
    if (d->H > t->max_rows * t->H) return fail(-2, "draft_step: %d draft heads do not fit the target's attention scratch", d->H);
    HIP_TRY(hipSetDevice(d->device));
    int rc;
    int32_t tk = token, adv;
    if ((rc = load_block(d, &tk, 1, pos, true))) return rc;
    d->draft_chain = chain != 0;
    rc = launch_step(d, kv, 1, true);
    d->draft_chain = false;
    if (rc) return rc;
    if ((rc = wait_report(d, "draft_step", 1, tok_out, &adv))) return rc;
    d->last_rows = 1; d->last_adv = 1;
    return 0;
}

// One speculative round with no host involvement: K = rows-1 drafts (the first from the target's hidden state, the
// others chained), the link kernels that move their tokens, and the verify step.
static int enqueue_round(lg_hip_model *d, lg_hip_kv *kv, int rows, bool dry) {
    lg_hip_model *t = d->target;
    LinkArgs a{ d->ctl, t->ctl, d->sched, d->out, t->sched, t->out, t->adv, rows, 0 };
    int rc = 0;
    for (int j = 1; j <= rows && !rc; ++j) {
        a.phase = j;
        if (!dry) hipLaunchKernelGGL(lg_k_link, dim3(1), dim3(1), 0, t->stream, a);
        if (j == rows) break;
        d->draft_chain = j > 1;
        rc = enqueue_step_rows(d, kv, 1, true, dry);
        d->draft_chain = false;
    }
    if (!rc) rc = enqueue_step_rows(t, kv, rows, true, dry);
    a.phase = 0;
    if (!rc && !dry) hipLaunchKernelGGL(lg_k_link, dim3(1), dim3(1), 0, t->stream, a);
    if (!rc && !dry) { hipError_t e = hipGetLastError(); if (e != hipSuccess) rc = fail(-100 - (int)e, "mtp_rounds: launch failed: %s", hipGetErrorString(e)); }
    return rc;
}

extern "C" int lg_hip_mtp_rounds(lg_hip_model *d, lg_hip_kv *kv, int token, int pos, int rows, int n_rounds,
                                 int32_t *blocks, int32_t *out, int32_t *adv, int32_t *final_pos) {
    if (!d || !kv || !d->target || !d->committed || kv->m != d->target) return fail(-1, "mtp_rounds: bad draft / cache pointer");
    lg_hip_model *t = d->target;
    if (!blocks || !out || !adv) return fail(-1, "mtp_rounds: null output");
    if (rows < 2 || rows > t->max_rows) return fail(-2, "mtp_rounds: blocks of %d rows; the target was committed for 2..%d", rows, t->max_rows);
    if (rows > 2 && !d->w_post) return fail(-4, "mtp_rounds: this head has no post-projection, drafts cannot chain");
    if (n_rounds < 1 || n_rounds + 1 > t->sched_cap) return fail(-2, "mtp_rounds: %d rounds (limit %d)", n_rounds, t->sched_cap - 1);
    if (token < 0 || token >= t->n_vocab) return fail(-2, "mtp_rounds: token id %d outside the target vocabulary of %d", token, t->n_vocab);
    // every round may accept its whole block, so the last one may start rows*(n_rounds-1) positions on
    if (pos < 1 || (long long)pos + (long long)rows * n_rounds > kv->max_seq) return fail(-2, "mtp_rounds: positions %d..%lld do not fit a cache of %d", pos, (long long)pos + (long long)rows * n_rounds - 1, kv->max_seq);
    if (d->H > t->max_rows * t->H) return fail(-2, "mtp_rounds: %d draft heads do not fit the target's attention scratch", d->H);
    HIP_TRY(hipSetDevice(t->device));
    int rc;
    int32_t tk = token;
    if ((rc = load_block(t, &tk, 1, pos, false))) return rc;
    t->lread = t->lcoming = d->lread = d->lcoming = -1;
    if ((rc = count_steps(t, n_rounds)) || (rc = count_steps(d, n_rounds * (rows - 1)))) return rc;
    const bool graphs = t->use_graph && !t->prof.on && !d->prof.on;
    for (int r = 0; r < n_rounds; ++r) {
        Turn turn;
        if ((rc = turn.begin(t, rows, d))) return rc;
        if (!graphs) {
            if ((rc = enqueue_round(d, kv, rows, false))) return rc;
            continue;
        }
        GraphKey key = graph_key(t, kv, rows, 2);
        key[3] = graph_key(d, kv, 1, 2)[1];
        auto it = d->graphs.find(key);            // kept by the head: the graph dies with it or with the cache
        if (it == d->graphs.end()) {               // the first of them as launches, its graph while the device works on it
            if ((rc = enqueue_round(d, kv, rows, true)) || (rc = enqueue_round(d, kv, rows, false))) return rc;
            d->graphs.emplace(key, capture_behind(t->stream, [&]() { return enqueue_round(d, kv, rows, false); }));
        } else if (it->second) HIP_TRY(hipGraphLaunch(it->second, t->stream));
        else if ((rc = enqueue_round(d, kv, rows, false))) return rc;
    }
    const size_t nb = (size_t)n_rounds * rows;
    int32_t *res = t->pin + 64;
    HIP_TRY(hipMemcpyAsync(t->pin, t->ctl, sizeof(StepCtl), hipMemcpyDeviceToHost, t->stream));
    HIP_TRY(hipMemcpyAsync(res, t->sched, nb * 4, hipMemcpyDeviceToHost, t->stream));
    HIP_TRY(hipMemcpyAsync(res + nb, t->out, nb * 4, hipMemcpyDeviceToHost, t->stream));
    HIP_TRY(hipMemcpyAsync(res + 2 * nb, t->adv, (size_t)n_rounds * 4, hipMemcpyDeviceToHost, t->stream));
    HIP_TRY(hipStreamSynchronize(t->stream));
    StepCtl c;
    memcpy(&c, t->pin, sizeof c);
    if (c.step != n_rounds) return fail(-9, "mtp_rounds: %d of %d rounds ran", c.step, n_rounds);
    { const int erc = step_err("mtp_rounds", c.err); if (erc) return erc; }
    memcpy(blocks, res, nb * 4);
    memcpy(out, res + nb, nb * 4);
    memcpy(adv, res + 2 * nb, (size_t)n_rounds * 4);
    if (final_pos) *final_pos = c.pos;
    t->last_rows = rows; t->last_adv = adv[n_rounds - 1];
    t->sched_steps = 0;
    d->last_rows = 1; d->last_adv = 1;
    return 0;
}

extern "C" int lg_hip_prefill(lg_hip_model *m, lg_hip_kv *kv, const int32_t *toks, int n, int pos0) {
    if (n <= 0) return 0;
    if (!m) return fail(-1, "prefill: null model");
    if (!kv || !toks || kv->m != m) return fail(-1, "bad model / cache / token pointer");
    if (pos0 < 0 || n > kv->max_seq - pos0) return fail(-2, "positions %d..%lld do not fit a cache of %d", pos0, (long long)pos0 + n - 1, kv->max_seq);
    for (int i = 0; i < n; ++i) if (toks[i] < 0 || toks[i] >= m->n_vocab) return fail(-2, "token id %d outside the vocabulary of %d", toks[i], m->n_vocab);
    HIP_TRY(hipSetDevice(m->device));
    bool wide_ok = !m->target && m->wide_prefill;
    // (attention that keeps its weights in LDS addresses a layer's cache with 32 bits, and reaches no row past LG_WIDE_ROWS + 32 (LG_WA_TILES + 4))
    for (size_t L = 0; L < kv->seq.size(); ++L) wide_ok = wide_ok && (size_t)(LG_WIDE_ROWS + 32 * (LG_WA_TILES + 4)) * kv->kv_dim[L] * 2 < (size_t)1 << 31;
    const int cap = m->sched_cap * LG_HIP_MAX_ROWS;        // tokens the staging holds
    int32_t *err = m->pin + 32 + LG_REPORT_ERR;             // (written by the verify blocks among the call's, the prompt kernels wait for nobody)
    __atomic_store_n(err, 0, __ATOMIC_RELAXED);
    PromptTurn prompt;
    if (wide_ok && n > m->max_rows) { const int rc = prompt.begin(m); if (rc) return rc; }
    for (int at = 0; at < n;) {
        // the tokens go over once, the blocks follow each other on the stream and the host waits at the end
        const int part = n - at < cap ? n - at : cap;
        memcpy(m->pin + 64, toks + at, (size_t)part * 4);
        HIP_TRY(hipMemcpyAsync(m->sched, m->pin + 64, (size_t)part * 4, hipMemcpyHostToDevice, m->stream));
        for (int done = 0; done < part;) {
            const int left = part - done;
            int rows = left < kv->prompt_rows ? left : kv->prompt_rows, rc;
            const bool wide = wide_ok && !far_in_narrow_heads(m, kv, rows, pos0 + at + done);
            const bool first = at + done == 0;
            Turn turn;
            if (wide && left > m->max_rows) rc = enqueue_prompt(m, kv, m->sched + done, rows, pos0 + at + done, first);
            else {                                           // a remainder that fits a verify block
                rows = left < m->max_rows ? left : m->max_rows;
                if (done) HIP_TRY(hipMemcpyAsync(m->sched, m->pin + 64 + done, (size_t)rows * 4, hipMemcpyHostToDevice, m->stream));   // (its kernels read the schedule from its start)
                hipLaunchKernelGGL(lg_k_set_ctl, dim3(1), dim3(1), 0, m->stream, m->ctl, pos0 + at + done, first);
                if (!wide) rc = launch_step(m, kv, rows, false);
                else if (!(rc = turn.begin(m, rows)) && !(rc = count_steps(m, 1)))
                    rc = enqueue_step_rows(m, kv, rows, false);                                         // (a single one: not worth a capture)
            }
            if (rc) return rc;
            done += rows;
        }
        at += part;
        HIP_TRY(hipStreamSynchronize(m->stream));
    }
    prompt.done = true;
    return step_err("prefill", __atomic_load_n(err, __ATOMIC_RELAXED));
}

extern "C" int lg_hip_tail_stamps(lg_hip_model *m, int which, unsigned long long *dst, int cap) {
    if (!m || !dst || !m->tstamps || which < 0 || which > 1) return fail(-1, "tail_stamps: the model has no one-XCD tail");
    if (cap < LG_XTAIL_UNITS * 8) return fail(-2, "tail_stamps: room for %d values needed", LG_XTAIL_UNITS * 8);
    HIP_TRY(hipSetDevice(m->device));
    HIP_TRY(hipStreamSynchronize(m->stream));
    HIP_TRY(copy_now(m->stream, dst, m->tstamps + (size_t)which * LG_XTAIL_UNITS * 8, (size_t)LG_XTAIL_UNITS * 8 * 8, hipMemcpyDeviceToHost));
    return LG_XTAIL_UNITS;
}

extern "C" int lg_hip_get_hidden(lg_hip_model *m, float *dst) {
    if (!m || !dst) return fail(-1, "get_hidden: null argument");
    HIP_TRY(hipSetDevice(m->device));
    HIP_TRY(hipStreamSynchronize(m->stream));
    HIP_TRY(copy_now(m->stream, dst, m->g_hidden, (size_t)m->E * 4, hipMemcpyDeviceToHost));
    return 0;
}
extern "C" int lg_hip_set_hidden_row(lg_hip_model *m, int row) {
    if (!m) return fail(-1, "set_hidden_row: null model");
    if (row < 0 || row >= m->last_rows) return fail(-2, "set_hidden_row: row %d of a %d-row step", row, m->last_rows);
    HIP_TRY(hipSetDevice(m->device));
    HIP_TRY(hipMemcpyAsync(m->g_hidden, m->hidden_rows + (size_t)row * m->E, (size_t)m->E * 4, hipMemcpyDeviceToDevice, m->stream));
    return 0;
}
// A row crosses the bus when it is asked for: written into pinned memory by the head itself, every row of every step did, read or
// not (E4B shape, 8 rows that nobody reads: 2.37 -> 2.50 ms a step).  For a caller that takes the rows in turn the next one is on
// its way while it is given this one: a step and all its rows read take 2.05 ms at 1 row (2.03 with pinned logits), 2.33 at
// 4 (2.37), 2.77 at 8 (2.83).
extern "C" int lg_hip_get_logits(lg_hip_model *m, int row, float *dst) {
    if (!m || !dst) return fail(-1, "get_logits: null argument");
    if (!m->store_logits) return fail(-4, "get_logits: the store_logits option is off");
    if (row < 0 || row >= m->last_rows) return fail(-2, "get_logits: row %d of a %d-row step", row, m->last_rows);
    HIP_TRY(hipSetDevice(m->device));
    const size_t n = (size_t)m->n_vocab;
    auto start = [&](int r) { return hipMemcpyAsync(m->lstage + (r & 1) * n, m->logits + r * n, n * 4, hipMemcpyDeviceToHost, m->stream); };
    if (m->lcoming != row) HIP_TRY(start(row));
    m->lcoming = -1;
    HIP_TRY(hipStreamSynchronize(m->stream));
    if (row + 1 < m->last_rows && row == m->lread + 1) { HIP_TRY(start(row + 1)); m->lcoming = row + 1; }
    m->lread = row;
    memcpy(dst, m->lstage + (row & 1) * n, n * 4);
    return 0;
}

// ---- device-resident schedule -----------------------------------------------------------------
extern "C" int lg_hip_schedule_load(lg_hip_model *m, const int32_t *toks, int n_steps, int rows, int pos0) {
    if (!m || !toks || !m->committed) return fail(-1, "schedule_load: bad argument");
    if (rows < 1 || rows > m->max_rows || n_steps < 1 || n_steps > m->sched_cap) return fail(-2, "schedule_load: %d steps of %d rows (limits %d, %d)", n_steps, rows, m->sched_cap, m->max_rows);
    if (pos0 < 0) return fail(-2, "schedule_load: position %d", pos0);
    for (size_t i = 0; i < (size_t)n_steps * rows; ++i) if (toks[i] < 0 || toks[i] >= m->n_vocab) return fail(-2, "schedule_load: token id %d outside the vocabulary", toks[i]);
    HIP_TRY(hipSetDevice(m->device));
    HIP_TRY(hipStreamSynchronize(m->stream));
    HIP_TRY(copy_now(m->stream, m->sched, toks, (size_t)n_steps * rows * 4, hipMemcpyHostToDevice));
    StepCtl c{ pos0, 0, 0, 0, 0 };
    HIP_TRY(copy_now(m->stream, m->ctl, &c, offsetof(StepCtl, launch), hipMemcpyHostToDevice));
    m->sched_steps = n_steps; m->sched_rows = rows; m->sched_pos0 = pos0; m->sched_loaded = n_steps;
    return 0;
}
extern "C" int lg_hip_schedule_run(lg_hip_model *m, lg_hip_kv *kv, int n_steps) {
    if (!m || !kv || kv->m != m) return fail(-1, "schedule_run: bad argument");
    if (n_steps < 1 || n_steps > m->sched_steps) return fail(-2, "schedule_run: %d steps requested, %d loaded", n_steps, m->sched_steps);
    // every step may accept its whole block: the last one of this call may start rows * (steps so far) positions on
    const long long last = (long long)m->sched_pos0 + (long long)m->sched_rows * (m->sched_loaded - m->sched_steps + n_steps);
    if (last > kv->max_seq) return fail(-2, "schedule_run: positions up to %lld do not fit a cache of %d", last - 1, kv->max_seq);
    HIP_TRY(hipSetDevice(m->device));
    for (int s = 0; s < n_steps; ++s) { int rc = launch_step(m, kv, m->sched_rows, true); if (rc) return rc; }
    m->sched_steps -= n_steps;       // steps left to run
    m->last_rows = m->sched_rows;
    return 0;
}
extern "C" int lg_hip_schedule_wait(lg_hip_model *m, int32_t *out, int32_t *adv, int32_t *final_pos) {
    if (!m) return fail(-1, "schedule_wait: null model");
    HIP_TRY(hipSetDevice(m->device));
    HIP_TRY(hipStreamSynchronize(m->stream));
    StepCtl c;
    HIP_TRY(copy_now(m->stream, &c, m->ctl, sizeof c, hipMemcpyDeviceToHost));
    { const int erc = step_err("schedule_wait", c.err); if (erc) return erc; }
    // the step counter is device state: never copy more than the schedule that was loaded holds
    if (c.step < 0 || c.step > m->sched_loaded)
        return fail(-6, "schedule_wait: the device reports %d steps done, %d were loaded", c.step, m->sched_loaded);
    if (out) HIP_TRY(copy_now(m->stream, out, m->out, (size_t)c.step * m->sched_rows * 4, hipMemcpyDeviceToHost));
    if (adv) HIP_TRY(copy_now(m->stream, adv, m->adv, (size_t)c.step * 4, hipMemcpyDeviceToHost));
    if (final_pos) *final_pos = c.pos;
    return c.step;
}
extern "C" int lg_hip_schedule_time(lg_hip_model *m, lg_hip_kv *kv, int n_steps, float *ms) {
    if (!m || !ms) return fail(-1, "schedule_time: null argument");
    HIP_TRY(hipSetDevice(m->device));
    hipEvent_t a, b;
    HIP_TRY(hipEventCreate(&a));
    HIP_TRY(hipEventCreate(&b));
    HIP_TRY(hipEventRecord(a, m->stream));
    int rc = lg_hip_schedule_run(m, kv, n_steps);
    if (!rc) {
        (void)hipEventRecord(b, m->stream);
        hipError_t e = hipEventSynchronize(b);
        if (e != hipSuccess) rc = fail(-100 - (int)e, "hipEventSynchronize: %s", hipGetErrorString(e));
        else (void)hipEventElapsedTime(ms, a, b);
    }
    (void)hipEventDestroy(a); (void)hipEventDestroy(b);
    return rc;
}

// ---- measurement ------------------------------------------------------------------------------
static void class_bytes(const lg_hip_model *m, const lg_hip_kv *kv, int pos, int rows, double *b) {
    const double q = 18.0 / 32.0;                         // bytes per q4_0 weight
    for (int i = 0; i < KC_COUNT; ++i) b[i] = 0;
    if (m->ple) b[KC_PMP] = (double)m->E * m->ple * m->n_layer * (m->pmp_f ? 4.0 : q);
    const bool narrow = use_narrow(m, rows);              // (everything but the attention and the first layer's projections)
    for (int L = 0; L < m->n_layer; ++L) {
        const Layer &y = m->L[L];
        b[L && (narrow || (!y.winp_f && tail_does_qkv(m, rows, y) && use_ple_tail(m, rows, true))) ? KC_TAIL : L && !narrow && (use_mid_down(m, m->L[L - 1], y, rows) || (y.winp_f && use_mid_proj(m, y, rows))) ? KC_ROWS : KC_QKV] += (double)m->E * y.qkv_m * q;
        if (narrow) b[KC_TAIL] += ((double)y.qd * m->E + 3.0 * m->E * y.nff + 2.0 * m->E * m->ple) * q;
        else {
        {
            const int w = (y.is_local && m->window > 0) ? m->window : 0, st = (w > 0 && pos - w + 1 > 0) ? pos - w + 1 : 0;
            const int tiles = ((pos + rows - 1) >> 5) - (st >> 5) + 1;
            b[use_attn_tail(m, y, rows, tiles) ? KC_ATAIL : use_merge_o(m, y, rows, tiles) ? KC_MERGE : use_attn_out(m, y, rows, step_tiles(m, kv, y, rows, 0)) ? KC_ATAIL : KC_O] += (double)y.qd * m->E * q;
        }
        const int tiles = step_tiles(m, kv, y, rows, 0);
        if (m->xffn_built && m->xcd_ffn && may_wait(m) && rows >= 4) b[KC_FFN] += 3.0 * m->E * y.nff * q;
        else { b[use_attn_out(m, y, rows, tiles) ? attn_out_geglu(m, y, rows, tiles) ? KC_ATAIL : KC_GATEUP : use_mid_o(m, y, rows) ? KC_O : KC_GATEUP] += 2.0 * m->E * y.nff * q; b[L + 1 < m->n_layer && use_mid_down(m, y, m->L[L + 1], rows) ? KC_ROWS : KC_DOWN] += (double)y.nff * m->E * q; }
        if (m->ple && !y.winp_f && use_ple_tail(m, rows, L + 1 < m->n_layer && tail_does_qkv(m, rows, m->L[L + 1]))) b[KC_TAIL] += 2.0 * m->E * m->ple * q;
        else if (m->ple) { const double pq = y.winp_f ? 4.0 : q; b[KC_PLEGATE] += (double)m->E * m->ple * pq; b[L + 1 < m->n_layer && y.winp_f && use_mid_proj(m, m->L[L + 1], rows) ? KC_ROWS : KC_PLEPROJ] += (double)m->ple * m->E * pq; }
        }
        const int window = (y.is_local && m->window > 0) ? m->window : 0;
        const int last = pos + rows - 1, start = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
        b[KC_ATTN] += 2.0 * (last - start + 1) * y.kd * 2.0;          // K and V rows, f16
    }
    b[KC_HEAD] = (double)m->E * m->n_vocab * q;
}

extern "C" int lg_hip_profile_step(lg_hip_model *m, lg_hip_kv *kv, const int32_t *toks, int rows, int pos, int repeats,
                                   const char **names, float *ms, int32_t *launches, double *bytes, int cap) {
    int rc = check_block(m, kv, toks, rows, rows, pos);
    if (rc) return rc;
    if (cap < KC_COUNT || repeats < 1) return fail(-2, "profile_step: need room for %d classes", KC_COUNT);
    HIP_TRY(hipSetDevice(m->device));
    double acc[KC_COUNT] = { 0 };
    int cnt[KC_COUNT] = { 0 };
    for (int r = 0; r < repeats + 1; ++r) {              // first pass warms up and is dropped
        if ((rc = load_block(m, toks, rows, pos, false))) return rc;
        std::optional<Turn> turn(std::in_place);
        if ((rc = turn->begin(m, rows)) || (rc = count_steps(m, 1))) return rc;
        m->prof.on = true;
        m->lread = m->lcoming = -1;
        rc = enqueue_step_rows(m, kv, rows, true);
        turn.reset();
        m->prof.on = false;
        hipError_t e = hipStreamSynchronize(m->stream);
        if (!rc && e != hipSuccess) rc = fail(-100 - (int)e, "profile_step: %s", hipGetErrorString(e));
        for (size_t i = 0; i < m->prof.cls.size(); ++i) {
            float t = 0;
            if (!rc && r > 0 && hipEventElapsedTime(&t, m->prof.ev[2 * i], m->prof.ev[2 * i + 1]) == hipSuccess) { acc[m->prof.cls[i]] += t; cnt[m->prof.cls[i]]++; }
        }
        for (hipEvent_t ev : m->prof.ev) (void)hipEventDestroy(ev);
        m->prof.ev.clear(); m->prof.cls.clear();
        if (rc) return rc;
    }
    double b[KC_COUNT];
    class_bytes(m, kv, pos, rows, b);
    for (int i = 0; i < KC_COUNT; ++i) {
        names[i] = k_class_names[i]; ms[i] = (float)(acc[i] / repeats); launches[i] = cnt[i] / repeats; bytes[i] = b[i];
    }
    m->last_rows = rows;
    return KC_COUNT;
}

// ---- isolated kernels -------------------------------------------------------------------------
struct Scratch {            // device buffers freed on scope exit
    std::vector<void *> p;
    ~Scratch() { for (void *q : p) (void)hipFree(q); }
    template <typename T> int get(T **out, size_t n) {
        HIP_TRY(hipMalloc((void **)out, n * sizeof(T) ? n * sizeof(T) : 16));
        p.push_back(*out);
        return 0;
    }
};

template <int M>
static int matmul_rows(hipStream_t st, const uint8_t *dw, int k, int mrows, const float *dx, float *dout, int32_t *ddots,
                       int8_t *dq, int repeats, float *kernel_ms) {
    const int n32 = M * (k / 32);
    hipLaunchKernelGGL(lg_k_quant_flat, dim3((n32 * 8 + LG_WG - 1) / LG_WG), dim3(LG_WG), 0, st, dx, M, k, dq);
    MmArgs a{ dw, k, mrows, dout, dq, ddots };
    lg_hip_model shim;                       // the launcher only needs a stream and the profiling switch
    shim.stream = st;
    Launcher lx{ &shim, false };
    if (ddots) launch_mm<M, true>(lx, 0, a);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    auto body = [&]() -> int {
        HIP_TRY(hipEventCreate(&e0)); HIP_TRY(hipEventCreate(&e1));
        a.dots = nullptr;
        launch_mm<M, false>(lx, 0, a);           // warm-up, also the result
        HIP_TRY(hipEventRecord(e0, st));
        for (int r = 0; r < repeats; ++r) launch_mm<M, false>(lx, 0, a);
        if (lx.rc) return lx.rc;
        HIP_TRY(hipEventRecord(e1, st));
        HIP_TRY(hipStreamSynchronize(st));
        HIP_TRY(hipGetLastError());
        float t = 0;
        if (repeats > 0) HIP_TRY(hipEventElapsedTime(&t, e0, e1));
        if (kernel_ms) *kernel_ms = repeats > 0 ? t / repeats : 0.0f;
        return 0;
    };
    const int rc = body();
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    return rc;
}

// q8 rows of a verify-width block from the device's activation order back to natural order
static int read_back_q8(const int8_t *dq, int rows, int k, int8_t *xq, float *xd, int32_t *xsum) {
    const ActLayout lay = lg_act_layout(k);
    const int nb = k / 32;
    if (xq) {
        std::vector<int8_t> dev((size_t)rows * k);
        HIP_TRY(hipMemcpy(dev.data(), dq, dev.size(), hipMemcpyDeviceToHost));
        for (int j = 0; j < rows; ++j)
            for (int w = 0; w < k / 16; ++w)
                memcpy(xq + (size_t)j * k + (size_t)w * 16, dev.data() + (size_t)j * k + (size_t)lg_act_unit(lay, w) * 16, 16);
    }
    if (xd || xsum) {
        std::vector<float2> ds((size_t)rows * nb);
        HIP_TRY(hipMemcpy(ds.data(), dq + (size_t)rows * k, ds.size() * 8, hipMemcpyDeviceToHost));
        for (int j = 0; j < rows; ++j)
            for (int b = 0; b < nb; ++b) {
                const float2 v = ds[(size_t)j * nb + lg_act_block(lay, b)];
                if (xd) xd[(size_t)j * nb + b] = v.x;
                if (xsum) memcpy(&xsum[(size_t)j * nb + b], &v.y, 4);
            }
    }
    return 0;
}

// the same for a wide block: values from their two digits, sums from the values (the kernels need none)
static int read_back_wide(const uint8_t *dq, int rows, int k, int8_t *xq, float *xd, int32_t *xsum) {
    const int nb = k / 32;
    std::vector<uint8_t> dev(lg_wide_q8_bytes(rows, k));
    HIP_TRY(hipMemcpy(dev.data(), dq, dev.size(), hipMemcpyDeviceToHost));
    for (int j = 0; j < rows; ++j)
        for (int b = 0; b < nb; ++b) {
            const uint8_t *t = dev.data() + ((size_t)(j >> 6) * nb + b) * LG_QTILE;
            int v[2][32], sum = 0;
            for (int half = 0; half < 2; ++half) {
                const int lane = half * 32 + (j & 31), base = ((j >> 5) & 1) * 1536;
                uint8_t bytes[25] = { 0 };
                memcpy(bytes, t + base + lane * 16, 16);
                memcpy(bytes + 16, t + base + 1024 + lane * 8, 8);
                for (int e = 0; e < 32; ++e) {
                    const int code = ((bytes[6 * e / 8] | (bytes[6 * e / 8 + 1] << 8)) >> (6 * e % 8)) & 63;
                    v[half][e] = (code & 32) ? -(code & 31) : code & 31;
                }
            }
            for (int e = 0; e < 32; ++e) {
                const int q = 16 * v[0][e] + v[1][e];
                sum += q;
                if (xq) xq[(size_t)j * k + b * 32 + e] = (int8_t)q;
            }
            if (xd) memcpy(&xd[(size_t)j * nb + b], t + 3072 + (j & 63) * 4, 4);
            if (xsum) xsum[(size_t)j * nb + b] = sum;
        }
    return 0;
}
// (as the q/k/v and the attention output projection of a prompt are launched; *parts: slabs of the result)
static int matmul_wide(hipStream_t st, const uint8_t *dw, uint8_t *dwide, int k, int mrows, int rows, const float *dx, float *dout, int32_t *ddots,
                       int8_t *dq, int repeats, float *kernel_ms, int *parts) {
    const size_t np = (size_t)((mrows + LG_WT - 1) / LG_WT * LG_WT) * (k / 32);
    hipLaunchKernelGGL(lg_k_wide_pack, dim3((unsigned)((np + LG_WG - 1) / LG_WG)), dim3(LG_WG), 0, st, dw, k, mrows, 0, dwide);
    hipLaunchKernelGGL(lg_k_wide_quant, dim3((rows * (k / 32) * 8 + LG_WG - 1) / LG_WG), dim3(LG_WG), 0, st, dx, rows, k, (uint8_t *)dq);
    lg_hip_model shim;
    shim.stream = st;
    Launcher lx{ &shim, false };
    if (ddots) launch_wide_mm<true>(lx, 0, dwide, dq, k, mrows, rows, dout, ddots, true);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    auto body = [&]() -> int {
        HIP_TRY(hipEventCreate(&e0)); HIP_TRY(hipEventCreate(&e1));
        *parts = launch_wide_mm<false>(lx, 0, dwide, dq, k, mrows, rows, dout, nullptr, true);
        HIP_TRY(hipEventRecord(e0, st));
        for (int r = 0; r < repeats; ++r) launch_wide_mm<false>(lx, 0, dwide, dq, k, mrows, rows, dout, nullptr, true);
        if (lx.rc) return lx.rc;
        HIP_TRY(hipEventRecord(e1, st));
        HIP_TRY(hipStreamSynchronize(st));
        HIP_TRY(hipGetLastError());
        float t = 0;
        if (repeats > 0) HIP_TRY(hipEventElapsedTime(&t, e0, e1));
        if (kernel_ms) *kernel_ms = repeats > 0 ? t / repeats : 0.0f;
        return 0;
    };
    const int rc = body();
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    return rc;
}

extern "C" int lg_hip_matmul_f32w(const float *w, int k, int mrows, const float *x, int rows, float *out) {
    if (!w || !x || !out) return fail(-1, "matmul_f32w: null argument");
    if (k < 256 || k % 256 || mrows < 1 || rows < 1) return fail(-2, "matmul_f32w: k %d (a multiple of 256), m %d, rows %d", k, mrows, rows);
    if (lg_hip_device_count() < 1) return fail(-3, "matmul_f32w: no HIP device");
    Scratch sc;
    float *dw, *dx, *dout;
    if (sc.get(&dw, (size_t)mrows * k) || sc.get(&dx, (size_t)rows * k) || sc.get(&dout, (size_t)rows * mrows)) return -7;
    HIP_TRY(hipMemcpy(dw, w, (size_t)mrows * k * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dx, x, (size_t)rows * k * 4, hipMemcpyHostToDevice));
    MmfArgs a{ dw, k, mrows, dx, k, rows, dout, mrows, nullptr, 0 };
    hipLaunchKernelGGL((lg_k_mmf<8>), dim3((mrows + LG_WG / 64 - 1) / (LG_WG / 64), (rows + 7) / 8), dim3(LG_WG), 0, nullptr, a);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(out, dout, (size_t)rows * mrows * 4, hipMemcpyDeviceToHost));
    return 0;
}

extern "C" int lg_hip_matmul_q4q8(const void *w, int k, int mrows, const float *x, int rows, float *out, int32_t *dots,
                                  int8_t *xq, float *xd, int32_t *xsum, int repeats, float *kernel_ms) {
    if (!w || !x) return fail(-1, "matmul: null input");
    const bool wide = rows > LG_HIP_MAX_ROWS && rows % LG_WIDE == 0 && rows <= LG_WIDE_ROWS;     // row tiles through the kernels of prompt blocks
    if (rows < 1 || (rows > LG_HIP_MAX_ROWS && !wide) || !lg_hip_repacked_bytes(k, mrows) || (!wide && lds_mm(rows, k) > 160 * 1024))
        return fail(-2, "matmul: rows %d (1..%d, or a multiple of %d up to %d), k %d (multiple of 256; up to %d rows: rows*k*1.25 <= 160 KiB), m %d (multiple of 8)",
                    rows, LG_HIP_MAX_ROWS, LG_WIDE, LG_WIDE_ROWS, k, LG_HIP_MAX_ROWS, mrows);
    if (lg_hip_device_count() < 1) return fail(-3, "matmul: no HIP device");
    const int nb = k / 32;
    std::vector<uint8_t> tiled(lg_hip_repacked_bytes(k, mrows));
    int rc = lg_hip_repack_q4_0(w, k, mrows, tiled.data());
    if (rc) return rc;
    Scratch sc;
    uint8_t *dw; float *dx, *dout; int32_t *ddots = nullptr; int8_t *dq;
    if (sc.get(&dw, tiled.size()) || sc.get(&dx, (size_t)rows * k) || sc.get(&dout, (size_t)rows * mrows * 4) ||
        sc.get(&dq, wide ? lg_wide_q8_bytes(rows, k) : (size_t)rows * k * 5 / 4)) return -7;
    if (dots && sc.get(&ddots, (size_t)rows * mrows * nb)) return -7;
    HIP_TRY(hipMemcpy(dw, tiled.data(), tiled.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dx, x, (size_t)rows * k * 4, hipMemcpyHostToDevice));
    hipStream_t st;
    HIP_TRY(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    int parts = 1;
    if (wide) {
        uint8_t *dwide;
        if (sc.get(&dwide, lg_wide_bytes(k, mrows))) rc = -7;
        else rc = matmul_wide(st, dw, dwide, k, mrows, rows, dx, dout, ddots, dq, repeats, kernel_ms, &parts);
    } else switch (rows) {
#define CASE(M) case M: rc = matmul_rows<M>(st, dw, k, mrows, dx, dout, ddots, dq, repeats, kernel_ms); break;
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
    }
    (void)hipStreamDestroy(st);
    if (rc) return rc;
    if (out && parts == 4) {                               // four slabs of partial sums: the top of the segment tree is added here
        std::vector<float> slabs((size_t)4 * rows * mrows);
        HIP_TRY(hipMemcpy(slabs.data(), dout, slabs.size() * 4, hipMemcpyDeviceToHost));
        const size_t n = (size_t)rows * mrows;
        for (size_t i = 0; i < n; ++i) out[i] = (slabs[i] + slabs[n + i]) + (slabs[2 * n + i] + slabs[3 * n + i]);
    } else if (out) HIP_TRY(hipMemcpy(out, dout, (size_t)rows * mrows * 4, hipMemcpyDeviceToHost));
    if (dots) HIP_TRY(hipMemcpy(dots, ddots, (size_t)rows * mrows * nb * 4, hipMemcpyDeviceToHost));
    // the device keeps activation rows in the matmul's own order; hand them back in natural order
    return wide ? read_back_wide((const uint8_t *)dq, rows, k, xq, xd, xsum) : read_back_q8(dq, rows, k, xq, xd, xsum);
}

template <int M>
static void rows_isolated(hipStream_t st, const RowArgs &s_in, StepCtl *ctl) {
    RowArgs s = s_in;
    const int slices = (s.E + 1023) / 1024;                   // as a verify step launches it: the tail sliced over workgroups
    s.slices = slices;
    hipLaunchKernelGGL((lg_k_rows<M>), dim3(M, slices), dim3(LG_WG), 0, st, ctl, LG_ROW_FIELDS(LG_XA, s) 0);
}
extern "C" int lg_hip_rows_norm_q8(const float *x, const float *dout, const float *w_post, const float *out_scale,
                                   const float *w_pre, int rows, int E, float eps, float *x_out, float *h_out,
                                   int8_t *xq, float *xd, int32_t *xsum) {
    if (!x) return fail(-1, "rows_norm_q8: null input");
    if (rows < 1 || rows > LG_HIP_MAX_ROWS || E < 256 || E % 256 || E > 4096) return fail(-2, "rows_norm_q8: rows %d (1..%d), E %d (a multiple of 256 up to 4096)", rows, LG_HIP_MAX_ROWS, E);
    if (dout && !w_post) return fail(-1, "rows_norm_q8: a sub-layer output needs its norm weight");
    if (lg_hip_device_count() < 1) return fail(-3, "rows_norm_q8: no HIP device");
    Scratch sc;
    float *dx, *dd = nullptr, *dwp = nullptr, *dos = nullptr, *dwr = nullptr, *dxo, *dho; int8_t *dq; StepCtl *ctl;
    const size_t n = (size_t)rows * E;
    if (sc.get(&dx, n) || sc.get(&dxo, n) || sc.get(&dho, n) || sc.get(&dq, n * 5 / 4) || sc.get(&ctl, 1)) return -7;
    HIP_TRY(hipMemcpy(dx, x, n * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemset(ctl, 0, sizeof(StepCtl)));
    if (dout) { if (sc.get(&dd, n) || sc.get(&dwp, (size_t)E)) return -7; HIP_TRY(hipMemcpy(dd, dout, n * 4, hipMemcpyHostToDevice)); HIP_TRY(hipMemcpy(dwp, w_post, (size_t)E * 4, hipMemcpyHostToDevice)); }
    if (out_scale) { if (sc.get(&dos, 1)) return -7; HIP_TRY(hipMemcpy(dos, out_scale, 4, hipMemcpyHostToDevice)); }
    if (w_pre) { if (sc.get(&dwr, (size_t)E)) return -7; HIP_TRY(hipMemcpy(dwr, w_pre, (size_t)E * 4, hipMemcpyHostToDevice)); }
    RowArgs s{};
    s.x = dx; s.dout = dd; s.dparts = 1; s.w_post = dwp; s.os = dos; s.x_out = dxo; s.w_pre = dwr; s.h_out = dho;
    s.q = dq; s.E = E; s.eps = eps;
    switch (rows) {
#define CASE(M) case M: rows_isolated<M>(nullptr, s, ctl); break;
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
    }
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipDeviceSynchronize());
    if (x_out) HIP_TRY(hipMemcpy(x_out, dxo, n * 4, hipMemcpyDeviceToHost));
    if (h_out) HIP_TRY(hipMemcpy(h_out, dho, n * 4, hipMemcpyDeviceToHost));
    return read_back_q8(dq, rows, E, xq, xd, xsum);
}

// ---- isolated per-layer-embedding kernels (tests) ----------------------------------------------------
// lg_k_rows_plegate on its own: the residual update x + rmsnorm(dout) * w_post of `rows` rows, then the inp_gate
// matmul (w_gate: ple plain q4_0 rows of E) on the q8 of the new rows, gelu(.) * ipl and the q8 of that.
extern "C" int lg_hip_rows_ple_gate(const float *x, const float *dout, const float *w_post, const void *w_gate, const float *ipl,
                                    int rows, int E, int ple, float eps, float *x_out, int8_t *pq, float *pd, int32_t *psum) {
    if (!x || !dout || !w_post || !w_gate || !ipl) return fail(-1, "rows_ple_gate: null input");
    if (rows < 1 || rows > LG_HIP_MAX_ROWS || E < 256 || E % 256 || E > 4096 || ple != 256)
        return fail(-2, "rows_ple_gate: rows %d (1..%d), E %d (a multiple of 256 up to 4096), ple %d (256 is built)", rows, LG_HIP_MAX_ROWS, E, ple);
    if (lg_hip_device_count() < 1) return fail(-3, "rows_ple_gate: no HIP device");
    std::vector<uint8_t> tiled(lg_hip_repacked_bytes(E, ple));
    int rc = lg_hip_repack_q4_0(w_gate, E, ple, tiled.data());
    if (rc) return rc;
    Scratch sc;
    float *dx, *dd, *dw, *di, *dxo; uint8_t *dg; int8_t *dq;
    const size_t n = (size_t)rows * E;
    if (sc.get(&dx, n) || sc.get(&dd, n) || sc.get(&dw, (size_t)E) || sc.get(&di, (size_t)rows * ple) || sc.get(&dxo, n) ||
        sc.get(&dg, tiled.size()) || sc.get(&dq, (size_t)rows * ple * 5 / 4)) return -7;
    HIP_TRY(hipMemcpy(dx, x, n * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dd, dout, n * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dw, w_post, (size_t)E * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(di, ipl, (size_t)rows * ple * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dg, tiled.data(), tiled.size(), hipMemcpyHostToDevice));
    PleGateArgs a{ dg, E, ple, nullptr, di, 0, 1, dq };
    RowsPleGateArgs r{ a, dx, dd, dw, dxo, eps, 1 };
    switch (rows) {
#define CASE(M) case M: rc = set_lds(lg_k_rows_plegate<M>, lds_mm(1, E)); \
        if (!rc) hipLaunchKernelGGL((lg_k_rows_plegate<M>), dim3(ple / 32, M), dim3(LG_WG), lds_mm(1, E), nullptr, LG_RPG_FIELDS(LG_XA, r) 0); break;
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
    }
    if (rc) return rc;
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipDeviceSynchronize());
    if (x_out) HIP_TRY(hipMemcpy(x_out, dxo, n * 4, hipMemcpyDeviceToHost));
    return read_back_q8(dq, rows, ple, pq, pd, psum);
}

// lg_k_ipl on its own: the per-layer inputs of `rows` tokens from the raw per_layer_model_proj output
// (pmp [rows][n_layer*ple]) and the tokens' rows of per_layer_token_embd (pte: n_tok plain q4_0 rows of n_layer*ple).
extern "C" int lg_hip_ple_inputs(const float *pmp, const float *proj_norm, const void *pte, int n_tok, const int32_t *toks,
                                 int rows, int n_layer, int ple, int E, float eps, float *out) {
    if (!pmp || !proj_norm || !pte || !toks || !out) return fail(-1, "ple_inputs: null argument");
    if (rows < 1 || rows > LG_HIP_MAX_ROWS || n_layer < 1 || ple < 32 || ple % 32 || ple > 256 || n_tok < 1 || E < 1)
        return fail(-2, "ple_inputs: rows %d (1..%d), n_layer %d, ple %d (a multiple of 32 up to 256), %d token rows", rows, LG_HIP_MAX_ROWS, n_layer, ple, n_tok);
    for (int j = 0; j < rows; ++j) if (toks[j] < 0 || toks[j] >= n_tok) return fail(-2, "ple_inputs: token %d of row %d (table of %d rows)", toks[j], j, n_tok);
    if (lg_hip_device_count() < 1) return fail(-3, "ple_inputs: no HIP device");
    Scratch sc;
    const size_t w = (size_t)n_layer * ple, tb = (size_t)n_tok * (w / 32 * 18);
    float *dp, *dn; uint8_t *dt; int32_t *dk; StepCtl *ctl;
    if (sc.get(&dp, rows * w) || sc.get(&dn, (size_t)ple) || sc.get(&dt, tb) || sc.get(&dk, (size_t)rows) || sc.get(&ctl, 1)) return -7;
    HIP_TRY(hipMemcpy(dp, pmp, rows * w * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dn, proj_norm, (size_t)ple * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dt, pte, tb, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dk, toks, (size_t)rows * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemset(ctl, 0, sizeof(StepCtl)));
    IplArgs i{ dp, ple, n_layer, rows, dn, dt, dk, 1.0f / sqrtf((float)E), sqrtf((float)ple), 1.0f / sqrtf(2.0f), eps };
    hipLaunchKernelGGL(lg_k_ipl, dim3(n_layer, rows), dim3(64), 0, nullptr, i, ctl);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(out, dp, rows * w * 4, hipMemcpyDeviceToHost));
    return 0;
}

// the two launches of an isolated attention: tile partials, then the ordered merge
// (the same choice of kernels as a verify step makes: many (tile, kv head) pairs -> one workgroup per pair serves all
// rows; many tiles per row -> the merge is cut by dims)
template <int M>
static int enqueue_attention(hipStream_t st, const AttnArgs &a_in, const MergeArgs &g, StepCtl *ctl, int tiles, int pos, size_t lds) {
    AttnArgs a = a_in;
    a.gx = tiles; a.gz = M;                               // the grid of lg_k_attn, which reads it from its arguments
    if (attention_rows_shared(M, tiles, a.nkv, a.hd, a.seq, pos + M)) {
        if constexpr (M > 1) {
            const int units = M * (a.H / a.nkv);
            const bool few = attention_rows_few(tiles, units, a.nkv, false);
            const dim3 grid(few ? tiles : attention_rows_wgs(tiles, units, a.nkv), a.nkv);
            a.gx = (int)grid.x;
            int rc = 0;
#define ATTN_ROWS(HD) do { const size_t l2 = few ? AttnFewGeo<HD>::bytes(units, false) : AttnRowsGeo<HD>::bytes(units, false); \
    if (few) { if (!(rc = set_lds(lg_k_attn_few<M, HD>, l2))) hipLaunchKernelGGL((lg_k_attn_few<M, HD>), grid, dim3(LG_WG), l2, st, ctl, LG_ATTN_FIELDS(LG_XA, a) 0); } \
    else if (!(rc = set_lds(lg_k_attn_rows<M, HD>, l2))) hipLaunchKernelGGL((lg_k_attn_rows<M, HD>), grid, dim3(LG_WG), l2, st, ctl, LG_ATTN_FIELDS(LG_XA, a) 0); } while (0)
            if (a.hd == 256)      ATTN_ROWS(256);
            else if (a.hd == 128) ATTN_ROWS(128);
            else                  ATTN_ROWS(64);
#undef ATTN_ROWS
            if (rc) return rc;
        }
    } else hipLaunchKernelGGL((lg_k_attn<false, 1>), dim3(tiles, a.nkv, M), dim3(LG_WG), lds, st, ctl, LG_ATTN_FIELDS(LG_XA, a) 0);
    if (tiles >= 128 && a.hd % 64 == 0) {
#define GO(k, grid, block) hipLaunchKernelGGL(HIP_KERNEL_NAME(k), grid, block, 0, st, ctl, LG_MERGE_FIELDS(LG_XA, g) 0)
        MERGE_SPLIT(M, GO, a.H, a.hd, tiles);
#undef GO
    } else hipLaunchKernelGGL((lg_k_attn_merge<M>), dim3(a.H, M), dim3(LG_WG), 0, st, ctl, LG_MERGE_FIELDS(LG_XA, g) 0);
    return 0;
}

template <int M>
static int attention_rows(hipStream_t st, AttnArgs a, MergeArgs g, StepCtl *ctl, int tiles, int pos, int repeats, float *kernel_ms) {
    const size_t lds = attn_lds(a.H / a.nkv, a.hd, false);
    int rc = set_lds(lg_k_attn<false, 1>, lds);
    if (rc) return rc;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    auto body = [&]() -> int {
        HIP_TRY(hipEventCreate(&e0)); HIP_TRY(hipEventCreate(&e1));
        for (int r = 0; r < repeats + 1; ++r) {
            if (r == 1) HIP_TRY(hipEventRecord(e0, st));
            const int erc = enqueue_attention<M>(st, a, g, ctl, tiles, pos, lds);
            if (erc) return erc;
        }
        HIP_TRY(hipEventRecord(e1, st));
        HIP_TRY(hipStreamSynchronize(st));
        HIP_TRY(hipGetLastError());
        float t = 0;
        if (repeats > 0) HIP_TRY(hipEventElapsedTime(&t, e0, e1));
        if (kernel_ms) *kernel_ms = repeats > 0 ? t / repeats : 0.0f;
        return 0;
    };
    rc = body();
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    return rc;
}

extern "C" int lg_hip_attention(const float *q, const uint16_t *kc, const uint16_t *vc, int rows, int n_head, int n_head_kv,
                                int hd, int seq, int window, int pos, float *out, int repeats, float *kernel_ms) {
    if (!q || !kc || !vc || !out) return fail(-1, "attention: null argument");
    if (rows < 1 || rows > LG_HIP_MAX_ROWS || n_head_kv < 1 || n_head % n_head_kv || n_head / n_head_kv > 8 ||
        (hd != 64 && hd != 128 && hd != 256 && hd != 512) || pos < 0 || seq < 1)
        return fail(-2, "attention: unsupported shape");
    if (window > 0 ? seq < window + rows - 1 && seq < pos + rows : seq < pos + rows)
        return fail(-2, "attention: a cache of %d rows cannot hold the keys of positions up to %d", seq, pos + rows - 1);
    if (lg_hip_device_count() < 1) return fail(-3, "attention: no HIP device");
    const int kd = n_head_kv * hd, qd = n_head * hd;
    const int start0 = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    const int tiles = ((pos + rows - 1) >> 5) - (start0 >> 5) + 1;
    Scratch sc;
    float *dq, *dpm, *dpl, *dpacc, *dxf; uint16_t *dk, *dv; int8_t *dxq; StepCtl *ctl;
    const size_t slots = (size_t)rows * n_head * tiles;
    if (sc.get(&dq, (size_t)rows * qd) || sc.get(&dk, (size_t)seq * kd) || sc.get(&dv, (size_t)seq * kd) ||
        sc.get(&dpm, slots) || sc.get(&dpl, slots) || sc.get(&dpacc, slots * hd) || sc.get(&dxf, (size_t)rows * qd) ||
        sc.get(&dxq, (size_t)rows * qd * 5 / 4) || sc.get(&ctl, (size_t)1)) return -7;
    HIP_TRY(hipMemcpy(dq, q, (size_t)rows * qd * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dk, kc, (size_t)seq * kd * 2, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dv, vc, (size_t)seq * kd * 2, hipMemcpyHostToDevice));
    StepCtl c{ pos, 0, 0, 0, 0 };
    HIP_TRY(hipMemcpy(ctl, &c, sizeof c, hipMemcpyHostToDevice));
    AttnArgs a{};
    a.q = dq; a.H = n_head; a.nkv = n_head_kv; a.hd = hd;
    a.kc = dk; a.vc = dv; a.seq = seq; a.kv_dim = kd; a.window = window;
    a.pm = dpm; a.pl = dpl; a.pacc = dpacc; a.tiles_max = tiles;
    MergeArgs g{ dpm, dpl, dpacc, tiles, n_head, hd, window, 0, dxq, dxf };
    hipStream_t st;
    HIP_TRY(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    int rc = 0;
    switch (rows) {
#define CASE(M) case M: rc = attention_rows<M>(st, a, g, ctl, tiles, pos, repeats, kernel_ms); break;
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
    }
    (void)hipStreamDestroy(st);
    if (rc) return rc;
    HIP_TRY(hipMemcpy(out, dxf, (size_t)rows * qd * 4, hipMemcpyDeviceToHost));
    return 0;
}

// ---- attention for callers that cannot allocate ---------------------------------------------------
// lg_hip_attention with every buffer given by the caller as DEVICE memory, and the kernels' own working
// memory (step state, tile partials, the q8 copy of the result that the merge kernel also writes) in a
// static device array instead of hipMalloc'ed scratch: nothing is allocated or freed, the launches are
// left on the caller's stream and the call returns without waiting.
#define LG_NOALLOC_BYTES (8u << 20)
#define LG_NOALLOC_DEVICES 16
static __device__ __align__(256) unsigned char lg_noalloc_scratch[LG_NOALLOC_BYTES];
// the array's device address, asked once per device (each device holds its own copy at its own address)
static unsigned char *g_noalloc_ptr[LG_NOALLOC_DEVICES];

static size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }

extern "C" size_t lg_hip_attention_noalloc_limit(void) { return LG_NOALLOC_BYTES; }

// Everything the entry point needs from the runtime besides launches, for the current device: the array's address
// and, for every kernel it may launch with more than the default dynamic LDS, the limit raised to the most any
// accepted shape asks for.  Neither call is legal while a stream is being captured, so a capturing caller calls
// this first; the entry point calls it by itself on its first use on a device.
template <int M>
static int noalloc_raise_rows() {
    int rc = set_lds(lg_k_attn_rows<M, 256>, AttnRowsGeo<256>::bytes(M * 8, false));
    if (!rc) rc = set_lds(lg_k_attn_rows<M, 128>, AttnRowsGeo<128>::bytes(M * 8, false));
    if (!rc) rc = set_lds(lg_k_attn_rows<M, 64>, AttnRowsGeo<64>::bytes(M * 8, false));
    return rc;
}
extern "C" int lg_hip_attention_noalloc_init(void) {
    int dev = -1;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= LG_NOALLOC_DEVICES) return fail(-3, "attention_noalloc: device %d (0..%d are served)", dev, LG_NOALLOC_DEVICES - 1);
    if (g_noalloc_ptr[dev]) return 0;
    int rc = set_lds(lg_k_attn<false, 1>, attn_lds(8, 512, false));
    if (!rc) rc = noalloc_raise_rows<2>();
    if (!rc) rc = noalloc_raise_rows<3>();
    if (!rc) rc = noalloc_raise_rows<4>();
    if (!rc) rc = noalloc_raise_rows<5>();
    if (!rc) rc = noalloc_raise_rows<6>();
    if (!rc) rc = noalloc_raise_rows<7>();
    if (!rc) rc = noalloc_raise_rows<8>();
    if (rc) return rc;
    void *p = nullptr;
    HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(lg_noalloc_scratch)));
    if (!p) return fail(-3, "attention_noalloc: the working array has no address on device %d", dev);
    g_noalloc_ptr[dev] = (unsigned char *)p;
    return 0;
}

extern "C" int lg_hip_attention_noalloc(const float *d_q, const uint16_t *d_kc, const uint16_t *d_vc, int rows, int n_head,
                                        int n_head_kv, int hd, int seq, int window, int pos, float *d_out, void *stream) {
    if (!d_q || !d_kc || !d_vc || !d_out) return fail(-1, "attention_noalloc: null argument");
    if (rows < 1 || rows > LG_HIP_MAX_ROWS || n_head_kv < 1 || n_head % n_head_kv || n_head / n_head_kv > 8 ||
        (hd != 64 && hd != 128 && hd != 256 && hd != 512) || pos < 0 || seq < 1)
        return fail(-2, "attention_noalloc: unsupported shape");
    if (window > 0 ? seq < window + rows - 1 && seq < pos + rows : seq < pos + rows)
        return fail(-2, "attention_noalloc: a cache of %d rows cannot hold the keys of positions up to %d", seq, pos + rows - 1);
    const int qd = n_head * hd;
    const int start0 = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    const int tiles = ((pos + rows - 1) >> 5) - (start0 >> 5) + 1;
    const size_t slots = (size_t)rows * n_head * tiles;
    const size_t o_pm = 256, o_pl = o_pm + up256(slots * 4), o_pacc = o_pl + up256(slots * 4),
                 o_xq = o_pacc + up256(slots * hd * 4), need = o_xq + up256((size_t)rows * qd * 5 / 4);
    if (need > LG_NOALLOC_BYTES)
        return fail(-2, "attention_noalloc: %d rows x %d heads x %d key tiles of %d need %zu bytes of working memory; the built-in array holds %u",
                    rows, n_head, tiles, hd, need, LG_NOALLOC_BYTES);
    int dev = -1;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= LG_NOALLOC_DEVICES) return fail(-3, "attention_noalloc: device %d (0..%d are served)", dev, LG_NOALLOC_DEVICES - 1);
    if (!g_noalloc_ptr[dev]) {
        const int irc = lg_hip_attention_noalloc_init();
        if (irc) return irc;
    }
    unsigned char *base = g_noalloc_ptr[dev];
    StepCtl *ctl = (StepCtl *)base;
    float *dpm = (float *)(base + o_pm), *dpl = (float *)(base + o_pl), *dpacc = (float *)(base + o_pacc);
    int8_t *dxq = (int8_t *)(base + o_xq);
    AttnArgs a{};
    a.q = d_q; a.H = n_head; a.nkv = n_head_kv; a.hd = hd;
    a.kc = d_kc; a.vc = d_vc; a.seq = seq; a.kv_dim = n_head_kv * hd; a.window = window;
    a.pm = dpm; a.pl = dpl; a.pacc = dpacc; a.tiles_max = tiles;
    MergeArgs g{ dpm, dpl, dpacc, tiles, n_head, hd, window, 0, dxq, d_out };
    const size_t lds = attn_lds(n_head / n_head_kv, hd, false);
    int rc = set_lds(lg_k_attn<false, 1>, lds);
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    // every tile slot that the merge reads is written by the tile kernel of the same call, so nothing has to be
    // cleared; only the step state is set, by a kernel (a caller may be capturing this stream)
    hipLaunchKernelGGL(lg_k_set_ctl, dim3(1), dim3(1), 0, st, ctl, pos, true);
    switch (rows) {
#define CASE(M) case M: rc = enqueue_attention<M>(st, a, g, ctl, tiles, pos, lds); break;
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
    }
    if (rc) return rc;
    HIP_TRY(hipGetLastError());
    return 0;
}

// ---- launch floor -----------------------------------------------------------------------------------
// What a chain of dependent kernels costs before it does any work: a captured graph of n kernels in a row, each
// empty (mode 0) or reading the 64 bytes its predecessor wrote and writing 64 for its successor (mode 1).
__global__ void lg_k_floor_empty() {}
__global__ void lg_k_floor_chain(const int *src, int *dst) {
    if (blockIdx.x == 0 && threadIdx.x < 16) dst[threadIdx.x] = src[threadIdx.x] + 1;
}
extern "C" int lg_hip_launch_floor(int n_kernels, int mode, int grid, int block, int replays, float *us_per_kernel) {
    if (n_kernels < 1 || n_kernels > 4096 || mode < 0 || mode > 1 || grid < 1 || grid > 65536 || block < 1 || block > 1024 ||
        replays < 1 || !us_per_kernel) return fail(-2, "launch_floor: bad argument");
    if (lg_hip_device_count() < 1) return fail(-3, "launch_floor: no HIP device");
    hipStream_t st = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int *a = nullptr, *b = nullptr;
    auto body = [&]() -> int {
        HIP_TRY(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
        HIP_TRY(hipMalloc((void **)&a, 256)); HIP_TRY(hipMalloc((void **)&b, 256));
        HIP_TRY(hipMemset(a, 0, 256)); HIP_TRY(hipMemset(b, 0, 256));
        HIP_TRY(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        for (int i = 0; i < n_kernels; ++i) {
            if (mode == 0) hipLaunchKernelGGL(lg_k_floor_empty, dim3(grid), dim3(block), 0, st);
            else hipLaunchKernelGGL(lg_k_floor_chain, dim3(grid), dim3(block), 0, st, (i & 1) ? b : a, (i & 1) ? a : b);
        }
        HIP_TRY(hipStreamEndCapture(st, &graph));
        HIP_TRY(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
        HIP_TRY(hipEventCreate(&e0)); HIP_TRY(hipEventCreate(&e1));
        HIP_TRY(hipGraphLaunch(exec, st));                   // warm-up
        HIP_TRY(hipStreamSynchronize(st));
        HIP_TRY(hipEventRecord(e0, st));
        for (int r = 0; r < replays; ++r) HIP_TRY(hipGraphLaunch(exec, st));
        HIP_TRY(hipEventRecord(e1, st));
        HIP_TRY(hipStreamSynchronize(st));
        float ms = 0;
        HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
        *us_per_kernel = ms * 1e3f / ((float)replays * (float)n_kernels);
        return 0;
    };
    const int rc = body();
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (a) (void)hipFree(a);
    if (b) (void)hipFree(b);
    if (st) (void)hipStreamDestroy(st);
    return rc;
}

// ---- XCD placement and hand-over probes ------------------------------------------------------------
// Which XCD every workgroup of a grid x block launch (with lds_bytes of dynamic LDS) ran on, `launches` times in a
// row on one stream: xcc / hwid receive [launches][grid] values (XCC_ID and HW_ID registers).
__global__ void lg_k_xcd_map_lds(int32_t *xcc, int32_t *hwid) {
    extern __shared__ unsigned char smem[];
    if (threadIdx.x == 0) { smem[0] = 1; xcc[blockIdx.x] = lg_xcc_id(); hwid[blockIdx.x] = (int32_t)lg_hw_id(); }
}
extern "C" int lg_hip_xcd_map(int grid, int block, int lds_bytes, int launches, int32_t *xcc, int32_t *hwid) {
    if (grid < 1 || grid > 65536 || block < 1 || block > 1024 || lds_bytes < 0 || lds_bytes > 160 * 1024 || launches < 1 || !xcc || !hwid)
        return fail(-2, "xcd_map: bad argument");
    if (lg_hip_device_count() < 1) return fail(-3, "xcd_map: no HIP device");
    Scratch sc;
    int32_t *dx, *dh;
    const size_t n = (size_t)grid * launches;
    if (sc.get(&dx, n) || sc.get(&dh, n)) return -7;
    if (lds_bytes > 48 * 1024) HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(lg_k_xcd_map_lds), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes));
    for (int l = 0; l < launches; ++l)
        hipLaunchKernelGGL(lg_k_xcd_map_lds, dim3(grid), dim3(block), (size_t)lds_bytes, nullptr, dx + (size_t)l * grid, dh + (size_t)l * grid);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(xcc, dx, n * 4, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(hwid, dh, n * 4, hipMemcpyDeviceToHost));
    return 0;
}

// One hand-over experiment (lg_k_xcd_handover): n workgroups of a 256-workgroup launch, chosen by set_mode / sel,
// exchange `bytes` each per round through flags; store_scope / load_scope 0..3 = plain, sc0, sc1, sc0 sc1.
// res receives [n][4] = { ticks, mismatching words, polls given up, XCD id }; *tick_ns the length of a tick.
extern "C" int lg_hip_xcd_handover(int set_mode, int sel, int n, int store_scope, int load_scope, int bytes, int rounds,
                                   int32_t *res, float *tick_ns) {
    if (set_mode < 0 || set_mode > 1 || n < 2 || n > 32 || sel < 0 || (set_mode == 0 ? sel >= LG_XCDS : (sel + 1) * n > 256) ||
        store_scope < 0 || store_scope > 3 || load_scope < 0 || load_scope > 3 || bytes < 0 || bytes % 4 || bytes > (1 << 20) ||
        rounds < 1 || rounds > 100000 || !res || !tick_ns)
        return fail(-2, "xcd_handover: bad argument");
    if (lg_hip_device_count() < 1) return fail(-3, "xcd_handover: no HIP device");
    int dev = 0, khz = 0;
    HIP_TRY(hipGetDevice(&dev));
    HIP_TRY(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    *tick_ns = khz > 0 ? 1e6f / (float)khz : 10.0f;
    Scratch sc;
    XcdProbeArgs a{};
    a.n = n; a.words = bytes / 4; a.rounds = rounds; a.set_mode = set_mode; a.sel = sel; a.spin_limit = 4000;
    if (sc.get(&a.flags, (size_t)64) || sc.get(&a.data, (size_t)2 * n * (a.words ? a.words : 1)) || sc.get(&a.res, (size_t)n * 4)) return -7;
    HIP_TRY(hipMemset(a.flags, 0, 256));
    HIP_TRY(hipMemset(a.res, 0xFF, (size_t)n * 16));
    std::unique_lock<std::mutex> turn;
    { const int rc = take_turn_alone(turn); if (rc) return rc; }
    HIP_TRY(hipDeviceSynchronize());
    const int combo = store_scope * 4 + load_scope;
    switch (combo) {
#define CASE(S, L) case S * 4 + L: hipLaunchKernelGGL((lg_k_xcd_handover<S, L>), dim3(256), dim3(256), 0, nullptr, a); break;
        CASE(0, 0) CASE(0, 1) CASE(0, 2) CASE(0, 3) CASE(1, 0) CASE(1, 1) CASE(1, 2) CASE(1, 3)
        CASE(2, 0) CASE(2, 1) CASE(2, 2) CASE(2, 3) CASE(3, 0) CASE(3, 1) CASE(3, 2) CASE(3, 3)
#undef CASE
    }
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(res, a.res, (size_t)n * 16, hipMemcpyDeviceToHost));
    return 0;
}

// ---- device functions on their own (tests) ----------------------------------------------------------
__global__ void lg_k_math(int fn, const float *x, size_t n, float *out) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        out[i] = fn == 0 ? lg_rcp_exact(x[i]) : fn == 1 ? lg_inv_scale(x[i]) : fn == 2 ? lg_gelu_d(x[i]) : lg_gelu(x[i]);
}
extern "C" int lg_hip_math(int fn, const float *x, size_t n, float *out) {
    if (!x || !out || n < 1) return fail(-1, "math: null argument");
    if (fn < 0 || fn > 3) return fail(-2, "math: no function %d", fn);
    if (lg_hip_device_count() < 1) return fail(-3, "math: no HIP device");
    Scratch sc;
    float *dx, *dout;
    if (sc.get(&dx, n) || sc.get(&dout, n)) return -7;
    HIP_TRY(hipMemcpy(dx, x, n * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(lg_k_math, dim3(2048), dim3(LG_WG), 0, nullptr, fn, dx, n, dout);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(out, dout, n * 4, hipMemcpyDeviceToHost));
    return 0;
}

// ---- the XCD-partitioned feed-forward half on its own (tests, timing) ------------------------------
// x_out = x + rmsnorm(dout) * w_post; h = rmsnorm(x_out) * w_pre; act = gelu(gate . q8(h)) * (up . q8(h));
// out = down . q8(act): lg_k_ffn_xcd on host data, the 8 slabs added here in tree order.
extern "C" int lg_hip_down_m(const float *act, const void *down, int rows, int E, int FF, int join, float *out, int repeats, float *kernel_ms) {
    if (!act || !down || !out) return fail(-1, "down_m: null argument");
    const DownMGeo g = lg_down_m_geo(E, FF);
    if (rows < 4 || rows > LG_HIP_MAX_ROWS || !down_m_shape(g)) return fail(-2, "down_m: rows %d (4..%d), E %d, FF %d: no instantiation for this shape", rows, LG_HIP_MAX_ROWS, E, FF);
    if (lg_hip_device_count() < 1) return fail(-3, "down_m: no HIP device");
    Scratch sc;
    std::vector<uint8_t> stage(256 * g.wg_bytes);
    uint8_t *dw; float *dx, *dslabs; uint32_t *dq; DownMSync *dsync; StepCtl *ctl;
    const size_t n = (size_t)rows * E;
    if (sc.get(&dw, 256 * g.wg_bytes) || sc.get(&dx, (size_t)rows * FF) || sc.get(&dslabs, 4 * n) || sc.get(&dq, (size_t)(FF / 32) * LG_MU_DWORDS) ||
        sc.get(&dsync, (size_t)1) || sc.get(&ctl, (size_t)1)) return -7;
    HIP_TRY(hipMemset(dsync, 0, sizeof(DownMSync)));
    HIP_TRY(hipMemset(ctl, 0, sizeof(StepCtl)));
    pack_down_m((const uint8_t *)down, g, stage.data());
    HIP_TRY(hipMemcpy(dw, stage.data(), 256 * g.wg_bytes, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dx, act, (size_t)rows * FF * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemset(dq, 0, (size_t)(FF / 32) * LG_MU_DWORDS * 4));
    std::unique_lock<std::mutex> turn;
    { const int rc = take_turn_alone(turn); if (rc) return rc; }
    hipStream_t st;
    HIP_TRY(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    lg_hip_model shim;
    shim.stream = st;
    Launcher lx{ &shim, false };
    DownMArgs a{ dw, dq, dslabs, E, FF, join ? dsync : nullptr, ctl, 1 << 16, 0 };
    hipEvent_t e0 = nullptr, e1 = nullptr;
    auto body = [&]() -> int {
        HIP_TRY(hipEventCreate(&e0)); HIP_TRY(hipEventCreate(&e1));
        hipLaunchKernelGGL(lg_k_quant_mu, dim3((rows * (FF / 32) * 8 + LG_WG - 1) / LG_WG), dim3(LG_WG), 0, st, dx, rows, FF, dq);
        for (int r = 0; r < repeats + 1 && !lx.rc; ++r) {
            if (r == 1) HIP_TRY(hipEventRecord(e0, st));
            a.seq = r;
            switch (rows) {
#define CASE(M) case M: launch_down_m<M>(lx, a); break;
                CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
            }
        }
        if (lx.rc) return lx.rc;
        HIP_TRY(hipEventRecord(e1, st));
        HIP_TRY(hipStreamSynchronize(st));
        HIP_TRY(hipGetLastError());
        float t = 0;
        if (repeats > 0) HIP_TRY(hipEventElapsedTime(&t, e0, e1));
        if (kernel_ms) *kernel_ms = repeats > 0 ? t / repeats : 0.0f;
        return 0;
    };
    int rc = body();
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipStreamDestroy(st);
    if (rc) return rc;
    std::vector<float> slabs(4 * n);
    HIP_TRY(hipMemcpy(slabs.data(), dslabs, 4 * n * 4, hipMemcpyDeviceToHost));
    StepCtl c;
    HIP_TRY(hipMemcpy(&c, ctl, sizeof c, hipMemcpyDeviceToHost));
    { const int erc = step_err("down_m", c.err); if (erc) return erc; }
    for (size_t i = 0; i < n; ++i) out[i] = join ? slabs[i] : (slabs[i] + slabs[n + i]) + (slabs[2 * n + i] + slabs[3 * n + i]);    // (what the consumer kernel does)
    return 0;
}

// Gate/up + GeGLU of a verify block in isolation (tests): `rows` float rows of E are quantized as the step's row
// kernel does it (the q8 order of the kernel that follows: lg_k_geglu_t for 1..3 rows, lg_k_geglu_m for 4..8), then
// the kernel runs on gate / up (FF plain q4_0 rows of E each) and the q8 of gelu(gate) * up comes back in natural order.
extern "C" int lg_hip_gate_up_geglu(const float *x, const void *gate, const void *up, int rows, int E, int FF,
                                    int8_t *aq, float *ad, int32_t *asum, int repeats, float *kernel_ms) {
    if (!x || !gate || !up) return fail(-1, "gate_up_geglu: null argument");
    if (rows < 1 || rows > LG_HIP_MAX_ROWS || E < 256 || E % 256 || E > 4096 || FF < 32 || FF % 32 || lg_segments(E) != 8)
        return fail(-2, "gate_up_geglu: rows %d (1..%d), E %d (a multiple of 256 up to 4096), FF %d (a multiple of 32)", rows, LG_HIP_MAX_ROWS, E, FF);
    if (lg_hip_device_count() < 1) return fail(-3, "gate_up_geglu: no HIP device");
    const size_t rb = (size_t)(E / 32) * 18;
    std::vector<const uint8_t *> wrows;
    for (int t = 0; t < FF / 32; ++t) {
        for (int r = 0; r < 32; ++r) wrows.push_back((const uint8_t *)gate + ((size_t)t * 32 + r) * rb);
        for (int r = 0; r < 32; ++r) wrows.push_back((const uint8_t *)up + ((size_t)t * 32 + r) * rb);
    }
    std::vector<uint8_t> stage(lg_hip_repacked_bytes(E, 2 * FF));
    if (stage.empty()) return fail(-2, "gate_up_geglu: cannot tile a %d x %d matrix", 2 * FF, E);
    repack_rowblocks(wrows.data(), E, 2 * FF, stage.data());
    Scratch sc;
    uint8_t *dw; float *dx; int8_t *dq, *dgq; StepCtl *ctl;
    const size_t qbytes = (size_t)(E / 32) * LG_MU_DWORDS * 4 + (size_t)rows * E * 2;     // (room for either block order)
    if (sc.get(&dw, stage.size()) || sc.get(&dx, (size_t)rows * E) || sc.get(&dq, qbytes) || sc.get(&dgq, (size_t)rows * FF * 5 / 4) || sc.get(&ctl, (size_t)1)) return -7;
    HIP_TRY(hipMemcpy(dw, stage.data(), stage.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dx, x, (size_t)rows * E * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemset(dq, 0, qbytes));                        // (row slots past the block are read as operand rows of the matrix cores)
    HIP_TRY(hipMemset(ctl, 0, sizeof(StepCtl)));
    hipStream_t st;
    HIP_TRY(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    RowArgs s{};
    s.x = dx; s.dparts = 1; s.q = dq; s.E = E; s.eps = 1e-6f; s.q_units = rows >= 4 ? 2 : 1;
    GegluArgs a{ dw, E, FF, dq, dgq, 0 };
    hipEvent_t e0 = nullptr, e1 = nullptr;
    auto body = [&]() -> int {
        HIP_TRY(hipEventCreate(&e0)); HIP_TRY(hipEventCreate(&e1));
        int rc = 0;
        auto run = [&](auto tag) {
            constexpr int M = decltype(tag)::value;
            rows_isolated<M>(st, s, ctl);
            for (int r = 0; r < repeats + 1; ++r) {
                if (r == 1) (void)hipEventRecord(e0, st);
                if constexpr (M >= 4) {
                    const size_t lds = (size_t)(E / 32) * LG_MU_DWORDS * 4;
                    rc = set_lds(lg_k_geglu_m<M>, lds);
                    if (rc) return;
                    hipLaunchKernelGGL((lg_k_geglu_m<M>), dim3(FF / 32), dim3(512), lds, st, LG_GEGLU_FIELDS(LG_XA, a) 0);
                } else hipLaunchKernelGGL((lg_k_geglu_t<M>), dim3(FF / 32), dim3(512), 0, st, LG_GEGLU_FIELDS(LG_XA, a) 0);
            }
        };
        switch (rows) {
#define CASE(M) case M: run(std::integral_constant<int, M>{}); break;
            CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
        }
        if (rc) return rc;
        HIP_TRY(hipEventRecord(e1, st));
        HIP_TRY(hipStreamSynchronize(st));
        HIP_TRY(hipGetLastError());
        float t = 0;
        if (repeats > 0) HIP_TRY(hipEventElapsedTime(&t, e0, e1));
        if (kernel_ms) *kernel_ms = repeats > 0 ? t / repeats : 0.0f;
        return 0;
    };
    int rc = body();
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipStreamDestroy(st);
    if (rc) return rc;
    return read_back_q8(dgq, rows, FF, aq, ad, asum);
}

extern "C" int lg_hip_ffn_xcd(const float *x, const float *dout, const float *w_post, const float *w_pre,
                              const void *gate, const void *up, const void *down, int rows, int E, int FF, float eps,
                              float *x_out, float *act, float *out, int repeats, float *kernel_ms, int flush_mb, int delay_w, int64_t *stamps) {
    if (!x || !dout || !w_post || !w_pre || !gate || !up || !down) return fail(-1, "ffn_xcd: null input");
    const XffnGeo g = lg_xffn_geo(E, FF);
    const int cls = xffn_class_of(g);
    if (rows < 4 || rows > LG_HIP_MAX_ROWS || cls < 0) return fail(-2, "ffn_xcd: rows %d (4..%d), E %d, FF %d: no instantiation for this shape", rows, LG_HIP_MAX_ROWS, E, FF);
    if (lg_hip_device_count() < 1) return fail(-3, "ffn_xcd: no HIP device");
    if (cu_count() != LG_XCDS * LG_XCD_WGS) return fail(-3, "ffn_xcd: the kernel needs %d compute units in %d XCDs, this device has %d", LG_XCDS * LG_XCD_WGS, LG_XCDS, cu_count());
    Scratch sc;
    std::vector<uint8_t> stage(256 * (g.gu_bytes > g.dn_bytes ? g.gu_bytes : g.dn_bytes));
    uint8_t *dgu, *ddn; float *dx, *dd, *dwp, *dwr, *dxo, *dslabs, *dact; uint32_t *dxq; XcdSync *dsync; StepCtl *ctl;
    const size_t n = (size_t)rows * E;
    if (sc.get(&dgu, 256 * g.gu_bytes) || sc.get(&ddn, 256 * g.dn_bytes) || sc.get(&dx, n) || sc.get(&dd, n) || sc.get(&dwp, (size_t)E) ||
        sc.get(&dwr, (size_t)E) || sc.get(&dxo, n) || sc.get(&dslabs, LG_XCDS * n) || sc.get(&dact, (size_t)LG_XCDS * rows * g.C) ||
        sc.get(&dxq, (size_t)LG_XCDS * g.nb * LG_MU_DWORDS) || sc.get(&dsync, (size_t)1) || sc.get(&ctl, (size_t)1)) return -7;
    xffn_pack_gu((const uint8_t *)gate, (const uint8_t *)up, g, stage.data());
    HIP_TRY(hipMemcpy(dgu, stage.data(), 256 * g.gu_bytes, hipMemcpyHostToDevice));
    xffn_pack_dn((const uint8_t *)down, g, stage.data());
    HIP_TRY(hipMemcpy(ddn, stage.data(), 256 * g.dn_bytes, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dx, x, n * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dd, dout, n * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dwp, w_post, (size_t)E * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dwr, w_pre, (size_t)E * 4, hipMemcpyHostToDevice));
    HIP_TRY(hipMemset(dsync, 0, sizeof(XcdSync)));
    HIP_TRY(hipMemset(dxq, 0, (size_t)LG_XCDS * g.nb * LG_MU_DWORDS * 4));
    HIP_TRY(hipMemset(ctl, 0, sizeof(StepCtl)));
    std::unique_lock<std::mutex> turn;
    { const int rc = take_turn_alone(turn); if (rc) return rc; }
    hipStream_t st;
    HIP_TRY(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    lg_hip_model shim;
    shim.stream = st;
    Launcher lx{ &shim, false };
    // measurement runs: something else streams through the caches between two launches (the step's weights never
    // come from a cache), and every workgroup records the device clock at its phase boundaries
    unsigned char *dflush = nullptr;
    unsigned long long *dstamps = nullptr;
    if (flush_mb > 0 && sc.get(&dflush, (size_t)flush_mb << 20)) return -7;
    if (stamps && sc.get(&dstamps, (size_t)512 * LG_XFFN_STAMPS)) return -7;
    if (dstamps) HIP_TRY(hipMemset(dstamps, 0, (size_t)512 * LG_XFFN_STAMPS * 8));
    XffnArgs f{ dgu, ddn, dx, dd, dwp, dwr, dxo, dslabs, dxq, dact, dsync, ctl, E, FF, eps, 1 << 16, 0, delay_w, dstamps };
    hipEvent_t e0 = nullptr, e1 = nullptr;
    auto body = [&]() -> int {
        HIP_TRY(hipEventCreate(&e0)); HIP_TRY(hipEventCreate(&e1));
        for (int r = 0; r < repeats + 1 && !lx.rc; ++r) {
            if (r == 1) HIP_TRY(hipEventRecord(e0, st));
            if (dflush) HIP_TRY(hipMemsetAsync(dflush, r, (size_t)flush_mb << 20, st));
            f.seq = r;
            switch (rows) {
#define CASE(M) case M: launch_xffn<M>(lx, f, cls); break;
                CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
            }
        }
        if (lx.rc) return lx.rc;
        HIP_TRY(hipEventRecord(e1, st));
        HIP_TRY(hipStreamSynchronize(st));
        HIP_TRY(hipGetLastError());
        float t = 0;
        if (repeats > 0) HIP_TRY(hipEventElapsedTime(&t, e0, e1));
        if (kernel_ms) *kernel_ms = repeats > 0 ? t / repeats : 0.0f;
        return 0;
    };
    int rc = body();
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipStreamDestroy(st);
    if (rc) return rc;
    StepCtl c;
    HIP_TRY(hipMemcpy(&c, ctl, sizeof c, hipMemcpyDeviceToHost));
    if (c.err) return fail(-9, "ffn_xcd: the kernel reported %s%s (err 0x%x)", (c.err & LG_XFFN_ERR_PLACE) ? "a workgroup on an unexpected XCD " : "",
                           (c.err & LG_XFFN_ERR_WAIT) ? "a hand-over that was given up" : "", c.err);
    if (stamps) HIP_TRY(hipMemcpy(stamps, dstamps, (size_t)512 * LG_XFFN_STAMPS * 8, hipMemcpyDeviceToHost));
    if (x_out) HIP_TRY(hipMemcpy(x_out, dxo, n * 4, hipMemcpyDeviceToHost));
    if (act) {                                            // [rows][FF] from the 8 per-XCD pieces [rows][FF/8]
        std::vector<float> pieces((size_t)LG_XCDS * rows * g.C);
        HIP_TRY(hipMemcpy(pieces.data(), dact, pieces.size() * 4, hipMemcpyDeviceToHost));
        for (int xc = 0; xc < LG_XCDS; ++xc)
            for (int j = 0; j < rows; ++j)
                memcpy(act + (size_t)j * FF + (size_t)xc * g.C, pieces.data() + ((size_t)xc * rows + j) * g.C, (size_t)g.C * 4);
    }
    if (out) {
        std::vector<float> p(LG_XCDS * n);
        HIP_TRY(hipMemcpy(p.data(), dslabs, p.size() * 4, hipMemcpyDeviceToHost));
        for (size_t i = 0; i < n; ++i)
            out[i] = ((p[i] + p[n + i]) + (p[2 * n + i] + p[3 * n + i])) + ((p[4 * n + i] + p[5 * n + i]) + (p[6 * n + i] + p[7 * n + i]));
    }
    return 0;
}
