"""Performance cases: what a program that serves a model with this framework has it do.

Everything goes through the C ABI of liblg_hip.so (include/lg_hip.h) as a program bound to it by FFI calls it.  A case
is one call sequence of a generation loop:

  decode   one row at a position: the chosen token in, its greedy successor or (sampled) its logits out
  verify   a block of 2..8 rows (the chosen token and drafts) in, successors and accept count out; with `sampled`
           the logits of every row as well, for a caller that accepts by its own rule
  prompt   a prompt of n tokens at pos0 (0: a fresh conversation, later: the next turn), then the logits of its last
           token: the time to the first token
  rounds   n speculative rounds with a draft head after one decode step, kept on the device (`device`) or driven from
           the host with a wait per draft and per verify step

on the shapes of little-gemma_amd/synth.py: the E4B shape (also with its per-layer matrices kept in bf16, as
quantization-aware conversions keep them), the 12B shape, and the tiny shape with every optional piece on.  Weights
are random of the generator's distribution and quantized to q4_0; a process uploads a model once and keeps it, as a
server does, while caches, cache contents and tokens are made anew from each seed.

The returned logits of a prompt depend on every cache row that the call wrote.  Results are exact: the framework
defines one order for every floating sum and its tests hold the device to it bit for bit.
"""
import ctypes as C
import importlib
import math

import numpy as np
import torch

lg = importlib.import_module("little-gemma_amd")
H = lg.load_hip()
E4B, G12B, TINY = lg.synth.E4B, lg.synth.G12B, lg.synth.TINY_FULL
SHAPES = {"e4b": E4B, "e4b_bf16_ple": dict(E4B, ple_float=3), "12b": G12B, "tiny": TINY}
F32, Q4_0, BF16 = 0, 2, 30          # ggml type ids


# ---- the cases ----------------------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: one token of a small model, where launches and the host path are all there is
        dict(name="tiny decode", kind="decode", model="tiny", rows=1, ctx=100, cache=512, sampled=False),
        # chat with sampling: one token, its logits on the host
        dict(name="e4b decode sampled", kind="decode", model="e4b", rows=1, ctx=777, cache=4096, sampled=True),
        # the benchmark's verify step: 4 drafts at 2048 positions
        dict(name="e4b verify 5", kind="verify", model="e4b", rows=5, ctx=2048, cache=4096, sampled=False),
        # the widest block, a long document in the cache
        dict(name="e4b verify 8 long", kind="verify", model="e4b", rows=8, ctx=20011, cache=32768, sampled=False),
        # a quantization-aware conversion, verified with sampling (block-4)
        dict(name="e4b bf16 verify 4 sampled", kind="verify", model="e4b_bf16_ple", rows=4, ctx=1531, cache=4096, sampled=True),
        # the larger model, token by token and with drafts
        dict(name="12b decode", kind="decode", model="12b", rows=1, ctx=3001, cache=8192, sampled=False),
        dict(name="12b verify 5", kind="verify", model="12b", rows=5, ctx=8192, cache=16384, sampled=False),
        # a chat line, a page, the next turn of a longer conversation, a document on the larger model
        dict(name="e4b prompt 23", kind="prompt", model="e4b", n=23, pos0=0, cache=4096),
        dict(name="e4b prompt 1000", kind="prompt", model="e4b", n=1000, pos0=0, cache=4096),
        dict(name="e4b prompt 333 at 3001", kind="prompt", model="e4b", n=333, pos0=3001, cache=8192),
        dict(name="12b prompt 4093", kind="prompt", model="12b", n=4093, pos0=0, cache=8192),
        # the -mtp loop: a batch of rounds on the device, as the command line runs it
        dict(name="e4b rounds", kind="rounds", model="e4b", rows=4, ctx=2048, cache=4096, n=8, device=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cache_for(rng, need):
    """A cache sized to the conversation (as the command line does) or a server's fixed one."""
    return need + rng.randint(1, 256) if rng.random() < 0.4 else max(4096, 1 << (need - 1).bit_length())


def draw(rng):
    kind = rng.choices(("decode", "verify", "prompt", "rounds"), (3, 4, 4, 2))[0]
    model = rng.choices(("e4b", "12b", "e4b_bf16_ple", "tiny"), (5, 3, 2, 1))[0]
    if kind == "prompt":
        n = _log_uniform(rng, 2, 2048 if model == "12b" else 4093)
        pos0 = 0 if rng.random() < 0.6 else _log_uniform(rng, 33, 4093)
        return dict(kind=kind, model=model, n=n, pos0=pos0, cache=_cache_for(rng, pos0 + n + 1))
    if kind == "rounds":
        rows, n = rng.randint(2, 8), rng.randint(1, 12)
        ctx = _log_uniform(rng, 33, 8192)
        return dict(kind=kind, model=model, rows=rows, ctx=ctx, cache=_cache_for(rng, ctx + 1 + rows * n), n=n,
                    device=rng.random() < 0.75)
    rows = 1 if kind == "decode" else rng.randint(2, 8)
    ctx = _log_uniform(rng, 17, 28000 if model != "12b" else 14000)
    return dict(kind=kind, model=model, rows=rows, ctx=ctx, cache=_cache_for(rng, ctx + rows), sampled=rng.random() < 0.3)


# ---- models: uploaded once per process ----------------------------------------------------------------------------
class _Config(C.Structure):
    _fields_ = [(n, C.c_int32) for n in ("n_layer", "n_embd", "n_head", "n_vocab", "sliding_window", "n_embd_per_layer", "n_kv_start")] + [
        (n, C.c_float) for n in ("rms_eps", "rope_freq_base", "rope_freq_base_swa", "logit_softcap")] + [
        (n, C.POINTER(C.c_int32)) for n in ("is_local", "ffn_len", "head_dim", "n_head_kv")]


def _bind():
    P, I = C.c_void_p, C.c_int
    for name, args in (("lg_hip_model_create", [C.POINTER(_Config), I, C.POINTER(P)]), ("lg_hip_draft_create", [P, C.POINTER(_Config), C.POINTER(P)]),
                       ("lg_hip_model_tensor", [P, C.c_char_p, C.c_uint32, C.c_uint32, C.POINTER(C.c_uint64), P]), ("lg_hip_model_commit", [P, I]),
                       ("lg_hip_kv_create", [P, I, C.POINTER(P)]), ("lg_hip_draft_step", [P, P, I, I, I, C.POINTER(C.c_int32)])):
        getattr(H, name).argtypes = args
    H.lg_hip_kv_destroy.argtypes = [P]
    H.lg_hip_kv_destroy.restype = None


_bind()


def _ok(rc, what):
    if rc < 0:
        lg.hiplib.hip_check(rc, what)


def _layer_kinds(s):
    return [int(s["local_period"] > 0 and i % s["local_period"] != s["local_period"] - 1) for i in range(s["n_layer"])]


def _head_dim(s, local):
    return s["head_dim"] if local else (s["head_dim_full"] or s["head_dim"])


class _Weights:
    """Seeded host tensors in GGUF layout, made on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.keep = []                                   # the library reads the bytes at commit

    def _hand_over(self, m, name, typ, dims, data):
        self.keep.append(data)
        d = (C.c_uint64 * len(dims))(*dims)
        _ok(H.lg_hip_model_tensor(m, name.encode(), typ, len(dims), d, data.data_ptr()), name)

    def q4_0(self, m, name, k, rows, std):
        """N(0, std) weights as q4_0 blocks: the value of largest magnitude maps to -8."""
        out = torch.empty((rows, k // 32, 18), dtype=torch.uint8)
        step = max(1, (1 << 26) // k)
        for r in range(0, rows, step):
            n = min(step, rows - r)
            w = torch.randn((n * (k // 32), 32), generator=self.gen, device="cuda") * std
            top = w.gather(1, w.abs().argmax(1, keepdim=True))
            d = top / -8.0
            q = (w / d + 8.5).clamp_(0, 15).to(torch.uint8)
            blk = torch.cat([d.to(torch.float16).view(torch.uint8).view(-1, 2), q[:, :16] | (q[:, 16:] << 4)], 1)
            out[r:r + n] = blk.view(n, k // 32, 18).cpu()
        self._hand_over(m, name, Q4_0, (k, rows), out)

    def matrix(self, m, name, k, rows, std, ple_float=0):
        if not ple_float:
            return self.q4_0(m, name, k, rows, std)
        w = torch.randn((rows, k), generator=self.gen, device="cuda") * std
        self._hand_over(m, name, BF16, (k, rows), w.to(torch.bfloat16).view(torch.int16).cpu())

    def vector(self, m, name, n, centre, jitter):
        v = centre * (1.0 + jitter * (torch.rand(n, generator=self.gen, device="cuda") * 2.0 - 1.0))
        self._hand_over(m, name, F32, (n,), v.cpu())


def _config(s, kinds, n_embd, n_head, n_ff, ple, n_kv_start, nkv):
    n = len(kinds)
    arr = lambda v: (C.c_int32 * n)(*v)  # noqa: E731
    return _Config(n, n_embd, n_head, s["n_vocab"], s["sliding_window"], ple, n_kv_start, s["rms_eps"], s["rope_base"], s["rope_base_swa"], s["softcap"],
                   arr(kinds), arr([n_ff] * n), arr([_head_dim(s, k) for k in kinds]), arr([nkv] * n))


def _upload_target(s):
    E, F, P, kinds, std, jit = s["n_embd"], s["n_ff"], s["ple"], _layer_kinds(s), s["w_std"], s["norm_jitter"]
    kv_start = s["n_layer"] - s["shared_kv_layers"]
    m, w = C.c_void_p(), _Weights(s["seed"])
    _ok(H.lg_hip_model_create(C.byref(_config(s, kinds, E, s["n_head"], F, P, kv_start, s["n_head_kv"])), 0, C.byref(m)), "model_create")
    w.q4_0(m, "token_embd.weight", E, s["n_vocab"], std)
    w.vector(m, "output_norm.weight", E, 1.0, jit)
    w.vector(m, "rope_freqs.weight", _head_dim(s, 0) // 2, 1.0, jit)
    if P:
        w.q4_0(m, "per_layer_token_embd.weight", P * s["n_layer"], s["n_vocab"], std)
        w.matrix(m, "per_layer_model_proj.weight", E, P * s["n_layer"], std, s["ple_float"])
        w.vector(m, "per_layer_proj_norm.weight", P, 1.0, jit)
    for i, local in enumerate(kinds):
        hd, b = _head_dim(s, local), "blk.%d." % i
        qk = s["qk_norm"] or math.sqrt(1.28 / math.sqrt(hd))
        qd, kd = hd * s["n_head"], hd * s["n_head_kv"]
        w.q4_0(m, b + "attn_q.weight", E, qd, std)
        w.vector(m, b + "attn_q_norm.weight", hd, qk, jit)
        if i < kv_start:
            w.q4_0(m, b + "attn_k.weight", E, kd, std)
            if s["has_v"]:
                w.q4_0(m, b + "attn_v.weight", E, kd, std)
            w.vector(m, b + "attn_k_norm.weight", hd, qk, jit)
        w.q4_0(m, b + "attn_output.weight", qd, E, std)
        w.q4_0(m, b + "ffn_gate.weight", E, F, std)
        w.q4_0(m, b + "ffn_up.weight", E, F, std)
        w.q4_0(m, b + "ffn_down.weight", F, E, std)
        for v in ("attn_norm", "post_attention_norm", "ffn_norm", "post_ffw_norm"):
            w.vector(m, b + v + ".weight", E, 1.0, jit)
        if P:
            w.matrix(m, b + "inp_gate.weight", E, P, std, s["ple_float"])
            w.matrix(m, b + "proj.weight", P, E, std, s["ple_float"])
            w.vector(m, b + "post_norm.weight", E, 1.0, jit)
        if s["out_scale"]:
            w.vector(m, b + "layer_output_scale.weight", 1, s["out_scale"], 0.0)
    _ok(H.lg_hip_model_commit(m, lg.hiplib.MAX_ROWS), "model_commit")
    return m


def _head_shape(s):
    """The draft head that goes with a target: (spec, kinds of its blocks: the last `n_full` read the global cache)."""
    a = lg.synth.assistant_for(s)
    return a, [int(i < a["n_layer"] - a["n_full"]) for i in range(a["n_layer"])]


def _upload_head(target, s):
    a, kinds = _head_shape(s)
    I, B, std, jit = a["n_inner"], a["n_backbone"], a["w_std"], a["norm_jitter"]
    m, w = C.c_void_p(), _Weights(a["seed"])
    _ok(H.lg_hip_draft_create(target, C.byref(_config(s, kinds, I, a["n_head"], a["n_ff"], 0, 0, s["n_head_kv"])), C.byref(m)), "draft_create")
    w.q4_0(m, "token_embd.weight", I, a["n_vocab"], std)
    w.vector(m, "output_norm.weight", I, 1.0, jit)
    w.q4_0(m, "pre_projection.weight", 2 * B, I, std)
    w.q4_0(m, "post_projection.weight", I, B, std)
    for i, local in enumerate(kinds):
        hd, b = _head_dim(s, local), "blk.%d." % i
        w.q4_0(m, b + "attn_q.weight", I, hd * a["n_head"], std)
        w.vector(m, b + "attn_q_norm.weight", hd, a["qk_norm"] or math.sqrt(1.28 / math.sqrt(hd)), jit)
        w.q4_0(m, b + "attn_output.weight", hd * a["n_head"], I, std)
        w.q4_0(m, b + "ffn_gate.weight", I, a["n_ff"], std)
        w.q4_0(m, b + "ffn_up.weight", I, a["n_ff"], std)
        w.q4_0(m, b + "ffn_down.weight", a["n_ff"], I, std)
        for v in ("attn_norm", "post_attention_norm", "ffn_norm", "post_ffw_norm"):
            w.vector(m, b + v + ".weight", I, 1.0, jit)
    _ok(H.lg_hip_model_commit(m, 1), "model_commit (draft head)")
    return m


_models, _heads = {}, {}


def _model(name):
    if name not in _models:
        _models[name] = _upload_target(SHAPES[name])
    return _models[name]


def _head(name):
    if name not in _heads:
        _heads[name] = _upload_head(_model(name), SHAPES[name])
    return _heads[name]


# ---- states: a conversation -----------------------------------------------------------------------------------------
class _State:
    def __init__(self, case):
        self.case, self.model = case, _model(case["model"])
        self.kv = C.c_void_p()
        _ok(H.lg_hip_kv_create(self.model, case["cache"], C.byref(self.kv)), "kv_create")

    def __del__(self):
        if self.kv:
            H.lg_hip_kv_destroy(self.kv)
            self.kv = None

    def fill(self, ctx, gen):
        """Cache rows of the positions before ctx, with the scale real ones have: K after its norm, V of unit size."""
        s = SHAPES[self.case["model"]]
        rows, width = C.c_int(), C.c_int()
        for i, local in enumerate(_layer_kinds(s)):
            _ok(H.lg_hip_kv_layout(self.kv, i, C.byref(rows), C.byref(width)), "kv_layout")
            n = min(rows.value, ctx)
            if not n:
                continue
            kv = torch.randn((2, n, width.value), generator=gen, device="cuda")
            kv[0] *= s["qk_norm"] or math.sqrt(1.28 / math.sqrt(_head_dim(s, local)))
            kv = kv.to(torch.float16).view(torch.int16).cpu().numpy().view(np.uint16)
            for which in (0, 1):
                _ok(H.lg_hip_kv_write(self.kv, i, which, 0, n, kv[which]), "kv_write")


def _spec(st, toks, pos, out):
    adv = C.c_int32(0)
    _ok(H.lg_hip_forward_spec(st.model, st.kv, toks, len(toks), pos, out, C.byref(adv)), "forward_spec")
    return adv.value


def prepare(case, seed):
    kind, vocab = case["kind"], SHAPES[case["model"]]["n_vocab"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    st = _State(case)
    if kind == "rounds":
        st.head = _head(case["model"])
    sampled = kind == "prompt" or bool(case.get("sampled"))
    _ok(H.lg_hip_set_option(st.model, b"store_logits", int(sampled)), "set_option")
    st.fill(case["pos0"] if kind == "prompt" else case["ctx"], gen)
    rows = 1 if kind == "prompt" else case["rows"]
    st.out = np.zeros(rows, np.int32)
    st.logits = np.zeros((rows, vocab), np.float32) if sampled else None
    if kind == "prompt":
        st.toks = rng.integers(1, vocab, case["n"]).astype(np.int32)
        st.last = st.toks[-1:].copy()
    elif kind == "rounds":
        n = case["n"]
        st.toks = rng.integers(1, vocab, 1).astype(np.int32)
        st.one = np.zeros(1, np.int32)
        st.blocks, st.outs, st.advs = np.zeros((n, rows), np.int32), np.zeros((n, rows), np.int32), np.zeros(n, np.int32)
    else:
        # the model's own greedy continuation, with the first wrong draft drawn as the benchmark draws it
        st.toks = rng.integers(1, vocab, 1).astype(np.int32)
        one = np.zeros(1, np.int32)
        for j in range(1, rows):
            _spec(st, st.toks[-1:].copy(), case["ctx"] + j - 1, one)
            st.toks = np.append(st.toks, one)
        bad = int(rng.geometric(0.6))
        for j in range(bad, rows):
            st.toks[j] = rng.integers(1, vocab)
    return st


# ---- one pass -------------------------------------------------------------------------------------------------------
def _logits(st, rows):
    for j in range(rows):
        _ok(H.lg_hip_get_logits(st.model, j, st.logits[j]), "get_logits")
    return st.logits


def run(st):
    c = st.case
    if c["kind"] == "prompt":
        n = c["n"]
        _ok(H.lg_hip_prefill(st.model, st.kv, st.toks, n - 1, c["pos0"]), "prefill")
        _spec(st, st.last, c["pos0"] + n - 1, st.out)
        return {"token": st.out, "logits": _logits(st, 1)}
    if c["kind"] == "rounds":
        _spec(st, st.toks, c["ctx"], st.one)               # the token before the rounds: its hidden state feeds the head
        token, pos, rows, n = int(st.one[0]), c["ctx"] + 1, c["rows"], c["n"]
        if c["device"]:
            end = C.c_int32(0)
            _ok(H.lg_hip_mtp_rounds(st.head, st.kv, token, pos, rows, n, st.blocks, st.outs, st.advs, C.byref(end)), "mtp_rounds")
            pos = end.value
        else:
            d = C.c_int32(0)
            for r in range(n):
                blk = st.blocks[r]
                blk[0] = token
                for j in range(1, rows):
                    _ok(H.lg_hip_draft_step(st.head, st.kv, int(blk[j - 1]), pos + j - 1, int(j > 1), C.byref(d)), "draft_step")
                    blk[j] = d.value
                st.advs[r] = adv = _spec(st, blk, pos, st.outs[r])
                pos, token = pos + adv, int(st.outs[r, adv - 1])
        return {"blocks": st.blocks, "successors": st.outs, "accepted": st.advs, "position": pos}
    adv = _spec(st, st.toks, c["ctx"], st.out)
    if c["sampled"]:
        return {"successors": st.out, "accepted": adv, "logits": _logits(st, c["rows"])}
    return {"successors": st.out, "accepted": adv}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
def _layer_weights(s, local):
    """(q4_0 weights, weights of the per-layer block) of a layer."""
    hd = _head_dim(s, local)
    qd, kd = hd * s["n_head"], hd * s["n_head_kv"]
    return s["n_embd"] * (qd + kd * (2 if s["has_v"] else 1)) + qd * s["n_embd"] + 3 * s["n_embd"] * s["n_ff"], 2 * s["n_embd"] * s["ple"]


def _block(s, rows, pos, head_rows):
    """Bytes and operations of `rows` positions from pos as one block, the head on head_rows of them."""
    q4, fl = 18.0 / 32.0, 2.0 if s["ple_float"] else 18.0 / 32.0
    w_q4, w_ple = 0.0, float(s["n_embd"] * s["ple"] * s["n_layer"])
    kv_bytes = attn = 0.0
    for local in _layer_kinds(s):
        a, b = _layer_weights(s, local)
        w_q4, w_ple = w_q4 + a, w_ple + b
        hd = _head_dim(s, local)
        window = s["sliding_window"] if local else 0
        reach = (lambda p: min(p + 1, window) if window else p + 1)  # noqa: E731
        first = pos - reach(pos) + 1
        kv_bytes += 2.0 * 2.0 * hd * s["n_head_kv"] * (pos + rows - first + rows)         # rows read once, the block's written
        pairs = sum(reach(p) for p in (pos, pos + rows - 1)) / 2.0 * rows
        attn += 4.0 * hd * s["n_head"] * pairs
    head = float(s["n_embd"] * s["n_vocab"])
    nbytes = w_q4 * q4 + w_ple * fl + (head * q4 if head_rows else 0.0) + kv_bytes
    flops = 2.0 * (w_q4 + w_ple) * rows + 2.0 * head * head_rows + attn
    return nbytes, flops


def _draft(s, pos):
    a, kinds = _head_shape(s)
    I, q4 = a["n_inner"], 18.0 / 32.0
    w = 3.0 * a["n_backbone"] * I + float(I) * a["n_vocab"]
    kv = attn = 0.0
    for local in kinds:
        hd = _head_dim(s, local)
        keys = min(pos, s["sliding_window"]) if local else pos
        w += 2.0 * I * hd * a["n_head"] + 3.0 * I * a["n_ff"]
        kv += 4.0 * hd * s["n_head_kv"] * keys
        attn += 4.0 * hd * a["n_head"] * keys
    return w * q4 + kv, 2.0 * w + attn


def work(case):
    s, kind = SHAPES[case["model"]], case["kind"]
    row_bytes = 4.0 * s["n_vocab"]
    if kind == "prompt":
        b, f = _block(s, case["n"], case["pos0"], 1)
        b += row_bytes
    elif kind == "rounds":
        b, f = _block(s, 1, case["ctx"], 1)
        for _ in range(case["n"]):                          # every round waits for the one before it
            for j in range(1, case["rows"]):
                db, df = _draft(s, case["ctx"] + j)
                b, f = b + db, f + df
            vb, vf = _block(s, case["rows"], case["ctx"] + 1, case["rows"])
            b, f = b + vb, f + vf
    else:
        b, f = _block(s, case["rows"], case["ctx"], case["rows"])
        if case["sampled"]:
            b += row_bytes * case["rows"]
    return {"bytes": b, "flops": f}


def tolerance(case):
    return "exact"
