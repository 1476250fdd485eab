"""Two edge cases of the reference interface on the GPU: argmax ties (the lower index wins,
src/cuda/model-cuda.cuh:703-720, src/cpu/model-cpu.c:477-478) and the sampling hook model_pick
(include/model.h:105-111, src/cuda/mtp-kernel.cuh:103-118)."""
import ctypes as C
import json
import os
import shutil
import subprocess
import sys
import time

import numpy as np
import pytest

from conftest import gguf_tensor_span
from test_gpu_draft import write_head
from test_gpu_wide import nan_rows

pytestmark = pytest.mark.gpu


def duplicate_upper_vocabulary(path):
    """Rows V/2 .. V-1 of token_embd become copies of rows 0 .. V/2-1: with the tied head every logit
    then appears twice, V/2 apart, so every argmax is a tie."""
    off, nbytes, dims = gguf_tensor_span(path, "token_embd.weight")
    with open(path, "r+b") as f:
        f.seek(off)
        lower = f.read(nbytes // 2)
        f.seek(off + nbytes // 2)
        f.write(lower)
    return dims[1]


def test_argmax_ties_resolve_to_the_lower_index(lg, ob, gpu_required, model_path, model_dir):
    src, spec = model_path("tiny_full")
    path = os.path.join(str(model_dir), "tiny_full_tied.gguf")
    shutil.copyfile(src, path)
    V = duplicate_upper_vocabulary(path)
    head_src = write_head(lg, model_dir, "tiny_full", spec)
    head = os.path.join(str(model_dir), "assistant_tied.gguf")
    shutil.copyfile(head_src, head)
    assert duplicate_upper_vocabulary(head) == V
    half = V // 2
    rng = np.random.default_rng(41)
    prompt = rng.integers(0, half, 40).astype(np.int32)
    o = ob.Oracle(path)
    od = o.mtp_open(head)
    gpu = lg.hiplib.HipBackend(path, 160, max_rows=5)
    t = gpu.mtp_open(head)
    try:
        kv = o.kv_new(160, ob.I8)
        o.prefill(kv, prompt[:-1], 0, ob.I8)
        gpu.prefill(prompt[:-1], 0)
        gpu.set_option("store_logits", 1)
        print("ties: one-row decode", flush=True)
        tok, pos = int(prompt[-1]), len(prompt) - 1
        for _ in range(6):                                # model_forward_next: argmax on the device
            want, row, hid = o.forward(kv, tok, pos, ob.I8, want_hidden=True)
            got = gpu.forward_next(tok, pos)
            dev = gpu.logits_row(0, V)
            assert np.array_equal(dev[:half].view(np.uint32), dev[half:].view(np.uint32))      # every value is tied
            assert int(np.argmax(dev)) < half and dev[got] == dev.max()
            assert got == want and got < half
            tok, pos = got, pos + 1
        print("ties: draft head", flush=True)
        d_want, d_hid, _ = od.draft(kv, tok, pos, hid, ob.I8, want_logits=True)
        d_got = gpu.mtp_draft(t, tok, pos, chain=False)
        assert d_got == d_want and d_got < half
        print("ties: verify rows", flush=True)
        for step in range(4):                             # verify rows: every row's successor is the lower twin
            blk = np.array([tok] + [int(x) for x in rng.integers(0, half, 4)], np.int32)
            adv, out, _ = o.forward_spec_all(kv, blk, pos, ob.I8, want_hidden=True)
            gadv, gout = gpu.forward_spec(blk, pos)
            assert gadv == adv and gout.tolist() == list(out)
            assert all(int(x) < half for x in gout)
            for j in range(5):
                dev = gpu.logits_row(j, V)
                assert dev[int(gout[j])] == dev.max() == dev[int(gout[j]) + half]
            tok, pos = int(out[adv - 1]), pos + adv
    finally:
        gpu.mtp_close(t); gpu.close(); od.close(); o.close()


PICK = C.CFUNCTYPE(C.c_int, C.POINTER(C.c_float), C.c_int)


def second_best(row):
    """A deterministic rule that is not the argmax: the index of the second largest value (lower index on ties)."""
    order = np.lexsort((np.arange(row.size), -row))
    return int(order[1])


def test_sampling_hook_replaces_the_argmax(lg, ob, gpu_required, model_path):
    """With model_pick set the backend reads every row's logits back, lets the hook choose, accepts while the
    choice agrees with the next draft, and re-points the hidden state at the last accepted row."""
    path, spec = model_path("tiny_full")
    V, E, rows = spec["n_vocab"], spec["n_embd"], 4
    rng = np.random.default_rng(43)
    prompt = rng.integers(0, V, 50).astype(np.int32)
    o = ob.Oracle(path)
    gpu = lg.hiplib.HipBackend(path, 200, max_rows=rows)
    calls = []

    def pick(ptr, n):
        row = np.ctypeslib.as_array(ptr, shape=(n,))
        calls.append(n)
        return second_best(row)

    hook = PICK(pick)
    slot = C.c_void_p.in_dll(gpu.B, "model_pick")
    try:
        kv = o.kv_new(200, ob.I8)
        o.prefill(kv, prompt[:-1], 0, ob.I8)
        gpu.prefill(prompt[:-1], 0)
        slot.value = C.cast(hook, C.c_void_p).value
        tok, pos = int(prompt[-1]), len(prompt) - 1
        seen = set()
        for step in range(10):
            # the oracle's own chain under the same rule gives drafts that hold; plant the first wrong one
            first_bad = int(rng.integers(1, rows + 1))
            blk, picks, hiddens = [tok], [], []
            for j in range(rows):
                _, row, hid = o.forward(kv, blk[j], pos + j, ob.I8, want_hidden=True)
                picks.append(second_best(row)); hiddens.append(hid)
                if j + 1 < rows:
                    nxt = picks[j] if j + 1 < first_bad else (picks[j] + 1 + int(rng.integers(0, V - 1))) % V
                    blk.append(nxt)
            want_adv = 1
            while want_adv < rows and picks[want_adv - 1] == blk[want_adv]:
                want_adv += 1
            print(f"hook step {step} pos {pos} first_bad {first_bad} adv {want_adv}", flush=True)
            calls.clear()
            adv, out = gpu.forward_spec(np.array(blk, np.int32), pos)
            assert len(calls) == rows and all(n == V for n in calls)
            assert adv == want_adv and out.tolist() == picks
            assert np.array_equal(gpu.last_hidden(E).view(np.uint32), hiddens[adv - 1].view(np.uint32))
            seen.add(adv)
            tok, pos = picks[adv - 1], pos + adv
        assert len(seen) >= 2                              # both partial and full acceptance were exercised
    finally:
        slot.value = None
        gpu.close(); o.close()


@pytest.mark.parametrize("rows,name,over", [(2, "tiny_full", {}), (5, "tiny_full", {}), (6, "tiny", {"n_ff": 5120}), (5, "tiny_full", {"n_ff": 5120})])
def test_every_kernel_choice_gives_the_same_bits(lg, gpu_required, model_path, monkeypatch, rows, name, over):
    """The options that pick between kernels for the same arithmetic (row work inside the q/k/v matmul, the
    attention kernels that share a staged tile, the matrix-core lm_head, wide prompt blocks, graph replay, ffn_down
    cut by K quarter: the last case has the long FFN rows and no per-layer embeddings that kernel is for; the
    per-layer inputs built on a second stream beside layer 0) change
    timing only: every combination leaves the same cache rows and the same logits rows of a verify block."""
    monkeypatch.setenv("LG_HIP_MERGE_O", "1")          # (builds the second copy of attn_output that the merge_o option needs)
    monkeypatch.setenv("LG_HIP_XCD_ATTN_TAIL", "1")    # (... and the one the xcd_attn_tail option needs)
    path, spec = model_path(name, **over)
    V = spec["n_vocab"]
    rng = np.random.default_rng(rows)
    prompt = rng.integers(0, V, 300).astype(np.int32)
    blk = rng.integers(0, V, rows).astype(np.int32)

    def run(**opts):
        gpu = lg.hiplib.HipBackend(path, 400, max_rows=8)
        try:
            for k, v in opts.items():
                gpu.set_option(k, v)
            gpu.set_option("store_logits", 1)
            gpu.prefill(prompt, 0)
            adv, out = gpu.forward_spec(blk, 300)
            logits = np.stack([gpu.logits_row(j, V) for j in range(rows)])
            cache = [gpu.kv_read(L, w).copy() for L in range(spec["n_layer"] - spec["shared_kv_layers"]) for w in (0, 1)]
            return adv, out.copy(), logits, cache
        finally:
            gpu.close()

    base = run()
    assert np.isfinite(base[2]).all()                  # (a bitwise comparison would call two rows of NaN equal)
    for opt, val in (("fuse_rows", 0), ("attn_rows", 0), ("attn_rows_fq", 0), ("head_mfma", 0), ("wide_prefill", 0), ("use_graph", 0), ("down_kq", 0),
                     ("fork_ple", 1),        # (the per-layer inputs as a second branch of the graph: off by default)
                     ("xcd_tail", 0), ("xcd_tail", 2), ("xcd_tail_spread", 0), ("rows_geglu", 1),   # (the row work ahead of gate/up inside the gate/up launch: off by default; the per-layer-input block as separate kernels / as one launch also for narrow blocks)
                     ("down_m", 0), ("down_m", 2),                      # (ffn_down of 4..8-row blocks on v_dot4 instead of the matrix cores; the last two cases have the long FFN rows)
                     ("xcd_attn_tail", 0), ("xcd_attn_tail", 2),   # (attention merge + output projection + row work: separate kernels / one launch on one XCD for every width)
                     ("merge_o", 0), ("merge_o", 2), ("merge_o_slices", 8)):   # (attention merge + output projection: separate / one launch for every width / another cut of the rows)
        print(f"rows={rows} option {opt}={val}", flush=True)
        got = run(**{opt: val})
        assert got[0] == base[0] and np.array_equal(got[1], base[1]), opt
        assert np.array_equal(got[2].view(np.uint32), base[2].view(np.uint32)), opt
        for a, b in zip(got[3], base[3]):
            assert np.array_equal(a, b), opt


@pytest.mark.parametrize("rows,over", [(5, {}), (8, {}), (2, {}), (5, {"head_dim": 256, "head_dim_full": 256}), (8, {"head_dim_full": 256}), (8, {"n_head": 4}),
                                       (7, {"head_dim": 128}), (5, {"n_head": 16}), (3, {"n_head": 20, "head_dim": 128})])
def test_shared_tile_attention_prepares_its_own_rows(lg, ob, gpu_required, model_path, rows, over):
    """Layers with 256 and more (tile, kv head) pairs take the attention kernels whose workgroups serve all rows of a block (up to 16
    units of (row, query head) on so few tiles on the vector units, more on the matrix cores); they norm and rotate the block's queries and
    build the block's K/V rows themselves.  A 2048-key window
    on 4 KV heads (66 tiles) and a global context of the same length, layers that own their cache and layers that
    read another's, a block that starts 2 positions before a tile boundary (its rows fall into two tiles) and the
    next one after it: against the oracle, and bit for bit against the same step with lg_k_qkv_post run ahead
    (attn_rows_fq = 0) and with the per-row attention kernel (attn_rows = 0)."""
    path, spec = model_path("tiny_full", **dict({"n_head_kv": 4, "sliding_window": 2048}, **over))
    V, E = spec["n_vocab"], spec["n_embd"]
    rng = np.random.default_rng(90 + rows)
    n0 = 65 * 32 + 30
    prompt = rng.integers(0, V, n0).astype(np.int32)
    first, tail = int(rng.integers(0, V)), rng.integers(0, V, rows).astype(np.int32)
    ctx = n0 + 64

    def run(**opts):
        gpu = lg.hiplib.HipBackend(path, ctx, max_rows=8)
        try:
            for k, v in opts.items():
                gpu.set_option(k, v)
            gpu.set_option("store_logits", 1)
            gpu.prefill(prompt, 0)
            chain = [first]                                # the model's own continuation: a block that is accepted whole
            for i in range(rows):
                chain.append(gpu.forward_next(chain[-1], n0 + i))
            blocks = [np.array(chain[:rows], np.int32), np.concatenate(([chain[rows]], tail[1:])).astype(np.int32)]
            res, pos = [], n0
            for blk in blocks:
                adv, out = gpu.forward_spec(blk, pos)
                res.append((adv, out.copy(), np.stack([gpu.logits_row(j, V) for j in range(rows)]), gpu.last_hidden(E).copy(), blk))
                pos += adv
            cache = [gpu.kv_read(L, w).copy() for L in range(spec["n_layer"] - spec["shared_kv_layers"]) for w in (0, 1)]
            return res, cache
        finally:
            gpu.close()

    print(f"rows={rows}: default kernels", flush=True)
    base, base_cache = run()
    assert all(np.isfinite(r[2]).all() for r in base)
    assert base[0][0] == rows                              # verify == plain decode
    o = ob.Oracle(path)
    try:
        kv = o.kv_new(ctx, ob.I8)
        o.prefill(kv, prompt, 0, ob.I8)
        pos = n0
        for adv, out, _, hid, blk in base:
            oadv, oout, ohid = o.forward_spec(kv, blk, pos, ob.I8, want_hidden=True)
            assert oadv == adv and oout[:adv].tolist() == out[:adv].tolist()
            assert np.array_equal(hid.view(np.uint32), ohid.view(np.uint32))
            pos += adv
    finally:
        o.close()
    for opts in ({"attn_rows_fq": 0}, {"attn_rows": 0}):
        print(f"rows={rows}: {opts}", flush=True)
        got, cache = run(**opts)
        for g, b in zip(got, base):
            assert g[0] == b[0] and np.array_equal(g[1], b[1]), opts
            assert np.array_equal(g[2].view(np.uint32), b[2].view(np.uint32)), opts
        for a, b in zip(cache, base_cache):
            assert np.array_equal(a, b), opts


@pytest.mark.parametrize("n0,j,fq,n_head", [(2100, 0, 1, 8), (2100, 3, 1, 8), (2100, 7, 1, 8), (2100, 3, 0, 8), (20, 3, 1, 8), (20, 4, 0, 8),
                                            (2100, 0, 1, 4), (2100, 7, 1, 4), (2100, 3, 0, 4), (20, 3, 1, 4), (2100, 0, 1, 12), (2100, 7, 1, 12), (20, 3, 1, 12)])
def test_a_block_row_of_nan_reaches_no_row_before_it(lg, gpu_required, model_path, model_dir, n0, j, fq, n_head):
    """Verify blocks whose rows share an attention tile (256 and more (tile, kv head) pairs), with a token whose embedding is
    infinite at row j of the block that a tile boundary cuts, behind a whole window and in the first keys of one: the cache rows in
    front of it, in every layer, are those of the same block with another token there, and all of them those of the attention kernel
    per row."""
    src, spec = model_path("tiny_full", n_head=n_head, n_head_kv=4, sliding_window=2048)
    path = os.path.join(str(model_dir), "tiny_full_infinite_token.gguf")
    shutil.copyfile(src, path)
    off, nbytes, dims = gguf_tensor_span(path, "token_embd.weight")
    odd = 77
    with open(path, "r+b") as f:
        for b in range(dims[0] // 32):
            f.seek(off + odd * (nbytes // dims[1]) + b * 18)
            f.write(b"\x00\x7c")                          # the block's scale: +inf
    n = 16                                                # two blocks of 8 rows, the second over a tile boundary
    prompt = np.random.default_rng(j).integers(100, spec["n_vocab"], n0 + n).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 2160, max_rows=8)
    try:
        got = []
        for shared, token in ((1, int(prompt[n0 + 8 + j])), (1, odd), (0, odd)):
            gpu.new_cache()
            gpu.set_option("wide_prefill", 1)
            gpu.prefill(prompt[:n0], 0)
            gpu.set_option("wide_prefill", 0)
            gpu.set_option("attn_rows", shared)
            gpu.set_option("attn_rows_fq", fq)
            blocks = prompt[n0:].copy()
            blocks[8 + j] = token
            print(f"token {token} at row {j}, shared tiles {shared}, own preparation {fq}", flush=True)
            gpu.prefill(blocks, n0)
            got.append([gpu.kv_read(L, w)[np.arange(n0, n0 + n) % gpu.kv_layout(L)[0]] for L in range(spec["n_layer"] - spec["shared_kv_layers"]) for w in (0, 1)])
        for plain, shared, per_row in zip(*got):
            assert np.array_equal(shared[:8 + j], plain[:8 + j])
            assert np.array_equal(nan_rows(shared), nan_rows(per_row))
        assert all(((a[8 + j] & 0x7FFF) > 0x7C00).any() for a in got[1][2:])
    finally:
        gpu.close()


@pytest.mark.parametrize("n_head,hd,rows,pairs", [(16, 64, 8, 101), (16, 256, 8, 101), (16, 128, 5, 150), (8, 64, 8, 101), (16, 256, 5, 142)])
def test_block_rows_in_a_later_tile_of_their_workgroup(lg, gpu_required, model_path, n_head, hd, rows, pairs):
    """Long global layers of 8 kv heads whose pairs of tiles outnumber the workgroups that the CUs hold (96 per kv head): a block over the
    border between two pairs, prepared inside the attention kernel by the workgroups that walk to them as their second pair (16 units; 10 where
    the tiles are too many for lg_k_attn_few; the last two cases are those of 8 and 10 units that go there), against lg_k_qkv_post ahead of it (attn_rows_fq = 0) and the kernel
    per row (attn_rows = 0).  The keys in front are drawn."""
    path, spec = model_path("tiny", n_head=n_head, n_head_kv=8, head_dim_full=hd)
    n0 = 64 * pairs - 2
    blk = np.random.default_rng(rows).integers(0, spec["n_vocab"], rows).astype(np.int32)

    def run(**opts):
        gpu = lg.hiplib.HipBackend(path, n0 + 40, max_rows=8)
        try:
            rng = np.random.default_rng(5)
            for L in range(spec["n_layer"]):
                shape = gpu.kv_read(L, 0).shape
                for w in (0, 1):
                    gpu.kv_write(L, w, rng.normal(0, 1, shape).astype(np.float16).view(np.uint16))
            for k, v in opts.items():
                gpu.set_option(k, v)
            gpu.set_option("store_logits", 1)
            adv, out = gpu.forward_spec(blk, n0)
            return adv, out.copy(), np.stack([gpu.logits_row(j, spec["n_vocab"]) for j in range(rows)]), [gpu.kv_read(L, w).copy() for L in range(spec["n_layer"]) for w in (0, 1)]
        finally:
            gpu.close()

    got = []
    for opts in ({"attn_rows": 0}, {"attn_rows_fq": 0}, {}):
        print(f"n_head={n_head} hd={hd} rows={rows} pairs={pairs}: {opts}", flush=True)
        got.append(run(**opts))
    assert np.isfinite(got[0][2]).all()
    for g in got[1:]:
        assert g[0] == got[0][0] and np.array_equal(g[1], got[0][1])
        assert np.array_equal(g[2].view(np.uint32), got[0][2].view(np.uint32))
        assert all(np.array_equal(a, b) for a, b in zip(g[3], got[0][3]))


SESSION = """
import ctypes, importlib, json, sys
import numpy as np
root, path, head, shim = sys.argv[1:]
if shim:
    ctypes.CDLL(shim, mode=ctypes.RTLD_GLOBAL)      # ahead of the runtime for every library loaded from here on
sys.path.insert(0, root)
lg = importlib.import_module("little-gemma_amd")
gpu = lg.hiplib.HipBackend(path, 256, max_rows=4)
t = gpu.mtp_open(head)
gpu.prefill(np.arange(1, 31, dtype=np.int32), 0)
res, tok, pos = [], 31, 30
for _ in range(3):
    adv, out = gpu.forward_spec(np.array([tok, 5, 6, 7], np.int32), pos)
    pos, tok = pos + adv, int(out[adv - 1])
    res.append([adv, out.tolist()])
for _ in range(2):
    blocks, out, adv, pos = gpu.mtp_rounds(t, tok, pos, 3, 3)
    tok = int(out[-1, adv[-1] - 1])
    res.append([blocks.tolist(), out.tolist(), adv.tolist(), pos])
gpu.schedule(np.array([[tok, 1], [2, 3]], np.int32), pos)
gpu.schedule_run(2)
out, adv, pos = gpu.schedule_wait()
res.append([out.tolist(), adv.tolist(), pos, gpu.mtp_draft(t, 9, pos), gpu.mtp_draft(t, 9, pos)])
gpu.mtp_close(t)
gpu.close()
calls = ctypes.CDLL(shim).refused() if shim else 0
print(json.dumps([calls, res]))
"""


def test_a_step_counts_though_no_graph_of_it_can_be_made(lg, gpu_required, model_path, model_dir):
    """The first step of its kind runs as launches and its graph is made behind it.  In a process whose runtime refuses to make
    one (a library in front of it answers hipGraphInstantiate with out of memory), steps, rounds, schedules and drafts give
    what they give elsewhere: the step has run and the cache has moved, so its results must reach the caller."""
    path, spec = model_path("tiny_full")
    head = write_head(lg, model_dir, "tiny_full", spec)
    src, shim = os.path.join(str(model_dir), "refuse.c"), os.path.join(str(model_dir), "librefuse.so")
    with open(src, "w") as f:
        f.write("static int n;\nint hipGraphInstantiate(void **e, void *g, void **m, char *b, unsigned long s) { (void)e; (void)g; (void)m; (void)b; (void)s; n++; return 2; }\n"
                "int refused(void) { return n; }\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", shim, src], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    got = []
    for s in ("", shim):
        print(f"session {'without graphs' if s else 'with graphs'}", flush=True)
        r = subprocess.run([sys.executable, "-c", SESSION, root, path, head, s], capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-500:]
        got.append(json.loads(r.stdout.splitlines()[-1]))
    assert got[1][0] > 0 and got[1][1] == got[0][1]


def test_logits_rows_in_any_order(lg, gpu_required, model_path, model_dir):
    """Rows are fetched when they are asked for, the next one ahead of time for a caller that takes them in turn: in order,
    backwards, twice, with gaps, of the step before the last none; after blocks, schedules and drafts.  Each row against the
    same token decoded alone."""
    path, spec = model_path("tiny_full")
    V = spec["n_vocab"]
    head = write_head(lg, model_dir, "tiny_full", spec)
    gpu = lg.hiplib.HipBackend(path, 128, max_rows=8)
    t = gpu.mtp_open(head)
    try:
        gpu.prefill(np.arange(1, 21, dtype=np.int32), 0)
        blocks = [np.arange(30, 38, dtype=np.int32), np.arange(50, 58, dtype=np.int32)]
        want = []
        for b in blocks:
            want.append([gpu.forward(int(tok), 20 + j, V).view(np.uint32) for j, tok in enumerate(b)])
        gpu.set_option("store_logits", 1)
        orders = [range(8), range(7, -1, -1), (0, 1, 1, 2, 0, 1, 2, 5), (3,), (0,), (7, 0, 1, 2, 3, 4, 5, 6), ()]
        for i, order in enumerate(orders):
            adv = C.c_int32(0)
            out = np.zeros(8, np.int32)
            lg.hiplib.hip_check(gpu.H.lg_hip_forward_spec(gpu.dev, gpu.dkv, blocks[i & 1], 8, 20, out, C.byref(adv)), "forward_spec")
            for j in order:
                assert np.array_equal(gpu.logits_row(j, V).view(np.uint32), want[i & 1][j]), (i, j)
        print("schedule", flush=True)
        gpu.schedule(blocks[1][None], 20)
        gpu.schedule_run(1)
        for j in (0, 1, 4):
            assert np.array_equal(gpu.logits_row(j, V).view(np.uint32), want[1][j])
        gpu.schedule_wait()
        with pytest.raises(lg.hiplib.HipError):
            gpu.logits_row(8, V)
        print("draft head", flush=True)
        gpu.mtp_store_logits(t)
        first = gpu.mtp_draft(t, 9, 24)
        a = gpu.mtp_logits(t, V)
        assert int(np.argmax(a)) == first and np.array_equal(a, gpu.mtp_logits(t, V))
        second = gpu.mtp_draft(t, first, 25, chain=True)
        assert int(np.argmax(gpu.mtp_logits(t, V))) == second
    finally:
        gpu.mtp_close(t)
        gpu.close()


def test_logits_nobody_reads_stay_on_the_device(lg, gpu_required, model_path):
    """store_logits left on costs a scheduled step of 8 rows x 262144 logits what storing them in device memory does: 8 MiB across
    the bus would take 130 us at the 64 GB/s of its link; half of that is the bound here."""
    path, spec = model_path("tiny", n_vocab=262144)
    gpu = lg.hiplib.HipBackend(path, 512, max_rows=8)
    try:
        gpu.prefill(np.arange(1, 21, dtype=np.int32), 0)
        blocks = np.tile(np.arange(30, 38, dtype=np.int32), (20, 1))
        us = {}
        for on in (0, 1, 0, 1):
            gpu.set_option("store_logits", on)
            for _ in range(4):
                gpu.schedule(blocks, 20)
                us[on] = min(us.get(on, 1e9), gpu.schedule_time(20) * 1e3 / 20)
        print(f"a step: {us[0]:.1f} us, with logits {us[1]:.1f} us", flush=True)
        assert us[1] - us[0] < 65, us
    finally:
        gpu.close()


def test_a_process_that_asked_for_blocking_waits_gets_them(lg, gpu_required, model_path):
    """hipSetDeviceFlags(hipDeviceScheduleBlockingSync): the processor is given away during a step of some milliseconds (what is
    left is the launch and the short while the runtime polls first), and the results are those of polling."""
    path, spec = model_path("tiny", n_layer=64)
    gpu = lg.hiplib.HipBackend(path, 256, max_rows=4)
    hip = C.CDLL(None)
    if not hasattr(hip, "hipSetDeviceFlags"):
        hip = C.CDLL("libamdhip64.so")
    before = C.c_uint(0)
    assert hip.hipGetDeviceFlags(C.byref(before)) == 0
    try:
        gpu.prefill(np.arange(1, 21, dtype=np.int32), 0)
        got, steps = [], 40
        for flags in (before.value, 4, before.value):
            assert hip.hipSetDeviceFlags(flags) == 0
            gpu.forward_spec(np.array([5, 6, 7, 8], np.int32), 20)
            cpu, wall = time.thread_time(), time.perf_counter()
            res = [gpu.forward_spec(np.array([5, 6, 7, 8], np.int32), 20) for _ in range(steps)]
            cpu, wall = time.thread_time() - cpu, time.perf_counter() - wall
            print(f"flags {flags}: {wall / steps * 1e6:.0f} us a step, {cpu / steps * 1e6:.0f} us of the processor", flush=True)
            got.append((cpu / wall, [(a, o.tolist()) for a, o in res]))
        assert got[0][1] == got[1][1] == got[2][1]
        assert got[1][0] < 0.6, got[1][0]
    finally:
        hip.hipSetDeviceFlags(before.value)
        gpu.close()
