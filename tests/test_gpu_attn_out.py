"""Attention merge, output projection and the row work behind them as one launch (lg_k_attn_out, lg_k_attn_out_m) against the separate kernels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W8 = dict(n_embd=2560, n_head=8, head_dim=256)


@pytest.mark.parametrize("over,pos0,cache", [
    (W8, 0, 64), (W8, 100, 512), (dict(W8, sliding_window=512), 543, 700), (dict(W8, sliding_window=512), 3001, 3100), (dict(W8, n_embd=768), 31, 1280),
    (dict(W8, n_embd=1024, sliding_window=608), 639, 700), (dict(W8, n_embd=2304, head_dim=64, n_head=32, n_head_kv=4), 1231, 1270),
    (dict(W8, n_embd=1280, sliding_window=1184, head_dim=128, n_head=16), 2400, 2500), (dict(n_embd=2560, n_head=4, head_dim=512), 40, 96)])
def test_one_launch_equals_the_separate_kernels(lg, gpu_required, model_path, over, pos0, cache):
    """Row groups on all and on a part of the wavefronts, heads of 64 to 512, contexts of one tile, windows at and past the tiles of the first
    batch (20) and of all (40), layers of more tiles beside them: logits, hidden state and cache rows of several steps, bit for
    bit.  The cache rows in front are drawn."""
    path, spec = model_path("tiny", **dict(dict(n_layer=2, n_ff=512, n_vocab=2048), **over))
    rng = np.random.default_rng(pos0)
    gpu = lg.hiplib.HipBackend(path, cache, max_rows=8)
    try:
        gpu.set_option("store_logits", 1)
        front = [rng.normal(0, 0.5, (2,) + gpu.kv_layout(L)).astype(np.float16).view(np.uint16) for L in range(2)]
        toks = rng.integers(1, spec["n_vocab"], 40)
        got = []
        for on in (1, 0):
            gpu.new_cache()
            gpu.set_option("attn_out", on)
            for L in range(2):
                for which in (0, 1):
                    gpu.kv_write(L, which, front[L][which])
            res, pos = [], pos0
            for rows in (1, 1, 2, 3, 4, 5, 6, 7, 8, 1):
                print(f"{over} at {pos}, {rows} rows, attn_out {on}", flush=True)
                gpu.forward_spec(toks[pos - pos0:pos - pos0 + rows].astype(np.int32), pos)
                res += [gpu.logits_row(j, spec["n_vocab"]) for j in range(rows)] + [gpu.last_hidden(spec["n_embd"])]
                pos += rows
            res += [gpu.kv_read(L, w) for L in range(2) for w in (0, 1)]
            got.append([np.ascontiguousarray(r).view(np.uint8) for r in res])
            launches = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:1].astype(np.int32), pos0, 1)}
            assert (launches.get("attn_tail", 0) > 0) == bool(on), launches
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        gpu.close()


def launches_of(gpu, toks, pos):
    return {k["name"]: k["launches"] for k in gpu.profile_step(toks, pos, 1)}


@pytest.mark.parametrize("window,cache", [(512, 607), (512, 608), (1024, 1247), (1024, 1248)])
def test_every_width_takes_the_launch_that_its_tiles_allow(lg, gpu_required, model_path, window, cache):
    """A sliding and a global layer: at most 40 tiles at 1 to 3 rows, 20 at 4 to 8.  (Each has to have run for the comparison above to mean anything.)"""
    path, spec = model_path("tiny", **dict(W8, n_layer=2, n_ff=512, n_vocab=2048, sliding_window=window))
    toks = np.random.default_rng(window).integers(1, spec["n_vocab"], 8).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, cache, max_rows=8)
    try:
        for rows in range(1, 9):
            print(f"window {window}, cache {cache}, {rows} rows", flush=True)
            every = cache // 32 + 2                              # (tiles_max of lg_hip_kv_partials)
            tiles = (min((window + rows - 1 + 31) // 32 + 1, every), every)
            got = launches_of(gpu, toks[:rows], 16)
            want = sum(t <= (40 if rows <= 3 else 20) for t in tiles)
            assert got.get("attn_tail", 0) == want and got.get("attn_output", 0) == 2 - want, (rows, got)
    finally:
        gpu.close()


@pytest.mark.parametrize("rows", [4, 5, 8])
def test_launches_asked_for_come_before_this_one(lg, gpu_required, model_path, monkeypatch, rows):
    """The row work ahead of gate/up is in this launch, in the gate/up launch (rows_geglu) or in the feed-forward launch (xcd_ffn): the one that was
    asked for does it, in every layer, with the same bits."""
    monkeypatch.setenv("LG_HIP_XCD_FFN", "1")
    path, spec = model_path("tiny", **dict(W8, n_layer=2, n_ff=10240, n_vocab=2048, sliding_window=512))
    rng = np.random.default_rng(rows)
    prompt, blk = rng.integers(1, spec["n_vocab"], 40).astype(np.int32), rng.integers(1, spec["n_vocab"], rows).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 600, max_rows=8)
    try:
        gpu.set_option("store_logits", 1)
        gpu.set_option("xcd_ffn", 0)
        gpu.prefill(prompt, 0)
        res, cnt = {}, {}
        for name, opts in (("separate", dict(attn_out=0)), ("attn_out", {}), ("rows_geglu", dict(rows_geglu=1)), ("xcd_ffn", dict(xcd_ffn=1))):
            print(f"{rows} rows, {name}", flush=True)
            for k, v in dict(dict(attn_out=1, rows_geglu=0, xcd_ffn=0), **opts).items():
                gpu.set_option(k, v)
            gpu.forward_spec(blk, 40)
            res[name] = [gpu.logits_row(j, spec["n_vocab"]).view(np.uint32) for j in range(rows)]
            cnt[name] = launches_of(gpu, blk, 40)
        assert all(np.array_equal(a, b) for r in res.values() for a, b in zip(r, res["separate"]))
        n = {k: (c.get("rows_norm_quant", 0), c.get("attn_tail", 0), c.get("ffn_xcd", 0)) for k, c in cnt.items()}
        alone = n["separate"][0]
        assert n == {"separate": (alone, 0, 0), "attn_out": (alone - 2, 2, 0), "rows_geglu": (alone - 2, 0, 0), "xcd_ffn": (alone - 2, 0, 2)}, n
    finally:
        gpu.close()
