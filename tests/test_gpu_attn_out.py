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
