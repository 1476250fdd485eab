"""The next layer's q/k/v projections as part of the layer tail's launch (lg_k_ple_tail_s, option tail_qkv) against a launch of their own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ALL = range(1, 9)


@pytest.mark.parametrize("over,fused", [
    (dict(n_embd=512), range(2, 9)),                                              # segments of 2 blocks (one row: lg_k_narrow)
    (dict(n_embd=768), (1, 2, 3)),                                                # of 3: not on the matrix cores
    (dict(n_embd=1024, n_head=4, n_head_kv=1), ALL),                              # 8 to 20 workgroups with a share
    (dict(n_embd=1536, n_head=12, n_head_kv=3), ALL),
    (dict(n_embd=2560, n_head=8, n_head_kv=2, head_dim=256, head_dim_full=256, has_v=1), ALL),       # the widest of the shorter build
    (dict(n_embd=3072, n_head=8, n_head_kv=4, head_dim=256, head_dim_full=256), ALL),                # between the two builds
    (dict(n_embd=4096, n_head=8, n_head_kv=1, head_dim=256, head_dim_full=256), ALL),                # the widest of all
    (dict(n_embd=1024, n_head=20, n_head_kv=4, head_dim=256, head_dim_full=256), range(4, 9))])      # more rows than 16 to a workgroup
def test_one_launch_equals_two(lg, gpu_required, model_path, over, fused):
    """Every width: logits, hidden state and cache rows of steps in a row, bit for bit; and the launches say which form ran."""
    path, spec = model_path("tiny_full", **dict(dict(n_layer=4, n_ff=512, n_vocab=2048), **over))
    rng = np.random.default_rng(spec["n_embd"])
    prompt, toks = rng.integers(1, spec["n_vocab"], 150).astype(np.int32), rng.integers(1, spec["n_vocab"], 40).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 400, max_rows=8)
    try:
        gpu.set_option("store_logits", 1)
        got = []
        for on in (1, 0):
            gpu.new_cache()
            gpu.set_option("tail_qkv", on)
            gpu.prefill(prompt, 0)
            res, pos = [], len(prompt)
            for rows in (1, 2, 3, 4, 5, 6, 7, 8, 1):
                print(f"{over} at {pos}, {rows} rows, tail_qkv {on}", flush=True)
                gpu.forward_spec(toks[pos - 150:pos - 150 + rows], pos)
                res += [gpu.logits_row(j, spec["n_vocab"]) for j in range(rows)] + [gpu.last_hidden(spec["n_embd"])]
                pos += rows
            res += [gpu.kv_read(L, w) for L in range(2) for w in (0, 1)]
            got.append([np.ascontiguousarray(r).view(np.uint8) for r in res])
            for rows in ALL:
                n = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:rows], 150, 1)}.get("qkv", 0)
                narrow = rows == 1 and spec["n_embd"] == 512
                assert n == (1 if narrow or (on and rows in fused) else 4), (rows, on, n)
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        gpu.close()


@pytest.mark.parametrize("over,rows,joins", [
    (dict(n_embd=768), 4, False),                                                                    # not on the matrix cores: q/k/v keep their launch
    (dict(n_embd=1024, n_head=20, n_head_kv=4, head_dim=256, head_dim_full=256), 3, False),          # more rows than 16 to a workgroup
    (dict(n_embd=1024, n_head=4, n_head_kv=1), 3, True)])
def test_three_and_four_rows_take_the_form_that_joins_where_it_joins(lg, gpu_required, model_path, over, rows, joins):
    """lg_k_ple_tail_s at 3 and 4 rows only with the projections in it.  The units' stamps say which form ran: 8 x 3 units of lg_k_ple_tail or 3 x 10 of lg_k_ple_tail_s
    at three rows; at four lg_k_ple_tail alone has a phase 6.  (The last layer's, which joins nothing, is lg_k_ple_tail in either case.)"""
    path, spec = model_path("tiny_full", **dict(dict(n_layer=4, n_ff=512, n_vocab=2048), **over))
    toks = np.random.default_rng(rows).integers(1, spec["n_vocab"], rows).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 64, max_rows=8)
    try:
        gpu.set_option("xcd_tail_stamps", 1)
        gpu.forward_spec(toks, 0)
        s = gpu.tail_stamps(0)
        assert s[:24, 0].all()
        if rows == 3:
            assert s[24:30, 0].any() == joins and not s[30:, 0].any()
        assert s[:, 6].any()
    finally:
        gpu.close()
