"""A product, the row work behind it and the next product as one launch (lg_k_o_geglu, lg_k_down_qkv; option mid) against the separate kernels."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import loaded_hip_runtime

pytestmark = pytest.mark.gpu

ALL = tuple(range(1, 9))


# attn_output inputs of 4 to 16 blocks a segment, rows of 3 to 15, one and two column blocks to a workgroup; ffn_down's segments of 5 to 15 blocks
@pytest.mark.parametrize("over,o,down", [
    (dict(n_embd=768, n_head=16, n_ff=5120), ALL, (1, 2, 3)),                                        # (streams of ffn_down's matrix-core form: rows past 2048 values)
    (dict(n_embd=1280, n_head=8, head_dim=128, n_ff=8192, n_head_kv=4), ALL, (1, 2, 3)),
    (dict(n_embd=2304, n_head=12, head_dim=256, n_ff=5120), ALL, ALL),
    (dict(n_embd=2560, n_head=16, head_dim=64, n_ff=10240, out_scale=0.9), ALL, ALL),
    (dict(n_embd=3072, n_head=16, head_dim=256, n_head_kv=8, n_ff=15360), ALL, ALL),
    (dict(n_embd=3840, n_head=16, head_dim=256, n_head_kv=8, n_ff=15360), ALL, ALL),
    (dict(n_embd=3840, n_head=4, head_dim=256, n_ff=512), ALL, ()),                                 # 16 column blocks: most workgroups without one; ffn_down of 8 segments
    (dict(n_embd=2560, n_head=20, n_head_kv=4, head_dim=256, n_ff=512), (), ())])                                # an input too wide
def test_one_launch_equals_the_separate_kernels(lg, gpu_required, model_path, over, o, down):
    """Every width: logits, hidden state and cache rows of steps in a row, bit for bit; and the launches say which form ran."""
    path, spec = model_path("tiny", **dict(dict(n_layer=3, n_vocab=2048, sliding_window=64), **over))
    rng = np.random.default_rng(spec["n_embd"] + spec["n_ff"])
    prompt, toks = rng.integers(1, spec["n_vocab"], 90).astype(np.int32), rng.integers(1, spec["n_vocab"], 40).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 2000, max_rows=8)
    try:
        gpu.set_option("store_logits", 1)
        got = []
        for on in (1, 0):
            gpu.new_cache()
            gpu.set_option("mid", on)
            gpu.prefill(prompt, 0)
            res, pos = [], len(prompt)
            for rows in (1, 2, 3, 4, 5, 6, 7, 8, 1):
                print(f"{over} at {pos}, {rows} rows, mid {on}", flush=True)
                gpu.forward_spec(toks[pos - 90:pos - 90 + rows], pos)
                res += [gpu.logits_row(j, spec["n_vocab"]) for j in range(rows)] + [gpu.last_hidden(spec["n_embd"])]
                pos += rows
            res += [gpu.kv_read(L, w) for L in range(3) for w in (0, 1)]
            got.append([np.ascontiguousarray(r).view(np.uint8) for r in res])
            for rows in ALL:
                n = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:rows], 90, 1)}
                assert (n.get("gate_up_geglu", 0) == 0) == bool(on and rows in o), (rows, on, n)
                assert n["qkv"] == (1 if on and rows in down else 3), (rows, on, n)
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        gpu.close()


@pytest.mark.parametrize("name,over", [("tiny_full_bf16", dict(n_embd=768)), ("tiny_full_f32", dict(n_embd=2560, n_head=8, head_dim=256, head_dim_full=256, n_head_kv=2)),
                                       ("tiny_full_f16", dict(n_embd=3840, n_head=16, head_dim=256, head_dim_full=256, n_head_kv=4))])
def test_per_layer_projection_of_a_float_type(lg, gpu_required, model_path, name, over):
    """The same launch with that projection as its first product: 3, 10 and 15 of its rows to a workgroup, shared-cache layers (queries only) and others behind it."""
    path, spec = model_path(name, **dict(dict(n_layer=4, n_ff=512, n_vocab=2048), **over))
    rng = np.random.default_rng(spec["n_embd"])
    prompt, toks = rng.integers(1, spec["n_vocab"], 90).astype(np.int32), rng.integers(1, spec["n_vocab"], 40).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 400, max_rows=8)
    try:
        gpu.set_option("store_logits", 1)
        got = []
        for on in (1, 0):
            gpu.new_cache()
            gpu.set_option("mid", on)
            gpu.prefill(prompt, 0)
            res, pos = [], len(prompt)
            for rows in (1, 2, 3, 4, 5, 6, 7, 8, 1):
                print(f"{name} {over} at {pos}, {rows} rows, mid {on}", flush=True)
                gpu.forward_spec(toks[pos - 90:pos - 90 + rows], pos)
                res += [gpu.logits_row(j, spec["n_vocab"]) for j in range(rows)] + [gpu.last_hidden(spec["n_embd"])]
                pos += rows
            res += [gpu.kv_read(L, w) for L in range(2) for w in (0, 1)]
            got.append([np.ascontiguousarray(r).view(np.uint8) for r in res])
            for rows in ALL:
                n = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:rows], 90, 1)}
                assert n["qkv"] == (1 if on else 4), (rows, on, n)
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        gpu.close()


@pytest.mark.parametrize("over,pos0,cache,merges", [
    (dict(n_embd=3840, n_head=16, head_dim=256, n_head_kv=8, sliding_window=1024), 3001, 3100, 1), (dict(n_embd=3072, n_head=16, head_dim=128, n_head_kv=4, sliding_window=608), 639, 700, 0),
    (dict(n_embd=2816, n_head=16, head_dim=64, sliding_window=1184), 1200, 1214, 0), (dict(n_embd=2816, n_head=32, head_dim=64, n_head_kv=4, sliding_window=1312), 2400, 2500, 2),
    (dict(n_embd=3840, n_head=4, head_dim=256), 0, 64, 0)])
def test_merge_inside_the_launch(lg, gpu_required, model_path, over, pos0, cache, merges):
    """Attention's partials merged by lg_k_o_geglu (1 to 3 rows): contexts of one tile, windows at and past the tiles of the first batch (20) and of all (40), global layers of more
    tiles beside them; against the separate kernels, bit for bit.  The cache rows in front are drawn.  merges: layers of more tiles than that, which keep their own."""
    path, spec = model_path("tiny", **dict(dict(n_layer=2, n_ff=512, n_vocab=2048), **over))
    rng = np.random.default_rng(pos0)
    gpu = lg.hiplib.HipBackend(path, cache, max_rows=8)
    try:
        gpu.set_option("store_logits", 1)
        front = [rng.normal(0, 0.5, (2,) + gpu.kv_layout(L)).astype(np.float16).view(np.uint16) for L in range(2)]
        toks = rng.integers(1, spec["n_vocab"], 20).astype(np.int32)
        got = []
        for on in (1, 0):
            gpu.new_cache()
            gpu.set_option("mid", on)
            for L in range(2):
                for which in (0, 1):
                    gpu.kv_write(L, which, front[L][which])
            res, pos = [], pos0
            for rows in (1, 2, 3, 4, 1):
                print(f"{over} at {pos}, {rows} rows, mid {on}", flush=True)
                gpu.forward_spec(toks[pos - pos0:pos - pos0 + rows], pos)
                res += [gpu.logits_row(j, spec["n_vocab"]) for j in range(rows)] + [gpu.last_hidden(spec["n_embd"])]
                pos += rows
            res += [gpu.kv_read(L, w) for L in range(2) for w in (0, 1)]
            got.append([np.ascontiguousarray(r).view(np.uint8) for r in res])
            for rows in (1, 2, 3, 4):
                n = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:rows], pos0, 1)}
                assert n.get("attn_merge", 0) == (merges if on and rows < 4 else 2), (rows, on, n)
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        gpu.close()


# (over, widths at which the launches are taken unless the option says otherwise: with gate/up, with q/k/v)
@pytest.mark.parametrize("name,over,o,down", [
    ("tiny", dict(n_embd=768, n_head=16, head_dim=64, n_ff=3072), (), ()),
    ("tiny", dict(n_embd=768, n_head=20, head_dim=64, n_head_kv=4, n_ff=5120), (), (3,)),
    ("tiny", dict(n_embd=1280, n_head=12, head_dim=256, n_ff=5632), range(4, 9), ()),
    ("tiny", dict(n_embd=1536, n_head=20, head_dim=64, n_head_kv=4, n_ff=6144), (), (2, 3)),
    ("tiny", dict(n_embd=2304, n_head=12, head_dim=256, n_ff=9216), ALL, range(2, 9)),
    ("tiny", dict(n_embd=2560, n_head=16, head_dim=64, n_ff=10240), range(1, 5), range(2, 9)),
    ("tiny", dict(n_embd=3072, n_head=16, head_dim=256, n_ff=8192), (), range(2, 9)),
    ("tiny", dict(n_embd=3328, n_head=16, head_dim=128, n_ff=4608), (1, 2), ()),
    ("tiny", dict(n_embd=3584, n_head=16, head_dim=256, n_ff=4608), range(1, 5), ()),
    ("tiny", dict(n_embd=3840, n_head=16, head_dim=128, n_ff=4608), range(1, 5), ()),
    ("tiny", dict(n_embd=3840, n_head=16, head_dim=256, n_head_kv=8, n_ff=5120), ALL, ALL),
    ("tiny_full_bf16", dict(n_layer=4, n_embd=768), (), range(3, 9)),
    ("tiny_full_bf16", dict(n_layer=4, n_embd=2560, head_dim_full=64), (), range(2, 9))])
def test_taken_where_it_is_the_faster_form(lg, gpu_required, model_path, name, over, o, down):
    """The default: the launches that join products where they were measured faster than the separate ones, by the widths of model and block; same bits as without."""
    path, spec = model_path(name, **dict(dict(n_layer=3, n_vocab=2048, n_ff=512, sliding_window=64), **over))
    toks = np.random.default_rng(spec["n_embd"]).integers(1, spec["n_vocab"], 40).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 400, max_rows=8)
    try:
        got = []
        for mid in (None, 0):
            if mid is not None:
                gpu.set_option("mid", mid)
            gpu.new_cache()
            res, pos = [], 0
            for rows in ALL:
                print(f"{name} {over}, {rows} rows, mid {mid}", flush=True)
                n = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:rows], 90, 1)}
                assert (n.get("gate_up_geglu", 0) == 0) == (mid is None and rows in o), (rows, n)
                assert n["qkv"] == (1 if mid is None and rows in down else spec["n_layer"]), (rows, n)
                gpu.forward_spec(toks[pos:pos + rows], pos)
                res.append(gpu.last_hidden(spec["n_embd"]).view(np.uint32))
                pos += rows
            got.append(res + [gpu.kv_read(0, w) for w in (0, 1)])
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        gpu.close()


def test_no_copy_of_what_another_launch_always_serves(lg, gpu_required, model_path):
    """attn_output as pairs of K segments is for layers that lg_k_attn_out cannot serve: sliding layers of a window that it holds at every width keep none, those of a wider one do."""
    lg.load_hip()
    hip, layers, used = C.CDLL(loaded_hip_runtime()), 24, []

    def free():
        free, total = C.c_size_t(0), C.c_size_t(0)
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value
    for window in (512, 512, 1024):                            # (the first for what the process takes once)
        path, spec = model_path("tiny", n_layer=layers, n_embd=2560, n_head=8, head_dim=256, n_ff=512, n_vocab=2048, sliding_window=window, local_period=100)
        before = free()
        gpu = lg.hiplib.HipBackend(path, 64, max_rows=8)
        try:
            gpu.forward_spec(np.ones(1, np.int32), 0)
            used.append(before - free())
        finally:
            gpu.close()
    copies = layers * 2560 * 2048 * 18 // 32
    assert used[2] - used[1] > copies * 3 // 4, (used, copies)
