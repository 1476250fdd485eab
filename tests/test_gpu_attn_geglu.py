"""Gate/up and GeGLU as part of the launch of attention merge, output projection and row work (option attn_geglu) against a launch of their own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W8 = dict(n_embd=2560, n_head=8, head_dim=256)


# (224 workgroups with a block of 32 columns each, or two: 16 blocks, 224, 232, 448, and 456, which do not fit)
@pytest.mark.parametrize("over,fused", [
    (dict(W8, n_ff=512), True), (dict(W8, n_ff=7168), True), (dict(W8, n_ff=7424), True), (dict(W8, n_ff=14336), True), (dict(W8, n_ff=14592), False),
    (dict(W8, n_embd=768, n_ff=7424), True), (dict(W8, n_embd=2304, n_ff=1024), True), (dict(W8, n_embd=1280, n_ff=7936), True)])
def test_one_launch_equals_two(lg, gpu_required, model_path, over, fused):
    """Every width, segments of 3, 5, 9 and 10 blocks: logits, hidden state and cache rows of steps in a row, bit for bit; and the launches say which form ran."""
    path, spec = model_path("tiny", **dict(dict(n_layer=2, n_vocab=2048, sliding_window=512), **over))
    rng = np.random.default_rng(spec["n_ff"])
    prompt, toks = rng.integers(1, spec["n_vocab"], 33).astype(np.int32), rng.integers(1, spec["n_vocab"], 40).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 400, max_rows=8)
    try:
        gpu.set_option("store_logits", 1)
        got = []
        for on in (1, 0):
            gpu.new_cache()
            gpu.set_option("attn_geglu", on)
            gpu.prefill(prompt, 0)
            res, pos = [], len(prompt)
            for rows in (1, 2, 3, 4, 5, 6, 7, 8, 1):
                print(f"{over} at {pos}, {rows} rows, attn_geglu {on}", flush=True)
                gpu.forward_spec(toks[pos - 33:pos - 33 + rows], pos)
                res += [gpu.logits_row(j, spec["n_vocab"]) for j in range(rows)] + [gpu.last_hidden(spec["n_embd"])]
                pos += rows
            res += [gpu.kv_read(L, w) for L in range(2) for w in (0, 1)]
            got.append([np.ascontiguousarray(r).view(np.uint8) for r in res])
            for rows in range(1, 9):
                n = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:rows], 33, 1)}.get("gate_up_geglu", 0)
                assert n == (0 if on and fused else 2), (rows, on, n)
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        gpu.close()


@pytest.mark.parametrize("over,fused", [
    (dict(W8, n_embd=768, n_ff=7168), range(1, 9)), (dict(W8, n_embd=768, n_ff=7424), range(1, 5)), (dict(W8, n_embd=1536, n_ff=8192), range(1, 5)),
    (dict(W8, n_embd=1536, n_ff=8448), range(1, 9)), (dict(W8, n_embd=1792, n_ff=7424), range(1, 9))])
def test_taken_where_it_is_the_faster_form(lg, gpu_required, model_path, over, fused):
    """The default: not at five rows and more of a narrow model whose blocks of FFN columns are two to some of 224 workgroups and one to a CU in a launch of their own."""
    path, spec = model_path("tiny", **dict(dict(n_layer=2, n_vocab=2048, sliding_window=512), **over))
    toks = np.random.default_rng(spec["n_ff"]).integers(1, spec["n_vocab"], 8).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 400, max_rows=8)
    try:
        for rows in range(1, 9):
            got = []
            for on in (None, 0):
                if on is not None:
                    gpu.set_option("attn_geglu", on)
                n = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:rows], 33, 1)}.get("gate_up_geglu", 0)
                assert n == (0 if on is None and rows in fused else 2), (rows, on, n)
                gpu.forward_spec(toks[:rows], 0)
                got.append(gpu.last_hidden(spec["n_embd"]).view(np.uint32))
            assert np.array_equal(*got), rows
            gpu.set_option("attn_geglu", 2)
    finally:
        gpu.close()
