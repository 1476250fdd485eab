"""One row of a narrow model: a layer from the merge on as one launch (lg_k_narrow) against the separate kernels and the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,over,pos0", [
    ("tiny", {}, 0), ("tiny_full", {}, 100), ("tiny", {"n_embd": 256, "n_ff": 256}, 31), ("tiny_full", {"n_embd": 256, "n_ff": 1280}, 64),
    ("tiny", {"n_ff": 1280, "head_dim": 128}, 127), ("tiny", {"sliding_window": 512}, 1000), ("tiny", {"sliding_window": 1024}, 1500),
    ("tiny", {}, 1023), ("tiny_full", {}, 4094), ("tiny", {}, 8250), ("tiny_full", {}, 8190), ("tiny", {"local_period": 0}, 20478)])
def test_a_layer_as_one_launch_equals_the_separate_kernels(lg, gpu_required, model_path, name, over, pos0):
    """Widths of one and two tiles a segment, feed-forward blocks on a part of the workgroups and on more than all of them, heads of 64 and
    128, contexts of one tile, on both sides of 32 (the merge by one wavefront), of 128 (half a round of tiles), of 256 (a round) and of 640 (two and a half): logits, hidden state and
    cache rows of several steps, bit for bit.  The cache rows in front are drawn."""
    path, spec = model_path(name, **over)
    rng = np.random.default_rng(pos0)
    owners = spec["n_layer"] - spec["shared_kv_layers"]
    gpu = lg.hiplib.HipBackend(path, pos0 + 8, max_rows=8)
    try:
        gpu.set_option("store_logits", 1)
        front = [rng.normal(0, 0.5, (2,) + gpu.kv_layout(L)).astype(np.float16).view(np.uint16) for L in range(owners)]
        toks = rng.integers(1, spec["n_vocab"], 4)
        got = []
        for narrow in (1, 0):
            gpu.new_cache()
            gpu.set_option("narrow", narrow)
            for L in range(owners):
                for which in (0, 1):
                    gpu.kv_write(L, which, front[L][which])
            print(f"{name} {over} at {pos0}, narrow {narrow}", flush=True)
            res = []
            for i, t in enumerate(toks):
                gpu.forward_spec(np.array([t], np.int32), pos0 + i)
                res += [gpu.logits_row(0, spec["n_vocab"]), gpu.last_hidden(spec["n_embd"])]
            res += [gpu.kv_read(L, w) for L in range(owners) for w in (0, 1)]
            got.append([np.ascontiguousarray(r).view(np.uint8) for r in res])
            launches = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:1].astype(np.int32), pos0, 1)}
            assert (launches.get("attn_merge", 0) == 0) == bool(narrow), launches
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        gpu.close()


@pytest.mark.parametrize("name,over", [("tiny", {"n_embd": 256, "n_ff": 512}), ("tiny_full", {"n_ff": 1280})])
def test_narrow_steps_match_the_oracle(lg, ob, gpu_required, model_path, name, over):
    path, spec = model_path(name, **over)
    V = spec["n_vocab"]
    prompt = np.random.default_rng(3).integers(1, V, 150).astype(np.int32)
    o = ob.Oracle(path)
    gpu = lg.hiplib.HipBackend(path, 200, max_rows=1)
    try:
        gpu.set_option("store_logits", 1)
        okv = o.kv_new(200, ob.I8)
        o.prefill(okv, prompt[:-1], 0, ob.I8)
        gpu.prefill(prompt[:-1], 0)
        tok = int(prompt[-1])
        for pos in range(149, 155):
            print(f"{name} {over} at {pos}", flush=True)
            adv, out = gpu.forward_spec(np.array([tok], np.int32), pos)
            oadv, oout, ohid = o.forward_spec(okv, np.array([tok], np.int32), pos, ob.I8, want_hidden=True)
            assert out[0] == oout[0] and np.array_equal(gpu.last_hidden(spec["n_embd"]).view(np.uint32), ohid.view(np.uint32))
            tok = int(out[0])
    finally:
        gpu.close(); o.close()
