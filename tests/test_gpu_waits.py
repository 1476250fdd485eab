"""Launches whose workgroups wait for one another: a wait that is given up is reported by the call it happened in, and by no later one."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W8 = dict(n_embd=768, n_head=8, head_dim=256, n_layer=2, n_ff=512, n_vocab=2048)


@pytest.mark.parametrize("name,over,rows", [("tiny_full", {}, 1), ("tiny", W8, 2), ("tiny", W8, 3), ("tiny", W8, 8), ("tiny_full", {}, 4), ("tiny_full", {}, 5),
                                            ("tiny", {"n_layer": 2, "n_ff": 8192, "n_embd": 2560}, 6)])
def test_a_wait_given_up_is_reported_once(lg, ob, gpu_required, model_path, name, over, rows):
    """One row of a narrow model, the attention output by v_dot4 and by the matrix cores, both forms of the layer tail, ffn_down over four
    workgroups, each with no polls granted: a verify step, a schedule and prompts (in verify blocks, and with only the remainder in
    one) return -9; with the polls back a prompt and a step are the oracle's."""
    path, spec = model_path(name, **over)
    rng = np.random.default_rng(rows)
    V, n = spec["n_vocab"], 128 + rows                     # (one prompt block and a remainder)
    toks = rng.integers(1, V, n).astype(np.int32)
    blk = rng.integers(1, V, rows).astype(np.int32)
    o = ob.Oracle(path)
    gpu = lg.hiplib.HipBackend(path, n + 2 * rows, max_rows=max(rows, 4))
    H = gpu.H
    try:
        out, adv = np.zeros(rows, np.int32), C.c_int32(0)
        gpu.set_option("wait_polls", 0)
        assert H.lg_hip_forward_spec(gpu.dev, gpu.dkv, blk, rows, 0, out, C.byref(adv)) == -9
        assert b"given up" in H.lg_hip_last_error()
        for wide, m in ((0, 2 * rows), (1, n)):
            gpu.set_option("wide_prefill", wide)
            print(f"{name} {over}: prompt of {m}, prompt blocks {wide}", flush=True)
            assert H.lg_hip_prefill(gpu.dev, gpu.dkv, toks, m, 0) == -9
        gpu.schedule(np.stack([blk, blk]), 0)
        gpu.schedule_run(2)
        with pytest.raises(lg.hiplib.HipError, match="given up"):
            gpu.schedule_wait()
        gpu.set_option("wait_polls", 1 << 16)
        gpu.prefill(toks, 0)
        okv = o.kv_new(n + 2 * rows, ob.I8)
        o.prefill(okv, toks, 0, ob.I8)
        got = gpu.forward_spec(blk, n)
        want = o.forward_spec(okv, blk, n, ob.I8, want_hidden=True)
        assert got[0] == want[0] and got[1].tolist()[:got[0]] == want[1].tolist()[:want[0]]
        assert np.array_equal(gpu.last_hidden(spec["n_embd"]).view(np.uint32), want[2].view(np.uint32))
    finally:
        gpu.close(); o.close()


def test_more_layers_than_launch_numbers(lg, gpu_required, model_path, monkeypatch):
    """256 layers: the numbers of two steps would overlap, so every kernel is one that waits for nobody, also where another was asked for."""
    monkeypatch.setenv("LG_HIP_XCD_FFN", "1")
    path, spec = model_path("tiny", n_layer=256, n_vocab=2048)
    toks = np.random.default_rng(1).integers(1, spec["n_vocab"], 4).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 64, max_rows=4)
    try:
        gpu.set_option("xcd_ffn", 1)
        for rows in (1, 4):
            launches = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:rows], 0, 1)}
            assert not any(launches.get(k, 0) for k in ("ffn_xcd", "ple_tail", "attn_tail")), launches
    finally:
        gpu.close()


@pytest.mark.parametrize("name,over", [("tiny_full", {"n_embd": 2560, "n_head": 8, "head_dim": 256, "head_dim_full": 0, "n_ff": 8192, "n_vocab": 2048}), ("tiny_full", {}),
                                       ("tiny", {"n_embd": 2560, "n_head": 8, "head_dim": 256, "n_ff": 8192, "n_vocab": 2048}), ("tiny_full_bf16", {"n_ff": 8192})])
def test_steps_without_such_launches_leave_the_same_bits(lg, gpu_required, model_path, name, over):
    """What a step takes while another model has such launches: every kernel that waits for nobody, at every width, against the default's logits,
    hidden state and cache rows."""
    path, spec = model_path(name, **over)
    rng = np.random.default_rng(4)
    V, owners = spec["n_vocab"], spec["n_layer"] - spec["shared_kv_layers"]
    prompt, toks = rng.integers(1, V, 70).astype(np.int32), rng.integers(1, V, 40).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 160, max_rows=8)
    got = []
    try:
        gpu.set_option("store_logits", 1)
        for opts in (dict(narrow=1, attn_out=1, xcd_tail=1, down_m=1), dict(narrow=0, attn_out=0, xcd_tail=0, down_m=2)):
            for k, v in opts.items():
                gpu.set_option(k, v)
            gpu.new_cache()
            gpu.prefill(prompt, 0)
            pos, res = 70, []
            for rows in range(1, 9):
                print(f"{name} {over} {opts}: {rows} rows", flush=True)
                adv, out = gpu.forward_spec(toks[pos - 70:pos - 70 + rows], pos)
                res += [out, gpu.last_hidden(spec["n_embd"])] + [gpu.logits_row(j, V) for j in range(rows)]
                pos += rows
            launches = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:8], 100, 1)}
            if not opts["narrow"]:
                assert not any(launches.get(k, 0) for k in ("ple_tail", "attn_tail", "ffn_xcd")), launches
            got.append([np.ascontiguousarray(r).view(np.uint8) for r in res + [gpu.kv_read(L, w) for L in range(owners) for w in (0, 1)]])
    finally:
        gpu.close()
    assert all(np.array_equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("name,over,rows", [("tiny", {"n_layer": 2, "n_ff": 5120, "n_embd": 3840, "n_head": 16, "head_dim": 256, "n_head_kv": 8, "n_vocab": 2048}, 2),
                                            ("tiny", {"n_layer": 2, "n_ff": 5120, "n_embd": 3840, "n_head": 16, "head_dim": 256, "n_head_kv": 8, "n_vocab": 2048}, 5),
                                            ("tiny", {"n_layer": 2, "n_ff": 8192, "n_embd": 2560, "n_vocab": 2048}, 3), ("tiny_full_bf16", {"n_embd": 768, "n_vocab": 2048}, 4)])
def test_a_wait_given_up_in_a_launch_of_two_products(lg, ob, gpu_required, model_path, name, over, rows):
    """The same of lg_k_o_geglu with the merge in it and without, of lg_k_down_qkv on v_dot4 and on the matrix cores, and with the per-layer projection of a float type in ffn_down's place."""
    test_a_wait_given_up_is_reported_once(lg, ob, gpu_required, model_path, name, over, rows)


WAITS = dict(narrow=1, attn_out=1, xcd_tail=1, down_m=1, mid=1)
NONE = dict(narrow=0, attn_out=0, xcd_tail=0, down_m=2, mid=0)


@pytest.mark.parametrize("name,over", [("tiny_full", {"n_embd": 2560, "n_head": 8, "head_dim": 256, "head_dim_full": 0, "n_ff": 8192, "n_vocab": 2048}), ("tiny_full", {}),
                                       ("tiny", {"n_embd": 2560, "n_head": 8, "head_dim": 256, "n_ff": 8192, "n_vocab": 2048}), ("tiny_full_bf16", {"n_ff": 8192, "n_embd": 768}),
                                       ("tiny", {"n_layer": 3, "n_embd": 3840, "n_head": 16, "head_dim": 256, "n_head_kv": 8, "n_ff": 5120, "n_vocab": 2048})])
def test_every_launch_that_waits_against_none(lg, gpu_required, model_path, name, over):
    """All launches whose workgroups wait for one another, those that join two products among them, against none at all: logits, hidden state and cache rows at every width;
    and at every width the launches say that none was left (q/k/v, gate/up and ffn_down have one of their own in every layer)."""
    path, spec = model_path(name, **over)
    rng = np.random.default_rng(5)
    V, nl, owners = spec["n_vocab"], spec["n_layer"], spec["n_layer"] - spec["shared_kv_layers"]
    prompt, toks = rng.integers(1, V, 70).astype(np.int32), rng.integers(1, V, 40).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 160, max_rows=8)
    got = []
    try:
        gpu.set_option("store_logits", 1)
        for opts in (WAITS, NONE):
            for k, v in opts.items():
                gpu.set_option(k, v)
            gpu.new_cache()
            gpu.prefill(prompt, 0)
            pos, res, joined = 70, [], 0
            for rows in range(1, 9):
                print(f"{name} {over} {opts}: {rows} rows", flush=True)
                adv, out = gpu.forward_spec(toks[pos - 70:pos - 70 + rows], pos)
                res += [out, gpu.last_hidden(spec["n_embd"])] + [gpu.logits_row(j, V) for j in range(rows)]
                pos += rows
                n = {k["name"]: k["launches"] for k in gpu.profile_step(toks[:rows], 110, 1)}
                if opts is NONE:
                    assert not any(n.get(k, 0) for k in ("ple_tail", "attn_tail", "ffn_xcd")) and [n.get(k, 0) for k in ("qkv", "gate_up_geglu", "ffn_down")] == [nl] * 3, (rows, n)
                joined += n["qkv"] < nl
            assert (joined > 0) == (opts is WAITS)
            got.append([np.ascontiguousarray(r).view(np.uint8) for r in res + [gpu.kv_read(L, w) for L in range(owners) for w in (0, 1)]])
    finally:
        gpu.close()
    assert all(np.array_equal(a, b) for a, b in zip(*got))


def test_marks_are_cleared_while_steps_go_on(lg, gpu_required, model_path):
    """2^15 steps and more in a row, across the clearing of what launches hand over: the last schedule's tokens are the first one's."""
    path, spec = model_path("tiny_full", n_embd=768, n_layer=4, n_ff=512, n_vocab=2048, sliding_window=32, local_period=100)
    toks = np.random.default_rng(7).integers(1, spec["n_vocab"], (4096, 1)).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 4096, max_rows=2)
    try:
        got = []
        for i in range(9):
            gpu.schedule(toks, 0)
            gpu.schedule_run(4096)
            out, adv, pos = gpu.schedule_wait()
            print(f"schedule {i}: {len(adv)} steps, position {pos}", flush=True)
            got.append(out)
        assert all(np.array_equal(g, got[0]) for g in got[1:])
    finally:
        gpu.close()
