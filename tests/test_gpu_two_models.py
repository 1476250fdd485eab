"""Two models at work at once on one device: one of them has launches whose workgroups wait for one another, results are those of a model alone."""
import ctypes as C
import threading

import numpy as np
import pytest

from conftest import random_q4_0

pytestmark = pytest.mark.gpu

NARROW = dict(E=512, heads=8, nkv=2, hd=64, ff=1024, rows=1)             # lg_k_narrow
WIDE = dict(E=2560, heads=8, nkv=2, hd=256, ff=2048, rows=5)             # lg_k_attn_out_m
ONE = dict(WIDE, rows=2)                                                 # lg_k_attn_out
JOINED = dict(E=3840, heads=16, nkv=8, hd=256, ff=5120, rows=5)          # lg_k_o_geglu, lg_k_down_qkv
LAYERS, VOCAB, SEQ, FRONT = 3, 2048, 512, 130


class Config(C.Structure):
    _fields_ = [(n, C.c_int32) for n in ("n_layer", "n_embd", "n_head", "n_vocab", "sliding_window", "ple", "n_kv_start")] + [
        (n, C.c_float) for n in ("eps", "base", "base_swa", "softcap")] + [(n, C.POINTER(C.c_int32)) for n in ("is_local", "ffn_len", "head_dim", "n_head_kv")]


class Served:
    """A model of seeded weights and a cache with a prompt in it, through the C ABI."""

    def __init__(self, H, s, seed):
        self.H, self.s, self.m, self.kv = H, s, C.c_void_p(), C.c_void_p()
        rng = np.random.default_rng(seed)
        arr = lambda v: (C.c_int32 * LAYERS)(*[v] * LAYERS)  # noqa: E731
        E, qd, kd, ff = s["E"], s["heads"] * s["hd"], s["nkv"] * s["hd"], s["ff"]
        cfg = Config(LAYERS, E, s["heads"], VOCAB, 256, 0, LAYERS, 1e-6, 1e6, 1e4, 30.0, arr(1), arr(ff), arr(s["hd"]), arr(s["nkv"]))
        assert H.lg_hip_model_create(C.cast(C.byref(cfg), C.c_void_p), 0, C.byref(self.m)) == 0, H.lg_hip_last_error()
        keep = []

        def tensor(name, typ, dims, data):
            keep.append(data)
            assert H.lg_hip_model_tensor(self.m, name.encode(), typ, len(dims), (C.c_uint64 * len(dims))(*dims), data.ctypes.data) == 0, H.lg_hip_last_error()

        def q4(name, k, n):
            tensor(name + ".weight", 2, (k, n), random_q4_0(rng, n, k))

        def vec(name, n):
            tensor(name + ".weight", 0, (n,), rng.uniform(0.5, 1.5, n).astype(np.float32))
        q4("token_embd", E, VOCAB)
        vec("output_norm", E)
        vec("rope_freqs", s["hd"] // 2)
        for i in range(LAYERS):
            b = f"blk.{i}."
            for n, k, r in (("attn_q", E, qd), ("attn_k", E, kd), ("attn_v", E, kd), ("attn_output", qd, E), ("ffn_gate", E, ff), ("ffn_up", E, ff), ("ffn_down", ff, E)):
                q4(b + n, k, r)
            for n, k in (("attn_q_norm", s["hd"]), ("attn_k_norm", s["hd"]), ("attn_norm", E), ("post_attention_norm", E), ("ffn_norm", E), ("post_ffw_norm", E)):
                vec(b + n, k)
        assert H.lg_hip_model_commit(self.m, 8) == 0, H.lg_hip_last_error()
        assert H.lg_hip_kv_create(self.m, s.get("seq", SEQ), C.byref(self.kv)) == 0, H.lg_hip_last_error()
        self.prompt = rng.integers(1, VOCAB, FRONT).astype(np.int32)
        self.blocks = rng.integers(1, VOCAB, (300, s["rows"])).astype(np.int32)

    def work(self):
        """A prompt, steps with a wait each, and the same blocks as a schedule: everything that comes out."""
        H, rows, got = self.H, self.s["rows"], []
        out, adv, pos = np.zeros(rows, np.int32), C.c_int32(0), C.c_int32(0)
        hid = np.zeros(self.s["E"], np.float32)
        for r in range(3):
            assert H.lg_hip_prefill(self.m, self.kv, self.prompt, FRONT, 0) == 0, H.lg_hip_last_error()
            for b in self.blocks[:40]:
                assert H.lg_hip_forward_spec(self.m, self.kv, b, rows, FRONT, out, C.byref(adv)) == 0, H.lg_hip_last_error()
                assert H.lg_hip_get_hidden(self.m, hid) == 0
                got += [out.copy(), hid.view(np.uint32).copy(), adv.value]
        n = (SEQ - FRONT) // rows
        blocks = np.resize(self.blocks, (n, rows))
        outs, advs = np.zeros((n, rows), np.int32), np.zeros(n, np.int32)
        assert H.lg_hip_schedule_load(self.m, blocks, n, rows, FRONT) == 0, H.lg_hip_last_error()
        assert H.lg_hip_schedule_run(self.m, self.kv, n) == 0, H.lg_hip_last_error()
        assert H.lg_hip_schedule_wait(self.m, outs.ctypes.data, advs.ctypes.data, C.byref(pos)) == n, H.lg_hip_last_error()
        return got + [outs, advs, pos.value]

    def close(self):
        self.H.lg_hip_kv_destroy(self.kv)
        self.H.lg_hip_model_destroy(self.m)


@pytest.fixture
def H(lg, gpu_required):
    H = lg.load_hip()
    P, I = C.c_void_p, C.c_int
    for name, args in (("lg_hip_model_create", [P, I, C.POINTER(P)]), ("lg_hip_kv_create", [P, I, C.POINTER(P)]), ("lg_hip_kv_destroy", [P]), ("lg_hip_model_destroy", [P]),
                       ("lg_hip_model_tensor", [P, C.c_char_p, C.c_uint32, C.c_uint32, C.POINTER(C.c_uint64), P]), ("lg_hip_model_commit", [P, I])):
        getattr(H, name).argtypes = args
    return H


@pytest.mark.parametrize("a,b", [(NARROW, NARROW), (NARROW, WIDE), (ONE, WIDE), (WIDE, WIDE)])
def test_two_threads_with_a_model_each(H, a, b):
    models = [Served(H, a, 1), Served(H, b, 2)]
    try:
        print(f"alone: {a} {b}", flush=True)
        alone = [m.work() for m in models]
        got = [None, None]

        def go(i):
            got[i] = models[i].work()
        threads = [threading.Thread(target=go, args=(i,)) for i in (0, 1)]
        print("together", flush=True)
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for x, y in zip(alone, got):
            assert y is not None and len(x) == len(y) and all(np.array_equal(p, q) for p, q in zip(x, y))
        models.pop(0).close()                                             # the other one goes on
        again = models[0].work()
        assert all(np.array_equal(p, q) for p, q in zip(alone[1], again))
    finally:
        for m in models:
            m.close()


@pytest.mark.parametrize("a,b", [(JOINED, JOINED), (dict(JOINED, rows=2), WIDE)])
def test_two_threads_with_launches_of_the_whole_chip(H, a, b):
    """The same with the launches that need all 256 CUs in one or both models."""
    test_two_threads_with_a_model_each(H, a, b)


def launches(m, rows):
    """Launches of a step by class."""
    cap = 32
    names, ms, n, by = (C.c_char_p * cap)(), np.zeros(cap, np.float32), np.zeros(cap, np.int32), np.zeros(cap, np.float64)
    k = m.H.lg_hip_profile_step(m.m, m.kv, m.blocks[0][:rows], rows, FRONT, 1, names, ms, n, by, cap)
    assert k > 0, m.H.lg_hip_last_error()
    return {names[i].decode(): int(n[i]) for i in range(k)}


def test_steps_beside_a_prompt_wait_for_nobody(H):
    """A prompt's kernels hold the CUs for long: while another model has one under way a step has no launch whose workgroups wait for one another, and the same results."""
    a, b = Served(H, JOINED, 1), Served(H, dict(WIDE, seq=4096), 2)
    try:
        rows = JOINED["rows"]
        out, adv = np.zeros(rows, np.int32), C.c_int32(0)

        def step():
            assert H.lg_hip_forward_spec(a.m, a.kv, a.blocks[0], rows, FRONT, out, C.byref(adv)) == 0, H.lg_hip_last_error()
            return out.copy()
        assert H.lg_hip_prefill(a.m, a.kv, a.prompt, FRONT, 0) == 0
        alone = step()
        assert launches(a, rows).get("gate_up_geglu", 0) == 0
        long = np.resize(b.prompt, 4000)
        rcs, begun = [], threading.Event()

        def prompts():
            for _ in range(40):
                begun.set()
                rcs.append(H.lg_hip_prefill(b.m, b.kv, long, len(long), 0))
        t = threading.Thread(target=prompts)
        print("together", flush=True)
        t.start()
        begun.wait()
        seen = []
        while t.is_alive():
            n = launches(a, rows).get("gate_up_geglu", 0)
            assert np.array_equal(step(), alone)
            if t.is_alive():
                seen.append(n)
        t.join()
        assert rcs == [0] * 40 and len(seen) > 3
        assert sum(n == LAYERS for n in seen) > len(seen) // 2, seen    # (one can fall between two prompts)
        assert launches(a, rows).get("gate_up_geglu", 0) == 0           # theirs again
    finally:
        a.close()
        b.close()
