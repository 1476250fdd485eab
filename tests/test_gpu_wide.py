"""The kernels of prompt blocks (lg_wide.h) at the sizes where they can go wrong: every workgroup shape of the matmul, weight
rows that are no multiple of its 64-row tile, ragged activation rows, and prompts of every remainder through blocks of
their own width, against the oracle bit for bit."""
import os
import shutil
import time

import numpy as np
import pytest

from conftest import gguf_tensor_span, random_q4_0
from test_gpu_kernels import oracle_matmul
from test_gpu_prefill import check_wide_prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,rows", [(20480, 256, 32), (20480, 512, 64), (8200, 3840, 96), (264, 2560, 512), (2560, 5120, 160), (4160, 256, 480),
                                      (3072, 2560, 32), (1000, 4096, 96), (72, 4352, 128), (8, 256, 32), (2048, 2560, 64), (2056, 2560, 64), (264, 256, 160)])
def test_wide_matmul_shapes(lg, ob, gpu_required, m, k, rows):
    """64 x 32 tiles by two wavefronts (8 K segments in four parts, up to 64 tiles and 128 rows), by four and by eight, 64 x 64 tiles, a last
    weight tile of 8 rows, 32 K segments; rows of 8 segments of an odd number of blocks, of one."""
    rng = np.random.default_rng(m + k + rows)
    w = random_q4_0(rng, m, k)
    x = rng.normal(0, 1, (rows, k)).astype(np.float32)
    x[1, :64] = 0.0
    x[2] = np.sign(x[2])                                  # every value at the end of the q8 range
    print(f"wide matmul m={m} k={k} rows={rows}", flush=True)
    r = lg.hiplib.matmul_q4q8(w, k, m, x)
    xq, xd, xs, out, _ = oracle_matmul(ob, w, k, m, x)
    assert np.array_equal(r["xq"], xq) and np.array_equal(r["xsum"], xs) and np.array_equal(r["xd"].view(np.uint32), xd.view(np.uint32))
    assert np.array_equal(r["out"].view(np.uint32), out.view(np.uint32))


@pytest.mark.parametrize("k", [256, 2560, 5120])
def test_wide_q8_of_values_that_are_not_finite(lg, gpu_required, k):
    """NaN and infinities in the activations: q8 values, scales and products of a wide block are those that blocks of 8 rows get.
    (A NaN counts as 0 beside finite neighbours; an infinity makes its block's scale a NaN.)"""
    rng = np.random.default_rng(k)
    m = 64
    w = random_q4_0(rng, m, k)
    x = rng.normal(0, 1, (32, k)).astype(np.float32)
    for j in range(24):                                   # NaN at every place of a lane's four values, in several lanes
        x[j, 32 * (j % 8) + j] = np.nan
    x[24, 7], x[25, 40], x[26, 100] = np.inf, -np.inf, np.nan
    x[26, 101] = np.inf
    x[27, 64:96] = np.nan
    print(f"wide q8 of NaN k={k}", flush=True)
    wide = lg.hiplib.matmul_q4q8(w, k, m, x)
    parts = [lg.hiplib.matmul_q4q8(w, k, m, np.ascontiguousarray(x[j:j + 8])) for j in range(0, 32, 8)]
    for key in ("xq", "xsum", "xd", "out"):
        want = np.concatenate([p[key].reshape(8, -1) for p in parts])
        got = wide[key].reshape(32, -1)
        assert np.array_equal(got, want, equal_nan=key in ("xd", "out")), key
    assert np.isfinite(wide["out"].reshape(32, m)[:24]).all() and np.isnan(wide["out"].reshape(32, m)[24:28]).all()


@pytest.mark.parametrize("name,n_prompt,over", [("tiny_full", 9, {}), ("tiny_full", 31, {}), ("tiny", 33, {}), ("tiny_full", 65, {}), ("tiny", 129, {}), ("tiny", 130, {}), ("tiny_full", 97, {}), ("tiny_full", 98, {}), ("tiny_full", 34, {"n_embd": 1280}),
                                                ("tiny", 70, {"n_ff": 10240}), ("tiny_full", 30, {"n_ff": 10240}), ("tiny", 1303, {}),
                                                ("tiny", 61, {"n_head": 12, "n_head_kv": 4}), ("tiny_full", 50, {"n_head_kv": 8}), ("tiny", 45, {"head_dim_full": 512})])
def test_ragged_prompts_leave_the_same_cache_and_logits(lg, ob, gpu_required, model_path, name, n_prompt, over):
    """Blocks of any width (padded inside the kernels only), the gate/up shapes of 64 x 64 tiles, more key tiles than the
    attention keeps in LDS, query groups that leave units idle (three heads per kv head) or one head each, 512-wide heads; widths around those up to which
    the per-layer gate does the row work ahead of it and small matrices are cut by K quarter."""
    path, spec = model_path(name, **over)
    check_wide_prefill(lg, ob, path, spec, f"{name} {over}", n_prompt)


@pytest.mark.parametrize("name,pos0,n", [("tiny", 0, 45), ("tiny", 301, 70), ("tiny_full", 300, 33)])
def test_rows_no_position_sees_may_hold_anything(lg, ob, gpu_required, model_path, name, pos0, n):
    """Infinities and NaN in the cache rows behind the prompt and in front of its windows (what a discarded branch of a
    conversation can leave) change no bit of what a prompt writes."""
    path, spec = model_path(name)
    rng = np.random.default_rng(n)
    prompt = rng.integers(1, spec["n_vocab"], pos0 + n).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, 640, max_rows=4)
    try:
        got = []
        for garbage in (0, 1):
            gpu.new_cache()
            if pos0:
                gpu.prefill(prompt[:pos0], 0)
            for L, y in enumerate(gpu.layers):
                if L >= spec["n_layer"] - spec["shared_kv_layers"] or not garbage:
                    continue
                rows = gpu.kv_layout(L)[0]
                seen = np.arange(max(0, pos0 + 1 - spec["sliding_window"]) if y["is_local"] else 0, pos0)
                hidden = np.setdiff1d(np.arange(rows), seen % rows)
                for which, bits in ((0, 0x7E00), (1, 0x7C00)):
                    d = gpu.kv_read(L, which)
                    d[hidden] = bits
                    gpu.kv_write(L, which, d)
            print(f"{name}: {n} positions at {pos0}, garbage {garbage}", flush=True)
            gpu.prefill(prompt[pos0:], pos0)
            got.append([gpu.kv_read(L, w)[np.arange(pos0, pos0 + n) % gpu.kv_layout(L)[0]]
                        for L in range(spec["n_layer"] - spec["shared_kv_layers"]) for w in (0, 1)])
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        gpu.close()


def test_long_cache_of_a_model_for_single_rows(lg, ob, gpu_required, model_path):
    """A model committed for one row with a cache too long for wide partials: the weights of 32 prompt rows over all its
    tiles need more memory than the partials of single rows, and the cache has it.  Against the same prompt row by row."""
    path, spec = model_path("tiny", n_head=16, n_head_kv=2, head_dim_full=512)
    max_seq, n = 70000, 33
    pos0 = max_seq - n - 1
    prompt = np.random.default_rng(1).integers(1, spec["n_vocab"], n).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, max_seq, max_rows=1)
    try:
        got = []
        for wide in (1, 0):
            gpu.new_cache()
            gpu.set_option("wide_prefill", wide)
            print(f"33 positions at {pos0}, wide {wide}", flush=True)
            gpu.prefill(prompt, pos0)
            got.append([gpu.kv_read(L, w) for L in range(spec["n_layer"] - spec["shared_kv_layers"]) for w in (0, 1)])
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        gpu.close()


@pytest.mark.parametrize("name,pos0,n,over", [("tiny", 351, 9, {}), ("tiny", 352, 33, {"sliding_window": 512}), ("tiny_full", 1500, 40, {}), ("tiny", 3000, 22, {"head_dim": 256, "sliding_window": 1024}),
                                              ("tiny", 700, 250, {"head_dim_full": 512}), ("tiny", 701, 61, {"n_head": 12, "n_head_kv": 4, "sliding_window": 512}),
                                              ("tiny", 1471, 260, {}), ("tiny", 1471, 420, {}), ("tiny", 32735, 24, {}), ("tiny", 32760, 24, {})])
def test_few_rows_late_in_a_context(lg, ob, gpu_required, model_path, name, pos0, n, over):
    """Scores and values as two kernels: from 12 tiles on, heads of 64 to 512 dims, windows and whole contexts, three heads per
    kv head, on both sides of the rows (128 workgroups, 205 of 256 beyond 44 tiles) and the tiles (1024) up to which they are used.  Against the same
    rows through verify blocks, bit for bit; the cache rows in front are drawn."""
    path, spec = model_path(name, **over)
    rng = np.random.default_rng(pos0 + n)
    prompt = rng.integers(1, spec["n_vocab"], n).astype(np.int32)
    owners = spec["n_layer"] - spec["shared_kv_layers"]
    gpu = lg.hiplib.HipBackend(path, pos0 + n + 2, max_rows=8)
    try:
        front = {}
        for L in range(owners):
            rows, width = gpu.kv_layout(L)
            front[L] = rng.normal(0, 0.5, (2, rows, width)).astype(np.float16).view(np.uint16)
        got = []
        for wide in (1, 0):
            gpu.new_cache()
            gpu.set_option("wide_prefill", wide)
            for L in front:
                for which in (0, 1):
                    gpu.kv_write(L, which, front[L][which])
            print(f"{name} {over}: {n} positions at {pos0}, wide {wide}", flush=True)
            gpu.prefill(prompt, pos0)
            got.append([gpu.kv_read(L, w) for L in range(owners) for w in (0, 1)] + [gpu.forward(5, pos0 + n, spec["n_vocab"]).view(np.uint32)])
        assert all(np.array_equal(a, b) for a, b in zip(*got))
    finally:
        gpu.close()


def nan_rows(a):
    """binary16 bit patterns with every NaN as one pattern (which NaN comes out of a sum is not defined)."""
    return np.where((a & 0x7FFF) > 0x7C00, 0x7E00, a)


@pytest.mark.parametrize("name,pos0,n,over", [("tiny", 301, 45, {}), ("tiny_full", 301, 33, {}), ("tiny", 400, 61, {"head_dim": 256}), ("tiny", 301, 37, {"n_head": 12, "n_head_kv": 4}),
                                              ("tiny", 701, 61, {"sliding_window": 512}), ("tiny", 1700, 300, {"sliding_window": 1536})])
def test_an_infinity_reaches_only_rows_that_see_it(lg, ob, gpu_required, model_path, name, pos0, n, over):
    """Value rows of infinities and NaN at the start of a window, seen by the prompt's first two rows and by none after them (rows
    that share a workgroup's products): the next layer's cache rows of the others keep their bits, and those of the two are what
    verify blocks make of them.  With all weights in LDS, in memory, and as two kernels; three heads per kv head."""
    path, spec = model_path(name, **over)
    rng = np.random.default_rng(pos0 + n)
    prompt = rng.integers(1, spec["n_vocab"], n).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, pos0 + n + 2, max_rows=8)
    try:
        front = {}
        for L in (0, 1):
            rows, width = gpu.kv_layout(L)
            front[L] = rng.normal(0, 0.5, (2, rows, width)).astype(np.float16).view(np.uint16)
        at = (pos0 + 2 - spec["sliding_window"]) % front[0].shape[1]
        odd = front[0][1].copy()
        odd[at, 0::5], odd[at, 1::5], odd[at, 7::5] = 0x7C00, 0xFC00, 0x7E00
        got = {}
        for wide, v0 in ((1, front[0][1]), (1, odd), (0, odd)):
            gpu.new_cache()
            gpu.set_option("wide_prefill", wide)
            for L in front:
                gpu.kv_write(L, 0, front[L][0])
                gpu.kv_write(L, 1, v0 if L == 0 else front[L][1])
            print(f"{name} {over}: {n} positions at {pos0}, wide {wide}, infinities {v0 is odd}", flush=True)
            gpu.prefill(prompt, pos0)
            ring = gpu.kv_layout(1)[0]
            got[wide, v0 is odd] = [gpu.kv_read(1, w)[np.arange(pos0, pos0 + n) % ring] for w in (0, 1)]
        for plain, wide, narrow in zip(got[1, False], got[1, True], got[0, True]):
            assert np.array_equal(wide[2:], plain[2:])
            assert np.array_equal(nan_rows(wide), nan_rows(narrow)) and ((wide[:2] & 0x7FFF) > 0x7C00).all()
    finally:
        gpu.close()


@pytest.mark.parametrize("name,n,j,over", [("tiny", 45, 18, {}), ("tiny_full", 33, 10, {}), ("tiny", 130, 34, {"head_dim_full": 512}), ("tiny", 37, 13, {"n_head": 12, "n_head_kv": 4})])
def test_a_row_of_nan_reaches_no_row_before_it(lg, ob, gpu_required, model_path, model_dir, name, n, j, over):
    """A prompt token whose embedding is infinite: the cache rows of the positions in front of it, in every layer, are those of the
    same prompt with another token there, and all of them those that verify blocks leave."""
    src, spec = model_path(name, **over)
    path = os.path.join(str(model_dir), os.path.basename(src) + ".odd")
    shutil.copyfile(src, path)
    off, nbytes, dims = gguf_tensor_span(path, "token_embd.weight")
    odd = 77
    with open(path, "r+b") as f:
        for b in range(dims[0] // 32):
            f.seek(off + odd * (nbytes // dims[1]) + b * 18)
            f.write(b"\x00\x7c")                          # the block's scale: +inf
    prompt = np.random.default_rng(n).integers(100, spec["n_vocab"], n).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, n + 2, max_rows=8)
    try:
        got = []
        for wide, token in ((1, prompt[j]), (1, odd), (0, odd)):
            gpu.new_cache()
            gpu.set_option("wide_prefill", wide)
            p = prompt.copy()
            p[j] = token
            print(f"{name} {over}: {n} positions, token {token} at {j}, wide {wide}", flush=True)
            gpu.prefill(p, 0)
            got.append([gpu.kv_read(L, w)[:n] for L in range(spec["n_layer"] - spec["shared_kv_layers"]) for w in (0, 1)])
        for plain, wide, narrow in zip(*got):
            assert np.array_equal(wide[:j], plain[:j])
            assert np.array_equal(nan_rows(wide), nan_rows(narrow))
        assert all(((a[j:] & 0x7FFF) > 0x7C00).all() for a in got[1][2:])
    finally:
        gpu.close()


@pytest.mark.parametrize("hd", [512, 64])
def test_prompt_blocks_on_a_cache_of_two_gibibytes_a_layer(lg, gpu_required, model_path, hd):
    """Caches whose value rows pass 2 GiB per layer (524288 positions at the 12B shape; here rows of 8 and 2 KiB): a prompt across
    that offset leaves the cache rows that verify blocks leave (heads of 512: by 64-bit addresses; of 64: as such blocks), and one at the start of the cache still runs in prompt blocks
    (20 times fewer launches per token than 8-row blocks: half their time is far off)."""
    heads = 8 if hd == 512 else 16
    path, spec = model_path("tiny", n_head=heads, n_head_kv=heads, head_dim=hd, n_layer=2)
    limit = (1 << 31) // (heads * hd * 2)                 # positions whose value rows fit 2 GiB
    n = 90
    pos0 = limit - 50
    rng = np.random.default_rng(hd)
    prompt = rng.integers(1, spec["n_vocab"], 480).astype(np.int32)
    gpu = lg.hiplib.HipBackend(path, limit + 300, max_rows=8)
    try:
        width = gpu.kv_layout(1)[1]
        front = rng.normal(0, 0.5, (2, 700, width)).astype(np.float16).view(np.uint16)
        got, took = [], []
        for wide in (1, 0):
            gpu.new_cache()
            gpu.set_option("wide_prefill", wide)
            for which in (0, 1):
                gpu.kv_write(1, which, front[which], pos0 - 700)
            print(f"{n} positions at {pos0}, heads of {hd}, wide {wide}", flush=True)
            gpu.prefill(prompt[:n], pos0)
            rows = [np.zeros((n, width), np.uint16) for _ in (0, 1)]
            for which in (0, 1):
                lg.hiplib.hip_check(gpu.H.lg_hip_kv_read(gpu.dkv, 1, which, pos0, n, rows[which]), "kv_read")
            hidden = gpu.forward(5, pos0 + n, spec["n_vocab"])
            got.append(rows + [hidden.view(np.uint32)])
            gpu.prefill(prompt, 0)
            t = []
            for _ in range(5):
                t0 = time.perf_counter()
                gpu.prefill(prompt, 0)
                t.append(time.perf_counter() - t0)
            took.append(min(t))
        assert all(np.array_equal(a, b) for a, b in zip(*got))
        assert took[0] < 0.5 * took[1], took
    finally:
        gpu.close()
