"""mi_hip_attn_fwd_reference_order: the ATTN_QK -> SOFTMAX -> ATTN_KQV triple in
the reference's own operation order (src/ops_cpu.cpp:304-410), against the
oracle (the same order, the host C library's expf) BIT FOR BIT.

Short rows run the staged kernel (K, then V rows in LDS; up to 256 keys at
head_dim 64, as many as fit at 128, and only as many rows as run at once), few
longer rows the row kernel (a workgroup per row), many the tile kernel (a row
per wave). Key counts cover one key, partial and whole chunks of 16, odd and
even chunk counts, the staged limit and past it,
prefill rows on both sides of it, and a row whose exponentials are all equal
but one (its one-lane sum rounds the same way step after step). 32 seeded
random shapes (1-8 KV heads, 1-8 Q heads each, decode rows and short
prefills, 1-3000 keys) cover head layouts the chosen cases do not.
"""
import ctypes

import numpy as np
import pytest

from oracle import cpu_attention
import mi_hip_attn as mh

pytestmark = pytest.mark.gpu


def _inputs(seed, n_tokens, n_kv, h, hkv, d):
    rng = np.random.default_rng(seed)
    q = rng.standard_normal((n_tokens, h, d), dtype=np.float32)
    k = rng.standard_normal((n_kv, hkv, d), dtype=np.float32)
    v = rng.standard_normal((n_kv, hkv, d), dtype=np.float32)
    return q, k, v


def _run(hip, stream, q, k, v, n_past, scale):
    import torch
    qd, kd, vd = (torch.from_numpy(x).cuda() for x in (q, k, v))
    out = torch.full_like(qd, float("nan"))
    a = mh.attn_args(qd, out, q.shape[1] // k.shape[1], n_past, scale, stream, k=kd, v=vd)
    hip.check(hip.mi_hip_attn_fwd_reference_order(ctypes.byref(a)))
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _bits(x):
    return np.ascontiguousarray(x, dtype=np.float32).view(np.uint32)


def _check(hip, stream, q, k, v, n_past, scale, what):
    print(what, flush=True)
    got = _run(hip, stream, q, k, v, n_past, scale)
    want = cpu_attention.oracle().attention(q, k, v, n_past, scale, 8)[2]
    diff = np.flatnonzero(_bits(got) != _bits(want))
    assert diff.size == 0, (f"{what}: {diff.size} of {got.size} outputs differ in their bits, first at "
                            f"{np.unravel_index(diff[0], got.shape)}: {got.flat[diff[0]]!r} vs {want.flat[diff[0]]!r}")


@pytest.mark.parametrize("d,n_kv", [(64, 1), (64, 15), (64, 16), (64, 17), (64, 33), (64, 129), (64, 256),
                                    (64, 383), (64, 512), (64, 513), (64, 1000), (128, 31), (128, 255),
                                    (128, 256), (128, 257), (128, 300), (128, 301)])
def test_decode_bit_for_bit(hip, stream, d, n_kv):
    q, k, v = _inputs(1000 + n_kv, 1, n_kv, 14, 2, d)
    _check(hip, stream, q, k, v, n_kv - 1, float(np.float32(1) / np.sqrt(np.float32(d))),
           f"decode D {d} n_kv {n_kv}")


@pytest.mark.parametrize("n_tokens,n_past,h,hkv", [(37, 100, 14, 2), (20, 600, 14, 2), (9, 0, 8, 8),
                                                    (16, 481, 28, 4)])
def test_prefill_rows_bit_for_bit(hip, stream, n_tokens, n_past, h, hkv):
    # rows of one call span several key counts (n_past + j + 1)
    q, k, v = _inputs(7 + n_past, n_tokens, n_past + n_tokens, h, hkv, 64)
    _check(hip, stream, q, k, v, n_past, 0.125, f"prefill {n_tokens} rows after {n_past}, {h}/{hkv} heads")


def test_equal_keys_but_one(hip, stream):
    # Every key equal but key 0: each head's exponentials are all one value but
    # one, so the one-lane sum rounds the same way step after step (its value
    # drifts far from the exact sum, which any reassociation would expose).
    n_kv, d = 512, 64
    q, k, v = _inputs(99, 1, n_kv, 14, 2, d)
    k[1:] = k[1]
    k[0] = -0.5 * k[1]
    _check(hip, stream, q, k, v, n_kv - 1, 0.125, "equal keys but one, n_kv 512")


def test_rejects_what_it_does_not_cover(hip, stream):
    import torch
    q = torch.zeros((1, 14, 64), device="cuda")
    out = torch.empty_like(q)
    k16 = torch.zeros((8, 2, 64), device="cuda", dtype=torch.float16)
    a = mh.attn_args(q, out, 7, 7, 0.125, stream, k=k16, v=k16)
    assert hip.mi_hip_attn_fwd_reference_order(ctypes.byref(a)) == 5  # MI_HIP_E_UNSUPPORTED
    assert "F32" in hip.last_error()
    k = torch.zeros((40000, 2, 64), device="cuda")
    a = mh.attn_args(q, out, 7, 39999, 0.125, stream, k=k, v=k)
    assert hip.mi_hip_attn_fwd_reference_order(ctypes.byref(a)) == 5
    assert "32768" in hip.last_error()


def _random_cases(n, seed):
    # (case, n_head_kv, n_rep, head_dim, n_past, n_tokens, scale): decode rows and
    # short prefills, key counts spread log-uniformly over 1..3000
    rng = np.random.default_rng(seed)
    out = []
    for i in range(n):
        hkv = int(rng.choice([1, 2, 3, 4, 8]))
        n_rep = int(rng.integers(1, 9))
        d = int(rng.choice([64, 128]))
        n_kv = max(1, int(np.exp(rng.uniform(0.0, np.log(3000.0)))))
        n_tok = 1 if rng.uniform() < 0.6 else int(rng.integers(2, min(n_kv, 40) + 1)) if n_kv > 1 else 1
        scale = float(np.float32(rng.uniform(0.5, 2.0) / np.sqrt(d)))
        out.append((i, hkv, n_rep, d, n_kv - n_tok, n_tok, scale))
    return out


@pytest.mark.parametrize("case", _random_cases(32, 20261204), ids=lambda c: f"r{c[0]}")
def test_random_shapes_bit_for_bit(hip, stream, case):
    i, hkv, n_rep, d, n_past, n_tok, scale = case
    q, k, v = _inputs(3000 + i, n_tok, n_past + n_tok, hkv * n_rep, hkv, d)
    _check(hip, stream, q, k, v, n_past, scale,
           f"random case {i}: n_head_kv {hkv} n_rep {n_rep} D {d} n_past {n_past} n_tokens {n_tok}")


@pytest.mark.parametrize("hkv,n_rep,d,n_past,n_tok", [
    (2, 7, 64, 8200, 1),     # one row per workgroup: half-size K buffers (past 7,000 keys)
    (1, 2, 64, 24500, 1),    # quarter-size ones
    (1, 1, 64, 32127, 1),    # the last key count with those
    (1, 1, 64, 32128, 1),    # and the smallest ones
    (1, 2, 64, 32767, 1),
    (2, 2, 128, 513, 2),     # a buffer more than both hold at head_dim 128
    (1, 3, 128, 8200, 1),    # head_dim 128: half-size buffers
    (1, 2, 128, 24500, 1),   # quarter-size ones, whose last requests are past the row
    (1, 1, 128, 32127, 1),
    (1, 1, 128, 32128, 1),
    (1, 2, 128, 32767, 1),
    (1, 1, 64, 0, 300),      # more rows than workgroups and up to 300 keys: tiles
    (2, 7, 64, 63, 37),      # more rows than workgroups and few keys: staged, several a CU
    (2, 7, 64, 55, 73),      # 1022 rows of up to 128 keys: the last that run staged at once
    (2, 7, 64, 54, 74),      # 1036 rows: tiles, rows past the last
    (2, 7, 64, 55, 74),      # one key more: across a tile's edge
    (3, 5, 128, 3, 51),      # head_dim 128: 765 rows staged,
    (3, 5, 128, 3, 52),      # 780 in tiles, rows past the last
    (3, 5, 128, 40, 60),     # across a tile's edge
    (3, 5, 128, 60, 20),     # 300 staged, 100 rows per KV head
    (1, 8, 64, 4300, 40),    # more rows than workgroups, scores too long for tiles of 8 rows
    (3, 6, 64, 4090, 30),    # more than two rounds of them: tiles of 4
    (2, 9, 64, 4090, 70),    # more than one round of those: a wave per row
    (2, 9, 64, 8150, 29),    # too long for tiles: rows
    (3, 6, 128, 3100, 30),   # head_dim 128: tiles of 4,
    (3, 6, 128, 6090, 29),   # then rows,
    (3, 6, 128, 7600, 29),   # a wave per row where their buffers halve,
    (3, 6, 128, 15000, 29),  # rows where fewer waves fit
])
def test_row_and_tile_kernels_bit_for_bit(hip, stream, hkv, n_rep, d, n_past, n_tok):
    q, k, v = _inputs(77 + n_past, n_tok, n_past + n_tok, hkv * n_rep, hkv, d)
    _check(hip, stream, q, k, v, n_past, float(np.float32(d ** -0.5)),
           f"{hkv} x {n_rep} heads of {d}, {n_tok} rows after {n_past}")


@pytest.mark.parametrize("d,n_tok", [
    (64, 4000), (64, 7000), (128, 5000),   # tiles of 8 rows, of 4, of 4
    (64, 4200), (128, 7000),               # a wave per row
    (64, 20700), (64, 32300), (128, 20700), (128, 32300),  # rows, with K buffers of 16 and 14 KB
])
def test_short_rows_of_a_long_launch_bit_for_bit(hip, stream, d, n_tok):
    # The kernel and its K buffers are those of a launch's longest row; its
    # short rows come through the same ones. Rows of one key up to past both
    # buffers, against one-row launches of their own (the oracle checks those
    # above).
    import torch
    g = torch.Generator(device="cuda").manual_seed(n_tok + d)
    q, k, v = (torch.randn((n_tok, 1, d), device="cuda", generator=g) for _ in range(3))
    scale = float(np.float32(d ** -0.5))
    out = torch.full_like(q, float("nan"))
    a = mh.attn_args(q, out, 1, 0, scale, stream, k=k, v=v)
    hip.check(hip.mi_hip_attn_fwd_reference_order(ctypes.byref(a)))
    for j in (0, 1, 14, 15, 27, 28, 55, 56, 63, 64, 111, 112, 127, 128, 300, n_tok - 1):
        one = torch.full((1, 1, d), float("nan"), device="cuda")
        a = mh.attn_args(q[j:j + 1], one, 1, j, scale, stream, k=k, v=v)
        hip.check(hip.mi_hip_attn_fwd_reference_order(ctypes.byref(a)))
        torch.cuda.synchronize()
        assert torch.equal(out[j].view(torch.int32), one[0].view(torch.int32)), j
