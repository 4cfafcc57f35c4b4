"""Indexer projection and query RoPE on the GPU vs the oracle.

* ``dsa_indexer_query_rope_inplace`` (reference schema, nanovllm_ops.cpp:713-714):
  bit-exact against the oracle's restatement of the AscendC kernel, bf16 and
  fp16, several token / head counts and a smaller rope width.
* ``dsa_indexer_project_query_only``, fused launch: with the reference test's
  one-hot projections (ut_ops/test_glm_dsa_indexer.py:127-192) every
  projection is exact, so q and the weights are bit-exact against the oracle
  (which the CPU tests pin to the closed form), including the score-scale
  rounding and token counts that cross the 64-token groups.  With random
  projections the fp32 accumulation order differs from the oracle's float64
  sums, so the test allows the 16-bit rounding to land a step apart: at
  most 2^-7 (bf16) / 2^-10 (fp16) relative to the value (to the pair's norm
  for rotated dims), and at least 98% (95% rotated) of the values exact.
* the fp32 ``weights_proj`` path and the prefill ``dsa_indexer_project``
  (k through a library layer norm: the reference test's tolerances,
  atol 0.05 / rtol 0.025).
* the reference's argument errors.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _helpers import bits, dname
from oracle import dsa_oracle as O
from oracle import indexer_oracle as I

pytestmark = pytest.mark.gpu

H, D, R, HID, ROPE = 32, 128, 2048, 6144, 64


def _dev(x_bits: np.ndarray, dtype: torch.dtype) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(x_bits).view(np.int16)).view(dtype).to("cuda")


def _to_bits(x: np.ndarray, dtype: torch.dtype) -> np.ndarray:
    return O.f32_to_bits(np.asarray(x, np.float32), dname(dtype)).reshape(np.shape(x))


def _cos_sin(T, dtype, rope=ROPE, seed=0):
    rng = np.random.default_rng(seed)
    pos = rng.integers(1, 40000, size=(T, 1)).astype(np.float64)
    freq = 10000.0 ** (-np.arange(rope // 2) * 2.0 / rope)
    ang = np.repeat(pos * freq[None, :], 2, axis=1)
    return _to_bits(np.cos(ang), dtype).reshape(T, 1, 1, rope), _to_bits(np.sin(ang), dtype).reshape(T, 1, 1, rope)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,heads,head_dim,rope", [(1, 32, 128, 64), (24, 32, 128, 64), (100, 64, 128, 64),
                                                   (7, 16, 64, 32)])
def test_query_rope_bit_exact(dtype, T, heads, head_dim, rope):
    from nanovllm_amd import ops

    print(f"ROPE {dtype} T={T} H={heads} D={head_dim} rope={rope}", flush=True)
    rng = np.random.default_rng(T + heads)
    q = _to_bits(rng.standard_normal((T, heads, head_dim)) * 3, dtype)
    c, s = _cos_sin(T, dtype, rope, seed=T)
    qd = _dev(q, dtype)
    ops.dsa_indexer_query_rope_inplace(qd, _dev(c, dtype), _dev(s, dtype), rope)
    torch.cuda.synchronize()
    expect = q.copy()
    I.query_rope_inplace(expect, c, s, rope, dname(dtype))
    assert np.array_equal(bits(qd), expect)


def test_query_rope_errors():
    from nanovllm_amd import ops

    q = torch.zeros(4, 32, 128, dtype=torch.bfloat16, device="cuda")
    c = torch.zeros(4, 1, 1, 64, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(RuntimeError, match="aligned to 16"):
        ops.dsa_indexer_query_rope_inplace(q, c, c, 56)
    with pytest.raises(RuntimeError, match="cos dtype mismatch"):
        ops.dsa_indexer_query_rope_inplace(q, c.half(), c, 64)
    with pytest.raises(RuntimeError, match="token dimension mismatch"):
        ops.dsa_indexer_query_rope_inplace(q, c[:3], c[:3], 64)


def _one_hot():
    q_rows = H * D
    wq = np.zeros((q_rows, R), np.float32)
    wq[np.arange(q_rows), (np.arange(q_rows) * 17 + 11) % R] = np.where(np.arange(q_rows) % 3 == 0, -1.0, 1.0)
    wp = np.zeros((H, HID), np.float32)
    wp[np.arange(H), (np.arange(H) * 43 + 5) % HID] = np.where(np.arange(H) % 2 == 0, 1.0, -1.0)
    wk = np.zeros((D, HID), np.float32)
    wk[np.arange(D), (np.arange(D) * 29 + 7) % HID] = np.where(np.arange(D) % 2 == 0, 1.0, -1.0)
    return wq, wp, wk


def _random_weights(seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((H * D, R)) / np.sqrt(R), rng.uniform(-1, 1, (H, HID)) / np.sqrt(HID),
            rng.standard_normal((D, HID)) / np.sqrt(HID))


def _inputs(T, dtype, seed):
    rng = np.random.default_rng(seed)
    hidden = _to_bits(rng.standard_normal((T, HID)), dtype)
    qc = _to_bits(rng.standard_normal((T, R)), dtype)
    c, s = _cos_sin(T, dtype, seed=seed)
    return hidden, qc, c, s


def _run_query_only(hidden, qc, c, s, wq, wp, dtype, scale, wp_dev=None):
    from nanovllm_amd.dsa_indexer_project import dsa_indexer_project_query_only

    T = hidden.shape[0]
    q_out = torch.empty(T, H, D, dtype=dtype, device="cuda")
    w_out = torch.empty(T, H, dtype=dtype, device="cuda")
    dsa_indexer_project_query_only(_dev(hidden, dtype), _dev(qc, dtype), _dev(c, dtype), _dev(s, dtype),
                                   _dev(wq, dtype), wp_dev if wp_dev is not None else _dev(wp, dtype), q_out, w_out,
                                   n_head=H, head_dim=D, rope_dim=ROPE, score_scale=scale)
    torch.cuda.synchronize()
    return bits(q_out), bits(w_out)


def _close(got, expect, dtype, min_exact=0.98, pairs=False):
    """Within two 16-bit steps of the value (of the pair's norm for rotated
    pairs: an input one step off moves both outputs by up to a step of the
    larger one), and mostly exact.  The values are O(1)."""
    g = O.bits_to_f32(got, dname(dtype)).astype(np.float64)
    e = O.bits_to_f32(expect, dname(dtype)).astype(np.float64)
    mag = np.abs(e)
    if pairs:
        mag = np.repeat(np.hypot(e[..., 0::2], e[..., 1::2]), 2, axis=-1)
    rel = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    # values near zero: the fp32 sums' own error (~1e-6 here) is the floor
    err = np.abs(g - e) - rel * np.maximum(mag, 2.0 ** -6)
    assert np.all(err <= 0), f"worst excess {float(err.max()):.3g}"
    exact = float(np.mean(got == expect))
    assert exact >= min_exact, exact


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,scale", [(1, 1.0), (24, 1.0), (64, 0.0883883), (65, 1.0), (130, 0.5)])
def test_project_query_only_one_hot_bit_exact(dtype, T, scale):
    print(f"PROJECT one-hot {dtype} T={T} scale={scale}", flush=True)
    hidden, qc, c, s = _inputs(T, dtype, seed=T)
    wq, wp, _ = _one_hot()
    wq16, wp16 = _to_bits(wq, dtype), _to_bits(wp, dtype)
    q, w = _run_query_only(hidden, qc, c, s, wq16, wp16, dtype, scale)
    eq, ew = I.project_query_only(hidden, qc, c, s, wq16, wp16, H, D, ROPE, scale, dname(dtype))
    assert np.array_equal(q, eq)
    assert np.array_equal(w, ew)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [3, 24, 64])
def test_project_query_only_random_close(dtype, T):
    print(f"PROJECT random {dtype} T={T}", flush=True)
    hidden, qc, c, s = _inputs(T, dtype, seed=100 + T)
    wq, wp, _ = _random_weights(T)
    wq16, wp16 = _to_bits(wq, dtype), _to_bits(wp, dtype)
    q, w = _run_query_only(hidden, qc, c, s, wq16, wp16, dtype, 1.0)
    eq, ew = I.project_query_only(hidden, qc, c, s, wq16, wp16, H, D, ROPE, 1.0, dname(dtype))
    _close(q[..., ROPE:], eq[..., ROPE:], dtype)
    _close(q[..., :ROPE], eq[..., :ROPE], dtype, min_exact=0.95, pairs=True)
    _close(w, ew, dtype)


def test_project_query_only_fp32_weights_proj():
    """weights_proj in fp32 (the reference's dtype-mismatch branch, :82-86)."""
    dtype = torch.bfloat16
    T = 24
    hidden, qc, c, s = _inputs(T, dtype, seed=7)
    wq, wp, _ = _random_weights(7)
    wq16 = _to_bits(wq, dtype)
    wp32 = np.asarray(wp, np.float32)
    q, w = _run_query_only(hidden, qc, c, s, wq16, None, dtype, 0.25,
                           wp_dev=torch.from_numpy(wp32).to("cuda"))
    eq, ew = I.project_query_only(hidden, qc, c, s, wq16, wp32, H, D, ROPE, 0.25, "bf16")
    _close(w, ew, dtype)
    _close(q[..., ROPE:], eq[..., ROPE:], dtype)
    _close(q[..., :ROPE], eq[..., :ROPE], dtype, min_exact=0.95, pairs=True)


def test_project_full_prefill():
    from nanovllm_amd.dsa_indexer_project import dsa_indexer_project

    dtype = torch.bfloat16
    T = 200
    print(f"PROJECT full T={T}", flush=True)
    hidden, qc, c, s = _inputs(T, dtype, seed=9)
    wq, wp, wk = _one_hot()
    kw = _to_bits(np.linspace(0.75, 1.25, D), dtype)
    kb = _to_bits(np.linspace(-0.125, 0.125, D), dtype)
    q_out = torch.empty(T, H, D, dtype=dtype, device="cuda")
    k_out = torch.empty(T, D, dtype=dtype, device="cuda")
    w_out = torch.empty(T, H, dtype=dtype, device="cuda")
    dsa_indexer_project(_dev(hidden, dtype), _dev(qc, dtype), _dev(c, dtype), _dev(s, dtype),
                        _dev(_to_bits(wq, dtype), dtype), _dev(_to_bits(wk, dtype), dtype), _dev(kw, dtype),
                        _dev(kb, dtype), torch.from_numpy(wp).to("cuda"), q_out, k_out, w_out, n_head=H,
                        head_dim=D, rope_dim=ROPE, score_scale=1.0)
    torch.cuda.synchronize()
    eq, ek, ew = I.project_full(hidden, qc, c, s, _to_bits(wq, dtype), _to_bits(wk, dtype), kw, kb, wp, H, D, ROPE,
                                1.0)
    assert np.array_equal(bits(q_out), eq)
    assert np.array_equal(bits(w_out), ew)
    torch.testing.assert_close(k_out.float().cpu(), torch.from_numpy(O.bits_to_f32(ek)), atol=0.05, rtol=0.025)


def test_project_errors():
    from nanovllm_amd.dsa_indexer_project import dsa_indexer_project, dsa_indexer_project_query_only

    dtype = torch.bfloat16
    T = 2
    hidden = torch.zeros(T, HID, dtype=dtype, device="cuda")
    qc = torch.zeros(T, R, dtype=dtype, device="cuda")
    cos = torch.zeros(T, 1, 1, ROPE, dtype=dtype, device="cuda")
    wq = torch.zeros(H * D, R, dtype=dtype, device="cuda")
    wp = torch.zeros(H, HID, dtype=dtype, device="cuda")
    with pytest.raises(ValueError, match=r"q_index_out shape must be \(2, 32, 128\)"):
        dsa_indexer_project_query_only(hidden, qc, cos, cos, wq, wp, torch.empty(T, H, 64, dtype=dtype, device="cuda"),
                                       torch.empty(T, H, dtype=dtype, device="cuda"), n_head=H, head_dim=D,
                                       rope_dim=ROPE, score_scale=1.0)
    with pytest.raises(ValueError, match=r"index_weights_out shape must be \(2, 32\)"):
        dsa_indexer_project_query_only(hidden, qc, cos, cos, wq, wp, torch.empty(T, H, D, dtype=dtype, device="cuda"),
                                       torch.empty(T, 16, dtype=dtype, device="cuda"), n_head=H, head_dim=D,
                                       rope_dim=ROPE, score_scale=1.0)
    with pytest.raises(ValueError, match="index_k_out must use dtype"):
        dsa_indexer_project(hidden, qc, cos, cos, wq, torch.zeros(D, HID, dtype=dtype, device="cuda"),
                            torch.ones(D, dtype=dtype, device="cuda"), None, wp.float(),
                            torch.empty(T, H, D, dtype=dtype, device="cuda"),
                            torch.empty(T, D, dtype=torch.float16, device="cuda"),
                            torch.empty(T, H, dtype=dtype, device="cuda"), n_head=H, head_dim=D, rope_dim=ROPE,
                            score_scale=1.0)
    with pytest.raises(RuntimeError, match="multiple of 256"):
        dsa_indexer_project_query_only(hidden, qc[:, :2000].contiguous(), cos, cos, wq[:, :2000].contiguous(), wp,
                                       torch.empty(T, H, D, dtype=dtype, device="cuda"),
                                       torch.empty(T, H, dtype=dtype, device="cuda"), n_head=H, head_dim=D,
                                       rope_dim=ROPE, score_scale=1.0)


def _tile(tokens, outputs):
    """The tile that the dispatch takes (0: the launch of up to 64 tokens)."""
    from nanovllm_amd import _lib

    return _lib.lib.nvdsa_dsa_indexer_project_tile(tokens, outputs)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,heads,head_dim,rank,rope", [
    (65, 16, 16, 256, 6),        # 64 x 64 tiles, one token in the last
    (1000, 16, 48, 256, 18),     # heads that end inside a 32-wide tile
    (15999, 16, 16, 512, 16),    # 128 x 128 tiles, all dims rotated
    (49001, 16, 16, 256, 10),    # the same, ragged in another place
    (300, 32, 128, 2048, 64),    # the GLM indexer's shape
    (55001, 16, 16, 256, 10),    # 256 x 256 tiles, one round and more
    (4001, 32, 128, 256, 62),    # 256 x 256 tiles, heads of 128, a rotation that ends inside a chunk
])
def test_project_many_tokens_close(dtype, T, heads, head_dim, rank, rope):
    """The tiled GEMM path (more than 64 tokens), every tile shape, ragged
    token counts; guard rows around the output stay untouched."""
    from nanovllm_amd import ops

    print(f"PROJECT GEMM {dtype} T={T} heads={heads}x{head_dim} rank={rank} rope={rope}", flush=True)
    assert _tile(T, heads * head_dim) == {65: 64, 1000: 64, 300: 64, 15999: 128, 49001: 128}.get(T, 256)
    rng = np.random.default_rng(T)
    qc = _to_bits(rng.standard_normal((T, rank)), dtype)
    wq = _to_bits(rng.standard_normal((heads * head_dim, rank)) / np.sqrt(rank), dtype)
    c, s = _cos_sin(T, dtype, rope, seed=T)
    buf = torch.full((T + 2, heads, head_dim), 7.0, dtype=dtype, device="cuda")
    hidden = torch.zeros(T, 64, dtype=dtype, device="cuda")
    ops.indexer_project_query_only(hidden, _dev(qc, dtype), _dev(c, dtype), _dev(s, dtype), _dev(wq, dtype), None,
                                   buf[1:T + 1], None, heads, head_dim, rope, 1.0)
    torch.cuda.synchronize()
    eq, _ = I.project_query_only(np.zeros((T, 64), np.uint16), qc, c, s, wq, np.zeros((heads, 64), np.float32), heads,
                                 head_dim, rope, 1.0, dname(dtype))
    got = bits(buf)
    seven = _to_bits(np.full((heads, head_dim), 7.0), dtype)
    assert np.array_equal(got[0], seven) and np.array_equal(got[T + 1], seven)
    if rope < head_dim:
        _close(got[1:T + 1][..., rope:], eq[..., rope:], dtype)
    _close(got[1:T + 1][..., :rope], eq[..., :rope], dtype, min_exact=0.95, pairs=True)


@pytest.mark.parametrize("shift", [2, 4, 6])
@pytest.mark.parametrize("T,rank,tile", [(64, 256, 0), (65, 256, 64), (130, 512, 64), (8001, 256, 128), (27001, 256, 256)])
def test_project_outputs_at_4_byte_addresses(T, rank, tile, shift):
    """An output 4, 8 or 12 bytes past a 16-byte address holds what an aligned
    one does, and the elements around it stay untouched."""
    from nanovllm_amd import ops

    dtype, heads, head_dim, rope = torch.bfloat16, 16, 32, 18
    assert _tile(T, heads * head_dim) == tile
    print(f"PROJECT unaligned output T={T} rank={rank} shift={shift}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)  # noqa: E731
    args = (rand(T, 64), rand(T, rank), rand(T, rope), rand(T, rope), rand(heads * head_dim, rank), None)
    size = T * heads * head_dim
    aligned = torch.empty(T, heads, head_dim, dtype=dtype, device="cuda")
    buf = torch.full((size + 16,), 7.0, dtype=dtype, device="cuda")
    out = buf[shift:shift + size].view(T, heads, head_dim)
    assert buf.data_ptr() % 16 == 0 and aligned.data_ptr() % 16 == 0
    for q in (aligned, out):
        ops.indexer_project_query_only(*args, q, None, heads, head_dim, rope, 1.0)
    torch.cuda.synchronize()
    assert torch.equal(out, aligned)
    assert (buf[:shift] == 7).all() and (buf[shift + size:] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,heads,hid,fp32,bias", [(1, 16, 64, True, True), (127, 32, 6144, True, False),
                                                   (128, 64, 192, False, True), (129, 32, 6144, True, True),
                                                   (700, 64, 1088, True, True), (33000, 16, 128, False, False)])
def test_project_key_and_weights_kernel(dtype, T, heads, hid, fp32, bias):
    """Index key and head weights of many tokens against the fp64 oracle:
    token tiles' edges, one to many hidden_size slices, fp32 and 16-bit head
    weights."""
    from nanovllm_amd import ops

    print(f"PROJECT kw {dtype} T={T} heads={heads} hid={hid} fp32={fp32}", flush=True)
    rng = np.random.default_rng(T + heads)
    hidden = _to_bits(rng.standard_normal((T, hid)), dtype)
    wk = _to_bits(rng.standard_normal((D, hid)) / np.sqrt(hid), dtype)
    wp = np.asarray(rng.standard_normal((heads, hid)) / np.sqrt(hid), np.float32)
    wp_bits = None if fp32 else _to_bits(wp, dtype)
    kw = _to_bits(rng.uniform(0.75, 1.25, D), dtype)
    kb = _to_bits(rng.uniform(-0.125, 0.125, D), dtype) if bias else None
    c, s = _cos_sin(T, dtype, ROPE, seed=T)
    k_out = torch.full((T + 2, D), 7.0, dtype=dtype, device="cuda")
    w_out = torch.full((T + 2, heads), 7.0, dtype=dtype, device="cuda")
    wp_dev = torch.from_numpy(wp).to("cuda") if fp32 else _dev(wp_bits, dtype)
    ops.indexer_project_kw(_dev(hidden, dtype), _dev(c, dtype), _dev(s, dtype), _dev(wk, dtype), _dev(kw, dtype),
                           _dev(kb, dtype) if bias else None, wp_dev, k_out[1:T + 1], w_out[1:T + 1], ROPE, 0.25)
    only_w = torch.empty(T, heads, dtype=dtype, device="cuda")
    ops.indexer_project_kw(_dev(hidden, dtype), None, None, None, None, None, wp_dev, None, only_w, ROPE, 0.25)
    torch.cuda.synchronize()
    qc, wq = np.zeros((T, 16), np.uint16), np.zeros((heads * D, 16), np.uint16)
    _, ek, ew = I.project_full(hidden, qc, c, s, wq, wk, kw, kb, wp, heads, D, ROPE, 0.25, dname(dtype))
    if not fp32:
        _, ew = I.project_query_only(hidden, qc, c, s, wq, wp_bits, heads, D, ROPE, 0.25, dname(dtype))
    gk, gw = bits(k_out), bits(w_out)
    for g in (gk, gw):
        assert np.array_equal(g[0], _to_bits(np.full(g.shape[1], 7.0), dtype))
        assert np.array_equal(g[T + 1], _to_bits(np.full(g.shape[1], 7.0), dtype))
    _close(gw[1:T + 1], ew, dtype)
    _close(bits(only_w), ew, dtype)
    # A key value is (x - mean) rstd g + b of a sum x rounded to 16 bits.  The
    # fp32 sum may round one step of x away: 2^-8 (bf16) or 2^-11 (fp16) of |x|
    # on either side of a power of two, so 2^-7 / 2^-10 of |x| at most, times
    # rstd g.  With 128 sums of unit variance |mean| stays below 0.5 (5.6
    # sigma), |rstd g| below 1.25 * 1.3, and |b| below 0.125, so
    # |x rstd g| <= |y| + 0.125 + 0.5 * 1.63 < |y| + 0.95.  The value's own
    # rounding adds one step of |y|, the rotation mixes a pair's two values.
    rel = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    g64 = O.bits_to_f32(gk[1:T + 1], dname(dtype)).astype(np.float64)
    e64 = O.bits_to_f32(ek, dname(dtype)).astype(np.float64)
    mag = np.repeat(np.hypot(e64[:, 0::2], e64[:, 1::2]), 2, axis=-1)
    excess = np.abs(g64 - e64) - rel * (2 * mag + 1.41 * 0.95)
    assert np.all(excess <= 0), float(excess.max())
    assert np.mean(gk[1:T + 1] == ek) >= 0.9


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("fp32", [True, False])
def test_project_weights_infinities(dtype, fp32):
    """Infinite and NaN activations and head weights give the infinities and
    NaNs of the products themselves (a NaN only where inf * 0, inf - inf or a
    NaN is summed); the other tokens and heads are those of finite inputs."""
    from nanovllm_amd import ops

    print(f"PROJECT kw infinities {dtype} fp32={fp32}", flush=True)
    T, heads, hid = 70, 16, 192
    rng = np.random.default_rng(5)
    x = torch.from_numpy(rng.integers(1, 4, (T, hid)).astype(np.float32)).to(dtype)
    w = torch.from_numpy(rng.integers(1, 4, (heads, hid)).astype(np.float32) / 64)
    x[3, 7] = float("inf")
    x[4, 9], x[4, 150] = float("inf"), float("-inf")
    x[5, 0] = float("nan")
    w[2, 100] = float("-inf")
    w[6, 20] = float("nan")
    w[8, 7] = 0.0
    w = w if fp32 else w.to(dtype)
    out = torch.empty(T, heads, dtype=dtype, device="cuda")
    ops.indexer_project_kw(x.cuda(), None, None, None, None, None, w.cuda(), None, out, ROPE, 1.0)
    want = (x.double() @ w.double().T).to(dtype)  # (small integers over 64: exact sums, one rounding)
    assert torch.isinf(want).any() and torch.isnan(want).any()
    assert torch.equal(out.cpu().isnan(), want.isnan())
    assert torch.equal(torch.nan_to_num(out.cpu(), nan=1.0), torch.nan_to_num(want, nan=1.0))
