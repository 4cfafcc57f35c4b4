"""Which indexer projections take the kernels of many tokens: what the one
launch of up to 64 tokens refuses stays refused past them, and outputs that
ask for a gradient keep the library path (whose copy refuses or records
them)."""

from __future__ import annotations

import pytest
import torch

from nanovllm_amd import dsa_indexer_project as P


@pytest.mark.parametrize("tokens,hidden,shift,split", [(64, 512, 0, False), (65, 512, 0, True), (65, 576, 0, False),
                                                       (65, 512, 1, False)])
def test_16_bit_head_weights_keep_their_limits(monkeypatch, tokens, hidden, shift, split):
    """hidden_size of 576 and outputs on odd 16-bit words go to the one launch,
    which refuses them, at any token count."""
    calls = []
    monkeypatch.setattr(P.ops, "indexer_project_query_only", lambda *a: calls.append(a[5] is not None))
    monkeypatch.setattr(P.ops, "indexer_project_kw", lambda *a: calls.append("kw"))
    z = lambda *shape: torch.zeros(*shape, dtype=torch.bfloat16)  # noqa: E731
    out = z(tokens * 16 + 8)[shift:shift + tokens * 16].view(tokens, 16)
    P.dsa_indexer_project_query_only(z(tokens, hidden), z(tokens, 256), z(tokens, 8), z(tokens, 8), z(256, 256),
                                     z(16, hidden), z(tokens, 16, 16), out, n_head=16, head_dim=16, rope_dim=8,
                                     score_scale=1.0)
    assert calls == ([False, "kw"] if split else [True])


@pytest.mark.parametrize("tokens,heads,rank,one", [
    (65, 32, 2048, True), (160, 32, 2048, True), (161, 32, 2048, False), (192, 32, 512, True), (193, 32, 512, False),
    (80, 64, 1536, True), (81, 64, 1536, False), (256, 16, 2048, True), (257, 16, 2048, False), (384, 16, 512, True),
    (385, 16, 512, False),
])
def test_16_bit_head_weights_by_size(monkeypatch, tokens, heads, rank, one):
    """q and the head weights in one launch up to the size where the three
    launches of many tokens are the shorter way."""
    calls = []
    monkeypatch.setattr(P.ops, "indexer_project_query_only", lambda *a: calls.append(a[5] is not None))
    monkeypatch.setattr(P.ops, "indexer_project_kw", lambda *a: calls.append("kw"))
    z = lambda *shape: torch.zeros(*shape, dtype=torch.bfloat16)  # noqa: E731
    P.dsa_indexer_project_query_only(z(tokens, 512), z(tokens, rank), z(tokens, 64), z(tokens, 64), z(heads * 128, rank),
                                     z(heads, 512), z(tokens, heads, 128), z(tokens, heads), n_head=heads, head_dim=128,
                                     rope_dim=64, score_scale=1.0)
    assert calls == ([True] if one else [False, "kw"])


def test_outputs_with_gradients_keep_the_library_path():
    hidden = torch.zeros(65, 512, dtype=torch.bfloat16)
    weights, out = torch.zeros(16, 512), torch.zeros(65, 16, dtype=torch.bfloat16)
    assert P._weights_kernel_takes(hidden, weights, out, 16)
    assert not P._weights_kernel_takes(hidden, weights, out.requires_grad_(), 16)
    with torch.no_grad():
        assert P._weights_kernel_takes(hidden, weights, out, 16)


@pytest.mark.parametrize("dual", ["hidden", "weights", "wk", "norm"])
def test_forward_mode_derivatives_are_handed_on(monkeypatch, dual):
    """A tangent of an input reaches the outputs that depend on it."""
    from torch.autograd import forward_ad

    monkeypatch.setattr(P.ops, "indexer_project_query_only", lambda *a: None)
    monkeypatch.setattr(P.ops, "indexer_project_kw", lambda *a: None)
    monkeypatch.setattr(P.ops, "dsa_indexer_query_rope_inplace", lambda *a: None)
    z = lambda *shape: torch.zeros(*shape, dtype=torch.bfloat16)  # noqa: E731
    gen = torch.Generator().manual_seed(1)
    half = lambda *shape: torch.randn(*shape, generator=gen).to(torch.bfloat16)  # noqa: E731
    T = 3
    ins = {"hidden": half(T, 64), "weights": torch.randn(16, 64, generator=gen), "wk": half(128, 64), "norm": half(128)}
    plain = dict(ins)
    with forward_ad.dual_level():
        tangent = torch.ones_like(ins[dual])
        ins[dual] = forward_ad.make_dual(ins[dual], tangent)
        q, k, w = z(T, 16, 128), z(T, 128), z(T, 16)
        P.dsa_indexer_project(ins["hidden"], z(T, 256), z(T, 8), z(T, 8), z(2048, 256), ins["wk"], ins["norm"], None,
                              ins["weights"], q, k, w, n_head=16, head_dim=128, rope_dim=8, score_scale=0.5)
        dk, dw = (forward_ad.unpack_dual(t).tangent for t in (k, w))
        w2 = z(T, 16)
        P.dsa_indexer_project_query_only(ins["hidden"], z(T, 256), z(T, 8), z(T, 8), z(2048, 256), ins["weights"], q, w2,
                                         n_head=16, head_dim=128, rope_dim=8, score_scale=0.5)
        dw2 = forward_ad.unpack_dual(w2).tangent
    if dual in ("hidden", "weights"):
        a, b = (tangent, plain["weights"]) if dual == "hidden" else (plain["hidden"], tangent)
        expect = (a.float() @ b.float().T * 0.5).to(torch.bfloat16)
        for d in (dw, dw2):
            torch.testing.assert_close(d, expect, rtol=2.0 ** -7, atol=2.0 ** -7)
    if dual != "weights":
        assert dk is not None


class _Scaled(torch.Tensor):
    """A tensor whose values are not its memory's (as of quantised weights)."""

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        return super().__torch_function__(func, types, args, kwargs or {})


class _Loaded(torch.nn.Parameter):
    """A parameter class that only adds attributes (weight loaders)."""


@pytest.mark.parametrize("which", ["hidden", "weights"])
@pytest.mark.parametrize("form", ["plain", "parameter", "loaded", "negated", "subclass", "sparse"])
def test_only_plain_memory_goes_to_the_kernel(which, form):
    make = {"plain": lambda t: t, "parameter": lambda t: torch.nn.Parameter(t, requires_grad=False),
            "loaded": lambda t: _Loaded(t, requires_grad=False), "negated": torch._neg_view,
            "subclass": lambda t: t.as_subclass(_Scaled), "sparse": lambda t: t.to_sparse()}[form]
    ins = {"hidden": torch.ones(3, 64, dtype=torch.bfloat16), "weights": torch.ones(16, 64)}
    ins[which] = make(ins[which])
    out = torch.zeros(3, 16, dtype=torch.bfloat16)
    assert P._weights_kernel_takes(ins["hidden"], ins["weights"], out, 16) == (form in ("plain", "parameter", "loaded"))


def test_outputs_count_as_written(monkeypatch):
    """Autograd refuses a backward pass through values that a later call
    overwrote, as it does after the library path's copies."""
    monkeypatch.setattr(P.ops, "indexer_project_query_only", lambda *a: None)
    monkeypatch.setattr(P.ops, "indexer_project_kw", lambda *a: None)
    z = lambda *shape: torch.zeros(*shape, dtype=torch.bfloat16)  # noqa: E731
    q, k, w, scale = z(3, 16, 128), z(3, 128), z(3, 16), torch.ones(3, 16, requires_grad=True)
    loss = (w * scale).sum()
    P.dsa_indexer_project_query_only(z(3, 64), z(3, 256), z(3, 16), z(3, 16), z(2048, 256), torch.zeros(16, 64), q, w,
                                     n_head=16, head_dim=128, rope_dim=16, score_scale=0.5)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()
    before = k._version, w._version
    P.dsa_indexer_project(z(3, 64), z(3, 256), z(3, 16), z(3, 16), z(2048, 256), z(128, 64), z(128), None,
                          torch.zeros(16, 64), q, k, w, n_head=16, head_dim=128, rope_dim=16, score_scale=0.5)
    assert k._version > before[0] and w._version > before[1]


@pytest.mark.parametrize("rope_dim,kernel", [(64, True), (16, True), (6, False), (40, False)])
def test_key_rotation_keeps_its_limits(monkeypatch, rope_dim, kernel):
    """A rope_dim that is no multiple of 16 goes to the key's RoPE operator,
    which refuses it."""
    calls = []
    monkeypatch.setattr(P.ops, "indexer_project_query_only", lambda *a: None)
    monkeypatch.setattr(P.ops, "indexer_project_kw", lambda *a: calls.append("kw"))
    monkeypatch.setattr(P.ops, "dsa_indexer_query_rope_inplace", lambda *a: calls.append(a[3]))
    z = lambda *shape: torch.zeros(*shape, dtype=torch.bfloat16)  # noqa: E731
    P.dsa_indexer_project(z(3, 64), z(3, 256), z(3, 64), z(3, 64), z(2048, 256), z(128, 64), z(128), None,
                          torch.zeros(16, 64), z(3, 16, 128), z(3, 128), z(3, 16), n_head=16, head_dim=128,
                          rope_dim=rope_dim, score_scale=0.5)
    assert calls == (["kw"] if kernel else [rope_dim])
