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


def test_outputs_with_gradients_keep_the_library_path():
    hidden = torch.zeros(65, 512, dtype=torch.bfloat16)
    weights, out = torch.zeros(16, 512), torch.zeros(65, 16, dtype=torch.bfloat16)
    assert P._weights_kernel_takes(hidden, weights, out, 16)
    assert not P._weights_kernel_takes(hidden, weights, out.requires_grad_(), 16)
    with torch.no_grad():
        assert P._weights_kernel_takes(hidden, weights, out, 16)
