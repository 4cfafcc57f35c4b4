"""Which runtime inputs of a captured decode step go to the one staging launch
(every element's copy independent of the others) and which to torch copies, on
CPU tensors with the launch recorded."""

from __future__ import annotations

import pytest
import torch

from nanovllm_amd import decode_graph as G

BATCH, HEADS = 4, 4


def _graph(monkeypatch, on_gpu=True):
    """A graph of CPU buffers, and the staging launches it makes (as if the
    buffers were on the current GPU)."""
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16)  # noqa: E731
    g = G.DsaLayerGraph(BATCH, index_key_cache=z(1, 128, 1, 128), cache_slots_pool=torch.zeros(1, 1280),
                        hbm_k_rope=z(1, 128, 1, 64), hbm_kv_cache=z(1, 128, 1, 512), dram_k_rope=z(1, 128, 64),
                        dram_kv_cache=z(1, 128, 512), hbm_block_columns=7, dram_block_columns=9, heads=HEADS,
                        index_heads=32, scale=1.0)
    launches = []
    if on_gpu:
        monkeypatch.setattr(g, "_launches_here", lambda: True)
    monkeypatch.setattr(G._op_impl, "stage_inputs",
                        lambda fields, like: launches.append([fields[i:i + 8] for i in range(0, len(fields), 8)]))
    return g, launches


def _runtime(g, real):
    gen = torch.Generator().manual_seed(real)
    ints = lambda *s: torch.randint(-5, 1000, s, generator=gen, dtype=torch.int32)  # noqa: E731
    runtime = {n: ints(real) for n in G._ROW_INPUTS}
    runtime.update({n: ints(real, cols) for n, cols in zip(G._TABLES, (10, 4, 9))})
    runtime.update({n: torch.randn(real, *g.inputs[n].shape[1:], generator=gen).to(torch.bfloat16)
                    for n in G._QUERY_INPUTS})
    return runtime


def _reads_what_it_writes(items) -> bool:
    """Whether any 2-byte unit is read for one place and written for another
    (units read for their own place are left as they are)."""
    written, read = set(), []
    for dst, src, rows, real, dst_bytes, src_bytes, src_stride, _ in items:
        written.update(range(dst, dst + rows * dst_bytes, 2))
        read += [(src + r * src_stride + c, dst + r * dst_bytes + c) for r in range(real) for c in range(0, src_bytes, 2)]
    return any(a != b and a in written for a, b in read)


@pytest.mark.parametrize("real", [1, 3, BATCH])
@pytest.mark.parametrize("name,cols", [("index_block_table", 9), ("hbm_block_table", 4), ("dram_block_table", 9)])
@pytest.mark.parametrize("compact", [True, False])
def test_own_table_memory(monkeypatch, name, cols, real, compact):
    """A table given as its own buffer's memory: the leading columns stay in
    place; rows of another width are not staged, and arrive as they were."""
    g, launches = _graph(monkeypatch)
    runtime, whole = _runtime(g, real), g.inputs[name]
    whole.copy_(torch.arange(whole.numel(), dtype=torch.int32).view_as(whole))
    runtime[name] = whole.view(-1)[:real * cols].view(real, cols) if compact else whole[:real, :cols]
    expect = torch.zeros_like(whole)
    expect[:real, :cols] = runtime[name]
    g.copy_runtime_inputs(**runtime)
    if compact and real > 1 and cols < whole.shape[1]:
        assert not launches
    if launches:
        assert not _reads_what_it_writes(launches[0])
    else:
        assert torch.equal(whole, expect)


@pytest.mark.parametrize("name", ["num_cache_tokens", "dram_block_table", "query"])
@pytest.mark.parametrize("how", ["entry", "memory"])
def test_replaced_inputs_get_the_step(monkeypatch, name, how):
    """An input whose buffer a caller replaced (a tensor of its own in
    ``inputs``, or other memory under the same tensor) receives the step's
    data, which the captured step reads there."""
    g, launches = _graph(monkeypatch)
    if how == "entry":
        g.inputs[name] = torch.full_like(g.inputs[name], 7)
    else:
        g.inputs[name].data = torch.full_like(g.inputs[name], 7)
    runtime = _runtime(g, 3)
    g.copy_runtime_inputs(**runtime)
    assert not launches
    part = tuple(slice(0, d) for d in runtime[name].shape)
    assert torch.equal(g.inputs[name][part], runtime[name])
    assert not (g.inputs[name] == 7).any() or (runtime[name] == 7).any()


def test_staged_inputs_count_as_written(monkeypatch):
    g, launches = _graph(monkeypatch)
    before = {n: t._version for n, t in g.inputs.items()}
    g.copy_runtime_inputs(**_runtime(g, 2))
    assert launches
    assert all(t._version > before[n] for n, t in g.inputs.items())


def test_host_buffers_take_the_copies(monkeypatch):
    """A graph object over host memory copies its inputs there, also where
    there is no GPU."""
    g, launches = _graph(monkeypatch, on_gpu=False)
    runtime = _runtime(g, 3)
    assert g.copy_runtime_inputs(**runtime) == 3 and not launches
    for name, t in runtime.items():
        assert torch.equal(g.inputs[name][tuple(slice(0, d) for d in t.shape)], t)
    assert (g.inputs["req_pool_entries"][3:] == -1).all() and not g.inputs["query"][3:].any()
