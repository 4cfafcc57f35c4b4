"""HIP-graph replay of the DSA decode layer-step at fixed batch sizes.

The reference replays its whole stable decode step from captured graphs,
one per exact batch size, with every per-step input copied into
fixed-address buffers first (FullDecodeOnlyGraphManager and
FullDecodeGraphEntry, nanovllm/engine/full_decode_graph.py:33-57, :140-385,
:546-720).  This module does the same for the path this library owns: the
layer-step ``fused_li_manage(_mtp) -> fused_copy_sfa(_mtp)``.

* :func:`normalize_capture_sizes` / :func:`select_capture_size` keep the
  reference's rules (:33-57): sorted distinct positive sizes; a runtime batch
  runs in the smallest captured size that holds it.
* :class:`DsaLayerGraph` owns the static inputs and outputs of one batch
  size, captures the step once (after one eager warm-up that also sizes the
  operator workspaces) and replays it.  Rows past the runtime batch are
  padded so that every kernel skips them: no candidates, pool entry -1, no
  cache budget, zero visible length (LIM row guard, zero attention output).
  Tables narrower than the graph buffers are copied left-aligned and the
  rest zeroed (the reference's ``_copy_table``, :227-248).
* The KV caches, index keys and the LIDU pool are the caller's persistent
  tensors; their addresses are baked into the graph, as in the reference.

Inputs are copied on the current stream before each replay, all in one
launch (``nvdsa_stage_inputs``; with a tensor of another device, dtype or
layout among them, by ordinary torch copies); nothing inside the graph is a
memset.
"""

from __future__ import annotations

import math
import operator
from typing import Iterable

import torch
from torch.autograd.graph import increment_version

from . import dsa_offload_ops as ops
from . import ops as _op_impl

MTP_QUERIES = 4
TOPK = 2048


def normalize_capture_sizes(values: Iterable[int]) -> tuple[int, ...]:
    """Validate, sort and deduplicate capture batch sizes (reference :33-45)."""
    sizes = tuple(sorted({int(v) for v in values}))
    if not sizes:
        raise ValueError("FULL_DECODE_ONLY requires at least one decode graph capture size. "
                         "Pass decode_graph_capture_sizes, for example (16,).")
    if sizes[0] <= 0:
        raise ValueError(f"Decode graph capture sizes must be positive, got {sizes}.")
    return sizes


def select_capture_size(real_batch_size: int, capture_sizes: Iterable[int]) -> int | None:
    """The smallest captured size that holds the batch (reference :48-56)."""
    for size in capture_sizes:
        if int(size) >= int(real_batch_size):
            return int(size)
    return None


# Per-request inputs and their padding value for rows past the runtime batch.
_ROW_INPUTS = {
    "num_candidate_tokens": 0,
    "num_cache_tokens": 0,
    "req_pool_entries": -1,
    "actual_seq_lengths_query": 1,
    "actual_seq_lengths_kv": 0,
}
_TABLES = ("index_block_table", "hbm_block_table", "dram_block_table")
# Per-query-row inputs (rows = requests x queries per request).
_QUERY_INPUTS = ("query_index", "index_weights", "query_rope", "query")


class DsaLayerGraph:
    """One captured DSA layer-step for ``batch_size`` requests."""

    def __init__(self, batch_size: int, *, index_key_cache: torch.Tensor, cache_slots_pool: torch.Tensor,
                 hbm_k_rope: torch.Tensor, hbm_kv_cache: torch.Tensor, dram_k_rope: torch.Tensor,
                 dram_kv_cache: torch.Tensor, hbm_block_columns: int, dram_block_columns: int, heads: int,
                 index_heads: int, scale: float, mtp: bool = False, dtype: torch.dtype = torch.bfloat16) -> None:
        if batch_size <= 0:
            raise ValueError(f"batch_size must be positive, got {batch_size}")
        # The LIM operators require the index table to span the pool row
        # (S_cap == table columns * 128).
        index_block_columns = int(cache_slots_pool.shape[1]) // 128
        dev = hbm_kv_cache.device
        B = int(batch_size)
        q = MTP_QUERIES if mtp else 1
        rows = B * q
        i32 = dict(dtype=torch.int32, device=dev)
        f16 = dict(dtype=dtype, device=dev)
        self.batch_size, self.mtp, self.scale = B, bool(mtp), float(scale)
        self.persistent = dict(index_key_cache=index_key_cache, cache_slots_pool=cache_slots_pool,
                               hbm_k_rope=hbm_k_rope, hbm_kv_cache=hbm_kv_cache, dram_k_rope=dram_k_rope,
                               dram_kv_cache=dram_kv_cache)
        shapes = {
            "query_index": ((rows, index_heads, 128), dtype),
            "index_weights": ((rows, index_heads), dtype),
            "query_rope": ((rows, heads, 64), dtype),
            "query": ((rows, heads, 512), dtype),
            "index_block_table": ((B, index_block_columns), torch.int32),
            "hbm_block_table": ((B, hbm_block_columns), torch.int32),
            "dram_block_table": ((B, dram_block_columns), torch.int32),
            **{name: ((B,), torch.int32) for name in _ROW_INPUTS},
        }
        # One block of memory holds every static input (256-byte steps), so
        # whether a runtime tensor lies in any of them is one comparison.
        self._nbytes = {k: math.prod(shape) * dt.itemsize for k, (shape, dt) in shapes.items()}
        offsets, total = {}, 0
        for k, n in self._nbytes.items():
            offsets[k] = total
            total += -(-n // 256) * 256
        self._block = torch.zeros(max(total, 256), dtype=torch.uint8, device=dev)
        self._span = (self._block.data_ptr(), self._block.data_ptr() + self._block.numel())
        self._address = {k: self._span[0] + o for k, o in offsets.items()}
        self.inputs = {k: self._block[offsets[k]:offsets[k] + self._nbytes[k]].view(dt).view(shape)
                       for k, (shape, dt) in shapes.items()}
        self._buffers = list(self.inputs.values())
        self._pointers = [t.data_ptr() for t in self._buffers]
        for name, pad in _ROW_INPUTS.items():
            self.inputs[name].fill_(pad)
        self.outputs = {
            "topk_src_ids": torch.full((rows, 1, TOPK), -1, **i32),
            "topk_dst_slots": torch.full((rows, 1, TOPK), -1, **i32),
            "miss_counts": torch.zeros(B, **i32),
            "attention_out": torch.zeros(rows, heads, 512, **f16),
        }
        if mtp:
            self.outputs["miss_src_ids"] = torch.full((B, MTP_QUERIES * TOPK), -1, **i32)
            self.outputs["miss_dst_slots"] = torch.full((B, MTP_QUERIES * TOPK), -1, **i32)
        self._device = self._block.device
        self.graph: torch.cuda.CUDAGraph | None = None
        self.real_batch = 0
        self.replay_count = 0

    # -- the captured step ----------------------------------------------------
    def _step(self) -> None:
        i, o, p = self.inputs, self.outputs, self.persistent
        lim = (i["query_index"], i["index_weights"], p["index_key_cache"], i["index_block_table"],
               i["num_candidate_tokens"], i["num_cache_tokens"], i["req_pool_entries"], p["cache_slots_pool"],
               o["topk_src_ids"], o["topk_dst_slots"])
        common = (i["query_rope"], i["query"], i["actual_seq_lengths_query"], i["actual_seq_lengths_kv"],
                  i["num_cache_tokens"], o["topk_dst_slots"])
        caches = (i["hbm_block_table"], i["dram_block_table"], p["hbm_k_rope"], p["hbm_kv_cache"], p["dram_k_rope"],
                  p["dram_kv_cache"], self.scale, o["attention_out"])
        if self.mtp:
            ops.fused_li_manage_mtp(*lim, o["miss_src_ids"], o["miss_dst_slots"], o["miss_counts"])
            ops.fused_copy_sfa_mtp(*common, o["topk_src_ids"], o["miss_src_ids"], o["miss_dst_slots"],
                                   o["miss_counts"], *caches)
        else:
            ops.fused_li_manage(*lim, o["miss_counts"])
            ops.fused_copy_sfa(*common, o["topk_src_ids"].view(self.batch_size, TOPK), o["miss_counts"], *caches)

    def capture(self) -> None:
        """Warm up eagerly on a side stream (sizes the operator workspaces),
        then capture the step.  The warm-up runs with every row padded, so
        it changes no pool row and copies nothing."""
        stream = torch.cuda.Stream(device=self.outputs["miss_counts"].device)
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            self._step()
        stream.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=stream):
            self._step()
        torch.cuda.current_stream().wait_stream(stream)

    # -- per-step inputs --------------------------------------------------------
    def _launches_here(self) -> bool:
        """Whether the buffers are on the current GPU."""
        return self._device.type == "cuda" and torch.cuda.current_device() == self._device.index

    def _own_buffers(self) -> bool:
        """Whether the inputs are still the buffers that this object made: a
        caller may put tensors of its own into ``inputs`` before the capture."""
        inputs = self.inputs.values()
        return (len(inputs) == len(self._buffers) and all(map(operator.is_, inputs, self._buffers))
                and list(map(torch.Tensor.data_ptr, inputs)) == self._pointers)

    def _source(self, name: str, src: torch.Tensor) -> int | None:
        """The address from which the staging kernel may read ``src`` for buffer
        ``name``, if it is a plain tensor of the buffer's dtype on its device,
        outside the static inputs' memory or the buffer itself."""
        if type(src) is not torch.Tensor or src.dtype != self.inputs[name].dtype or src.device != self._device:
            return None
        at = src.data_ptr()
        lo, hi = self._span
        return None if (lo <= at < hi and at != self._address[name]) or src.requires_grad or src.is_neg() else at

    def _copy_inputs(self, runtime: dict[str, torch.Tensor], real: int) -> None:
        """The same with torch copies (any device, dtype and layout)."""
        q = MTP_QUERIES if self.mtp else 1
        for name, pad in _ROW_INPUTS.items():
            self.inputs[name][:real].copy_(runtime[name])
            self.inputs[name][real:].fill_(pad)
        for name in _TABLES:
            src, dst = runtime[name], self.inputs[name]
            if src.data_ptr() == dst.data_ptr() and src.stride() != dst.stride():
                src = src.clone()  # the buffer's own memory in other rows
            dst[:real, :src.shape[1]].copy_(src)
            dst[:real, src.shape[1]:].zero_()
            dst[real:].zero_()
        for name in _QUERY_INPUTS:
            dst = self.inputs[name]
            dst[:real * q].copy_(runtime[name])
            dst[real * q:].zero_()

    def copy_runtime_inputs(self, **runtime: torch.Tensor) -> int:
        """Copy one step's inputs into the static buffers; returns the runtime
        batch.  Every name in ``_ROW_INPUTS``, ``_TABLES`` and
        ``_QUERY_INPUTS`` is required."""
        missing = [n for n in (*_ROW_INPUTS, *_TABLES, *_QUERY_INPUTS) if n not in runtime]
        if missing:
            raise ValueError(f"missing runtime inputs: {missing}")
        real = int(runtime["num_candidate_tokens"].shape[0])
        if real > self.batch_size:
            raise ValueError(f"runtime batch {real} exceeds the graph's batch size {self.batch_size}")
        q = MTP_QUERIES if self.mtp else 1
        # Every check first, then one launch that moves what the kernel reads
        # as it is (same device and dtype, contiguous rows).  Anything else
        # sends the whole step through torch copies, one after another.
        staged: list[int] = []
        plain = self._launches_here() and self._own_buffers()
        for name, pad in _ROW_INPUTS.items():
            src = runtime[name]
            if src.shape != (real,):
                raise ValueError(f"{name} must be [{real}], got {tuple(src.shape)}")
            at = self._source(name, src) if plain else None
            plain = at is not None and src.is_contiguous()
            if plain:
                staged += (self._address[name], at, 1, 1, 4 * self.batch_size, 4 * real, 0, pad)
        for name in _TABLES:
            src, width = runtime[name], self.inputs[name].shape[1]
            shape = src.shape
            if len(shape) != 2 or shape[0] != real:
                raise ValueError(f"{name} must be rank 2 with {real} rows, got {tuple(shape)}")
            if shape[1] > width:
                raise ValueError(f"{name} is wider than its graph buffer: runtime={shape[1]}, graph={width}.")
            # (Rows of the buffer's own memory at another stride would be read
            # where other rows are written.)
            at = self._source(name, src) if plain else None
            plain = (at is not None and src.stride(1) == 1
                     and (at != self._address[name] or src.stride(0) == width or real <= 1))
            if plain:
                staged += (self._address[name], at, self.batch_size, real, 4 * width, 4 * shape[1],
                           4 * src.stride(0), 0)
        for name in _QUERY_INPUTS:
            src, dst = runtime[name], self.inputs[name]
            if src.shape[0] != real * q or src.shape[1:] != dst.shape[1:]:
                raise ValueError(f"{name} must be [{real * q}, {', '.join(map(str, dst.shape[1:]))}], "
                                 f"got {tuple(src.shape)}")
            at = self._source(name, src) if plain else None
            plain = at is not None and src.is_contiguous()
            if plain:
                nbytes = self._nbytes[name]
                staged += (self._address[name], at, 1, 1, nbytes, nbytes // self.batch_size * real, 0, 0)
        if plain:
            _op_impl.stage_inputs(staged, self._block)
            increment_version(self._block)  # written, for autograd (its views, the inputs, share the counter)
        else:
            self._copy_inputs(runtime, real)
        self.real_batch = real
        return real

    def replay(self, **runtime: torch.Tensor) -> dict[str, torch.Tensor]:
        """Copy the inputs (when given), replay, and return views of the
        outputs for the runtime rows."""
        if self.graph is None:
            raise RuntimeError("the graph is not captured; call capture() first")
        if runtime:
            self.copy_runtime_inputs(**runtime)
        self.graph.replay()
        self.replay_count += 1
        real = self.real_batch
        q = MTP_QUERIES if self.mtp else 1
        out = {k: (v[:real] if k in ("miss_counts", "miss_src_ids", "miss_dst_slots") else v[:real * q])
               for k, v in self.outputs.items()}
        return out


__all__ = ["DsaLayerGraph", "normalize_capture_sizes", "select_capture_size"]
