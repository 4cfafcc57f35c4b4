"""DSA indexer projection on MI355X: the producer of the LIM inputs.

Mirrors the two public functions of the reference module
nanovllm/models/dsa_indexer_project.py (same names, arguments, output
buffers and ``ValueError`` conditions):

* :func:`dsa_indexer_project_query_only` (reference :296-355), the stable
  decode path: ``q_index = RoPE(q_c . wq_b^T)`` and
  ``index_weights = hidden . weights_proj^T * score_scale``.  When
  ``weights_proj_weight`` shares the activations' dtype (the decode graph's
  cached low-precision copy, nanovllm/models/glm_mla.py:262-271) both come
  from one fused gfx950 launch (``nvdsa_dsa_indexer_project_query_only``).
  fp32 weights, and any weights of many tokens (from 65 to 385 on, by the
  sizes: :func:`_one_launch`), take launches of their own
  (``nvdsa_dsa_indexer_project_kw``: exact products, fp32 sums, one cast, as
  the reference computes them, :82-86) where the tensors are plain
  (contiguous, aligned, no derivative asked for), and fp32 ones an fp32 library
  GEMM otherwise.  ``wq_b_bmm_t`` / ``enable_q_bmm`` are accepted for signature
  parity; the kernels read ``wq_b_weight`` in its natural [H*D, R] layout, so
  the transposed BMM copy (an Ascend layout, :102-130) is not used.
* :func:`dsa_indexer_project` (reference :245-293), the prefill path: q as
  above, ``index_k = RoPE(LayerNorm(hidden . wk^T))`` and fp32 weights in one
  pass over ``hidden_states`` under the same conditions.  Otherwise the k
  projection and layer norm are library calls and its RoPE the HIP kernel
  behind ``torch.ops.nanovllm_dsa.dsa_indexer_query_rope_inplace``.

RoPE is the interleaved-pair rotation of the reference's AscendC kernel
(ops/dsa_indexer_project/op_kernel/dsa_indexer_project_kernel.cpp:105-176):
fp32 products and sum, rounded once to the 16-bit dtype.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.autograd.graph import increment_version  # what the library path's copies do to their outputs

from . import ops


def _check_project_outputs(q_index_out, index_k_out, index_weights_out, *, num_tokens, n_head, head_dim, dtype,
                           device) -> None:
    """The reference's output checks (dsa_indexer_project.py:135-155)."""
    if q_index_out.shape != (num_tokens, n_head, head_dim):
        raise ValueError(f"q_index_out shape must be {(num_tokens, n_head, head_dim)}, got {tuple(q_index_out.shape)}")
    if index_k_out.shape != (num_tokens, head_dim):
        raise ValueError(f"index_k_out shape must be {(num_tokens, head_dim)}, got {tuple(index_k_out.shape)}")
    if index_weights_out.shape != (num_tokens, n_head):
        raise ValueError(f"index_weights_out shape must be {(num_tokens, n_head)}, got {tuple(index_weights_out.shape)}")
    for name, tensor in (("q_index_out", q_index_out), ("index_k_out", index_k_out),
                         ("index_weights_out", index_weights_out)):
        if tensor.dtype != dtype or tensor.device != device:
            raise ValueError(f"{name} must use dtype={dtype} and device={device}, got dtype={tensor.dtype} "
                             f"device={tensor.device}")
        if not tensor.is_contiguous():
            raise ValueError(f"{name} must be contiguous")


def _rope_cos_sin(cos: torch.Tensor, sin: torch.Tensor, tokens: int, rope_dim: int):
    """cos/sin as the [T, 1, 1, rope_dim] tensors the RoPE op reads (the
    reference's reshape(T, -1)[..., :rope_dim], :28-32)."""
    c = cos.reshape(tokens, -1)[..., :rope_dim].contiguous().view(tokens, 1, 1, rope_dim)
    s = sin.reshape(tokens, -1)[..., :rope_dim].contiguous().view(tokens, 1, 1, rope_dim)
    return c, s


def _weights_fp32(hidden_states, weights_proj_weight, score_scale: float) -> torch.Tensor:
    """Reference :82-86 (dtype mismatch): fp32 projection, scale, one cast."""
    weights = F.linear(hidden_states.float(), weights_proj_weight.float())
    if float(score_scale) != 1.0:
        weights = weights * float(score_scale)
    return weights.to(hidden_states.dtype)


_TYPES, _STRIDED = frozenset((torch.Tensor, torch.nn.Parameter)), torch.strided


def _plain_type(cls) -> bool:
    """Tensors, parameters, and parameter classes that leave torch's functions
    as they are."""
    return cls in _TYPES or (cls.__torch_function__ is torch.nn.Parameter.__torch_function__
                             and cls.__torch_dispatch__ is torch.Tensor.__torch_dispatch__)


def _plain(t, shape, dtypes, device, align=16) -> bool:
    """A contiguous tensor of this shape whose memory holds its values as the
    HIP kernels read them (no subclass, lazy negation or sparse layout)."""
    return ((type(t) in _TYPES or _plain_type(type(t))) and t.layout is _STRIDED and t.shape == shape
            and t.dtype in dtypes and t.device == device and not t.is_neg() and t.is_contiguous()
            and t.data_ptr() % align == 0)


def _derivatives_asked(*tensors) -> bool:
    """Whether autograd follows any of the tensors, in either mode: only the
    library path hands derivatives on."""
    # (The level is below 0 outside every forward_ad.dual_level().)
    dual = getattr(forward_ad, "_current_level", 0) >= 0
    grad = torch.is_grad_enabled()
    if grad or dual:
        for t in tensors:
            if (grad and t.requires_grad) or (dual and forward_ad.unpack_dual(t).tangent is not None):
                return True
    return False


def _weights_kernel_takes(hidden_states, weights_proj_weight, index_weights_out, n_head) -> bool:
    """Whether the head weights can come from the fp32-product kernel
    (nvdsa_dsa_indexer_project_kw): plain tensors of the indexer's shapes;
    any other form keeps the library GEMM."""
    if hidden_states.dim() != 2 or weights_proj_weight.dim() != 2 or hidden_states.shape[0] == 0:
        return False
    hidden = hidden_states.shape[1]
    dtype, device = hidden_states.dtype, hidden_states.device
    return (dtype in (torch.bfloat16, torch.float16) and n_head in (16, 32, 64) and hidden > 0 and hidden % 64 == 0
            and _plain(hidden_states, hidden_states.shape, (dtype,), device)
            and _plain(weights_proj_weight, (n_head, hidden), (dtype, torch.float32), device)
            and _plain(index_weights_out, (hidden_states.shape[0], n_head), (dtype,), device, 2)
            and not _derivatives_asked(hidden_states, weights_proj_weight, index_weights_out))


def _one_launch(tokens: int, n_head: int, head_dim: int, rank: int) -> bool:
    """Whether q and 16-bit head weights come from the fused decode launch:
    for one 64-token group, and for more while reading wq_b again for each
    group costs less than the three launches of many tokens (the tiled GEMM,
    the head weights and their sum), whose time hardly grows with the tokens.
    bf16, us of one launch / of three:

         heads  rank  hidden   65     96    128    160    192    256    320
        32x128  2048    6144  20/33  24/34  30/35  38/34  43/34  57/37  70/38
        32x128  1536    5120  16/30  19/30  23/32  30/31  34/31  44/33  55/35
        32x128   512    2048  11/22  12/22  14/22  18/22  20/22  26/22  32/22
        64x128  2048    6144  39/44  47/44  58/45  74/45  84/46 111/46 137/49
        64x128   512    2048  19/23  23/22  26/24  35/23  38/24  50/25  63/27
        16x128  2048    6144  15/33  15/33  15/33  22/33  28/33  28/35  41/34
         64x64  1536    6144  19/33  22/33  28/33  35/34  40/34  53/34  65/37

    fp16 the same within 3 us.  Called from Python the three take 40 us of host
    time whatever the tokens, so the line lies at the upper end of where they
    cross.  Heads narrower than 64 keep the one group (a call of 65 to 512
    tokens, 16x16 heads: 33 to 34 us either way)."""
    if tokens <= 64 or head_dim < 64:
        return tokens <= 64
    most, outputs = (256, 5 * 2 ** 17) if rank > 1024 else (384, 6 * 2 ** 17)
    return tokens <= most and tokens * n_head * head_dim <= outputs


def dsa_indexer_project_query_only(hidden_states, q_c, cos, sin, wq_b_weight, weights_proj_weight, q_index_out,
                                   index_weights_out, *, n_head, head_dim, rope_dim, score_scale, wq_b_bmm_t=None,
                                   enable_q_bmm=False):
    """Decode-only indexer projection (reference dsa_indexer_project.py:296-355)."""
    del wq_b_bmm_t, enable_q_bmm  # the fused kernel reads wq_b_weight directly
    tokens = hidden_states.shape[0]
    if q_index_out.shape != (tokens, n_head, head_dim):
        raise ValueError(f"q_index_out shape must be {(tokens, n_head, head_dim)}, got {tuple(q_index_out.shape)}")
    if index_weights_out.shape != (tokens, n_head):
        raise ValueError(f"index_weights_out shape must be {(tokens, n_head)}, got {tuple(index_weights_out.shape)}")
    same = weights_proj_weight.dtype == hidden_states.dtype
    # One launch for both while that is the shorter way; more tokens (or fp32
    # head weights) take the head weights' own kernel where it reads their
    # form.  (16-bit weights only in the sizes that the one launch takes too).
    if ((not same or (not _one_launch(tokens, n_head, head_dim, q_c.shape[-1])
                      and hidden_states.shape[-1] % 512 == 0 and index_weights_out.data_ptr() % 4 == 0))
            and _weights_kernel_takes(hidden_states, weights_proj_weight, index_weights_out, n_head)):
        ops.indexer_project_query_only(hidden_states, q_c, cos, sin, wq_b_weight, None, q_index_out, None, n_head,
                                       head_dim, rope_dim, score_scale)
        ops.indexer_project_kw(hidden_states, None, None, None, None, None, weights_proj_weight, None,
                               index_weights_out, rope_dim, score_scale)
        increment_version(index_weights_out)
        return q_index_out, index_weights_out
    ops.indexer_project_query_only(hidden_states, q_c, cos, sin, wq_b_weight, weights_proj_weight if same else None,
                                   q_index_out, index_weights_out if same else None, n_head, head_dim, rope_dim,
                                   score_scale)
    if not same:
        index_weights_out.copy_(_weights_fp32(hidden_states, weights_proj_weight, score_scale))
    return q_index_out, index_weights_out


def dsa_indexer_project(hidden_states, q_c, cos, sin, wq_b_weight, wk_weight, k_norm_weight, k_norm_bias,
                        weights_proj_weight, q_index_out, index_k_out, index_weights_out, *, n_head, head_dim,
                        rope_dim, score_scale, wq_b_bmm_t=None, enable_q_bmm=False):
    """Prefill indexer projection (reference dsa_indexer_project.py:245-293)."""
    del wq_b_bmm_t, enable_q_bmm
    tokens = int(hidden_states.shape[0])
    _check_project_outputs(q_index_out, index_k_out, index_weights_out, num_tokens=tokens, n_head=int(n_head),
                           head_dim=int(head_dim), dtype=hidden_states.dtype, device=hidden_states.device)
    # q: projection + RoPE in one launch (no weights part).
    ops.indexer_project_query_only(hidden_states, q_c, cos, sin, wq_b_weight, None, q_index_out, None, n_head,
                                   head_dim, rope_dim, 1.0)
    # k and the head weights: one pass over hidden_states where every tensor
    # has the plain form that the kernels read (weights_proj_weight in fp32,
    # or in 16 bits, which only the library path widens before the product).
    dtype, device = hidden_states.dtype, hidden_states.device
    norm = (k_norm_weight,) if k_norm_bias is None else (k_norm_weight, k_norm_bias)
    # (A rope_dim that the key's RoPE operator refuses goes there too.)
    if (weights_proj_weight.dtype == torch.float32 and int(head_dim) == 128 and k_norm_weight is not None
            and int(rope_dim) % 16 == 0
            and _weights_kernel_takes(hidden_states, weights_proj_weight, index_weights_out, int(n_head))
            and _plain(wk_weight, (128, hidden_states.shape[1]), (dtype,), device)
            and _plain(k_norm_weight, (128,), (dtype,), device, 4)
            and (k_norm_bias is None or _plain(k_norm_bias, (128,), (dtype,), device, 4))
            and (cos.numel() // tokens) % 2 == 0 and index_k_out.data_ptr() % 4 == 0
            and not _derivatives_asked(wk_weight, index_k_out, *norm)):
        ops.indexer_project_kw(hidden_states, cos, sin, wk_weight, k_norm_weight, k_norm_bias, weights_proj_weight,
                               index_k_out, index_weights_out, int(rope_dim), score_scale)
        increment_version((index_k_out, index_weights_out))
        return q_index_out, index_k_out, index_weights_out
    # k: library projection and layer norm, then the RoPE kernel on [T, 1, D].
    k = F.linear(hidden_states, wk_weight)
    k = F.layer_norm(k, (int(head_dim),), k_norm_weight, k_norm_bias, eps=1e-6)
    index_k_out.copy_(k)
    if tokens:
        c, s = _rope_cos_sin(cos, sin, tokens, int(rope_dim))
        ops.dsa_indexer_query_rope_inplace(index_k_out.view(tokens, 1, int(head_dim)), c, s, int(rope_dim))
    index_weights_out.copy_(_weights_fp32(hidden_states, weights_proj_weight, score_scale))
    return q_index_out, index_k_out, index_weights_out


__all__ = ["dsa_indexer_project", "dsa_indexer_project_query_only"]
