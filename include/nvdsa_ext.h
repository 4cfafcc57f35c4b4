/* Entry points of libnvdsa.so beyond the reference's operators: parts of its
 * PyTorch functions that this library runs as kernels of their own.  Same
 * conventions as nvdsa.h (descriptors, status codes, caller-owned workspace,
 * launches on the given stream). */
#ifndef NVDSA_EXT_H
#define NVDSA_EXT_H

#include "nvdsa.h"

#ifdef __cplusplus
extern "C" {
#endif

/* The products of hidden_states that the indexer takes for many tokens, in
 * two launches that read it once:
 *   index_weights_out[t] = round16(fp32(hidden_states[t] . weights_proj_weight^T) * score_scale)
 * for fp32 weights_proj_weight (reference nanovllm/models/dsa_indexer_project.py:82-86;
 * with 16-bit weights rounded after the projection and again after a scale
 * other than 1, :74-81), and, unless wk_weight is NULL,
 *   index_k_out[t] = RoPE(layer_norm(round16(hidden_states[t] . wk_weight^T)))
 * (:245-293; eps 1e-6, k_norm_bias may be NULL).  Limits: n_head 16, 32 or
 * 64, hidden_size a multiple of 64, 128-wide keys.  The workspace is sized by
 * nvdsa_dsa_indexer_project_kw_workspace_size and holds no state. */
size_t nvdsa_dsa_indexer_project_kw_workspace_size(int64_t tokens, int64_t n_head, int64_t hidden_size,
                                                   int32_t with_k);
int nvdsa_dsa_indexer_project_kw(const nvdsa_tensor* hidden_states,
                                 const nvdsa_tensor* cos,
                                 const nvdsa_tensor* sin,
                                 const nvdsa_tensor* wk_weight,
                                 const nvdsa_tensor* k_norm_weight,
                                 const nvdsa_tensor* k_norm_bias,
                                 const nvdsa_tensor* weights_proj_weight,
                                 const nvdsa_tensor* index_k_out,
                                 const nvdsa_tensor* index_weights_out,
                                 int64_t rope_dim,
                                 double score_scale,
                                 void* workspace,
                                 size_t workspace_bytes,
                                 void* stream);

/* The tile (64, 128 or 256 tokens by as many outputs) in which
 * nvdsa_dsa_indexer_project_query_only multiplies more than 64 tokens into
 * `outputs` = n_head * head_dim values; 0 for up to 64 tokens, which take no
 * tiled product. */
int nvdsa_dsa_indexer_project_tile(int64_t tokens, int64_t outputs);

/* One row-wise copy of nvdsa_stage_inputs: rows [0, real) of dst (dst_bytes
 * apart) take src_bytes of src's row (src_stride bytes apart) and the 32-bit
 * pattern `fill` after them, rows [real, rows) the pattern alone.  All sizes
 * and addresses are multiples of 2 (of 4 unless the pattern's halves are
 * equal). */
typedef struct nvdsa_stage_item {
  void* dst;
  const void* src;
  int64_t rows;
  int64_t real;
  int64_t dst_bytes;
  int64_t src_bytes;
  int64_t src_stride;
  int64_t fill;
} nvdsa_stage_item;
/* Up to 16 such copies in one launch: the inputs of a decode step into a
 * captured graph's fixed buffers (reference
 * nanovllm/engine/full_decode_graph.py:546-720 copies them one by one).  No
 * item may read what another one writes. */
int nvdsa_stage_inputs(const nvdsa_stage_item* items, int64_t count, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* NVDSA_EXT_H */
