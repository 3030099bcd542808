// Sparse-token decode (sparse_decode.hip): parameters and host entry.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "akt_common.hpp"

namespace akt {

struct SparseParams {
  const half_t* q;      // [B, Hq, D] rows (strides q_sb, q_sh)
  const half_t* kbase;  // dense: K tensor; paged: KV pool
  const half_t* vbase;  // dense: V tensor; paged: KV pool + stride of the K/V axis
  const int32_t* indptr;  // paged: page table
  const int32_t* indices;
  const int32_t* sparse_ind;
  const int32_t* sparse_nnz;
  const int64_t* csr_ptr;  // CSR kept-index rows: row u = sparse_ind[csr_ptr[u] .. csr_ptr[u+1])
  const float* lsh_k;      // MagicPIG [B, Hq]
  const float* lsh_l;
  half_t* o;       // [B, Hq, D] contiguous
  float* lse;      // [B, Hq] or null
  int* arrive;     // [rows]: partials stored so far per row (zero between launches)
  float* part_o;   // [rows * n_split, D]
  float* part_ml;  // [rows * n_split, 4]: running max, fp16-P normaliser, fp32 normaliser, pad
  int64_t q_sb, q_sh;
  // Row address of a K/V row.  dense: base + b * batch + kvh * head + token * sa;
  // paged (K and V alike): base + kvh * head + page * sa + slot * sb.
  int64_t k_sa, k_sb, k_batch, k_head;
  int64_t v_sa, v_batch, v_head;
  int64_t ind_sb, ind_sh, nnz_sb, nnz_sh;
  int Hq, G;
  int rows;       // B * Hq
  int S;          // dense: cache length
  int page_size;
  int num_pool_pages;
  int l_max;
  int n_split;       // workgroups per row
  float qk_scale;    // softmax_scale * log2(e)
  float inv_sqrt_d;  // 1 / sqrt(head_dim) (MagicPIG)
};

// Launches rows * n_split workgroups (head_dim 64, 128 or 256; magic: paged only).
int sparse_launch(const SparseParams& p, int head_dim, bool paged, bool magic, hipStream_t st);

}  // namespace akt
