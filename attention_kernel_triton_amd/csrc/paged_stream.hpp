// Stream-K paged and dense decode (paged_stream.hip): parameters and host entries.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "akt_common.hpp"

namespace akt {

// Largest batch whose sequence table fits the kernel's LDS.
constexpr int kStreamMaxBatch = 1024;
// Most waves a launch uses.  (The paged workspace is sized for a partial slot
// per wave and unit, the public contract, more than the slots below.)
constexpr int kStreamMaxWaves = 4096;

struct StreamParams {
  const half_t* q;      // [B, Hq, D] rows (strides q_sb, q_sh)
  const half_t* kbase;  // KV pool, K half; dense: the K tensor
  const half_t* vbase;  // KV pool + the K/V axis stride; dense: the V tensor
  const int32_t* indptr;  // page table (unused by a dense cache)
  const int32_t* indices;
  const int32_t* last_len;
  half_t* o;      // [B, Hq, D] contiguous
  float* lse;     // [B, Hq] or null
  int* arrive;    // [workgroups] arrival counters (zero between launches)
  float* part_o;  // [slots, GT, D], slots < workgroups + min(workgroups, B * Y)
  float* part_ml; // [slots, GT, 4]: max, normaliser, the same again, pad
  int64_t q_sb, q_sh;
  int64_t k_sa, k_head, v_sa, v_head;  // page (dense: batch) and kv-head strides (elements)
  int k_sb, v_sb;                      // row strides (elements, < 2^26)
  int B, Hq, G, Y, n_hg;
  int page_size, gpp;  // gpp = page_size / 16 groups per page; dense: ceil(S / 16)
  int total_pages;     // dense: B
  int S;               // dense: the cache length
  int TG;              // groups per head group: total_pages * gpp
  int N;               // groups of the launch: Y * TG (< 2^31)
  // Set by paged_stream_launch: waves with groups (at most N), N / W, the
  // fraction (N % W) / W in 20-bit fixed point, W / N.
  int W, wq;
  uint32_t wf20;
  float w_per_g;
  int wgs_log;  // dense: 2^wgs_log workgroups to a unit, -1: stream-K ranges
  int num_pool_pages;
  float qk_scale;      // softmax_scale * log2(e)
};

// Whether a paged decode can take the stream-K kernel: pages of whole
// 16-token groups, a batch that fits the LDS table and a group axis that fits
// 32 bits.
bool paged_stream_eligible(int64_t batch, int64_t page_size, int64_t total_pages, int64_t Y);

// Waves a launch of instance (D, gt) uses at most on the current device
// (its resident workgroups' waves, eight each up to D = 128 and four at 256, at
// most kStreamMaxWaves; kStreamMaxWaves when the device cannot be queried).
int64_t paged_stream_wave_cap(int D, int gt);

// Launches the kernel for head dim D with gt heads per unit; the range fields
// of p (W and below) are set here.
int paged_stream_launch(const StreamParams& p, int D, int gt, hipStream_t st);

// The same for a dense cache.  Eligible: row strides that 32-bit offsets of 16
// rows can hold and a group axis below 2^31.
bool dense_stream_eligible(int64_t batch, int64_t seq_len, int64_t Y, int64_t k_row,
                           int64_t v_row);
int64_t dense_stream_parts(int D, int gt, int64_t units, int64_t unit_groups);
int dense_stream_launch(const StreamParams& p, int D, int gt, hipStream_t st);

}  // namespace akt
