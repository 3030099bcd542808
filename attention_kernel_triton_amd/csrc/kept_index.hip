// Kept-token index selection on the GPU.
//
// The reference builds the sparse-decode index lists in host-driven torch code
// (sparsetoken_decode_flash_attention_redundant.py:283-295,
//  sparsetoken_decode_flash_attention_redundant_var_len_paged.py:341-353,
//  magicpig_..._with_norm.py:327-338): keep = rand(n) < p; if nothing is kept,
// keep index 0; indices = nonzero(keep) ascending; pad with -1; nnz = count.
// This kernel produces the same int32 arrays in one launch, one 1024-thread
// workgroup per row.  A step covers 32768 elements (a whole row of typical
// length, with all its loads in flight): wave w owns 2048 consecutive ones and
// reads them in chunks of 64 runs of kRun, one run to a lane, so that a load
// instruction reads one contiguous KB.  A lane packs its 32 keep bits into a
// word and its counts per chunk into 16-bit halves, whose prefix over the lanes
// (DPP adds) ranks all chunks at once; the 16 wave totals go through LDS.  The
// loads of step s + 1 are in flight while step s is ranked.  They go through a
// buffer resource that ends at the row's last element, so nothing past the row
// is read.
//
// What bounds it: with few rows, one workgroup's round trips and instructions.
// Measured against 32 consecutive elements to a thread (64 cache lines to a load,
// 32 byte loads a thread for masks) and shuffles for the prefix (us): 32 rows of
// 32000 draws, 2% kept 6.9 -> 5.3, of 100000 19.4 -> 13.5; masks 17.3 -> 5.6 and
// 54.0 -> 9.8.  (A ballot per element instead of the packed counts: 7.9.)  The
// slot of each kept element costs more: where half is kept, 32 rows of 8191 draws
// 6.9 -> 7.5.
#include "akt_common.hpp"
#include "akt_host.hpp"

namespace akt {
namespace {

constexpr int kKThreads = 1024;
constexpr int kKWaves = kKThreads / kWave;
constexpr int kPer = 32;                      // elements per thread per step
constexpr int kWaveElems = kPer * kWave;      // consecutive elements per wave per step
constexpr int kStep = kKThreads * kPer;       // elements per step

// Keep sources: fp32 draws (4 to a 16-byte load), mask bytes in rows that start
// 4-byte aligned (16 to a load), or mask bytes at any address (byte loads).
enum : int { kUniform = 0, kMaskWords = 1, kMaskBytes = 2 };

// Inclusive prefix sum over the wave's lanes (two 16-bit halves at once: no
// carry, a wave's counts stay below 2^16).
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t add_dpp(uint32_t v) {
  return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
  v = add_dpp<0x111, 0xf>(v);     // row_shr 1, 2, 4, 8: within 16 lanes
  v = add_dpp<0x112, 0xf>(v);
  v = add_dpp<0x114, 0xf>(v);
  v = add_dpp<0x118, 0xf>(v);
  v = add_dpp<0x142, 0xa>(v);     // lane 15 of rows 0 and 2 to rows 1 and 3
  return add_dpp<0x143, 0xc>(v);  // lane 31 to rows 2 and 3
}

template <int SRC>
__global__ __launch_bounds__(kKThreads) void kept_index_kernel(
    const uint8_t* __restrict__ mask, const float* __restrict__ draws, float ratio, int64_t n,
    int64_t row_stride, const int32_t* __restrict__ row_len, int32_t* __restrict__ ind,
    int64_t l_max, int32_t* __restrict__ nnz, int ensure_nonempty) {
  constexpr int kRun = SRC == kMaskWords ? 16 : 4;  // consecutive elements per lane and chunk
  constexpr int NC = kPer / kRun;                   // chunks per wave and step
  constexpr uint32_t kRunMask = (1u << kRun) - 1u;
  constexpr int esz = SRC == kUniform ? 4 : 1;
  __shared__ int wave_tot[2][kKWaves];
  const int r = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = uniform(tid >> 6);
  int64_t nr = n;
  if (row_len) {
    const int64_t v = row_len[r];
    nr = v < 0 ? 0 : (v > n ? n : v);
  }
  int32_t* out = ind + (int64_t)r * l_max;
  // The row's elements [0, nr) (row lengths below 2^28: byte offsets fit 31 bits).
  const void* row_base = SRC == kUniform ? (const void*)(draws + (int64_t)r * row_stride)
                                         : (const void*)(mask + (int64_t)r * row_stride);
  // (Whole words of a mask row: the aligned word that holds its last byte.)
  const int range = SRC == kMaskWords ? (int)((nr + 3) & ~3) : (int)(nr * esz);
  const auto rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)row_base, 0, range, kBufferWord3);
  // The lane's run of chunk ch of a step, as raw words (kMaskBytes: a byte each).
  struct Step {
    uint4_t w[NC];
  };
  auto load = [&](int64_t base, Step& st) {
#pragma unroll
    for (int ch = 0; ch < NC; ++ch) {
      const int off = ((int)base + wave * kWaveElems + (ch * kWave + lane) * kRun) * esz;
      if constexpr (SRC == kMaskBytes) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          st.w[ch][k] = __builtin_amdgcn_raw_buffer_load_b8(rsrc, off + k, 0, 0);
      } else {
        st.w[ch] = __builtin_bit_cast(uint4_t,
                                      __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
      }
    }
  };
  Step cur, nxt;
  if (nr > 0) load(0, cur);
  int count = 0;  // kept so far (uniform across the workgroup)
  int buf = 0;
  for (int64_t base = 0; base < nr; base += kStep) {
    if (base + kStep < nr) load(base + kStep, nxt);
    const int e0 = (int)base + wave * kWaveElems + lane * kRun;  // element 0 of chunk 0
    // Keep bits of this lane's elements, chunk ch's from bit ch * kRun, and the
    // chunks' counts (chunk ch in half ch % 2 of word ch / 2).
    uint32_t m = 0, cnt[NC / 2];
#pragma unroll
    for (int ch = 0; ch < NC; ++ch) {
#pragma unroll
      for (int j = 0; j < kRun; ++j) {
        bool keep;
        if constexpr (SRC == kUniform) keep = __uint_as_float(cur.w[ch][j]) < ratio;
        else if constexpr (SRC == kMaskWords) keep = ((cur.w[ch][j >> 2] >> (8 * (j & 3))) & 0xffu) != 0;
        else keep = cur.w[ch][j] != 0;
        m |= keep ? 1u << (ch * kRun + j) : 0u;
      }
      // Elements at or past the row's end are not kept.
      const int over = e0 + ch * kWave * kRun + kRun - (int)nr;
      if (over > 0) m &= ~(((1u << min(over, kRun)) - 1u) << (ch * kRun + kRun - min(over, kRun)));
      const uint32_t c = (uint32_t)__builtin_popcount((m >> (ch * kRun)) & kRunMask);
      cnt[ch / 2] = ch % 2 ? cnt[ch / 2] | c << 16 : c;
    }
    // rank: kept elements of the wave before this lane's run of each chunk.
    uint32_t rank[NC / 2];
    int total = 0;  // kept elements of the wave (scalar)
#pragma unroll
    for (int k = 0; k < NC / 2; ++k) {
      const uint32_t incl = wave_inclusive_scan(cnt[k]);
      const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
      const int lo = total, hi = lo + (int)(all & 0xffffu);
      rank[k] = incl - cnt[k] + ((uint32_t)lo | (uint32_t)hi << 16);
      total = hi + (int)(all >> 16);
    }
    if (lane == 0) wave_tot[buf][wave] = total;
    __syncthreads();
    int before = count, step_total = 0;
#pragma unroll
    for (int w = 0; w < kKWaves; ++w) {
      const int t = wave_tot[buf][w];
      before += (w < wave) ? t : 0;
      step_total += t;
    }
    for (uint32_t rest = m; rest; rest &= rest - 1) {
      const int i = __builtin_ctz(rest);
      const int ch = i / kRun;
      uint32_t word = rank[0];
#pragma unroll
      for (int k = 1; k < NC / 2; ++k) word = ch / 2 == k ? rank[k] : word;
      const uint32_t lower = m & ((1u << i) - 1u) & (kRunMask << (ch * kRun));
      const int64_t slot = (int64_t)before + ((word >> (16 * (ch & 1))) & 0xffffu) +
                           __builtin_popcount(lower);
      if (slot < l_max) out[slot] = e0 + ch * (kWave - 1) * kRun + i;
    }
    count += step_total;
    buf ^= 1;  // the other buffer is free: every wave read it before this step's barrier
    cur = nxt;
  }
  int total = count;
  if (total == 0 && ensure_nonempty) {
    if (tid == 0 && l_max > 0) out[0] = 0;
    total = 1;
  }
  for (int64_t i = (int64_t)total + tid; i < l_max; i += kKThreads) out[i] = -1;
  if (tid == 0) nnz[r] = total;
}

int launch_kept(bool from_mask, const uint8_t* mask, const float* uniform, float ratio,
                int64_t rows, int64_t n, int64_t row_stride, const int32_t* row_len,
                int32_t* sparse_ind, int64_t l_max, int32_t* sparse_nnz, int ensure_nonempty,
                void* stream) {
  clear_error();
  AKT_CHECK(rows >= 0 && rows < (1ll << 31) && n >= 0 && l_max >= 0, "sizes out of range");
  AKT_CHECK(row_stride >= n, "row stride (%lld) smaller than row length (%lld)",
            (long long)row_stride, (long long)n);
  AKT_CHECK(n < (1ll << 28), "row length (%lld) must be below 2^28", (long long)n);
  AKT_CHECK(sparse_nnz && (sparse_ind || l_max == 0), "output pointers are required");
  if (rows == 0) return AKT_OK;
  AKT_CHECK(from_mask ? (mask || n == 0) : (uniform || n == 0), "input pointer is required");
  hipStream_t st = (hipStream_t)stream;
  KernelTimer timer;
  // Aligned mask rows are read in words: torch masks are, unless the row length
  // is not a multiple of 4.
  const bool words = aligned4(mask) && row_stride % 4 == 0;
  auto kernel = !from_mask ? kept_index_kernel<kUniform>
                           : (words ? kept_index_kernel<kMaskWords> : kept_index_kernel<kMaskBytes>);
  timer.launch(kernel, dim3((unsigned)rows), dim3(kKThreads), 0, st, mask, uniform, ratio, n,
               row_stride, row_len, sparse_ind, l_max, sparse_nnz, ensure_nonempty);
  return check_launch("kept_index_kernel");
}

}  // namespace
}  // namespace akt

extern "C" int akt_kept_index_from_mask(const uint8_t* mask, int64_t rows, int64_t n,
                                        int64_t mask_row_stride, const int32_t* row_len,
                                        int32_t* sparse_ind, int64_t l_max, int32_t* sparse_nnz,
                                        int ensure_nonempty, void* stream) {
  return akt::launch_kept(true, mask, nullptr, 0.f, rows, n, mask_row_stride, row_len, sparse_ind,
                          l_max, sparse_nnz, ensure_nonempty, stream);
}

extern "C" int akt_kept_index_from_uniform(const float* uniform, float kept_ratio, int64_t rows,
                                           int64_t n, int64_t row_stride, const int32_t* row_len,
                                           int32_t* sparse_ind, int64_t l_max,
                                           int32_t* sparse_nnz, int ensure_nonempty,
                                           void* stream) {
  return akt::launch_kept(false, nullptr, uniform, kept_ratio, rows, n, row_stride, row_len,
                          sparse_ind, l_max, sparse_nnz, ensure_nonempty, stream);
}
