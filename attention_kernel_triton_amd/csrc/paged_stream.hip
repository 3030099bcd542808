// Stream-K decode for gfx950: the automatic-chunk path of the paged var-len
// decode (decode_flash_attention_redundant_var_len_paged.py:70-224) and of the
// dense one (decode_flash_attention_redundant.py:71-229).
//
// A dense cache is a paged one whose sequence b is one page, page b of
// ceil(S / 16) groups: its DENSE instances read no table and, in the last
// group, no row past S.  (Against the split kernel's tickets, workgroup merge
// per chunk and P.V on the VALU: B=32, Hq=64, Hkv=8, S=4100, D=128 119.9 ->
// 94.4 us, 5.7 TB/s; B=8, Hq=64, Hkv=16, S=1024, D=64 14.4 -> 11.5 us.)
//
// Work decomposition.  A "unit" is one (sequence b, head group y): the up to
// GT query heads of one kv head that read the same K/V rows.  Every unit's
// K/V is cut into 16-token groups (a page of page_size tokens holds
// page_size / 16 of them), and the groups of all units are laid out on one
// axis, kv-head-group major:
//   g = y * TG + position * gpp + slice,   TG = total_pages * gpp,
// where `position` indexes kv_page_indices, so sequence b's groups of head
// group y are the contiguous range [y*TG + indptr[b]*gpp, y*TG + indptr[b+1]*gpp).
// The W waves of the launch take equal contiguous ranges of that axis (wave w:
// [w*N/W, (w+1)*N/W)), fixed before the launch: no tickets, no workgroup
// barrier between the prologue and the end of the stream.  A wave streams its range with two groups in flight, keeps one
// online softmax for the unit it is in, and at each unit boundary either
// writes the unit's output (a unit wholly inside the wave) or leaves the
// segment's state (m, l, o) in LDS.  Only a wave's first and last segments
// can be partial.
//
// Merge.  After its waves' streams a workgroup combines each unit's segments
// from LDS (log-sum-exp in wave order).  A unit inside the workgroup's range is
// then done.  Only the (at most two) units that reach into a neighbouring
// workgroup's range cost a global partial: it is stored with device scope and
// counted in the unit's arrival counter.  The wave that counts the last one
// merges them at once if one round trip of loads takes them all; else its
// workgroup does, wave v taking partials v, v + 8, ...; in an order that does
// not depend on timing either way.  Measured against one partial per wave and
// one wave merging a unit's partials ten to a round trip: a lone sequence of
// 30001 tokens (B=1, Hq=32, Hkv=8, D=128; 256 partials to a unit, 26 dependent
// round trips) 78.0 -> 33.8 us; 32 sequences of 256-8192 tokens 108.1 -> 106.4
// us; 16 of 512-2048 tokens 26 -> 23 us.
//
// Per group: four (D=128) v_mfma_f32_16x16x32_f16 give the 16-token x 16-head
// score block as S^T (lane (R, c) holds head c, tokens 4R .. 4R+3); the online
// softmax runs in log2 units; P.V is D/16 v_mfma_f32_16x16x16_f16 with P^T
// straight from the score lanes and V^T read from an LDS copy of the group's V
// rows with ds_read_b64_tr_b16, once for P rounded to fp16 (as the reference
// rounds it, decode_flash_attention_redundant_var_len_paged.py:186) and once for
// what the rounding left: the matrix pipe is idle here, and the outputs' error
// against 64 bits falls from 2.6e-4 to 2.1e-4 (2-norm) at the same time.
#include <math.h>

#include <algorithm>

#include "akt_common.hpp"
#include "akt_host.hpp"
#include "paged_stream.hpp"

namespace akt {
namespace {

#define AKT_SNEG_INF (-__builtin_inff())

// Compute units of MI355X: the workgroups assumed where no device can be queried.
constexpr int64_t kCUs = 256;

// The kernel's arguments, re-read from the kernel-argument segment (the opaque
// pointer keeps the compiler from reusing, and so holding, earlier reads): what
// only the unit boundaries and the merge use would otherwise take scalar
// registers from the stream's loop, which spills them to vector lanes.
typedef const __attribute__((address_space(4))) StreamParams* StreamArgs;
__device__ __forceinline__ StreamArgs reread_args() {
  StreamArgs a = (StreamArgs)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  return a;
}

// First group of wave w's range (WAVES to a workgroup).
// - Stream-K: w (N / W) + floor(w f), f = (N % W) / W in 20-bit fixed point:
//   W <= N, so no wave below W is empty, and waves from W on have none.  (The
//   long ranges are spread evenly on purpose: with the N % W longer ones all
//   in the first workgroups, those held 3% more and a 115096-token launch took
//   3% longer; an exact floor(w N / W) costs each wave a chain of divisions
//   before its first load.)
// - Whole units (DENSE, wgs_log >= 0): 2^wgs_log workgroups to a unit, the
//   unit's groups shared evenly by their waves (one each while they last, in
//   a single workgroup, for a unit with fewer groups than waves).
template <bool DENSE, int WAVES, typename P>
__device__ __forceinline__ int wave_start(const P& p, int w) {
  if (DENSE && p.wgs_log >= 0) {
    const int s = p.wgs_log + (WAVES == 8 ? 3 : 2);
    const int u = w >> s, j = w & ((1 << s) - 1);
    return u * p.gpp + (p.gpp < (1 << s) ? min(j, p.gpp) : (int)(((int64_t)j * p.gpp) >> s));
  }
  return w >= p.W ? p.N : w * p.wq + (int)(((uint32_t)w * p.wf20) >> 20);  // w < 4096
}

// Last index i in [0, n] with s[i] <= x, given a non-decreasing s[0..n];
// -1 if s[0] > x.
__device__ __forceinline__ int last_le(const int* s, int n, int x) {
  int lo = 0, hi = n + 1;  // first index with s > x lies in [lo, hi]
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (s[mid] <= x) lo = mid + 1;
    else hi = mid;
  }
  return lo - 1;
}

// Waves per SIMD the instance is built for: two up to D = 128 (at most ~180
// VGPRs whatever the head count: P.V accumulates in D/4 registers), one at
// D = 256.
template <int D, int GT>
constexpr int stream_min_waves() {
  return D <= 128 ? 2 : 1;
}
// Threads per workgroup: with two waves per SIMD, one 512-thread workgroup per
// CU, so that the two waves sharing a SIMD (waves w and w + 4) are in one
// workgroup and can see each other's progress; otherwise 256.
template <int D, int GT>
constexpr int stream_threads() {
  return stream_min_waves<D, GT>() == 2 ? 512 : 256;
}

// Groups in flight per wave: after a group is consumed, the group PD ahead is
// issued into its buffer.  (Three measured slower on config 3.)
template <int D, int GT>
constexpr int stream_depth() {
  return 2;
}

template <int D, int GT, bool DENSE>
__global__ __launch_bounds__((stream_threads<D, GT>()))
__attribute__((amdgpu_waves_per_eu(stream_min_waves<D, GT>(), 8))) void paged_stream_kernel(
    StreamParams p) {
  constexpr int PD = stream_depth<D, GT>();
  constexpr int kTable = DENSE ? 1 : kStreamMaxBatch;  // sequences of the LDS table
  constexpr int kSThreads = stream_threads<D, GT>();
  constexpr int kSWaves = kSThreads / kWave;
  constexpr bool PAIRED = kSWaves == 8;
  constexpr int KS = D / 32;                 // MFMA k-steps (8 elements each)
  constexpr int VTOK = (D == 64) ? 2 : 4;    // V tokens per lane per group
  constexpr int VDIM = (D == 256) ? 16 : 8;  // V dims per lane
  constexpr int VLD = VDIM / 8;              // 16-byte loads per V token
  constexpr int NT = D / 16;                 // 16-dim output tiles (P.V MFMAs per group)
  constexpr int VROW = D + 16;               // staged V row (fp16): padded against bank conflicts

  // Sequence page ranges: sequence b owns positions [sm_s[b], sm_s[b + 1]) of
  // kv_page_indices (indptr clamped to [0, total_pages] and made
  // non-decreasing).
  __shared__ int sm_s[kTable + 1];
  __shared__ int sm_wmax[kSWaves];
  __shared__ int sm_fin[2];  // units whose last partial this workgroup counted (-1: none)
  // Groups each wave has consumed (paired waves only).
  __shared__ int sm_prog[kSWaves];
  // Segment states a wave leaves for the merge: slot 0 (its first partial
  // segment) and slot 1 (a later one, always its last).  Rows of OROW floats
  // per head, padded against bank conflicts.  Until its stream ends a wave
  // stages a group's V rows in its slot 1, for the transposing reads of P.V.
  constexpr int OROW = D + 4;
  constexpr int SEG = GT * OROW;
  constexpr int SEG1 = SEG * 4 > 16 * VROW * 2 ? SEG : 16 * VROW / 2;
  __shared__ __attribute__((aligned(16))) float sm_seg0[kSWaves][SEG];
  __shared__ __attribute__((aligned(16))) float sm_seg1[kSWaves][SEG1];
  __shared__ float4_t sm_ml[kSWaves][2][GT];  // max, normaliser, the same again, -
  __shared__ int sm_unit[kSWaves][2];         // unit of each slot (-1: unused)

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = uniform(tid >> 6);
  const int R = lane >> 4;
  const int c16 = lane & 15;
  const int gw = (int)blockIdx.x * kSWaves + wave;
  const int g0 = wave_start<DENSE, kSWaves>(p, gw);
  const int n = wave_start<DENSE, kSWaves>(p, gw + 1) - g0;  // groups of this wave

  // Axis position of group g: head group y, page position pp, 16-row slice.
  auto locate = [&](int g, int& y, int& pp, int& slice) __attribute__((always_inline)) {
    y = g / p.TG;
    const int pos = g - y * p.TG;
    pp = pos / p.gpp;
    slice = pos - pp * p.gpp;
  };
  // ---- lookahead ------------------------------------------------------------
  // The group PD ahead of the one being issued is "fetched": its page id and
  // its sequence's last-page length are read with one vector load each (a
  // uniform address), the same two loads for every group.  (A scalar load
  // would be counted with the LDS accesses and, since scalar loads complete
  // out of order, every LDS wait would then wait for it.)  Its position is
  // tracked in scalar registers, advanced one group per fetch: head group
  // la_y, page position la_pp, 16-row slice la_slice, and sequence la_b
  // (-1 before sequence 0's pages, B past the last) with la_end, the first
  // position past la_b's pages (la_b and la_end need the sequence table).
  // (Sized to the tensors: a read past them returns 0 and touches no memory.)
  const auto idx_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.indices, 0,
                                                          p.total_pages * 4, kBufferWord3);
  const auto ll_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.last_len, 0, p.B * 4,
                                                         kBufferWord3);
  int la_y = 0, la_pp = 0, la_slice = 0, la_b = -1, la_end = 0;
  auto seq_end = [&](int b) __attribute__((always_inline)) -> int {
    return b < p.B ? uniform(sm_s[b + 1]) : INT32_MAX;
  };
  // First position of sequence b (a dense cache: position b, one each).
  auto seq_start = [&](int b) __attribute__((always_inline)) -> int {
    return DENSE ? b : uniform(sm_s[b]);
  };
  // One group forward; `track`: keep la_b / la_end (the table exists).
  auto advance = [&](bool track) __attribute__((always_inline)) {
    if (++la_slice < p.gpp) return;
    la_slice = 0;
    if (++la_pp == p.total_pages) {
      la_pp = 0;
      ++la_y;
      la_b = -1;
      if (!DENSE && track) la_end = uniform(sm_s[0]);
    }
    if (!DENSE && track)
      while (la_b < p.B && la_pp >= la_end) la_end = seq_end(++la_b);
  };
  // Sequence of position pp from the table (the last b with start <= pp).
  auto seek = [&](int pp) __attribute__((always_inline)) {
    la_b = uniform(last_le(sm_s, p.B, pp));
    la_end = la_b < 0 ? uniform(sm_s[0]) : seq_end(la_b);
  };
  // A fetched group: page id and last-page length (vector registers, loaded),
  // and its position (wave-uniform).
  struct Fetch {
    int page, ll;
    int b, y, slot, last;
  };
  auto fetch = [&](Fetch& f) __attribute__((always_inline)) {
    if constexpr (DENSE) {
      f.page = f.b = la_pp;
      f.y = la_y;
      f.slot = la_slice * 16;
      f.last = 1;
      advance(true);
      return;
    }
    f.page = __builtin_amdgcn_raw_buffer_load_b32(idx_rsrc, (uint32_t)la_pp * 4u, 0, 0);
    const bool seq_ok = la_b >= 0 && la_b < p.B;
    const int lb = min(max(la_b, 0), p.B - 1);
    f.ll = __builtin_amdgcn_raw_buffer_load_b32(ll_rsrc, (uint32_t)lb * 4u, 0, 0);
    f.b = seq_ok ? la_b : -1;
    f.y = la_y;
    f.slot = la_slice * 16;
    f.last = seq_ok && la_pp == la_end - 1;
    advance(true);
  };

  // ---- per-lane load offsets ------------------------------------------------
  // A group is the 16 rows from row `slot` of one page: its addresses are a
  // uniform base plus this lane's K row (c16) and K dims (8R + 32s for MFMA
  // k-step s, so that the four lanes of a row read 64 contiguous bytes per
  // load), and its V token tt0 + i at dims dim0.  Groups without a valid page
  // read the q tensor's first row instead (always mapped), inside that row.
  const int dim0 = (D == 64) ? 8 * (c16 & 7) : VDIM * c16;
  const int tt0 = (D == 64) ? (4 * R + 2 * (c16 >> 3)) : 4 * R;
  const uint32_t lane_kofs = (uint32_t)(c16 * p.k_sb + 8 * R) * 2u;
  const uint32_t lane_qofs = (uint32_t)(8 * R) * 2u;
  const uint32_t lane_v0ofs = (uint32_t)(tt0 * p.v_sb + dim0) * 2u;
  const uint32_t lane_dofs = (uint32_t)dim0 * 2u;
  const uint32_t vstep = (uint32_t)p.v_sb * 2u;

  struct Buf {
    uint4_t k[KS];
    uint4_t v[VTOK][VLD];
    half8_t q[KS];  // the query fragment of the group's unit
    // wave-uniform: sequence (-1: none or a dummy), head group, first row of
    // the slice, whether the page is the sequence's last, valid page id,
    // usable tokens
    int b, y, slot, last, use, nv;
  };
  // Usable tokens of a buffer's group given its sequence's last-page length
  // ll (a loaded register): 16, or on the sequence's last page the rows below
  // ll (clamped to [0, page_size]), 0 for invalid pages.  The length is read
  // into a scalar here, when the group is issued (its load, PD groups back,
  // is complete then), so that no vector register holding a loaded value is
  // carried from one group to the next: the compiler may copy such a register
  // at the loop's head, and would wait there for the load that last wrote it.
  auto set_usable = [&](Buf& bf, int ll_reg) __attribute__((always_inline)) {
    const int ll = min(max(uniform(ll_reg), 0), p.page_size);
    const int tail = min(max(ll - bf.slot, 0), 16);
    bf.nv = (!bf.use || bf.b < 0) ? 0 : (bf.last ? tail : 16);
  };

  // Query fragment of unit (b, y) (MFMA B operand): head hq0 + c16, dims
  // 32s + 8R + e (the K loads' assignment).  Columns past the unit's heads
  // repeat head hq0: each column's scores, softmax and P.V stay in that
  // column's lanes, and those lanes store nothing.  (Zeroing them would make
  // the compiler wait for the loads right where they are issued.)  b < 0 (no
  // unit; y may then lie past the last head group) reads sequence 0's first
  // rows, so that every group issues the same loads.
  auto load_q = [&](int b, int y, half8_t (&qd)[KS]) __attribute__((always_inline)) {
    y = b < 0 ? 0 : y;
    b = max(b, 0);
    const int kvh = p.n_hg == 1 ? y : y / p.n_hg;
    const int hg = y - kvh * p.n_hg;
    const int hq0 = kvh * p.G + hg * GT;
    const int nh = min(GT, p.G - hg * GT);
    const half_t* qrow =
        p.q + (int64_t)b * p.q_sb + (int64_t)(hq0 + (c16 < nh ? c16 : 0)) * p.q_sh + 8 * R;
#pragma unroll
    for (int s = 0; s < KS; ++s) qd[s] = as_half8(ld16(qrow + 32 * s));
  };

  // Issues group j of this wave from its fetch record f (j >= n: a dummy
  // group that reads the q row), then fetches group j + PD into f.
  // `take_ll`: the usable tokens are set from f's last-page length (the
  // prologue sets them itself).  Rows of a
  // valid page are loaded whole; tokens past the usable prefix are masked when
  // consumed.  `seq`: the sequence is known (the table exists), so the unit's
  // q fragment is loaded with the group.  Every call issues the same loads
  // whatever the data: a load issued only on some paths would leave the
  // compiler unsure how many loads follow a buffer's, and it would then wait
  // for all of them before consuming it.
  Fetch fr[PD];
  auto issue = [&](int j, Buf& bf, bool seq, Fetch& f, bool take_ll)
                   __attribute__((always_inline)) {
    const int page = DENSE ? f.page : uniform(f.page);
    const int y = f.y, slot = f.slot;
    bf.b = j < n ? f.b : -1;
    bf.y = y;
    bf.slot = slot;
    bf.last = f.last;
    const bool use = j < n && (DENSE || (page >= 0 && page < p.num_pool_pages));
    bf.use = use;
    if constexpr (DENSE) bf.nv = use ? min(p.S - slot, 16) : 0;
    else if (take_ll) set_usable(bf, f.ll);
    // A dense cache ends with its last row: lanes of rows past it re-read it.
    const int row_max = DENSE ? max(bf.nv - 1, 0) : 15;
    if (seq) fetch(f);
    if (seq) load_q(bf.b, y, bf.q);
    const int kvh = p.n_hg == 1 ? y : y / p.n_hg;
    const char* kg = reinterpret_cast<const char*>(
        use ? p.kbase + (int64_t)kvh * p.k_head + (int64_t)page * p.k_sa + (int64_t)slot * p.k_sb
            : p.q);
    uint32_t ko = use ? lane_kofs : lane_qofs;
    if (DENSE && row_max < 15 && use) ko = (uint32_t)(min(c16, row_max) * p.k_sb + 8 * R) * 2u;
#pragma unroll
    for (int s = 0; s < KS; ++s) bf.k[s] = ld16(kg + ko + 64 * s);
    const char* vg = reinterpret_cast<const char*>(
        use ? p.vbase + (int64_t)kvh * p.v_head + (int64_t)page * p.v_sa + (int64_t)slot * p.v_sb
            : p.q);
#pragma unroll
    for (int i = 0; i < VTOK; ++i) {
      uint32_t vo = use ? lane_v0ofs + (uint32_t)i * vstep : lane_dofs;
      if (DENSE && row_max < 15 && use) vo = (uint32_t)(min(tt0 + i, row_max) * p.v_sb + dim0) * 2u;
#pragma unroll
      for (int jj = 0; jj < VLD; ++jj) bf.v[i][jj] = ld16(vg + vo + 16 * jj);
    }
  };

  // Four normalised output values of row `row` at dims d0 .. d0 + 3.
  auto store_o4 = [&](half_t* o, int64_t row, int d0, float4_t O, float inv)
                      __attribute__((always_inline)) {
    half4_t hv;
#pragma unroll
    for (int r = 0; r < 4; ++r) hv[r] = (half_t)(O[r] * inv);
    *reinterpret_cast<half4_t*>(o + row * D + d0) = hv;
  };
  auto store_lse = [&](float* lse, int64_t row, float M, float E) __attribute__((always_inline)) {
    if (lse) lse[row] = E > 0.f ? (M + log2f(E)) * kLn2 : AKT_SNEG_INF;
  };

  // ---- prologue ----------------------------------------------------------------
  // The first PD groups' page ids, then group 0's K and V, need only the
  // kernel arguments: they go out before the sequence table is built (its
  // barriers wait for LDS only).  The table gives the groups' sequences, hence
  // their q fragments and last-page lengths.
  if (lane < 2) {
    sm_unit[wave][lane] = -1;
    if (wave == 0) sm_fin[lane] = -1;
  }
  if (PAIRED && lane == 0)
    __hip_atomic_store(&sm_prog[wave], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  int y0 = 0, pp0 = 0, slice0 = 0;
  if (n > 0) locate(g0, y0, pp0, slice0);
  la_y = y0;
  la_pp = pp0;
  la_slice = slice0;
  Buf bufs[PD];
  if constexpr (!DENSE) {
#pragma unroll
    for (int i = 0; i < PD; ++i) {
      fr[i].page = __builtin_amdgcn_raw_buffer_load_b32(idx_rsrc, (uint32_t)la_pp * 4u, 0, 0);
      fr[i].y = la_y;
      fr[i].slot = la_slice * 16;
      fr[i].b = -1;
      fr[i].last = 0;
      fr[i].ll = 0;
      advance(false);
    }
    constexpr int ENT = (kStreamMaxBatch + 1 + kSThreads - 1) / kSThreads;  // table entries per thread
    int tv[ENT];
#pragma unroll
    for (int j = 0; j < ENT; ++j) {
      const int e = ENT * tid + j;
      tv[j] = e <= p.B ? min(max(p.indptr[e], 0), p.total_pages) : 0;
    }
    if (n > 0) issue(0, bufs[0], false, fr[0], false);
    // Sequence table: indptr clamped to [0, total_pages] and made
    // non-decreasing (a max-scan).
    {
#pragma unroll
      for (int j = 1; j < ENT; ++j) tv[j] = max(tv[j], tv[j - 1]);
      int incl = tv[ENT - 1];
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int t = __shfl_up(incl, off, 64);
        if (lane >= off) incl = max(incl, t);
      }
      if (lane == 63) sm_wmax[wave] = incl;
      __syncthreads();
      int before = 0;
#pragma unroll
      for (int w = 0; w < kSWaves; ++w)
        if (w < wave) before = max(before, sm_wmax[w]);
      const int up = __shfl_up(incl, 1, 64);
      const int excl = lane > 0 ? max(before, up) : before;
#pragma unroll
      for (int j = 0; j < ENT; ++j) {
        const int e = ENT * tid + j;
        if (e <= p.B) sm_s[e] = max(excl, tv[j]);
      }
      __syncthreads();
    }

    // Sequences without pages have no groups: o = 0 and lse = -inf here.
    for (int bb = gw; bb < p.B; bb += (int)gridDim.x * kSWaves) {
      if (sm_s[bb] != sm_s[bb + 1]) continue;
      half_t* orow = p.o + (int64_t)bb * p.Hq * D;
      for (int i = lane; i < p.Hq * (D / 8); i += 64) st16(orow + 8 * i, uint4_t{0, 0, 0, 0});
      if (p.lse)
        for (int h = lane; h < p.Hq; h += 64) p.lse[(int64_t)bb * p.Hq + h] = AKT_SNEG_INF;
    }
  }
  if (n > 0) {  // wave-uniform

  if constexpr (DENSE) {
#pragma unroll
    for (int i = 0; i < PD; ++i) fetch(fr[i]);
#pragma unroll
    for (int i = 0; i < PD; ++i) issue(i, bufs[i], true, fr[i], true);
  } else {
    // Sequences of groups 0 .. PD-1 (their last-page lengths are loaded into
    // pll), then the lookahead from group PD on.  Group 0's q
    // fragment, group PD's fetch, then groups 1 .. PD-1: each buffer's loads in
    // the order of the main loop's, so that the compiler's wait counts at the
    // loop's entry match those of its iterations.
    la_y = y0;
    la_pp = pp0;
    la_slice = slice0;
    seek(pp0);
    int pll[PD];
#pragma unroll
    for (int i = 0; i < PD; ++i) {
      const bool seq_ok = la_b >= 0 && la_b < p.B;
      fr[i].b = seq_ok ? la_b : -1;
      fr[i].last = seq_ok && la_pp == la_end - 1;
      const int lb = min(max(la_b, 0), p.B - 1);
      pll[i] = __builtin_amdgcn_raw_buffer_load_b32(ll_rsrc, (uint32_t)lb * 4u, 0, 0);
      advance(true);
    }
    bufs[0].b = fr[0].b;
    bufs[0].last = fr[0].last;
    load_q(bufs[0].b, bufs[0].y, bufs[0].q);
    fetch(fr[0]);
#pragma unroll
    for (int i = 1; i < PD; ++i) issue(i, bufs[i], true, fr[i], false);
#pragma unroll
    for (int i = 0; i < PD; ++i) set_usable(bufs[i], pll[i]);
  }

  // ---- state of the unit being streamed ------------------------------------
  float m_run = AKT_SNEG_INF;  // running max of head c16 (log2 units)
  float e_part = 0.f;          // sum of this lane's P
  // O^T tiles of P.V: lane (R, c16) holds dims 16t + 4R + r of head c16.
  float4_t acc[NT];
  int cur_b = -1, cur_y = 0;
  // Unit bookkeeping (wave-uniform): unit id y * B + b (the units' order on
  // the axis), first head, heads, whether the unit lies inside this wave.
  int cu_unit = 0, cu_hq0 = 0, cu_nh = 0, cu_direct = 0;
  int n_seg = 0;  // partial segments left in LDS so far

  auto begin_unit = [&](int b, int y) __attribute__((always_inline)) {
    m_run = AKT_SNEG_INF;
    e_part = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = float4_t{0.f, 0.f, 0.f, 0.f};
    const StreamArgs p = reread_args();
    const int kvh = p->n_hg == 1 ? y : y / p->n_hg;
    const int hg = y - kvh * p->n_hg;
    cu_hq0 = kvh * p->G + hg * GT;
    cu_nh = min(GT, p->G - hg * GT);
    cu_unit = y * p->B + b;
    const int s0 = seq_start(b), s1 = seq_start(b + 1);
    cu_direct = y * p->TG + s0 * p->gpp >= g0 && y * p->TG + s1 * p->gpp <= g0 + n;
  };

  // Scores, online softmax and P.V of one loaded group.  Tokens past the
  // usable prefix (rows past the last page's length) get score -inf and
  // their V rows, which may hold anything, are staged as zeros.
  //   S^T = K . Q^T (16 tokens x 16 heads): A = K rows, B = the q fragment;
  //   O^T += V^T . P^T: one v_mfma_f32_16x16x16_f16 per 16 dims, A = V^T read
  //   from the staged rows with ds_read_b64_tr_b16 (lane (R, c) gets tokens
  //   4R .. 4R+3 of dim 16t + c), B = P^T straight from the score lanes
  //   (lane (R, c) holds head c's probabilities of tokens 4R .. 4R+3).
  half_t* const vst = reinterpret_cast<half_t*>(&sm_seg1[wave][0]);
  // The largest finite fp16, four times, held in vector registers (a scalar
  // one would be spilled).
  uint32_t max2 = 0x7bff7bffu;
  asm("" : "+v"(max2));
  const half4_t vmax = __builtin_bit_cast(half4_t, (uint2){max2, max2});
  auto consume = [&](const Buf& bf, int nv) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < VTOK; ++i)
#pragma unroll
      for (int jj = 0; jj < VLD; ++jj)
        *reinterpret_cast<uint4_t*>(vst + (tt0 + i) * VROW + dim0 + 8 * jj) = bf.v[i][jj];
    if (nv < 16) {  // wave-uniform: zero the rows past the usable prefix (LDS is in order)
#pragma unroll
      for (int i = 0; i < VTOK; ++i)
#pragma unroll
        for (int jj = 0; jj < VLD; ++jj)
          if (tt0 + i >= nv)
            *reinterpret_cast<uint4_t*>(vst + (tt0 + i) * VROW + dim0 + 8 * jj) = uint4_t{0, 0, 0, 0};
    }
    float4_t sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) sacc = mfma16x16x32(as_half8(bf.k[s]), bf.q[s], sacc);
    float t[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r] = (4 * R + r < nv) ? sacc[r] * p.qk_scale : AKT_SNEG_INF;
    float mt = fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]));
    mt = rows_max(mt);
    const float m_new = fmaxf(m_run, mt);
    if (__any(m_new > m_run)) {
      const float alpha = (m_new > m_run) ? fast_exp2(m_run - m_new) : 1.0f;
      e_part *= alpha;
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) acc[tt] *= alpha;
      m_run = m_new;
    }
    const float m_use = (m_run == AKT_SNEG_INF) ? 0.f : m_run;
    float pr[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) pr[r] = fast_exp2(t[r] - m_use);
    const uint32_t p01 = pack_half2(pr[0], pr[1]);
    const uint32_t p23 = pack_half2(pr[2], pr[3]);
    e_part += (pr[0] + pr[1]) + (pr[2] + pr[3]);
    const half4_t pb = __builtin_bit_cast(half4_t, (uint2){p01, p23});
    // Source lane (R, c) of the transposing read addresses token 4R + c / 4,
    // dims 16t + 4 (c % 4) .. + 3.  All tiles are read before the first MFMA.
    const half_t* vrd = vst + (4 * R + (c16 >> 2)) * VROW + 4 * (c16 & 3);
    half4_t va[NT];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) va[tt] = __builtin_bit_cast(half4_t, ds_read_tr16(vrd + 16 * tt));
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
      acc[tt] = __builtin_amdgcn_mfma_f32_16x16x16f16(va[tt], pb, acc[tt], 0, 0, 0);
    // The residual is zero or negative for many tokens (zero for the row's
    // maximum), where an infinite V would make the sum NaN: it multiplies V
    // clamped to the finite range, so that infinities enter through P alone.
    // (Clamping costs 0.3%: 32 sequences of 256-8192 tokens 106.7 -> 107.0 us.)
    const half4_t pl = {(half_t)(pr[0] - (float)pb[0]), (half_t)(pr[1] - (float)pb[1]),
                        (half_t)(pr[2] - (float)pb[2]), (half_t)(pr[3] - (float)pb[3])};
#pragma unroll
    for (int tt = 0; tt < NT; ++tt)
      acc[tt] = __builtin_amdgcn_mfma_f32_16x16x16f16(
          __builtin_elementwise_minimum(__builtin_elementwise_maximum(va[tt], -vmax), vmax), pl,
          acc[tt], 0, 0, 0);
  };

  // End of the current unit's segment: wave reduction, then the output (a
  // unit wholly inside this wave) or the segment's state in LDS.
  auto flush = [&]() __attribute__((always_inline)) {
    // Lane (R, c16) holds head c16's dims 16t + 4R + r: only the normalisers
    // are summed over the four rows.
    // One sum normalises O and gives the LSE.  (The merged rows keep a word for
    // each: with two-word rows the compiler's schedule of the whole kernel was
    // worse, 105 against 94.4 us on the dense case above.)
    const float e_w = rows_sum(e_part);
    const float l_w = e_w;
    if (cu_direct) {
      const StreamArgs a = reread_args();
      if (c16 < cu_nh) {
        const int64_t row = (int64_t)cur_b * a->Hq + cu_hq0 + c16;
        const float inv = l_w > 0.f ? 1.0f / l_w : 0.f;
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) store_o4(a->o, row, 16 * tt + 4 * R, acc[tt], inv);
        if (R == 0) store_lse(a->lse, row, m_run, e_w);
      }
    } else {
      float* seg = n_seg == 0 ? &sm_seg0[wave][0] : &sm_seg1[wave][0];
      if (c16 < cu_nh) {
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
          *reinterpret_cast<uint4_t*>(seg + c16 * OROW + 16 * tt + 4 * R) = as_uint4f(acc[tt]);
        if (R == 0) sm_ml[wave][n_seg][c16] = float4_t{m_run, l_w, e_w, 0.f};
      }
      if (lane == 0) sm_unit[wave][n_seg] = cu_unit;
      n_seg = 1;  // a second partial segment is the wave's last
    }
  };

  // ---- stream the range, PD groups in flight --------------------------------
  {
    // Balance of the two waves of a SIMD: the older one wins issue
    // arbitration, and with equal ranges it would finish ~15% before the
    // younger one (measured on MI355X).  After each group a wave publishes
    // its progress and runs at raised priority while it is behind its partner.
    int done = 0;
    auto balance = [&]() __attribute__((always_inline)) {
      if constexpr (PAIRED) {
        ++done;
        if (lane == 0)
          __hip_atomic_store(&sm_prog[wave], done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const int other = uniform(__hip_atomic_load(&sm_prog[wave ^ 4], __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_WORKGROUP));
        if (done < other) __builtin_amdgcn_s_setprio(1);
        else __builtin_amdgcn_s_setprio(0);
      }
    };
    auto step = [&](Buf& bf) __attribute__((always_inline)) {
      if (bf.b != cur_b || bf.y != cur_y) {  // wave-uniform
        if (cur_b >= 0) flush();
        if (bf.b >= 0) begin_unit(bf.b, bf.y);
        cur_b = bf.b;
        cur_y = bf.y;
      }
      if (bf.nv > 0) consume(bf, bf.nv);
      balance();
    };
    // Every iteration issues its loads (groups past the range read the q
    // row), so the loads after each buffer's are always the same ones.
    for (int j = 0; j < n; j += PD) {
#pragma unroll
      for (int i = 0; i < PD; ++i) {
        if (j + i < n) step(bufs[i]);
        issue(j + i + PD, bufs[i], true, fr[i], true);
      }
    }
    if (cur_b >= 0) flush();
    if constexpr (PAIRED) {
      __builtin_amdgcn_s_setprio(0);
      if (lane == 0)  // done: the partner no longer competes with this wave
        __hip_atomic_store(&sm_prog[wave], 1 << 30, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }

  }  // n > 0

  // ---- merge ------------------------------------------------------------------
  // Layout of a merging wave: lane l owns NVL consecutive float4 vectors of the
  // unit's output (vectors l*NVL .. l*NVL + NVL - 1), all of one head (64 is a
  // multiple of GT), so it needs one (m, l, e) row per state; U states are
  // loaded per round trip.
  const StreamArgs a = reread_args();
  constexpr int NV = GT * D / 4;               // float4 vectors of a unit's output
  constexpr int NVL = NV >= 64 ? NV / 64 : 1;  // per lane
  constexpr int U = 32 / (NVL + 1) > 0 ? 32 / (NVL + 1) : 1;
  const int vec0 = NV < 64 ? min(lane, NV - 1) : lane * NVL;
  const bool has_vec = NV >= 64 || lane < NV;
  const int mh = (vec0 * 4) / D;
  const int md = vec0 * 4 - mh * D;
  float M, L, E;
  float4_t Acc[NVL];
  auto merge_begin = [&]() __attribute__((always_inline)) {
    M = AKT_SNEG_INF;
    L = E = 0.f;
#pragma unroll
    for (int i = 0; i < NVL; ++i) Acc[i] = float4_t{0.f, 0.f, 0.f, 0.f};
  };
  // Adds one state (its ml row and this lane's vectors).
  auto merge_add = [&](float4_t ml, const float4_t (&ov)[NVL]) __attribute__((always_inline)) {
    const float m = ml[0];
    if (m > M) {
      const float sc = fast_exp2(M - m);  // 0 while M = -inf (Acc, L, E are 0 then)
#pragma unroll
      for (int i = 0; i < NVL; ++i) Acc[i] *= sc;
      L *= sc;
      E *= sc;
      M = m;
    }
    // A state without usable tokens (m = -inf, sums 0) adds nothing; one whose
    // every score is NaN has m = -inf too, and its NaN sums come through.
    const float f = fast_exp2(m - (M == AKT_SNEG_INF ? 0.f : M));
#pragma unroll
    for (int i = 0; i < NVL; ++i) Acc[i] += f * ov[i];
    L += f * ml[1];
    E += f * ml[2];
  };
  auto merge_lds = [&](const float* seg, float4_t ml) __attribute__((always_inline)) {
    float4_t ov[NVL];
#pragma unroll
    for (int i = 0; i < NVL; ++i)
      ov[i] = as_float4u(*reinterpret_cast<const uint4_t*>(seg + mh * OROW + md + 4 * i));
    merge_add(ml, ov);
  };
  // The unit's place: head group y, sequence b, groups [first, last] of the axis.
  auto unit_place = [&](int unit, int& y, int& b, int& first, int& last)
                        __attribute__((always_inline)) {
    y = unit / a->B;
    b = unit - y * a->B;
    first = y * a->TG + seq_start(b) * a->gpp;
    last = y * a->TG + seq_start(b + 1) * a->gpp - 1;
  };
  auto merge_out = [&](int y, int b) __attribute__((always_inline)) {
    const int kvh = a->n_hg == 1 ? y : y / a->n_hg;
    const int hg = y - kvh * a->n_hg;
    if (has_vec && mh < min(GT, a->G - hg * GT)) {
      const int64_t row = (int64_t)b * a->Hq + kvh * a->G + hg * GT + mh;
      const float inv = L > 0.f ? 1.0f / L : 0.f;
#pragma unroll
      for (int i = 0; i < NVL; ++i) store_o4(a->o, row, md + 4 * i, Acc[i], inv);
      if (md == 0) store_lse(a->lse, row, M, E);
    }
  };
  auto mstart = [&](int w) __attribute__((always_inline)) -> int {
    return wave_start<DENSE, kSWaves>(*a, w);
  };
  // The workgroups [wf, wf + nc) whose ranges hold the unit's groups.
  auto unit_run = [&](int unit, int first, int last, int& wf, int& nc)
                      __attribute__((always_inline)) {
    if (DENSE && a->wgs_log >= 0) {
      nc = 1 << a->wgs_log;
      wf = unit << a->wgs_log;
      return;
    }
    // The wave whose range holds group g: the float estimate is off by at most
    // one (W <= 4096, 24-bit products), and the range starts settle it.
    auto wave_of = [&](int g) __attribute__((always_inline)) -> int {
      int w = min((int)((float)g * a->w_per_g), a->W - 1);
      while (w > 0 && mstart(w) > g) --w;
      while (mstart(w + 1) <= g) ++w;
      return w;
    };
    wf = wave_of(first) / kSWaves;
    nc = wave_of(last) / kSWaves - wf + 1;
  };
  // Partial slots of a unit whose run starts in workgroup wf: workgroup w's is
  // w + min(wf, unit), both of which grow along the axis, the second by at
  // least one from a unit to the next that shares a workgroup with it, so no
  // two partials share a slot (whole units: w itself).
  auto first_slot = [&](int unit, int wf) __attribute__((always_inline)) -> int {
    return DENSE && a->wgs_log >= 0 ? wf : wf + min(wf, unit);
  };
  // Partials c0, c0 + step, ... (U of them, clamped to the last) of a unit
  // whose slots start at slot0.
  auto load_partials = [&](int slot0, int c0, int step, int nc, float4_t (&ml)[U],
                           float4_t (&ov)[U][NVL]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = min(c0 + u * step, nc - 1);
      const int64_t ph = ((int64_t)slot0 + c) * GT + mh;
      ml[u] = as_float4u(ld16_device(a->part_ml, (uint32_t)(ph * 16)));
#pragma unroll
      for (int i = 0; i < NVL; ++i)
        ov[u][i] = as_float4u(ld16_device(a->part_o, (uint32_t)((ph * D + md + 4 * i) * 4)));
    }
  };
  const int wave0 = (int)blockIdx.x * kSWaves;
  const int wg0 = mstart(wave0), wg1 = mstart(wave0 + kSWaves);  // the workgroup's groups

  __syncthreads();  // every wave's segments are in LDS
  // Each unit's segments are combined by the wave that holds the unit's first
  // one in this workgroup; the waves after it hold theirs in slot 0 (a unit
  // that began before a wave's range is that wave's first segment).
#pragma unroll
  for (int sl = 0; sl < 2; ++sl) {
    const int unit = uniform(sm_unit[wave][sl]);
    if (unit < 0) continue;
    int y, b, first, last;
    unit_place(unit, y, b, first, last);
    if (wave > 0 && first < mstart(wave0 + wave)) continue;  // an earlier wave's
    merge_begin();
    merge_lds(sl == 0 ? &sm_seg0[wave][0] : &sm_seg1[wave][0], sm_ml[wave][sl][mh]);
    for (int w = wave + 1; w < kSWaves && uniform(sm_unit[w][0]) == unit; ++w)
      merge_lds(&sm_seg0[w][0], sm_ml[w][0][mh]);
    if (first >= wg0 && last < wg1) {
      merge_out(y, b);
      continue;
    }
    // A partial of the workgroup.
    int wf, nc;
    unit_run(unit, first, last, wf, nc);
    const int slot0 = first_slot(unit, wf);
    if (has_vec) {
      const int64_t ph = ((int64_t)slot0 + (int)blockIdx.x - wf) * GT + mh;
#pragma unroll
      for (int i = 0; i < NVL; ++i)
        st16_device(a->part_o, (uint32_t)((ph * D + md + 4 * i) * 4), as_uint4f(Acc[i]));
      if (md == 0) st16_device(a->part_ml, (uint32_t)(ph * 16), as_uint4f(float4_t{M, L, E, 0.f}));
    }
    // The stores (device scope) are complete before the count.  Only one unit
    // reaches out of a workgroup's end, so wf names the unit's counter.
    __builtin_amdgcn_s_waitcnt(0);
    int prev = 0;
    if (lane == 0) prev = atomicAdd(&a->arrive[wf], 1);
    if (uniform(prev) != nc - 1) continue;
    if (lane == 0) atomicExch(&a->arrive[wf], 0);
    if (nc > U) {
      if (lane == 0) sm_fin[first < wg0 ? 0 : 1] = unit;
      continue;
    }
    // One round trip's worth: merged here, without the workgroup's barriers.
    float4_t ml[U], ov[U][NVL];
    load_partials(slot0, 0, 1, nc, ml, ov);
    merge_begin();
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < nc) merge_add(ml[u], ov[u]);
    merge_out(y, b);
  }
  __syncthreads();
  // Longer units whose last partial this workgroup counted: wave v takes partials v,
  // v + kSWaves, ... of the unit's run, then one wave combines the waves.
#pragma unroll 1
  for (int k = 0; k < 2; ++k) {
    const int unit = uniform(sm_fin[k]);
    if (unit < 0) continue;  // workgroup-uniform
    int y, b, first, last;
    unit_place(unit, y, b, first, last);
    int wf, nc;
    unit_run(unit, first, last, wf, nc);
    const int slot0 = first_slot(unit, wf);
    merge_begin();
    for (int c0 = wave; c0 < nc; c0 += U * kSWaves) {
      float4_t ml[U], ov[U][NVL];
      load_partials(slot0, c0, kSWaves, nc, ml, ov);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (c0 + u * kSWaves < nc) merge_add(ml[u], ov[u]);
    }
    if (has_vec) {
#pragma unroll
      for (int i = 0; i < NVL; ++i)
        *reinterpret_cast<uint4_t*>(&sm_seg0[wave][mh * OROW + md + 4 * i]) = as_uint4f(Acc[i]);
      if (md == 0) sm_ml[wave][0][mh] = float4_t{M, L, E, 0.f};
    }
    __syncthreads();
    if (wave == 0) {
      merge_begin();
      for (int w = 0; w < min(nc, kSWaves); ++w) merge_lds(&sm_seg0[w][0], sm_ml[w][0][mh]);
      merge_out(y, b);
    }
    __syncthreads();  // the buffers are reused by the second unit
  }
}

// Waves of a launch of instance (D, GT, DENSE) over N groups on `blocks`
// workgroups, and each wave's share.
template <int D, int GT, bool DENSE>
struct Stream {
  static constexpr int kThreads = stream_threads<D, GT>();
  static constexpr int kWaves = kThreads / kWave;

  // Workgroups resident at once (at most kStreamMaxWaves waves); `unknown`
  // where no device can be queried.
  static int64_t blocks(int64_t unknown) {
    const int64_t cap = resident_blocks<paged_stream_kernel<D, GT, DENSE>>(kThreads);
    return cap <= 0 ? unknown : std::min<int64_t>(cap, kStreamMaxWaves / kWaves);
  }
  static int64_t wave_cap() { return blocks(kStreamMaxWaves / kWaves) * kWaves; }

  static int64_t grid(int64_t N) {
    return std::max<int64_t>(1, std::min(blocks(kCUs), ceil_div(N, kWaves)));
  }
  // Workgroups per unit of a dense launch as a power of two (whole units: no
  // unit straddles a workgroup's end), or -1 for stream-K ranges.  The most
  // workgroups per unit that stay resident at once, if they fill the device, or
  // fill three quarters of it and a wave has at most 8 groups (balance matters
  // less than the shorter merge then).  Measured (us, whole units / stream-K):
  // D = 64, 128 units of 64 groups 10.6 / 11.0, 52 of 44 8.9 / 9.4; D = 128
  // 17.2 / 17.6, 10.7 / 11.0; D = 256 26.8 / 27.1, 13.5 / 14.7.
  static int dense_wgs_log(int64_t units, int64_t unit_groups) {
    const int64_t most = blocks(kCUs);
    if (units > most) return -1;
    int k = 0;
    while ((units << (k + 1)) <= most && unit_groups >= ((int64_t)kWaves << (k + 1))) ++k;
    const int64_t used = units << k;
    const bool even = used == most || (4 * used >= 3 * most && unit_groups <= ((int64_t)kWaves << (k + 3)));
    return even ? k : -1;
  }
  static int64_t dense_grid(int64_t units, int64_t unit_groups, int wgs_log) {
    return wgs_log >= 0 ? units << wgs_log : grid(units * unit_groups);
  }
  // Partial slots of a dense launch (first_slot in the kernel).
  static int64_t dense_parts(int64_t units, int64_t unit_groups) {
    const int k = dense_wgs_log(units, unit_groups);
    const int64_t g = dense_grid(units, unit_groups, k);
    return k >= 0 ? g : g + std::min(units, g);
  }

  static int launch(StreamParams p, hipStream_t st) {
    constexpr auto kernel = paged_stream_kernel<D, GT, DENSE>;
    if (resident_blocks<kernel>(kThreads) <= 0)
      return set_error(AKT_ERR_HIP, "occupancy query failed");
    p.wgs_log = DENSE ? dense_wgs_log((int64_t)p.Y * p.B, p.gpp) : -1;
    const int64_t g = DENSE ? dense_grid((int64_t)p.Y * p.B, p.gpp, p.wgs_log) : grid(p.N);
    p.W = (int)std::max<int64_t>(1, std::min<int64_t>(g * kWaves, p.N));
    p.wq = p.N / p.W;
    p.wf20 = (uint32_t)(((int64_t)(p.N % p.W) << 20) / p.W);
    p.w_per_g = p.N > 0 ? (float)p.W / (float)p.N : 0.f;
    KernelTimer timer;
    timer.launch(kernel, dim3((unsigned)g), dim3(kThreads), 0, st, p);
    return check_launch("paged_stream_kernel");
  }
};

// Calls f with the instance for head dim D and gt heads per unit (both checked
// by the callers; D = 256 units hold at most 8 heads).
template <bool DENSE, int D, typename F>
auto with_gt(int gt, F f) {
  switch (gt) {
    case 1: return f(Stream<D, 1, DENSE>());
    case 2: return f(Stream<D, 2, DENSE>());
    case 4: return f(Stream<D, 4, DENSE>());
    case 8: return f(Stream<D, 8, DENSE>());
  }
  return f(Stream<D, D == 256 ? 8 : 16, DENSE>());
}
template <bool DENSE, typename F>
auto with_instance(int D, int gt, F f) {
  if (D == 64) return with_gt<DENSE, 64>(gt, f);
  if (D == 128) return with_gt<DENSE, 128>(gt, f);
  return with_gt<DENSE, 256>(gt, f);
}

}  // namespace

bool paged_stream_eligible(int64_t batch, int64_t page_size, int64_t total_pages, int64_t Y) {
  return batch >= 1 && batch <= kStreamMaxBatch && page_size % 16 == 0 &&
         Y * total_pages * (page_size / 16) < ((int64_t)1 << 31);
}

int64_t paged_stream_wave_cap(int D, int gt) {
  return with_instance<false>(D, gt, [](auto s) { return s.wave_cap(); });
}

int paged_stream_launch(const StreamParams& p, int D, int gt, hipStream_t st) {
  return with_instance<false>(D, gt, [&](auto s) { return s.launch(p, st); });
}

bool dense_stream_eligible(int64_t batch, int64_t seq_len, int64_t Y, int64_t k_row,
                           int64_t v_row) {
  const int64_t most = (int64_t)1 << 26;
  return batch >= 1 && seq_len >= 1 && k_row >= 0 && k_row < most && v_row >= 0 && v_row < most &&
         batch < ((int64_t)1 << 31) / Y / ceil_div(seq_len, 16);
}

int64_t dense_stream_parts(int D, int gt, int64_t units, int64_t unit_groups) {
  return with_instance<true>(D, gt, [&](auto s) { return s.dense_parts(units, unit_groups); });
}

int dense_stream_launch(const StreamParams& p, int D, int gt, hipStream_t st) {
  return with_instance<true>(D, gt, [&](auto s) { return s.launch(p, st); });
}

}  // namespace akt
