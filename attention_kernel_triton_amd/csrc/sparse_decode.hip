// Sparse-token decode for gfx950: each query head attends the kept tokens of its
// own index list, over a dense cache
// (sparsetoken_decode_flash_attention_redundant.py:11-124) or a paged one
// (sparsetoken_decode_flash_attention_redundant_var_len_paged.py:11-167), and the
// MagicPIG form with its log-sum-exp
// (magicpig_sparsetoken_decode_flash_attention_redundant_var_len_paged_with_norm.py:16-164).
//
// A row is one (sequence, query head).  Its n kept tokens are cut into 16-token
// groups, shared evenly by the 4 n_split waves of the row's n_split workgroups,
// each a contiguous run.  Block x is workgroup x / rows of row x % rows, so that
// consecutive blocks, which the dispatcher deals to the XCDs in turn, are
// different rows.
//
// What bounds it is a chain of dependent round trips (arguments, row length,
// token indices, page ids, K/V rows, then the merge), not bytes: a wave has
// few groups at the usual sizes.  So a wave resolves 64 tokens at once, one to
// a lane: one load of indices and one of page ids for four groups, the next
// four groups' during the current ones, and every group's row loads go out
// from registers, one group ahead.  (With an index and a page lookup before
// each group's rows, waiting for them also waited, in order, for the previous
// group's rows.  Graph replays: B=3, Hq=32, D=256, 2% of 8192-32768 tokens 17.4 ->
// 15.0 us, with MagicPIG 18.2 -> 17.5; B=1, Hq=32, D=128, 2% of 32000 tokens 9.1 ->
// 7.8.  Rows that keep nearly everything lose: 1024 of 2000 out of 2048 tokens,
// D = 128 146 -> 152, D = 256 280 -> 298.)
//
// Per group: D/32 v_mfma_f32_16x16x32_f16 give the scores, the query in all 16
// columns, so that lane (R, c) holds tokens 4R .. 4R+3 in any column; the online
// softmax is uniform over the wave; P is rounded to fp16 as the reference rounds
// it; P.V runs on the VALU (v_dot2_f32_f16 over token pairs), 16-lane row R on
// the tokens whose probabilities it holds.  Loads of one row are contiguous
// over its lanes (64 bytes of K, 256 of V per instruction).
#include <math.h>

#include "akt_common.hpp"
#include "akt_host.hpp"
#include "sparse_decode.hpp"

namespace akt {
namespace {

#define AKT_NEG_INF (-__builtin_inff())

constexpr int kSpThreads = 256;
constexpr int kSpWaves = kSpThreads / kWave;

// g(y) = log1p(y) - y for y > -1, without the cancellation of the direct
// difference near 0.  With s = y / (2 + y), log1p(y) = 2 atanh(s) =
// 2 (s + s^3/3 + s^5/5 + ...) and 2 s - y = -y s, so
//   g(y) = -y s + 2 s^3 (1/3 + s^2/5 + s^4/7 + s^6/9 + s^8/11 + ...),
// whose two parts never cancel for |y| < 0.25 (|s| < 1/7: the dropped terms
// are below 1e-10 relative).  From |y| = 0.25 on, the direct difference
// loses at most 3 bits.
__device__ __forceinline__ float log1p_minus_id(float y) {
  if (fabsf(y) < 0.25f) {
    const float s = y / (2.0f + y);
    const float s2 = s * s;
    const float poly =
        (1.0f / 3.0f) + s2 * ((1.0f / 5.0f) + s2 * ((1.0f / 7.0f) + s2 * ((1.0f / 9.0f) + s2 * (1.0f / 11.0f))));
    return __builtin_fmaf(-y, s, 2.0f * s * s2 * poly);
  }
  return log1pf(y) - y;
}

// MagicPIG correction ln u for one token (eq. 11 of the reference's
// attention_with_norm.png, as evaluated in
// magicpig_sparsetoken_decode_flash_attention_redundant_var_len_paged_with_norm.py:110-160):
//   p = 1 - acos(c) / pi (clamped to [0, 1]),  x = p^K,
//   u = 1 - (1 - x)^L - L x (1 - x)^(L - 1),  clamped to >= 1e-10.
// u is a difference of nearly equal terms when x is small or L is near 1, so
// it is evaluated in fp32 in a form without that cancellation.  With m = L - 1,
//   u = 1 - (1 - x)^m (1 + m x) = -expm1(f),
//   f = m log1p(-x) + log1p(m x) = m g(-x) + g(m x),   g(y) = log1p(y) - y
// (the linear terms -m x and +m x cancel exactly), and for L >= 1 both parts
// of f are <= 0, so nothing cancels for any x in [0, 1) and any L >= 1.  The
// relative error of u stays within a few fp32 ulps.  Outside that domain
// (x >= 1 from K < 0, or m x <= -1 from L < 0) the reference's formula is
// evaluated as written, with its clamp of 1 - x to [0, 1].
__device__ __forceinline__ float magicpig_log_u(float cosv, float K, float L) {
  const float pp = fminf(fmaxf(1.0f - acosf(cosv) * (float)M_1_PI, 0.0f), 1.0f);
  const float x = pp > 0.0f ? __expf(K * __logf(pp)) : 0.0f;
  const float m = L - 1.0f;
  const float mx = m * x;
  float u;
  if (x < 1.0f && mx > -1.0f) {
    u = -expm1f(__builtin_fmaf(m, log1p_minus_id(-x), log1p_minus_id(mx)));
  } else {
    const float om = fminf(fmaxf(1.0f - x, 0.0f), 1.0f);
    u = 1.0f - powf(om, L) - L * x * powf(om, m);
  }
  return __logf(fmaxf(u, 1e-10f));
}

template <int D, bool PAGED, bool MAGIC>
__global__ __launch_bounds__(kSpThreads)
__attribute__((amdgpu_waves_per_eu(2, 8))) void sparse_kernel(SparseParams p) {
  constexpr int KS = D / 32;                 // MFMA k-steps (8 elements a lane each)
  constexpr int VTOK = (D == 64) ? 2 : 4;    // V tokens per lane per group
  constexpr int VLD = (D == 256) ? 2 : 1;    // 16-byte loads per V token
  constexpr int VDIM = 8 * VLD;              // V dims per lane
  constexpr int NV = D / 4;                  // float4 vectors of a row's output
  const uint32_t kOnes = 0x3c003c00u;        // half2(1, 1)

  __shared__ float4_t sm_o[kSpWaves][NV];
  __shared__ float sm_m[kSpWaves], sm_l[kSpWaves], sm_e[kSpWaves];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = uniform(tid >> 6);
  const int R = lane >> 4;
  const int c16 = lane & 15;

  // ---- the row, its kept tokens and this wave's groups -----------------------
  const int c = (int)blockIdx.x / p.rows;
  const int u = (int)blockIdx.x - c * p.rows;
  const int b = u / p.Hq;
  const int hq = u - b * p.Hq;
  const int kvh = hq / p.G;
  int n;
  const int* ind_row;
  if (p.csr_ptr) {  // CSR rows: any length, no padding
    const int64_t r0 = p.csr_ptr[u], r1 = p.csr_ptr[u + 1];
    ind_row = p.sparse_ind + r0;
    n = (int)min(max(r1 - r0, (int64_t)0), (int64_t)INT32_MAX);
  } else {  // padded rows [B, Hq, l_max] with a count per row
    ind_row = p.sparse_ind + (int64_t)b * p.ind_sb + (int64_t)hq * p.ind_sh;
    n = p.sparse_nnz[(int64_t)b * p.nnz_sb + (int64_t)hq * p.nnz_sh];
    n = min(max(n, 0), p.l_max);
    // A dense-cache row with no kept token attends to its first index slot, as
    // the reference's PyTorch path does (it treats nnz == 0 as nnz == 1,
    // sparsetoken_decode_flash_attention_redundant.py:191-194); with the
    // harness's -1 padding that slot names the last row.
    if constexpr (!PAGED) n = max(n, min(1, p.l_max));
  }
  n = uniform(n);
  int pstart = 0, np = 0;
  if constexpr (PAGED) {
    pstart = p.indptr[b];
    np = p.indptr[b + 1] - pstart;
  }
  // Wave w of W takes G / W groups, one more for the first G % W.
  const int groups = (int)(((uint32_t)n + 15u) >> 4);
  const int w = c * kSpWaves + wave, W = p.n_split * kSpWaves;
  const int gq = groups / W, gr = groups - gq * W;
  const int gs = w * gq + min(w, gr);
  const int ng = gq + (w < gr ? 1 : 0);

  const half_t* qrow = p.q + (int64_t)b * p.q_sb + (int64_t)hq * p.q_sh;
  const half_t* kb = p.kbase + (PAGED ? 0 : (int64_t)b * p.k_batch) + (int64_t)kvh * p.k_head;
  const half_t* vb = p.vbase + (PAGED ? 0 : (int64_t)b * p.v_batch) + (int64_t)kvh * p.v_head;

  // Query fragment (MFMA B operand): dims 32 s + 8 R + e in every column.
  half8_t qf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) qf[s] = as_half8(ld16(qrow + 32 * s + 8 * R));

  // ---- kept tokens, 64 at a time: lane l holds token 64 k + l of the wave's run
  struct Batch {
    int row, slot;   // dense: token; paged: page id and slot
    uint64_t ok;     // usable tokens (a bit per lane)
  };
  // Entries past the row's last are read clamped to it and not usable.
  auto load_index = [&](int k) __attribute__((always_inline)) -> int {
    return ind_row[min(16u * gs + 64u * k + lane, (uint32_t)n - 1u)];
  };
  auto resolve = [&](int k, int t) __attribute__((always_inline)) -> Batch {
    Batch r;
    bool ok = 16u * gs + 64u * k + lane < (uint32_t)n;
    if constexpr (PAGED) {
      const int lp = t >= 0 ? (int)((uint32_t)t / (uint32_t)p.page_size) : 0;
      ok = ok && t >= 0 && lp < np;
      // np == 0 (no pages) reads the row's first kept index (always mapped)
      // instead of an empty page table; such tokens are never used.
      const int* pptr = np > 0 ? p.indices + pstart + min(lp, np - 1) : ind_row;
      r.row = *pptr;
      r.slot = t - lp * p.page_size;
      ok = ok && r.row >= 0 && r.row < p.num_pool_pages;
    } else {
      // Torch indexing, as the reference's gather K[b, h, ind] does
      // (sparsetoken_decode_flash_attention_redundant.py:196): -S <= t < 0 names
      // row S + t.
      if (t < 0) t += p.S;
      ok = ok && t >= 0 && t < p.S;
      r.row = t;
      r.slot = 0;
    }
    r.ok = __ballot(ok);
    return r;
  };

  // ---- one 16-token group in flight ------------------------------------------
  // Every load is issued whatever the data (a lane whose token is unusable
  // reads the q row, always mapped and finite), so that no load sits behind a
  // branch and the wait counts cover only the buffer being consumed.
  const int dim0 = (D == 64) ? 8 * (c16 & 7) : 8 * c16;  // and + 128 for the second load
  const int tt0 = (D == 64) ? (4 * R + 2 * (c16 >> 3)) : 4 * R;
  struct Buf {
    uint4_t k[KS];
    uint4_t v[VTOK][VLD];
    uint32_t mask;  // bit t: token t usable
  };
  auto issue = [&](const Batch& bt, int k4, Buf& bf) __attribute__((always_inline)) {
    const int src = 16 * k4;
    bf.mask = (uint32_t)(bt.ok >> src) & 0xffffu;
    auto row_off = [&](int t, int64_t sa) __attribute__((always_inline)) -> int64_t {
      int64_t off = (int64_t)__shfl(bt.row, src + t, 64) * sa;
      if constexpr (PAGED) off += (int64_t)__shfl(bt.slot, src + t, 64) * p.k_sb;
      return off;
    };
    const int64_t ko = row_off(c16, p.k_sa);
    const half_t* kr = ((bf.mask >> c16) & 1 ? kb + ko : qrow) + 8 * R;
#pragma unroll
    for (int s = 0; s < KS; ++s) bf.k[s] = ld16(kr + 32 * s);
#pragma unroll
    for (int i = 0; i < VTOK; ++i) {
      const int64_t vo = row_off(tt0 + i, p.v_sa);
      const half_t* vr = ((bf.mask >> (tt0 + i)) & 1 ? vb + vo : qrow) + dim0;
#pragma unroll
      for (int j = 0; j < VLD; ++j) bf.v[i][j] = ld16(vr + 128 * j);
    }
  };

  // ---- state ---------------------------------------------------------------
  float q_norm = 0.f, lsh_k = 0.f, lsh_l = 0.f;  // MagicPIG
  if constexpr (MAGIC) {
    lsh_k = p.lsh_k[u];
    lsh_l = p.lsh_l[u];
    float qs = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint4_t x = as_uint4(qf[s]);
#pragma unroll
      for (int j = 0; j < 4; ++j) qs = dot2(x[j], x[j], qs);
    }
    q_norm = sqrtf(rows_sum(qs));
  }
  float m_run = AKT_NEG_INF;  // running max (log2 units), the same in every lane
  // This lane's share (tokens 4R + r) of the sums of the fp16-rounded P, which
  // normalises O, and of the fp32 P, for the log-sum-exp.
  float l_part = 0.f, e_part = 0.f;
  float acc[VDIM];
#pragma unroll
  for (int d = 0; d < VDIM; ++d) acc[d] = 0.f;

  auto consume = [&](const Buf& bf) __attribute__((always_inline)) {
    float t[4];
    float4_t sacc = {0.f, 0.f, 0.f, 0.f};
    if constexpr (MAGIC) {
      // Operands swapped: lane (R, c) holds the score of token c in any R, so
      // each lane evaluates one token's correction (and has its |k|^2).
      float ks = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        sacc = mfma16x16x32(qf[s], as_half8(bf.k[s]), sacc);
#pragma unroll
        for (int j = 0; j < 4; ++j) ks = dot2(bf.k[s][j], bf.k[s][j], ks);
      }
      const float dotp = sacc[0];
      float cosv = dotp / (q_norm * sqrtf(rows_sum(ks)) + 1e-8f);
      cosv = fminf(fmaxf(cosv, -1.0f + 1e-7f), 1.0f - 1e-7f);
      const float sc = dotp * p.inv_sqrt_d - magicpig_log_u(cosv, lsh_k, lsh_l);
#pragma unroll
      for (int r = 0; r < 4; ++r) t[r] = __shfl(sc, 4 * R + r, 64) * kLog2e;
    } else {
#pragma unroll
      for (int s = 0; s < KS; ++s) sacc = mfma16x16x32(as_half8(bf.k[s]), qf[s], sacc);
#pragma unroll
      for (int r = 0; r < 4; ++r) t[r] = sacc[r] * p.qk_scale;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (!((bf.mask >> (4 * R + r)) & 1)) t[r] = AKT_NEG_INF;

    const float m_new =
        fmaxf(m_run, rows_max(fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]))));
    if (__any(m_new > m_run)) {
      const float alpha = (m_new > m_run) ? fast_exp2(m_run - m_new) : 1.0f;
      l_part *= alpha;
      e_part *= alpha;
#pragma unroll
      for (int d = 0; d < VDIM; ++d) acc[d] *= alpha;
      m_run = m_new;
    }
    const float m_use = (m_run == AKT_NEG_INF) ? 0.f : m_run;
    float pr[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) pr[r] = fast_exp2(t[r] - m_use);
    const uint32_t p01 = pack_half2(pr[0], pr[1]);
    const uint32_t p23 = pack_half2(pr[2], pr[3]);
    l_part = dot2(p23, kOnes, dot2(p01, kOnes, l_part));
    e_part += (pr[0] + pr[1]) + (pr[2] + pr[3]);
    // P.V over token pairs; D = 64: lanes c >= 8 hold the second pair.
#pragma unroll
    for (int q2 = 0; q2 < VTOK / 2; ++q2) {
      const uint32_t pp = D == 64 ? ((c16 >> 3) ? p23 : p01) : (q2 ? p23 : p01);
#pragma unroll
      for (int j = 0; j < VLD; ++j)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const uint32_t v0 = bf.v[2 * q2][j][x], v1 = bf.v[2 * q2 + 1][j][x];
          float* a = &acc[8 * j + 2 * x];
          a[0] = dot2(pp, pair_lo(v0, v1), a[0]);
          a[1] = dot2(pp, pair_hi(v0, v1), a[1]);
        }
    }
  };

  // ---- stream the wave's groups, one ahead -----------------------------------
  if (ng > 0) {  // wave-uniform; n > 0
    Batch cur = resolve(0, load_index(0));
    Buf A, B;
    issue(cur, 0, A);
    // Groups past the last re-read it (an L2 hit): every iteration issues the
    // same loads.
    for (int k0 = 0;; k0 += 4) {
      const int left = ng - k0;  // >= 1
      const int t_next = load_index(k0 / 4 + 1);
      issue(cur, min(1, left - 1), B);
      consume(A);
      if (left <= 1) break;
      issue(cur, min(2, left - 1), A);
      const Batch nxt = resolve(k0 / 4 + 1, t_next);
      consume(B);
      if (left <= 2) break;
      issue(cur, min(3, left - 1), B);
      consume(A);
      if (left <= 3) break;
      issue(left > 4 ? nxt : cur, left > 4 ? 0 : 3, A);
      consume(B);
      if (left <= 4) break;
      cur = nxt;
    }
  }

  // ---- the waves' states through LDS -----------------------------------------
  {
    const float l_w = rows_sum(l_part), e_w = rows_sum(e_part);
#pragma unroll
    for (int d = 0; d < VDIM; ++d) {
      if constexpr (D == 64) acc[d] += shfl_xor_f(acc[d], 8);
      acc[d] = rows_sum(acc[d]);
    }
    if (R == 0 && (D != 64 || c16 < 8)) {
#pragma unroll
      for (int j = 0; j < VDIM / 4; ++j)
        sm_o[wave][(dim0 + 128 * (j >> 1)) / 4 + (j & 1)] =
            float4_t{acc[4 * j], acc[4 * j + 1], acc[4 * j + 2], acc[4 * j + 3]};
    }
    if (lane == 0) {
      sm_m[wave] = m_run;
      sm_l[wave] = l_w;
      sm_e[wave] = e_w;
    }
  }
  __syncthreads();
  if (wave != 0) return;

  // ---- wave 0: workgroup state, then the row's output or a partial -------------
  const int vec = min(lane, NV - 1);  // this lane's float4 of the output
  float M = AKT_NEG_INF, L = 0.f, E = 0.f;
  float4_t O = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < kSpWaves; ++i) M = fmaxf(M, sm_m[i]);
  // A wave without usable tokens has weight and sums 0; NaN sums (a NaN in every
  // score of a wave leaves its maximum at -inf) come through.
  const float Mu = M == AKT_NEG_INF ? 0.f : M;
#pragma unroll
  for (int i = 0; i < kSpWaves; ++i) {
    const float f = fast_exp2(sm_m[i] - Mu);
    L += f * sm_l[i];
    E += f * sm_e[i];
    O += f * sm_o[i][vec];
  }
  auto write_out = [&]() __attribute__((always_inline)) {
    const float inv = L > 0.f ? 1.0f / L : 0.f;
    half4_t hv;
#pragma unroll
    for (int r = 0; r < 4; ++r) hv[r] = (half_t)(O[r] * inv);
    if (lane < NV) *reinterpret_cast<half4_t*>(p.o + (int64_t)u * D + 4 * vec) = hv;
    if (p.lse && lane == 0) p.lse[u] = E > 0.f ? (M + log2f(E)) * kLn2 : AKT_NEG_INF;
  };
  if (p.n_split == 1) {
    write_out();
    return;
  }
  // Stored with device scope and counted; the wave that counts the row's last
  // partial merges them all, in split order.
  const int64_t part = (int64_t)u * p.n_split + c;
  if (lane < NV) st16_device(p.part_o, (uint32_t)((part * D + 4 * vec) * 4), as_uint4f(O));
  if (lane == 0) st16_device(p.part_ml, (uint32_t)(part * 16), as_uint4f(float4_t{M, L, E, 0.f}));
  __builtin_amdgcn_s_waitcnt(0);
  int prev = 0;
  if (lane == 0) prev = atomicAdd(&p.arrive[u], 1);
  if (uniform(prev) != p.n_split - 1) return;
  if (lane == 0) atomicExch(&p.arrive[u], 0);
  constexpr int U = 8;
  M = AKT_NEG_INF;
  L = E = 0.f;
  O = float4_t{0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < p.n_split; c0 += U) {
    float4_t ml[U], ov[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int64_t ph = (int64_t)u * p.n_split + min(c0 + i, p.n_split - 1);
      ml[i] = as_float4u(ld16_device(p.part_ml, (uint32_t)(ph * 16)));
      ov[i] = as_float4u(ld16_device(p.part_o, (uint32_t)((ph * D + 4 * vec) * 4)));
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const float m = ml[i][0];
      if (c0 + i >= p.n_split) continue;
      if (m > M) {
        const float s = fast_exp2(M - m);  // 0 while M = -inf (O, L, E are 0 then)
        O *= s;
        L *= s;
        E *= s;
        M = m;
      }
      const float f = fast_exp2(m - (M == AKT_NEG_INF ? 0.f : M));
      O += f * ov[i];
      L += f * ml[i][1];
      E += f * ml[i][2];
    }
  }
  write_out();
}

template <int D>
int launch_sparse(const SparseParams& p, bool paged, bool magic, hipStream_t st) {
  auto kernel = !paged ? sparse_kernel<D, false, false>
                       : (magic ? sparse_kernel<D, true, true> : sparse_kernel<D, true, false>);
  KernelTimer timer;
  timer.launch(kernel, dim3((unsigned)(p.rows * (int64_t)p.n_split)), dim3(kSpThreads), 0, st, p);
  return check_launch("sparse_kernel");
}

}  // namespace

int sparse_launch(const SparseParams& p, int head_dim, bool paged, bool magic, hipStream_t st) {
  switch (head_dim) {
    case 64: return launch_sparse<64>(p, paged, magic, st);
    case 128: return launch_sparse<128>(p, paged, magic, st);
    case 256: return launch_sparse<256>(p, paged, magic, st);
  }
  return set_error(AKT_ERR_UNSUPPORTED, "head_dim %d not supported (64, 128, 256)", head_dim);
}

}  // namespace akt
