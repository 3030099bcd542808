"""GPU parity of kept-index selection (R8), sparse decode (R5), sparse paged decode (R6)
and MagicPIG with-norm decode (R7)."""
import math

import numpy as np
import pytest
import torch

from attention_kernel_triton_amd import _ops, kept_index
from attention_kernel_triton_amd import magicpig_sparsetoken_decode_flash_attention_redundant_var_len_paged_with_norm as mp
from attention_kernel_triton_amd import sparsetoken_decode_flash_attention_redundant as sp
from attention_kernel_triton_amd import sparsetoken_decode_flash_attention_redundant_var_len_paged as spp
from attention_kernel_triton_amd import synthetic as syn
from helpers import assert_close, max_abs_err
from oracle import naive
from oracle.kept import kept_from_uniform, kept_indices

pytestmark = pytest.mark.gpu


# --------------------------------------------------------------------------- kept-index
def _select(s, dev):
    return kept_index.select_kept(s.l_max, uniform=s.uniform.to(dev), kept_ratio=s.kept_ratio,
                                  row_len=s.row_len.to(dev))


def test_kept_index_config4a_bit_exact(dev):
    s = syn.sparse_config()
    ind, nnz = _select(s, dev)
    B, H, N = s.uniform.shape
    rind, rnnz = kept_from_uniform(s.uniform.reshape(B * H, N).numpy(), s.kept_ratio, s.l_max,
                                   s.row_len.reshape(-1).numpy())
    assert np.array_equal(ind.cpu().reshape(B * H, -1).numpy(), rind)
    assert np.array_equal(nnz.cpu().reshape(-1).numpy(), rnnz)


def test_kept_index_config4b_bit_exact(dev):
    s = syn.sparse_paged_config()
    ind, nnz = _select(s, dev)
    B, H, N = s.uniform.shape
    rind, rnnz = kept_from_uniform(s.uniform.reshape(B * H, N).numpy(), s.kept_ratio, s.l_max,
                                   s.row_len.reshape(-1).numpy())
    assert np.array_equal(ind.cpu().reshape(B * H, -1).numpy(), rind)
    assert np.array_equal(nnz.cpu().reshape(-1).numpy(), rnnz)


@pytest.mark.parametrize("ensure", [True, False])
def test_kept_index_from_mask_edge_rows(dev, ensure):
    rng = np.random.default_rng(3)
    keep = rng.random((7, 1000)) < 0.1
    keep[1] = False                    # empty row
    keep[2] = True                     # overflow past l_max
    keep[3, 255:257] = True            # across the 256-element step boundary
    ind, nnz = kept_index.select_kept(64, mask=torch.from_numpy(keep).to(dev),
                                      ensure_nonempty=ensure)
    rind, rnnz = kept_indices(keep, 64, ensure_nonempty=ensure)
    assert np.array_equal(ind.cpu().numpy(), rind)
    assert np.array_equal(nnz.cpu().reshape(-1).numpy(), rnnz)


# --------------------------------------------------------------------------- sparse dense
def _sparse_lists(s):
    B, H, N = s.uniform.shape
    ind, nnz = kept_from_uniform(s.uniform.reshape(B * H, N).numpy(), s.kept_ratio, s.l_max,
                                 s.row_len.reshape(-1).numpy())
    return (torch.from_numpy(ind).reshape(B, H, -1),
            torch.from_numpy(nnz).reshape(B, H, 1))


def test_sparse_config4a_full(dev):
    s = syn.sparse_config()
    ind, nnz = _sparse_lists(s)
    o, lse = sp.sparsetoken_flash_attention_decode(s.q.to(dev), s.K.to(dev), s.V.to(dev),
                                                   ind.to(dev), nnz.to(dev), s.scale, s.group,
                                                   return_lse=True)
    ro, rl = naive.sparsetoken_naive_decode(s.q, s.K, s.V, ind, nnz, s.scale, s.group)
    assert o.shape == (1, 32, 1, 128)
    err = assert_close(o, ro, what="config 4a")
    assert_close(lse, rl, atol=1e-4, what="config 4a lse")
    print(f"config 4a max abs err {err:.3e}")


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("splits", [0, 1, 3])
def test_sparse_shapes_and_splits(dev, D, splits):
    s = syn.sparse_config(seed=D + splits, B=2, Hq=8, Hkv=2, S=3000, D=D, kept_ratio=0.05)
    ind, nnz = _sparse_lists(s)
    from attention_kernel_triton_amd import _ops
    o, lse = _ops.sparse_decode(s.q.to(dev), s.K.to(dev), s.V.to(dev), ind.to(dev), nnz.to(dev),
                                s.scale, return_lse=True, num_splits=splits)
    ro, rl = naive.sparsetoken_naive_decode(s.q, s.K, s.V, ind, nnz, s.scale, s.group)
    assert_close(o, ro, what=f"sparse D={D} splits={splits}")
    assert_close(lse, rl, atol=1e-4, what="sparse lse")


def test_sparse_empty_heads_and_out_of_range_indices(dev):
    """nnz == 0 and negative indices follow the reference's PyTorch path
    (sparsetoken_decode_flash_attention_redundant.py:193-196: nnz == 0 reads
    the first index slot; K[b, h, ind] wraps -S <= i < 0 to S + i), so those
    heads are compared with the oracle; indices outside [-S, S), which that
    gather would reject, are skipped."""
    s = syn.sparse_config(seed=5, B=1, Hq=6, Hkv=1, S=500, D=128, kept_ratio=0.05)
    ind, nnz = _sparse_lists(s)
    nnz[0, 1, 0] = 0                                 # empty head, slot 0 a kept index
    nnz[0, 4, 0] = 0                                 # empty head, slot 0 the -1 pad
    ind[0, 4, 0] = -1
    n5 = int(nnz[0, 5, 0])
    ind[0, 5, n5 - 1] = -3                           # row S - 3
    ind2 = ind.clone()
    n2 = int(nnz[0, 2, 0])
    ind2[0, 2, n2 - 1] = 10 ** 6                     # out of range -> skipped
    o, lse = sp.sparsetoken_flash_attention_decode(s.q.to(dev), s.K.to(dev), s.V.to(dev),
                                                   ind2.to(dev), nnz.to(dev), s.scale, s.group,
                                                   return_lse=True)
    o, lse = o.cpu(), lse.cpu()
    nnz_ref = nnz.clone()
    nnz_ref[0, 2, 0] = n2 - 1
    ro, rl = naive.sparsetoken_naive_decode(s.q, s.K, s.V, ind, nnz_ref, s.scale, s.group)
    for h in range(6):
        assert_close(o[0, h], ro[0, h], what=f"head {h}")
        assert_close(lse[0, h], rl[0, h], atol=1e-4, what=f"head {h} lse")
    # The harness-padded empty head reads the last row alone: its output is that V row.
    assert_close(o[0, 4, 0], s.V[0, 0, -1].double(), atol=1e-3, what="nnz 0 -> V[S - 1]")


# --------------------------------------------------------------------------- sparse paged
def test_sparse_paged_single_token_addressing_is_bit_exact(dev):
    """nnz = 1 returns the addressed V row bit for bit: checks page/slot translation."""
    p = syn.paged_config(seed=21, B=3, Hq=8, Hkv=2, D=256, page=16, min_len=100, max_len=900)
    g = torch.Generator().manual_seed(22)
    B, H = 3, 8
    ind = torch.full((B, H, 4), -1, dtype=torch.int32)
    toks = torch.zeros((B, H), dtype=torch.int64)
    for b in range(B):
        toks[b] = torch.randint(0, p.lens[b], (H,), generator=g)
    ind[..., 0] = toks.to(torch.int32)
    nnz = torch.ones((B, H, 1), dtype=torch.int32)
    o = spp.sparsetoken_flash_attention_decode_paged(p.q.to(dev), p.pool.to(dev),
                                                     p.indptr.to(dev), p.indices.to(dev),
                                                     ind.to(dev), nnz.to(dev)).cpu()
    for b in range(B):
        for h in range(H):
            t = int(toks[b, h])
            pid = int(p.indices[int(p.indptr[b]) + t // 16])
            assert torch.equal(o[b, h], p.pool[pid, 1, h // 4, t % 16])


@pytest.mark.parametrize("page", [1, 16, 256])
def test_sparse_paged_shapes(dev, page):
    s = syn.sparse_paged_config(seed=page, B=2, Hq=8, Hkv=2, D=128, page=page, min_len=500,
                                max_len=3000, kept_ratio=0.05, magicpig=False)
    ind, nnz = _sparse_lists(s)
    p = s.paged
    o, lse = spp.sparsetoken_flash_attention_decode_paged(p.q.to(dev), p.pool.to(dev),
                                                          p.indptr.to(dev), p.indices.to(dev),
                                                          ind.to(dev), nnz.to(dev),
                                                          return_lse=True)
    ro, rl = naive.sparsetoken_naive_paged_attention(p.q, p.pool, p.indptr, p.indices, ind, nnz)
    assert_close(o, ro, what=f"sparse paged page={page}")
    assert_close(lse, rl, atol=1e-4, what="sparse paged lse")


def test_sparse_paged_config4b_full(dev):
    s = syn.sparse_paged_config()
    ind, nnz = _sparse_lists(s)
    p = s.paged
    o, lse = spp.sparsetoken_flash_attention_decode_paged(p.q.to(dev), p.pool.to(dev),
                                                          p.indptr.to(dev), p.indices.to(dev),
                                                          ind.to(dev), nnz.to(dev),
                                                          return_lse=True)
    ro, rl = naive.sparsetoken_naive_paged_attention(p.q, p.pool, p.indptr, p.indices, ind, nnz)
    err = assert_close(o, ro, what="config 4b")
    assert_close(lse, rl, atol=1e-4, what="config 4b lse")
    print(f"config 4b max abs err {err:.3e}")


def test_magicpig_config4b_full(dev):
    s = syn.sparse_paged_config()
    ind, nnz = _sparse_lists(s)
    p = s.paged
    o, lse = mp.magicpig_sparsetoken_flash_attention_decode_paged(
        p.q.to(dev), p.pool.to(dev), p.indptr.to(dev), p.indices.to(dev), ind.to(dev),
        nnz.to(dev), s.lsh_k.to(dev), s.lsh_l.to(dev), return_lse=True)
    r64, l64 = naive.magicpig_sparsetoken_naive_paged_attention(
        p.q, p.pool, p.indptr, p.indices, ind, nnz, s.lsh_k, s.lsh_l)
    err = assert_close(o, r64, what="MagicPIG vs fp64 oracle")
    assert_close(lse, l64, atol=1e-3, what="MagicPIG lse vs fp64 oracle")
    # The reference's own precision (fp32) agrees except on heads whose u_i formula
    # cancels catastrophically; report how many such heads there are.
    r32, _ = naive.magicpig_sparsetoken_naive_paged_attention(
        p.q, p.pool, p.indptr, p.indices, ind, nnz, s.lsh_k, s.lsh_l, dtype=torch.float32)
    ill = [(b, h) for b in range(r64.shape[0]) for h in range(r64.shape[1])
           if max_abs_err(r32[b, h], r64[b, h]) > 1e-3]
    well = torch.ones(r64.shape[:2], dtype=torch.bool)
    for b, h in ill:
        well[b, h] = False
    err32 = max_abs_err(o.cpu()[well], r32[well])
    print(f"MagicPIG err vs fp64 {err:.3e}; vs fp32 on {int(well.sum())} well-conditioned "
          f"heads {err32:.3e}; ill-conditioned heads {len(ill)}")
    assert err32 <= 2e-3


@pytest.mark.parametrize("D,B,Hq,Hkv,min_len,max_len", [
    (128, 1, 32, 8, 32000, 32000),  # config 4's first variant: one 32000-token sequence
    (64, 2, 8, 2, 3000, 5000),
])
def test_magicpig_head_dims_64_and_128(dev, D, B, Hq, Hkv, min_len, max_len):
    """MagicPIG at head dims 64 and 128 (the kernel instances with D/4-element K
    slices per lane and, at D = 64, two V tokens per lane).  The D = 128 case is
    config 4's first variant (B = 1, Hq = 32, Hkv = 8, 32000 tokens, page 16,
    p = 0.02 kept lists from the device selection, K, L ~ U[1, 6)): O within
    2e-3 and LSE within 1e-3 of the fp64 oracle."""
    s = syn.sparse_paged_config(seed=40 + D, B=B, Hq=Hq, Hkv=Hkv, D=D, page=16,
                                min_len=min_len, max_len=max_len, kept_ratio=0.02)
    p = s.paged
    ind, nnz = _select(s, dev)
    o, lse = mp.magicpig_sparsetoken_flash_attention_decode_paged(
        p.q.to(dev), p.pool.to(dev), p.indptr.to(dev), p.indices.to(dev), ind, nnz,
        s.lsh_k.to(dev), s.lsh_l.to(dev), return_lse=True)
    assert o.shape == (B, Hq, D)
    r64, l64 = naive.magicpig_sparsetoken_naive_paged_attention(
        p.q, p.pool, p.indptr, p.indices, ind.cpu(), nnz.cpu(), s.lsh_k, s.lsh_l)
    err = assert_close(o, r64, what=f"MagicPIG D={D} vs fp64 oracle")
    assert_close(lse, l64, atol=1e-3, what=f"MagicPIG D={D} lse vs fp64 oracle")
    print(f"MagicPIG D={D}: max abs err {err:.3e}, kept per head "
          f"{float(nnz.float().mean()):.0f}")


@pytest.mark.parametrize("L", [50.0, 150.0])
def test_magicpig_many_hash_tables(dev, L):
    """Large L (the MagicPIG paper's L = 150 and 50) with K ~ U[4, 8), where
    x = p^K is small but L x is not: the regime where a truncated power series
    of u in x diverges.  O within 2e-3 and LSE within 1e-3 of the fp64 oracle;
    the test first checks that a good share of kept tokens sit in that regime."""
    s = syn.sparse_paged_config(seed=int(L), B=2, Hq=8, Hkv=2, D=128, page=16, min_len=2000,
                                max_len=6000, kept_ratio=0.05)
    p = s.paged
    g = torch.Generator().manual_seed(int(L) + 1)
    lsh_k = torch.rand(s.lsh_k.shape, generator=g) * 4 + 4
    lsh_l = torch.full_like(s.lsh_l, L)
    ind, nnz = _sparse_lists(s)
    # Share of kept tokens with x < 0.05 and L x > 1 (cosine from fp64 q, k).
    hits = total = 0
    for b in range(2):
        for h in range(8):
            n = int(nnz[b, h, 0])
            t = ind[b, h, :n].long()
            pages = p.indices[int(p.indptr[b]) + t // 16].long()
            k = p.pool[pages, 0, h // 4, t % 16].double()
            q = p.q[b, h, 0].double()
            c = (k @ q) / (q.norm() * k.norm(dim=-1) + 1e-8)
            x = (1 - torch.acos(c.clamp(-1 + 1e-7, 1 - 1e-7)) / math.pi) ** float(lsh_k[b, h])
            hits += int(((x < 0.05) & (L * x > 1)).sum())
            total += n
    assert hits > 0.2 * total, (hits, total)
    o, lse = mp.magicpig_sparsetoken_flash_attention_decode_paged(
        p.q.to(dev), p.pool.to(dev), p.indptr.to(dev), p.indices.to(dev), ind.to(dev),
        nnz.to(dev), lsh_k.to(dev), lsh_l.to(dev), return_lse=True)
    r64, l64 = naive.magicpig_sparsetoken_naive_paged_attention(
        p.q, p.pool, p.indptr, p.indices, ind, nnz, lsh_k, lsh_l)
    err = assert_close(o, r64, what=f"MagicPIG L={L} vs fp64 oracle")
    assert_close(lse, l64, atol=1e-3, what=f"MagicPIG L={L} lse vs fp64 oracle")
    print(f"MagicPIG L={L}: max abs err {err:.3e}, {hits}/{total} tokens with x < 0.05, L x > 1")


def test_magicpig_empty_head_and_L1_reduction(dev):
    s = syn.sparse_paged_config(seed=31, B=1, Hq=4, Hkv=1, D=256, page=16, min_len=600,
                                max_len=900, kept_ratio=0.05)
    ind, nnz = _sparse_lists(s)
    nnz[0, 0, 0] = 0
    p = s.paged
    Lone = torch.ones_like(s.lsh_l)
    o, lse = mp.magicpig_sparsetoken_flash_attention_decode_paged(
        p.q.to(dev), p.pool.to(dev), p.indptr.to(dev), p.indices.to(dev), ind.to(dev),
        nnz.to(dev), s.lsh_k.to(dev), Lone.to(dev), return_lse=True)
    o, lse = o.cpu(), lse.cpu()
    assert torch.equal(o[0, 0], torch.zeros_like(o[0, 0])) and torch.isinf(lse[0, 0])
    ro, rl = naive.sparsetoken_naive_paged_attention(p.q, p.pool, p.indptr, p.indices, ind, nnz)
    assert_close(o, ro, what="MagicPIG L=1 == plain sparse")
    assert_close(lse[0, 1:], rl[0, 1:] - math.log(1e-10), atol=1e-3, what="L=1 lse shift")


def test_sparse_paged_page_ids_past_32_bit_byte_offsets(dev):
    """Kept tokens on pages near the end of a 4.6 GB pool (64-bit row addresses)."""
    Hq, Hkv, page, D, P, L = 8, 8, 16, 128, 70000, 200
    npg = (L + page - 1) // page
    used = torch.arange(P - 1, P - 1 - npg, -1, dtype=torch.int32)
    g = torch.Generator().manual_seed(23)
    content = torch.randn(npg, 2, Hkv, page, D, generator=g).half()
    q = torch.randn(1, Hq, 1, D, generator=g).half()
    pool = torch.empty(P, 2, Hkv, page, D, dtype=torch.float16, device=dev)
    pool[used.long().to(dev)] = content.to(dev)
    indptr = torch.tensor([0, npg], dtype=torch.int32)
    keep = torch.rand(1, Hq, L, generator=g) < 0.1
    keep[..., L - 1] = True  # the last token lives on the highest page of the sequence
    l_max = int(keep.sum(-1).max())
    ind = torch.full((1, Hq, l_max), -1, dtype=torch.int32)
    nnz = torch.zeros(1, Hq, 1, dtype=torch.int32)
    for h in range(Hq):
        idx = keep[0, h].nonzero().flatten().to(torch.int32)
        ind[0, h, : len(idx)] = idx
        nnz[0, h, 0] = len(idx)
    o, lse = spp.sparsetoken_flash_attention_decode_paged(q.to(dev), pool, indptr.to(dev),
                                                          used.to(dev), ind.to(dev), nnz.to(dev),
                                                          return_lse=True)
    compact = torch.arange(npg, dtype=torch.int32)
    ro, rl = naive.sparsetoken_naive_paged_attention(q, content, indptr, compact, ind, nnz)
    assert_close(o, ro, what="sparse paged, page ids near 70000")
    assert_close(lse, rl, atol=1e-4, what="sparse paged lse, page ids near 70000")
    del pool


def test_sparse_empty_batch_returns_empty_outputs(dev):
    """B = 0: nothing to compute, no workspace; both sparse entry points return
    empty outputs (as dense and paged decode do)."""
    q = torch.zeros(0, 8, 1, 128, dtype=torch.float16, device=dev)
    K = torch.zeros(0, 2, 64, 128, dtype=torch.float16, device=dev)
    ind = torch.zeros(0, 8, 16, dtype=torch.int32, device=dev)
    nnz = torch.zeros(0, 8, 1, dtype=torch.int32, device=dev)
    o, lse = sp.sparsetoken_flash_attention_decode(q, K, K, ind, nnz, 0.1, 4, return_lse=True)
    assert o.shape == (0, 8, 1, 128) and lse.shape == (0, 8)
    pool = torch.zeros(4, 2, 2, 16, 128, dtype=torch.float16, device=dev)
    indptr = torch.zeros(1, dtype=torch.int32, device=dev)
    pages = torch.zeros(0, dtype=torch.int32, device=dev)
    o2 = spp.sparsetoken_flash_attention_decode_paged(q, pool, indptr, pages, ind, nnz)
    assert o2.shape == (0, 8, 128)


def test_sparse_splits_merge_deterministically(dev):
    """Split partials are merged by whichever workgroup of a row finishes last;
    the merge order is fixed, so repeated calls are bit-identical."""
    s = syn.sparse_config()
    ind, nnz = _sparse_lists(s)
    args = (s.q.to(dev), s.K.to(dev), s.V.to(dev), ind.to(dev), nnz.to(dev), s.scale, s.group)
    o0, l0 = sp.sparsetoken_flash_attention_decode(*args, return_lse=True)
    for _ in range(5):
        o, lse = sp.sparsetoken_flash_attention_decode(*args, return_lse=True)
        assert torch.equal(o, o0) and torch.equal(lse, l0)


# A query head with a NaN has NaN outputs however many waves and splits its tokens
# take (one token leaves three waves without any), and no other head changes.
@pytest.mark.parametrize("kind", ["dense", "paged", "magicpig"])
@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("n,splits", [(1, 1), (5, 3), (200, 1), (200, 3), (700, 0), (700, 12)])
def test_sparse_nan_query_head(dev, kind, D, n, splits):
    g = torch.Generator().manual_seed(n + splits + D)
    B, Hkv, G, S = 2, 2, 2, 1000
    Hq = Hkv * G
    q = torch.randn(B, Hq, 1, D, generator=g).half()
    ind = torch.stack([torch.randperm(S, generator=g)[:n].sort().values for _ in range(B * Hq)])
    ind = ind.reshape(B, Hq, n).to(torch.int32).to(dev)
    nnz = torch.full((B, Hq, 1), n, dtype=torch.int32, device=dev)
    if kind == "dense":
        K, V = (torch.randn(B, Hkv, S, D, generator=g).half().to(dev) for _ in range(2))
        run = lambda x: _ops.sparse_decode(x.to(dev), K, V, ind, nnz, 0.1,  # noqa: E731
                                           num_splits=splits)[:, :, 0]
    else:
        indptr, indices, _, P = syn.block_table(g, [S] * B, 16)
        pool = torch.randn(P, 2, Hkv, 16, D, generator=g).half().to(dev)
        lsh = {}
        if kind == "magicpig":
            lsh = {"lsh_k": torch.full((B, Hq), 10.0, device=dev),
                   "lsh_l": torch.full((B, Hq), 150.0, device=dev)}
        run = lambda x: _ops.sparse_decode_paged(  # noqa: E731
            x.to(dev), pool, indptr.to(dev), indices.to(dev), ind, nnz, num_splits=splits, **lsh)
    bad = 1
    dirty = q.clone()
    dirty[:, bad, 0, D // 3] = float("nan")
    want, got = run(q).reshape(B, Hq, D), run(dirty).reshape(B, Hq, D)
    rest = [h for h in range(Hq) if h != bad]
    assert torch.isnan(got[:, bad]).all()
    assert torch.equal(got[:, rest], want[:, rest])


def _reference_harness_fixture(dev):
    """The reference harness's sparse paged / MagicPIG case at its own shape
    (sparsetoken_decode_flash_attention_redundant_var_len_paged.py:296-330,
    magicpig_..._with_norm.py:296-317): a 1024-page pool of page size 256 and
    head dim 256, 8 kv heads and 32 query heads, three sequences of 270 / 350 /
    321 pages over a random permutation of the first 941 page ids with last
    page lengths 63 / 22 / 55, kept ratio 0.02 over each sequence's tokens,
    L_max = 512 * 256 index slots, MagicPIG K, L ~ U[1, 6)."""
    g = torch.Generator(device=dev).manual_seed(61)
    gc = torch.Generator().manual_seed(62)
    B, Hkv, G, D, page = 3, 8, 4, 256, 256
    Hq = Hkv * G
    pool = torch.randn(1024, 2, Hkv, page, D, generator=g, device=dev, dtype=torch.float16)
    npg = torch.tensor([270, 350, 321], dtype=torch.int32)
    indices = torch.randperm(int(npg.sum()), generator=gc).to(torch.int32)
    indptr = torch.zeros(B + 1, dtype=torch.int32)
    indptr[1:] = torch.cumsum(npg, 0)
    last = torch.tensor([63, 22, 55], dtype=torch.int32)
    lens = (npg - 1) * page + last
    l_max = 512 * page
    u = torch.rand((B, Hq, l_max), generator=g, device=dev)
    row_len = lens.view(B, 1).expand(B, Hq).contiguous().to(dev)
    ind, nnz = kept_index.select_kept(l_max, uniform=u, kept_ratio=0.02, row_len=row_len)
    q = torch.randn(B, Hq, 1, D, generator=g, device=dev, dtype=torch.float16)
    K = torch.rand(B, Hq, generator=gc) * 5 + 1
    L = torch.rand(B, Hq, generator=gc) * 5 + 1
    return q, pool, indptr, indices, ind, nnz, K, L


def test_sparse_paged_and_magicpig_on_the_reference_harness_fixture(dev):
    q, pool, indptr, indices, ind, nnz, K, L = _reference_harness_fixture(dev)
    o, lse = spp.sparsetoken_flash_attention_decode_paged(q, pool, indptr.to(dev),
                                                          indices.to(dev), ind, nnz,
                                                          return_lse=True)
    mo, ml = mp.magicpig_sparsetoken_flash_attention_decode_paged(
        q, pool, indptr.to(dev), indices.to(dev), ind, nnz, K.to(dev), L.to(dev),
        return_lse=True)
    qc, pc, ic, zc = q.cpu(), pool.cpu(), ind.cpu(), nnz.cpu()
    ro, rl = naive.sparsetoken_naive_paged_attention(qc, pc, indptr, indices, ic, zc)
    err = assert_close(o, ro, what="harness fixture, sparse paged")
    assert_close(lse, rl, atol=1e-4, what="harness fixture, sparse paged lse")
    r64, l64 = naive.magicpig_sparsetoken_naive_paged_attention(qc, pc, indptr, indices, ic, zc,
                                                                 K, L)
    merr = assert_close(mo, r64, what="harness fixture, MagicPIG vs fp64 oracle")
    assert_close(ml, l64, atol=1e-3, what="harness fixture, MagicPIG lse vs fp64 oracle")
    print(f"harness fixture: sparse paged err {err:.3e}, MagicPIG err {merr:.3e}, "
          f"kept per head {float(zc.float().mean()):.0f}")


# A wave resolves its kept tokens 64 at a time: lists that give the four waves of
# a row's workgroups 0, 1, 4, 5, 8 and 9 groups, with ragged last groups.
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("splits", [1, 3])
def test_sparse_groups_per_wave_edges(dev, D, splits):
    counts = [1, 15, 16, 17, 64, 65, 255, 256, 257, 321, 511, 512, 513, 577, 769, 1000]
    g = torch.Generator().manual_seed(D + splits)
    Hq, Hkv, page, lens = len(counts), 4, 16, [3000, 2001]
    indptr, indices, last, P = syn.block_table(g, lens, page)
    pool = torch.randn(P, 2, Hkv, page, D, generator=g).half()
    q = torch.randn(2, Hq, 1, D, generator=g).half()
    ind = torch.full((2, Hq, 1100), -1, dtype=torch.int32)
    for b in range(2):
        for h, n in enumerate(counts):
            ind[b, h, :n] = torch.randperm(lens[b], generator=g)[:n].sort().values.int()
    nnz = torch.tensor(counts, dtype=torch.int32).expand(2, Hq).unsqueeze(-1).contiguous()
    lk, ll = (torch.rand(2, Hq, generator=g) * 5 + 1 for _ in range(2))
    dargs = [t.to(dev) for t in (q, pool, indptr, indices, ind, nnz)]
    args = (q, pool, indptr, indices, ind, nnz)
    o, lse = _ops.sparse_decode_paged(*dargs, return_lse=True, num_splits=splits)
    ro, rl = naive.sparsetoken_naive_paged_attention(*args)
    assert_close(o, ro, what="paged")
    assert_close(lse, rl, atol=1e-4, what="paged lse")
    o, lse = _ops.sparse_decode_paged(*dargs, return_lse=True, num_splits=splits,
                                      lsh_k=lk.to(dev), lsh_l=ll.to(dev))
    ro, rl = naive.magicpig_sparsetoken_naive_paged_attention(*args, lk, ll)
    assert_close(o, ro, what="MagicPIG")
    assert_close(lse, rl, atol=1e-3, what="MagicPIG lse")
    K, V = (torch.randn(2, Hkv, 3000, D, generator=g).half() for _ in range(2))
    K2 = K.transpose(1, 2).contiguous().transpose(1, 2)  # K and V of different strides
    o, lse = _ops.sparse_decode(dargs[0], K2.to(dev), V.to(dev), dargs[4], dargs[5],
                                1 / math.sqrt(D), return_lse=True, num_splits=splits)
    ro, rl = naive.sparsetoken_naive_decode(q, K, V, ind, nnz, 1 / math.sqrt(D), Hq // Hkv)
    assert_close(o, ro, what="dense")
    assert_close(lse, rl, atol=1e-4, what="dense lse")


# Both ways of reading mask rows (whole words, single bytes) and the fp32 draws, at
# the edges of runs, chunks, waves and steps, against torch.nonzero.
@pytest.mark.parametrize("n", [1, 3, 4, 15, 16, 17, 255, 1024, 2047, 2049, 32767, 32768, 32772, 70001])
@pytest.mark.parametrize("offset", [0, 1, 4])
@pytest.mark.parametrize("density", [0.02, 0.6])
def test_kept_index_sources_and_edges(dev, n, offset, density):
    g = torch.Generator().manual_seed(n + offset)
    rows = 3
    flat = torch.rand(rows * n + offset, generator=g)
    u = flat[offset:].view(rows, n)
    lens = torch.tensor([n, max(0, n - 5), n // 2], dtype=torch.int32)
    l_max = max(1, n - 2 if density > 0.5 else n // 2)
    mask = (flat.to(dev) < density)[offset:].view(rows, n)  # starts `offset` bytes into its storage
    for src in (dict(mask=mask), dict(uniform=u.to(dev), kept_ratio=density)):
        for rl in (None, lens):
            ind, nnz = kept_index.select_kept(l_max, row_len=None if rl is None else rl.to(dev), **src)
            for r in range(rows):
                m = n if rl is None else int(rl[r])
                want = torch.nonzero(u[r, :m] < density).view(-1).int()
                want = want if want.numel() else torch.zeros(1, dtype=torch.int32)
                assert int(nnz[r]) == want.numel()
                k = min(want.numel(), l_max)
                got = ind[r].cpu()
                assert torch.equal(got[:k], want[:k]) and bool((got[k:] == -1).all())
