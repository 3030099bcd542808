"""GPU parity of dense decode (R3) and paged var-len decode (R4)."""
import math

import pytest
import torch

from attention_kernel_triton_amd import decode_flash_attention_redundant as dec
from attention_kernel_triton_amd import decode_flash_attention_redundant_var_len_paged as pg
from attention_kernel_triton_amd import _ops
from attention_kernel_triton_amd import synthetic as syn
from helpers import assert_close, takes_stream_kernel
from oracle import naive

pytestmark = pytest.mark.gpu


def _dec_inputs(seed, B, Hkv, G, S, D):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, Hkv * G, 1, D, generator=g).half()
    K = torch.randn(B, Hkv, S, D, generator=g).half()
    V = torch.randn(B, Hkv, S, D, generator=g).half()
    return q, K, V


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("G", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("S", [1, 37, 1000])
def test_decode_shapes(dev, D, G, S):
    B, Hkv = 2, 2
    q, K, V = _dec_inputs(D + G + S, B, Hkv, G, S, D)
    o, lse = dec.flash_attention_decode(q.to(dev), K.to(dev), V.to(dev), 1 / math.sqrt(D), G,
                                        return_lse=True)
    ro, rl = naive.decode(q, K, V, 1 / math.sqrt(D), G)
    assert o.shape == (B, Hkv * G, 1, D)
    assert_close(o, ro, what=f"decode D={D} G={G} S={S}")
    assert_close(lse, rl, atol=1e-4, what="decode lse")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("chunk", [128, 256, 512, 640])
def test_decode_chunking_does_not_change_results(dev, chunk, D):
    """Every chunk length; at D = 64 the 512- and 640-token chunks run the
    persistent loop with four groups in flight per wave."""
    q, K, V = _dec_inputs(3, 2, 4, 4, 777, D)
    o, lse = _ops.decode(q.to(dev), K.to(dev), V.to(dev), 0.09, return_lse=True,
                         chunk_tokens=chunk)
    ro, rl = naive.decode(q, K, V, 0.09, 4)
    assert_close(o, ro, what=f"chunk {chunk} D={D}")
    assert_close(lse, rl, atol=1e-4, what=f"chunk {chunk} D={D} lse")


def test_decode_config2_full(dev):
    c = syn.decode_config()
    o = dec.flash_attention_decode(c.q.to(dev), c.K.to(dev), c.V.to(dev), c.scale, c.group)
    ro, _ = naive.decode(c.q, c.K, c.V, c.scale, c.group)
    print(f"config 2 max abs err {assert_close(o, ro, what='config 2'):.3e}")


def test_decode_empty_cache_gives_zeros(dev):
    q, K, V = _dec_inputs(4, 1, 2, 2, 0, 64)
    o, lse = dec.flash_attention_decode(q.to(dev), K.to(dev), V.to(dev), 0.1, 2, return_lse=True)
    assert torch.equal(o.cpu(), torch.zeros_like(o.cpu())) and torch.isinf(lse).all()


# --------------------------------------------------------------------------- paged
def _paged_call(p, dev, **kw):
    return pg.flash_attention_decode_paged(p.q.to(dev), p.pool.to(dev), p.indptr.to(dev),
                                           p.indices.to(dev), p.last_len.to(dev), **kw)


def test_paged_reference_fixture(dev):
    """Page table of decode_flash_attention_redundant_var_len_paged.py:349-353."""
    g = torch.Generator().manual_seed(6)
    pool = torch.randn(16, 2, 2, 64, 64, generator=g).half()
    indptr = torch.tensor([0, 4, 5, 8], dtype=torch.int32)
    indices = torch.tensor([0, 1, 3, 5, 2, 6, 7, 4], dtype=torch.int32)
    last = torch.tensor([2, 22, 3], dtype=torch.int32)
    q = torch.randn(3, 4, 1, 64, generator=g).half()
    o, lse = pg.flash_attention_decode_paged(q.to(dev), pool.to(dev), indptr.to(dev),
                                             indices.to(dev), last.to(dev), return_lse=True)
    ro, rl = naive.naive_paged_attention(q, pool, indptr, indices, last)
    assert o.shape == (3, 4, 64)
    assert_close(o, ro, what="paged fixture")
    assert_close(lse, rl, atol=1e-4, what="paged fixture lse")


# B = 5: the chunked kernel; B = 64 (128 units): the stream-K kernel where pages hold
# whole 16-token groups.
@pytest.mark.parametrize("page", [1, 8, 16, 48, 64])
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("B", [5, 64])
def test_paged_page_sizes(dev, page, D, B):
    p = syn.paged_config(seed=page * 3 + D, B=B, Hq=8, Hkv=2, D=D, page=page, min_len=1,
                         max_len=700, extra_pages=7)
    assert takes_stream_kernel(p.q, p.pool, p.indices) == (B == 64 and page % 16 == 0)
    o, lse = _paged_call(p, dev, return_lse=True)
    ro, rl = naive.naive_paged_attention(p.q, p.pool, p.indptr, p.indices, p.last_len)
    assert_close(o, ro, what=f"paged page={page} D={D}")
    assert_close(lse, rl, atol=1e-4, what="paged lse")


@pytest.mark.parametrize("copies", [1, 16])  # 8 and 128 units: chunked and stream-K kernel
def test_paged_empty_sequences_and_clamped_last_len(dev, copies):
    g = torch.Generator().manual_seed(9)
    pool = torch.randn(10, 2, 2, 16, 128, generator=g).half()
    q = torch.randn(4 * copies, 8, 1, 128, generator=g).half()
    ends = torch.tensor([0, 3, 3, 5])  # sequences 0 and 2 (of each 4) are empty
    indptr = torch.cat([torch.zeros(1), *(5 * c + ends for c in range(copies))]).to(torch.int32)
    indices = torch.tensor([9, 2, 4, 0, 7] * copies, dtype=torch.int32)
    last = torch.tensor([5, 40, 3, 0] * copies, dtype=torch.int32)  # 40 clamps to 16, 0 drops a page
    assert takes_stream_kernel(q, pool, indices) == (copies == 16)
    o, lse = pg.flash_attention_decode_paged(q.to(dev), pool.to(dev), indptr.to(dev),
                                             indices.to(dev), last.to(dev), return_lse=True)
    ro, rl = naive.naive_paged_attention(q, pool, indptr, indices, last)
    o, lse = o.cpu(), lse.cpu()
    assert not o[0::4].any() and not o[2::4].any()
    assert torch.isinf(lse[0::4]).all() and torch.isinf(lse[2::4]).all()
    assert_close(o, ro, what="paged edge cases")


@pytest.mark.parametrize("B", [12, 32])  # 48 and 128 units: chunked and stream-K kernel
def test_paged_single_token_sequences_are_exact(dev, B):
    """A one-token sequence returns its V row bit for bit (p = 1, l = 1)."""
    g = torch.Generator().manual_seed(10)
    pool = torch.randn(40, 2, 4, 16, 128, generator=g).half()
    indptr = torch.arange(B + 1, dtype=torch.int32)
    indices = torch.randperm(40, generator=g)[:B].to(torch.int32)
    last = torch.ones(B, dtype=torch.int32)
    q = torch.randn(B, 16, 1, 128, generator=g).half()
    assert takes_stream_kernel(q, pool, indices) == (B == 32)
    o = pg.flash_attention_decode_paged(q.to(dev), pool.to(dev), indptr.to(dev), indices.to(dev),
                                        last.to(dev)).cpu()
    for b in range(B):
        for h in range(16):
            assert torch.equal(o[b, h], pool[int(indices[b]), 1, h // 4, 0])


def test_paged_config3_full(dev):
    p = syn.paged_config()
    o, lse = _paged_call(p, dev, return_lse=True)
    ro, rl = naive.naive_paged_attention(p.q, p.pool, p.indptr, p.indices, p.last_len)
    err = assert_close(o, ro, what="config 3")
    assert_close(lse, rl, atol=1e-4, what="config 3 lse")
    print(f"config 3 max abs err {err:.3e}")


@pytest.mark.parametrize("chunk", [256, 512, 640])
def test_paged_chunk_lengths(dev, chunk):
    p = syn.paged_config(B=8, min_len=1, max_len=5000)
    d = p.to(dev)
    o, lse = _ops.decode_paged(d.q, d.pool, d.indptr, d.indices, d.last_len, return_lse=True,
                               chunk_tokens=chunk)
    ro, rl = naive.naive_paged_attention(p.q, p.pool, p.indptr, p.indices, p.last_len)
    assert_close(o, ro, what=f"paged chunk {chunk}")
    assert_close(lse, rl, atol=1e-4, what=f"paged chunk {chunk} lse")


@pytest.mark.parametrize("Hq,D", [(32, 128), (32, 64), (64, 128)])
@pytest.mark.parametrize("chunk", [0, 640])
def test_paged_lengths_at_every_boundary(dev, Hq, D, chunk):
    """Lengths on both sides of each 16-token group and 640-token chunk
    boundary, empty and one-token sequences, padded with 8192-token ones to a
    config-3-sized launch: the automatic path (chunk 0, the stream-K kernel,
    whose wave ranges then cut units at many positions) and the persistent
    chunked kernel at 640 tokens; a second call is bit-identical."""
    from attention_kernel_triton_amd import _ops
    g = torch.Generator().manual_seed(70 + D + Hq)
    Hkv = 8
    lens = [0, 1, 15, 16, 17, 255, 256, 257, 639, 640, 641, 913, 914, 915, 916, 1279, 1280,
            1281, 1828, 1829, 1919, 1920, 1921, 4096] + [8192] * 13
    B = len(lens)
    indptr, indices, last, P = syn.block_table(g, lens, 16)
    pool = torch.randn(P, 2, Hkv, 16, D, generator=g).half()
    q = torch.randn(B, Hq, 1, D, generator=g).half()
    args = (q.to(dev), pool.to(dev), indptr.to(dev), indices.to(dev), last.to(dev))
    o, lse = _ops.decode_paged(*args, chunk_tokens=chunk, return_lse=True)
    ro, rl = naive.naive_paged_attention(q, pool, indptr, indices, last)
    nonempty = torch.tensor(lens) > 0
    assert_close(o, ro, what=f"chunk {chunk} Hq={Hq} D={D}")
    assert_close(lse, rl, atol=1e-4, what=f"chunk {chunk} lse", mask=nonempty)
    assert torch.isinf(lse.cpu()[~nonempty]).all()
    again = _ops.decode_paged(*args, chunk_tokens=chunk)
    assert torch.equal(again, o)


def test_paged_config3_page_relabelling_is_bit_exact(dev):
    """Renaming physical pages (and moving their contents) must not change a single bit."""
    p = syn.paged_config(B=8, min_len=256, max_len=4096)
    P = p.pool.shape[0]
    perm = torch.randperm(P, generator=torch.Generator().manual_seed(1))
    pool2 = torch.empty_like(p.pool)
    pool2[perm] = p.pool                      # page i moves to slot perm[i]
    indices2 = perm[p.indices.long()].to(torch.int32)
    a = _paged_call(p, dev)
    b = pg.flash_attention_decode_paged(p.q.to(dev), pool2.to(dev), p.indptr.to(dev),
                                        indices2.to(dev), p.last_len.to(dev))
    assert torch.equal(a, b)


def test_paged_invalid_page_ids_are_skipped(dev):
    g = torch.Generator().manual_seed(12)
    pool = torch.randn(6, 2, 1, 16, 64, generator=g).half()
    q = torch.randn(1, 2, 1, 64, generator=g).half()
    indptr = torch.tensor([0, 3], dtype=torch.int32)
    good = torch.tensor([4, 1], dtype=torch.int32)
    o = pg.flash_attention_decode_paged(q.to(dev), pool.to(dev), indptr.to(dev),
                                        torch.tensor([4, 99, 1], dtype=torch.int32).to(dev),
                                        torch.tensor([16], dtype=torch.int32).to(dev))
    ro, _ = naive.naive_paged_attention(q, pool, torch.tensor([0, 2], dtype=torch.int32), good,
                                        torch.tensor([16], dtype=torch.int32))
    assert_close(o, ro, what="invalid page skipped")


# As above in launches of the stream-K kernel: pages of one and of several groups,
# ids below 0 and past the pool anywhere but on a sequence's last page, whole
# sequences of them among it.
@pytest.mark.parametrize("page,Hkv,D", [(16, 4, 128), (64, 4, 64), (48, 2, 256)])
def test_paged_invalid_page_ids_are_skipped_in_large_launches(dev, page, Hkv, D):
    g = torch.Generator().manual_seed(page + D)
    B, G = 64, 4
    lens = torch.randint(1, 900, (B,), generator=g).tolist()
    indptr, indices, last, P = syn.block_table(g, lens, page)
    pool = torch.randn(P, 2, Hkv, page, D, generator=g).half()
    q = torch.randn(B, Hkv * G, 1, D, generator=g).half()
    bad = torch.rand(len(indices), generator=g) < 0.25
    bad[indptr[1:].long() - 1] = False
    bad[indptr[5]:indptr[6]] = True  # a sequence without any valid page
    dirty = torch.where(bad, torch.tensor([-1, -(1 << 31), P, (1 << 31) - 1])[
        torch.randint(0, 4, (len(indices),), generator=g)], indices.long()).to(torch.int32)
    good = torch.zeros(B + 1, dtype=torch.int32)
    for b in range(B):
        good[b + 1] = good[b] + int((~bad[indptr[b]:indptr[b + 1]]).sum())
    assert takes_stream_kernel(q, pool, dirty)
    o, lse = pg.flash_attention_decode_paged(q.to(dev), pool.to(dev), indptr.to(dev),
                                             dirty.to(dev), last.to(dev), return_lse=True)
    ro, rl = naive.naive_paged_attention(q, pool, good, indices[~bad], last)
    there = good[1:] > good[:-1]
    assert_close(o, ro, what=f"page={page} D={D}")
    assert_close(lse, rl, atol=1e-4, what="lse", mask=there)
    assert not o.cpu()[~there].any() and torch.isinf(lse.cpu()[~there]).all()


def test_paged_repeated_calls_are_bit_identical(dev):
    """Which workgroup merges a unit depends on timing, never the result; the arrival
    counters are left at zero by every call."""
    p = syn.paged_config(B=16, min_len=256, max_len=6000).to(dev)
    outs = [pg.flash_attention_decode_paged(p.q, p.pool, p.indptr, p.indices, p.last_len)
            for _ in range(4)]
    for o in outs[1:]:
        assert torch.equal(o, outs[0])
    from attention_kernel_triton_amd import _native
    bufs = _native.workspace_buffers()
    assert bufs
    for _, _, buf in bufs:
        assert int(buf[:256].count_nonzero()) == 0


def test_paged_on_a_side_stream_matches_the_default_stream(dev):
    """Each stream gets its own workspace (its scheduling counters must not be shared
    by calls that can overlap), and the kernels launch on the caller's current stream."""
    from attention_kernel_triton_amd import _native
    p = syn.paged_config(B=8, min_len=256, max_len=3000).to(dev)
    ref = pg.flash_attention_decode_paged(p.q, p.pool, p.indptr, p.indices, p.last_len)
    side = torch.cuda.Stream(device=dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        o = pg.flash_attention_decode_paged(p.q, p.pool, p.indptr, p.indices, p.last_len)
        key = (torch.device(dev).index or 0, side.cuda_stream)
    torch.cuda.synchronize(dev)
    assert torch.equal(o, ref)
    assert key in [(d, s) for d, s, _ in _native.workspace_buffers()]
    # ctypes reads the null (default) stream back as None
    assert (_native.stream_of(p.q).value or 0) == torch.cuda.current_stream(dev).cuda_stream


def test_paged_on_two_streams_at_once(dev):
    """Two launches in flight together on two streams: each stream has its own
    workspace, so their scheduling counters never mix."""
    p = syn.paged_config(B=16, min_len=256, max_len=6000).to(dev)
    q2 = p.q.flip(1).contiguous()
    ref1 = pg.flash_attention_decode_paged(p.q, p.pool, p.indptr, p.indices, p.last_len)
    ref2 = pg.flash_attention_decode_paged(q2, p.pool, p.indptr, p.indices, p.last_len)
    s1, s2 = torch.cuda.Stream(device=dev), torch.cuda.Stream(device=dev)
    s1.wait_stream(torch.cuda.current_stream(dev))
    s2.wait_stream(torch.cuda.current_stream(dev))
    outs1, outs2 = [], []
    for _ in range(4):
        with torch.cuda.stream(s1):
            outs1.append(pg.flash_attention_decode_paged(p.q, p.pool, p.indptr, p.indices,
                                                         p.last_len))
        with torch.cuda.stream(s2):
            outs2.append(pg.flash_attention_decode_paged(q2, p.pool, p.indptr, p.indices,
                                                         p.last_len))
    torch.cuda.synchronize(dev)
    for o in outs1:
        assert torch.equal(o, ref1)
    for o in outs2:
        assert torch.equal(o, ref2)


# 16 and 128 units: the chunked and the stream-K kernel.
@pytest.mark.parametrize("lens", [[100, 37], [100, 37] * 8])
def test_paged_page_ids_past_32_bit_byte_offsets(dev, lens):
    """Pages near the end of a 4.6 GB pool: page id x page stride overflows 32 bits, so
    the row address must be formed in 64 bits.  Only the used pages are filled; the
    oracle runs on a compact copy of them."""
    Hq, Hkv, page, D = 8, 8, 16, 128
    P = 70000  # 70000 pages x 2 x 8 x 16 x 128 x 2 B = 4.6 GB
    npg = [(L + page - 1) // page for L in lens]
    used = torch.arange(P - 1, P - 1 - sum(npg), -1, dtype=torch.int32)  # highest ids first
    g = torch.Generator().manual_seed(21)
    content = torch.randn(len(used), 2, Hkv, page, D, generator=g).half()
    q = torch.randn(len(lens), Hq, 1, D, generator=g).half()
    pool = torch.empty(P, 2, Hkv, page, D, dtype=torch.float16, device=dev)
    pool[used.long().to(dev)] = content.to(dev)
    indptr = torch.tensor([0, *npg]).cumsum(0).to(torch.int32)
    last = torch.tensor([L - (n - 1) * page for L, n in zip(lens, npg)], dtype=torch.int32)
    assert takes_stream_kernel(q, pool, used) == (len(lens) > 2)
    o, lse = pg.flash_attention_decode_paged(q.to(dev), pool, indptr.to(dev), used.to(dev),
                                             last.to(dev), return_lse=True)
    compact = torch.arange(len(used), dtype=torch.int32)
    ro, rl = naive.naive_paged_attention(q, content, indptr, compact, last)
    assert_close(o, ro, what="paged, page ids near 70000")
    assert_close(lse, rl, atol=1e-4, what="paged lse, page ids near 70000")
    del pool


def test_decode_long_sequence(dev):
    """One 131072-token cache (four 640-token-or-less chunk rounds per unit and more)."""
    q, K, V = _dec_inputs(22, 1, 2, 4, 131072, 128)
    o, lse = dec.flash_attention_decode(q.to(dev), K.to(dev), V.to(dev), 1 / math.sqrt(128), 4,
                                        return_lse=True)
    ro, rl = naive.decode(q, K, V, 1 / math.sqrt(128), 4)
    assert_close(o, ro, what="decode S=131072")
    assert_close(lse, rl, atol=1e-4, what="decode S=131072 lse")


@pytest.mark.parametrize("page", [16, 8])
def test_paged_batch_past_the_lds_chunk_table(dev, page):
    """Batches over 1024 sequences take the non-persistent kernel: each workgroup
    locates its chunk by scanning the page table, chunks are 256 tokens, and the
    first workgroups write the rows of empty sequences.  Both the page-aligned
    (16) and the unaligned (8) group addressing are covered, with the LSE."""
    g = torch.Generator().manual_seed(40 + page)
    B, Hq, Hkv, D = 1100, 4, 2, 128
    lens = torch.randint(1, 700, (B,), generator=g).tolist()
    for b in (0, 3, 517, B - 1):
        lens[b] = 0
    indptr, indices, last, P = syn.block_table(g, lens, page, extra_pages=5)
    pool = torch.randn(P, 2, Hkv, page, D, generator=g).half()
    q = torch.randn(B, Hq, 1, D, generator=g).half()
    o, lse = pg.flash_attention_decode_paged(q.to(dev), pool.to(dev), indptr.to(dev),
                                             indices.to(dev), last.to(dev), return_lse=True)
    ro, rl = naive.naive_paged_attention(q, pool, indptr, indices, last)
    nonempty = torch.tensor(lens) > 0
    assert_close(o, ro, what=f"paged B={B} page={page}")
    assert_close(lse, rl, atol=1e-4, what="paged lse", mask=nonempty)
    assert torch.isinf(lse.cpu()[~nonempty]).all()


@pytest.mark.parametrize("B,Hkv", [(1, 2), (63, 2), (64, 2), (200, 2), (1024, 2), (2, 64),
                                   (63, 4)])
def test_paged_batches_up_to_the_lds_sequence_table(dev, B, Hkv):
    """Both paged kernels build every workgroup's sequence table in LDS, up to
    1024 sequences (the stream-K kernel from 128 units on): batches from one
    sequence to that limit, with empty sequences and clamped last-page lengths,
    match the oracle (O and LSE)."""
    g = torch.Generator().manual_seed(70 + B)
    Hq, D, page = 4 * Hkv, 128, 16
    lens = torch.randint(1, 300, (B,), generator=g).tolist()
    for b in {0, B // 2, B - 1} if B > 2 else set():
        lens[b] = 0
    indptr, indices, last, P = syn.block_table(g, lens, page, extra_pages=3)
    if B > 1:
        last[1] = 40  # clamps to the page size
    pool = torch.randn(P, 2, Hkv, page, D, generator=g).half()
    q = torch.randn(B, Hq, 1, D, generator=g).half()
    assert takes_stream_kernel(q, pool, indices) == (B * Hkv >= 128)
    o, lse = pg.flash_attention_decode_paged(q.to(dev), pool.to(dev), indptr.to(dev),
                                             indices.to(dev), last.to(dev), return_lse=True)
    ro, rl = naive.naive_paged_attention(q, pool, indptr, indices, last)
    nonempty = (indptr[1:] - indptr[:-1]) > 0
    assert_close(o, ro, what=f"paged B={B}")
    assert_close(lse, rl, atol=1e-4, what=f"paged lse B={B}", mask=nonempty)
    assert torch.isinf(lse.cpu()[~nonempty]).all()


@pytest.mark.parametrize("G,D", [(1, 128), (2, 64), (3, 128), (8, 256), (16, 128), (32, 64),
                                 (20, 128), (12, 256)])
@pytest.mark.parametrize("B", [6, 64])
def test_paged_automatic_path_every_head_group_width(dev, B, G, D):
    """Every heads-per-unit width of the automatic path (GT = 1, 2, 4, 8,
    16; G = 3 leaves a unit's last column empty, G = 32 at D = 64 takes two
    head groups of 16 per kv head, G = 20 and 12 leave their second one part
    empty) against the oracle, O and LSE, with two groups to a page: on the
    stream-K kernel with 64 sequences, and with 6 on the chunked one (except 16
    heads to a unit at D = 64, which stay with the stream-K kernel)."""
    g = torch.Generator().manual_seed(90 + G + D)
    Hkv, page = 2, 32
    lens = torch.randint(1, 900, (B,), generator=g).tolist()
    indptr, indices, last, P = syn.block_table(g, lens, page, extra_pages=2)
    pool = torch.randn(P, 2, Hkv, page, D, generator=g).half()
    q = torch.randn(len(lens), Hkv * G, 1, D, generator=g).half()
    assert takes_stream_kernel(q, pool, indices) == (B == 64 or (G, D) == (32, 64))
    o, lse = pg.flash_attention_decode_paged(q.to(dev), pool.to(dev), indptr.to(dev),
                                             indices.to(dev), last.to(dev), return_lse=True)
    ro, rl = naive.naive_paged_attention(q, pool, indptr, indices, last)
    assert_close(o, ro, what=f"paged G={G} D={D}")
    assert_close(lse, rl, atol=1e-4, what=f"paged lse G={G} D={D}")


# Small launches with many heads to a unit, on both sides of the lines that choose
# their kernel, against the oracle and the chunked kernel: ragged lengths with an
# empty sequence, pages of one and several groups, a pool with padded strides, head
# counts that leave part of a unit empty.
@pytest.mark.parametrize("B,Hkv,G,D,page,mean,stream", [
    (1, 1, 16, 64, 16, 1, True), (5, 2, 9, 64, 48, 700, True), (3, 2, 20, 64, 16, 400, True),
    (8, 8, 8, 64, 16, 240, True), (8, 8, 5, 64, 32, 60, False), (2, 4, 7, 64, 16, 900, False),
    (10, 4, 4, 64, 16, 700, True), (10, 4, 3, 64, 16, 400, False),
    (12, 8, 16, 128, 64, 60, True), (12, 8, 13, 128, 16, 330, False), (2, 2, 16, 128, 16, 90, False),
])
def test_paged_small_launches_with_many_heads(dev, B, Hkv, G, D, page, mean, stream):
    g = torch.Generator().manual_seed(B + G + D + mean)
    lens = [mean] * B if mean == 1 else torch.randint(mean // 2, 3 * mean // 2, (B,),
                                                      generator=g).tolist()
    if B > 3:
        lens[1] = 0
    indptr, indices, last, P = syn.block_table(g, lens, page, extra_pages=2)
    pool = torch.full((P, 2, Hkv, page + 3, D + 8), float("nan")).half()[:, :, :, :page, :D]
    pool.copy_(torch.randn(P, 2, Hkv, page, D, generator=g))
    q = torch.randn(B, Hkv * G, 1, D, generator=g).half()
    assert takes_stream_kernel(q, pool, indices) == stream
    big = torch.full((P, 2, Hkv, page + 3, D + 8), float("nan"), dtype=torch.float16, device=dev)
    big[:, :, :, :page, :D] = pool.to(dev)
    args = (q.to(dev), big[:, :, :, :page, :D], indptr.to(dev), indices.to(dev), last.to(dev))
    o, lse = _ops.decode_paged(*args, return_lse=True)
    oc, lc = _ops.decode_paged(*args, return_lse=True, chunk_tokens=128)
    ro, rl = naive.naive_paged_attention(q, pool, indptr, indices, last)
    there = torch.tensor(lens) > 0
    # Two orders of fp32 sums: the fp16 results differ by at most one ulp (|o| < 4: 2^-9).
    assert_close(o, oc, atol=2 ** -9, what="chunked kernel")
    assert_close(lse, lc, atol=1e-4, what="chunked lse", mask=there)
    assert_close(o, ro, what="oracle")
    assert_close(lse, rl, atol=1e-4, what="oracle lse", mask=there)
    assert torch.isinf(lse.cpu()[~there]).all()


def test_paged_merges_are_coherent_across_launches(dev):
    """The last workgroup of a unit merges partials other workgroups (on any XCD)
    stored in the same launch.  Alternating two inputs over one workspace, every
    launch must reproduce its input's first result bit for bit: a partial read
    before it was visible, or a stale one from the previous launch, would not."""
    a = syn.paged_config(B=32, min_len=256, max_len=8192).to(dev)
    b = syn.paged_config(seed=7, B=32, min_len=256, max_len=8192).to(dev)
    ra = pg.flash_attention_decode_paged(a.q, a.pool, a.indptr, a.indices, a.last_len)
    rb = pg.flash_attention_decode_paged(b.q, b.pool, b.indptr, b.indices, b.last_len)
    outs = []
    for _ in range(10):
        outs.append((pg.flash_attention_decode_paged(a.q, a.pool, a.indptr, a.indices,
                                                     a.last_len),
                     pg.flash_attention_decode_paged(b.q, b.pool, b.indptr, b.indices,
                                                     b.last_len)))
    for oa, ob in outs:
        assert torch.equal(oa, ra) and torch.equal(ob, rb)
    ref, _ = naive.naive_paged_attention(a.q.cpu(), a.pool.cpu(), a.indptr.cpu(),
                                         a.indices.cpu(), a.last_len.cpu())
    assert_close(ra, ref, what="config-3-sized merge")


def test_decode_more_units_than_the_fixed_arrival_area(dev):
    """35200 units (B = 1100, 32 kv heads, G = 1, two chunks each).  Arrival
    counters past the fixed 32768-slot area sit where the earlier, smaller calls
    stored their partials, so the call must clear them first.  Splitting the
    batch does not change what any unit computes, so the results are bit-identical."""
    g = torch.Generator().manual_seed(50)
    B, Hkv, S, D = 1100, 32, 150, 64
    q = torch.randn(B, Hkv, 1, D, generator=g).half().to(dev)
    K = torch.randn(B, Hkv, S, D, generator=g).half().to(dev)
    V = torch.randn(B, Hkv, S, D, generator=g).half().to(dev)
    parts = [_ops.decode(q[i:i + 100], K[i:i + 100], V[i:i + 100], 0.125, chunk_tokens=128)
             for i in range(0, B, 100)]
    full = _ops.decode(q, K, V, 0.125, chunk_tokens=128)
    assert torch.equal(full, torch.cat(parts))
    ro, _ = naive.decode(q[:100].cpu(), K[:100].cpu(), V[:100].cpu(), 0.125, 1)
    assert_close(parts[0], ro, what="first slice")


# Long units: a unit's run covers a few workgroups (merged by one wave in one
# round trip) up to more than a round trip holds (merged by a workgroup), with
# unit starts inside and at the edges of a workgroup's range, for every head
# count a unit can have and both workgroup sizes.
@pytest.mark.parametrize("lens", [[40001], [16 * 8 * 256], [9000, 1, 700, 16 * 8 * 200, 40],
                                  [128] * 300 + [5000]])
@pytest.mark.parametrize("G,D", [(1, 128), (3, 128), (8, 128), (16, 128), (4, 64), (4, 256)])
def test_paged_units_over_many_workgroups(dev, lens, G, D):
    from attention_kernel_triton_amd import _ops
    g = torch.Generator().manual_seed(sum(lens) + 10 * G + D)
    indptr, indices, last, P = syn.block_table(g, lens, 16)
    pool = torch.randn(P, 2, 1, 16, D, generator=g).half()
    q = torch.randn(len(lens), G, 1, D, generator=g).half()
    args = (q.to(dev), pool.to(dev), indptr.to(dev), indices.to(dev), last.to(dev))
    o, lse = _ops.decode_paged(*args, return_lse=True)
    ro, rl = naive.naive_paged_attention(q, pool, indptr, indices, last)
    assert_close(o, ro, what=f"G={G} D={D}")
    assert_close(lse, rl, atol=1e-4, what="lse")
    again = _ops.decode_paged(*args, return_lse=True)
    assert torch.equal(again[0], o) and torch.equal(again[1], lse)


# The automatic dense path on large enough launches (whole units per workgroup
# and ranges that cut units), against the oracle and the chunked kernel: every
# remainder class of a 16-token group, head counts with several units per kv
# head, layouts with other strides, and rows past S that must not be read into
# any result.
@pytest.mark.parametrize("B,Hkv,G,S,D", [
    (256, 1, 4, 17, 64), (16, 16, 1, 33, 128), (16, 16, 2, 1, 256),   # a workgroup per unit
    (64, 2, 4, 1029, 64), (64, 2, 3, 1040, 128), (52, 1, 8, 1297, 256),
    (3, 2, 20, 12001, 64), (7, 8, 8, 1999, 128), (1, 5, 16, 14001, 128), (300, 1, 1, 250, 256),
    (1, 5, 16, 28001, 128), (96, 1, 1, 1211, 128), (1, 1, 4, 68805, 256),  # more split items than CUs
    (200, 1, 1, 200, 128), (1, 1, 8, 16390, 64), (16, 1, 2, 2045, 64),      # lines of the rule
    (32, 1, 16, 2043, 128), (16, 1, 1, 3071, 256),
])
@pytest.mark.parametrize("layout", ["contiguous", "padded", "sequence-major"])
def test_dense_auto_path_layouts_and_edges(dev, B, Hkv, G, S, D, layout):
    from attention_kernel_triton_amd import _ops
    g = torch.Generator().manual_seed(S + G)
    K, V = (torch.randn(B, Hkv, S, D, generator=g).half() for _ in range(2))
    q = torch.randn(B, Hkv * G, 1, D, generator=g).half()
    kd, vd = K.to(dev), V.to(dev)
    if layout == "padded":  # NaN rows between one sequence's last row and the next one's first
        def pad(t):
            big = torch.full((B, Hkv, S + 15, D), float("nan"), dtype=t.dtype, device=dev)
            big[:, :, :S] = t
            return big[:, :, :S]
        kd, vd = pad(kd), pad(vd)
    elif layout == "sequence-major":
        kd = kd.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)
        vd = vd.permute(2, 1, 0, 3).contiguous().permute(2, 1, 0, 3)
    scale = 1 / math.sqrt(D)
    o, lse = _ops.decode(q.to(dev), kd, vd, scale, return_lse=True)
    oc, lc = _ops.decode(q.to(dev), kd, vd, scale, return_lse=True, chunk_tokens=256)
    # Two orders of fp32 sums: the fp16 results differ by at most one ulp (|o| < 2: 2^-10).
    assert_close(o, oc, atol=2 ** -9, what="chunked kernel")
    assert_close(lse, lc, atol=1e-5 * math.log(S + 2) + 1e-5, what="chunked lse")
    if layout == "contiguous":
        kr, vr = (t.repeat_interleave(G, 1).double() for t in (K, V))
        sc = torch.matmul(q.double(), kr.transpose(2, 3)) * scale
        assert_close(o, torch.matmul(torch.softmax(sc, -1), vr), what="oracle")
        assert_close(lse, torch.logsumexp(sc, -1)[..., 0], atol=1e-4, what="oracle lse")


def _assert_same_with_nonfinite(got, ref, what):
    """Infinities and NaN where the reference has them, the rest within ATOL."""
    g, r = got.detach().cpu().double(), ref.detach().cpu().double().reshape(got.shape)
    assert torch.equal(torch.isnan(g), torch.isnan(r)), f"{what}: NaN positions"
    inf = torch.isinf(r)
    assert torch.equal(torch.isinf(g), inf) and torch.equal(g[inf], r[inf]), f"{what}: infinities"
    assert_close(g, r, what=what, mask=torch.isfinite(r))


# An infinite V element of a used token makes its output element infinite, both
# signs together or a NaN make it NaN, and nothing else changes; on every kernel
# that a decode can take (stream-K for the longest, the chunked one for the shortest).
# Scores are within +-6, so every probability is far above fp16's smallest.
@pytest.mark.parametrize("D,G", [(64, 4), (128, 4), (128, 16), (256, 8)])
@pytest.mark.parametrize("S", [300, 16 * 2050 + 5, 16 * 4300 + 5])
@pytest.mark.parametrize("paged", [False, True])
def test_decode_infinite_v_elements(dev, paged, S, D, G):
    g = torch.Generator().manual_seed(S + D + G)
    Hkv, page = 2, 16
    q = torch.randn(1, Hkv * G, 1, D, generator=g).half()
    K = torch.randn(1, Hkv, S, D, generator=g).clamp(-2, 2).half()
    V = torch.randn(1, Hkv, S, D, generator=g).half()
    q *= 6 * math.sqrt(D) / torch.matmul(q.float(), K.float().repeat_interleave(G, 1)
                                         .transpose(2, 3)).abs().amax(-1, keepdim=True).half()
    inf = float("inf")
    top = torch.matmul(q[0, 0].float(), K[0, 0].float().t()).argmax()  # head 0's largest P
    V[0, 0, top, 0] = inf
    for i in range(12):  # every dim class, positions all over the cache
        V[0, i % 2, (37 * i + i * S // 13) % S, 1 + 5 * i] = inf if i % 3 else -inf
    V[0, 1, S - 1, 2], V[0, 1, S // 2, 2] = inf, -inf
    V[0, 1, S // 3, 4] = float("nan")
    ref, rl = naive.decode(q, K, V, 1 / math.sqrt(D), G)
    if paged:
        indptr, indices, last, P = syn.block_table(g, [S], page)
        pool = torch.full((P, 2, Hkv, page, D), inf).half()  # rows past S hold anything
        for i, pg_id in enumerate(indices.tolist()):
            n = min(page, S - i * page)
            pool[pg_id, 0, :, :n] = K[0, :, i * page:i * page + n]
            pool[pg_id, 1, :, :n] = V[0, :, i * page:i * page + n]
        o, lse = pg.flash_attention_decode_paged(q.to(dev), pool.to(dev), indptr.to(dev),
                                                 indices.to(dev), last.to(dev), return_lse=True)
    else:
        o, lse = dec.flash_attention_decode(q.to(dev), K.to(dev), V.to(dev), 1 / math.sqrt(D), G,
                                            return_lse=True)
    _assert_same_with_nonfinite(o, ref, f"paged={paged} S={S} D={D} G={G}")
    assert_close(lse, rl, atol=1e-4, what="lse")


# A query head with a NaN has NaN outputs, whatever kernel and however many waves
# its tokens take, and no other head changes: neither the first head of a unit,
# whose row stands in for rows that are not there, nor the last.
@pytest.mark.parametrize("head", [0, -1])
@pytest.mark.parametrize("D,G", [(64, 1), (128, 4), (128, 16), (256, 8)])
@pytest.mark.parametrize("paged,chunk,lens", [
    (True, 0, [1, 16, 17, 300, 0]), (True, 128, [1, 130, 700]),     # chunked kernel
    (True, 0, [3] * 1100),                                          # its batches past 1024
    (True, 0, [5, 16 * 1100, 16 * 1100 - 3]),                       # stream-K kernel
    (False, 0, [1]), (False, 0, [300]), (False, 0, [16 * 2100]),    # dense, either kernel
    (False, 0, [16 * 4300]),                                        # dense, stream-K kernel
])
def test_decode_nan_query_head(dev, paged, chunk, lens, D, G, head):
    g = torch.Generator().manual_seed(sum(lens) + D + G)
    Hkv, B = 2, len(lens)
    q = torch.randn(B, Hkv * G, 1, D, generator=g).half()
    bad = head % (Hkv * G)
    rest = [h for h in range(Hkv * G) if h != bad]
    dirty = q.clone()
    dirty[:, bad, 0, D // 3] = float("nan")
    if paged:
        indptr, indices, last, P = syn.block_table(g, lens, 16)
        pool = torch.randn(P, 2, Hkv, 16, D, generator=g).half()
        args = [t.to(dev) for t in (pool, indptr, indices, last)]
        run = lambda x: _ops.decode_paged(x.to(dev), *args, chunk_tokens=chunk)  # noqa: E731
    else:
        K, V = (torch.randn(B, Hkv, lens[0], D, generator=g).half().to(dev) for _ in range(2))
        run = lambda x: _ops.decode(x.to(dev), K, V, 0.1)[:, :, 0]  # noqa: E731
    want, got = run(q), run(dirty)
    nonempty = torch.tensor(lens, device=dev) > 0
    assert torch.isnan(got[nonempty, bad]).all()
    assert torch.equal(got[:, rest], want[:, rest])
    assert torch.equal(got[~nonempty], want[~nonempty])


# The tokens past a sequence's end have probability 0, and no infinite or NaN V row
# of a token that is there stands in for theirs: the last group's first row holds
# an infinity, which reaches its own output element and nothing else.
@pytest.mark.parametrize("D,G", [(64, 1), (128, 4), (128, 16), (256, 8)])
@pytest.mark.parametrize("page,chunk,last", [(16, 0, 1), (16, 0, 7), (16, 256, 15), (48, 0, 5),
                                             (8, 0, 3), (0, 0, 9)])
def test_decode_infinite_v_at_the_start_of_a_partial_group(dev, page, chunk, last, D, G):
    g = torch.Generator().manual_seed(10 * page + last + D + G)
    Hkv, S = 2, 16 * 20 + last
    q = torch.randn(1, Hkv * G, 1, D, generator=g).half()
    K, V = (torch.randn(1, Hkv, S, D, generator=g).half() for _ in range(2))
    K *= 0.25  # scores within a few units: every probability is well above fp16's smallest
    V[0, 0, S - last, 3], V[0, 1, S - last, D - 1] = float("inf"), -float("inf")
    scale = 1 / math.sqrt(D)
    ref, rl = naive.decode(q, K, V, scale, G)
    if page:
        indptr, indices, lastl, P = syn.block_table(g, [S], page)
        pool = torch.zeros(P, 2, Hkv, page, D).half()
        for i, pg_id in enumerate(indices.tolist()):
            n = min(page, S - i * page)
            pool[pg_id, 0, :, :n] = K[0, :, i * page:i * page + n]
            pool[pg_id, 1, :, :n] = V[0, :, i * page:i * page + n]
        o, lse = _ops.decode_paged(q.to(dev), pool.to(dev), indptr.to(dev), indices.to(dev),
                                   lastl.to(dev), return_lse=True, chunk_tokens=chunk)
    else:
        o, lse = _ops.decode(q.to(dev), K.to(dev), V.to(dev), scale, return_lse=True)
    _assert_same_with_nonfinite(o, ref, f"page={page} last={last} D={D} G={G}")
    assert_close(lse, rl, atol=1e-4, what="lse")
