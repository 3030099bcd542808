"""The decode workspace contract of the C ABI (include/akt_amd.h): only the
first min(AKT_WORKSPACE_ZERO_BYTES, size) bytes of a workspace must be zero
before its first use, and every call leaves them zero again.

Each case fills a workspace with 0xFF, zeroes exactly that prefix, calls the
paged decode entry point through the C ABI twice in a row on it, and compares
both results bit for bit with the drop-in wrapper (which runs the same kernels
on a workspace zeroed whole).
"""
import math

import pytest
import torch

from attention_kernel_triton_amd import _native as N
from attention_kernel_triton_amd import _ops
from attention_kernel_triton_amd import synthetic as syn
from helpers import takes_stream_kernel

pytestmark = pytest.mark.gpu


def _dirty_workspace(nbytes, dev):
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=dev)
    ws[: min(N.WORKSPACE_ZERO_BYTES, nbytes)] = 0
    return ws


def _paged_capi(p, ws, chunk=0):
    lib = N.load()
    B, Hq, D = p.q.shape[0], p.q.shape[1], p.q.shape[-1]
    P, _, Hkv, page, _ = p.pool.shape
    o = torch.empty((B, Hq, D), dtype=torch.float16, device=p.q.device)
    lse = torch.empty((B, Hq), dtype=torch.float32, device=p.q.device)
    rc = lib.akt_decode_paged_fwd(N.ptr(p.q), N.ptr(p.pool), N.ptr(p.indptr), N.ptr(p.indices),
                                  N.ptr(p.last_len), N.ptr(o), N.ptr(lse), B, Hq, Hkv, D, page,
                                  p.indices.numel(), P, N.strides(p.q), N.strides(p.pool),
                                  1.0 / math.sqrt(D), chunk, N.ptr(ws), ws.numel(),
                                  N.stream_of(p.q))
    N.check(rc, "akt_decode_paged_fwd")
    return o, lse


def _need(p, chunk=0):
    B, Hq, D = p.q.shape[0], p.q.shape[1], p.q.shape[-1]
    _, _, Hkv, page, _ = p.pool.shape
    return N.load().akt_decode_paged_workspace_size(B, Hq, Hkv, D, page, p.indices.numel(), chunk)


@pytest.mark.parametrize("case", ["config3", "over_32768_units"])
def test_paged_decode_needs_only_the_documented_zero_prefix(dev, case):
    if case == "config3":
        p = syn.paged_config().to(dev)  # 256 units, stream-K kernel
    else:
        # 1100 sequences x 32 kv heads = 35200 units: past the fixed counter
        # area, so the call zero-fills its extra counters itself (and, past
        # 1024 sequences, runs the non-persistent split kernel).
        g = torch.Generator().manual_seed(13)
        B, Hkv, D, page = 1100, 32, 64, 16
        lens = torch.randint(257, 321, (B,), generator=g).tolist()
        indptr, indices, last, P = syn.block_table(g, lens, page)
        gd = torch.Generator(device=dev).manual_seed(14)
        pool = torch.randn(P, 2, Hkv, page, D, generator=gd, device=dev, dtype=torch.float16)
        q = torch.randn(B, Hkv, 1, D, generator=gd, device=dev, dtype=torch.float16)
        p = syn.Paged(q, pool, indptr.to(dev), indices.to(dev), last.to(dev), lens)
    need = _need(p)
    assert need > N.WORKSPACE_ZERO_BYTES
    ro, rl = _ops.decode_paged(p.q, p.pool, p.indptr, p.indices, p.last_len, return_lse=True)
    ws = _dirty_workspace(need, dev)
    for _ in range(2):
        o, lse = _paged_capi(p, ws)
        torch.cuda.synchronize(dev)
        assert torch.equal(o, ro) and torch.equal(lse, rl)
        # The counters are zero again after the call.
        assert int(ws[: N.WORKSPACE_ZERO_BYTES].count_nonzero()) == 0


# Small launches of the automatic path, on the chunked kernel, and launches of the
# stream-K kernel: more waves than groups (some waves empty) and fewer, units cut
# at many positions, pages of several groups, one to 16 heads to a unit and two
# units to a kv head, 512-thread and 256-thread (D = 256) instances.
@pytest.mark.parametrize("lens,page,Hq,Hkv,D,stream", [
    ([40, 300, 1], 16, 8, 2, 128, False),
    ([360, 27, 4, 450, 140], 48, 8, 2, 128, False),
    ([1, 16, 17, 33], 16, 8, 1, 128, False),
    ([700, 5, 1300], 16, 16, 4, 64, False),
    ([513, 2, 90], 64, 4, 2, 256, False),
    ([8192, 4000, 31, 6000], 16, 32, 8, 128, True),    # 9112 groups on 2048 waves
    ([40, 300, 1] * 22 + [9], 16, 8, 2, 128, True),    # 1014 groups, 1016 waves: two empty ones
    ([360, 27, 4, 450, 140] * 13, 48, 8, 2, 128, True),
    ([17] * 129, 16, 8, 1, 128, True),                 # 258 groups of G = 8, 264 waves
    ([700, 5, 1300], 16, 64, 4, 64, True),             # 16 heads to a unit
    ([3, 50], 32, 64, 2, 64, True),                    # two units to a kv head: 24 groups
    ([513, 2, 90] * 22, 64, 4, 2, 256, True),          # G = 2, 256 threads
    ([5] * 135, 16, 1, 1, 256, True),                  # 135 groups, 136 waves of 256-thread ones
])
def test_paged_auto_path_on_dirty_workspace_matches_oracle(dev, lens, page, Hq, Hkv, D, stream):
    """The results match the oracle on a workspace whose partial area holds
    garbage, and the arrival counters are zero again after each of two calls."""
    from oracle import naive

    g = torch.Generator().manual_seed(sum(lens) + page + D)
    indptr, indices, last, P = syn.block_table(g, lens, page, 3)
    pool = torch.randn(P, 2, Hkv, page, D, generator=g).half()
    q = torch.randn(len(lens), Hq, 1, D, generator=g).half()
    ro, rl = naive.naive_paged_attention(q, pool, indptr, indices, last)
    assert takes_stream_kernel(q, pool, indices) == stream
    p = syn.Paged(q.to(dev), pool.to(dev), indptr.to(dev), indices.to(dev), last.to(dev), lens)
    ws = _dirty_workspace(_need(p), dev)
    for _ in range(2):
        o, lse = _paged_capi(p, ws)
        torch.cuda.synchronize(dev)
        err = float((o.cpu().double() - ro).abs().max())
        lerr = float((lse.cpu().double() - rl).abs().max())
        assert err <= 2e-3 and lerr <= 1e-4, (err, lerr)
        assert int(ws[: N.WORKSPACE_ZERO_BYTES].count_nonzero()) == 0


# Page tables that break the contract (indptr outside [0, total_pages] or
# decreasing): every kernel takes the entries clamped to the table and made
# non-decreasing, reads no position outside it and stores no partial past the
# workspace that the table's size asks for.
_LOW, _HIGH = -(1 << 31), (1 << 31) - 1
_TABLES = {
    "consistent": [0, 3, 3, 9, 12, 17, 20],
    "negative": [-5, 3, 3, 9, 12, 17, 20],
    "past the end": [0, 3, 3, 9, 12, 17, 999],
    "decreasing": [0, 9, 4, 2, 12, 17, 20],
    "overlapping": [0, 20, 0, 20, 0, 20, 20],
    "extremes": [_LOW, _HIGH, _LOW, 5, _HIGH, _LOW, 20],
    "late start": [7, 7, 9, 8, 12, 40, 13],
}


def _check_table(dev, indptr, page, Hkv, chunk, T, seed):
    from oracle import naive

    g = torch.Generator().manual_seed(seed)
    B, G, D = len(indptr) - 1, 4, 64
    pool = torch.randn(T + 3, 2, Hkv, page, D, generator=g).half()
    indices = torch.randperm(T + 3, generator=g)[:T].to(torch.int32)
    last = torch.randint(-1, page + 2, (B,), generator=g).to(torch.int32)
    q = torch.randn(B, Hkv * G, 1, D, generator=g).half()
    raw = torch.tensor(indptr, dtype=torch.int64)
    start = raw.clamp(0, T).cummax(0).values.to(torch.int32)
    ro, rl = naive.naive_paged_attention(q, pool, start, indices, last)
    p = syn.Paged(q.to(dev), pool.to(dev), raw.to(torch.int32).to(dev), indices.to(dev),
                  last.to(dev), None)
    need = _need(p, chunk)
    buf = torch.full((need + (1 << 20),), 0xA5, dtype=torch.uint8, device=dev)
    buf[: min(N.WORKSPACE_ZERO_BYTES, need)] = 0
    # Past 1024 sequences the rows of one that only the running maximum leaves
    # without pages are not written.
    keep = torch.ones(B, dtype=torch.bool)
    if B > 1024:
        keep = (raw[1:] <= raw[:-1]) | (start[1:] > start[:-1])
    for _ in range(2):
        o, lse = _paged_capi(p, buf[:need], chunk)
        torch.cuda.synchronize(dev)
        o, lse = o.cpu().double()[keep], lse.cpu().double()[keep]
        assert float((o - ro[keep]).abs().max()) <= 2e-3
        empty = torch.isinf(rl[keep])
        assert torch.equal(torch.isinf(lse), empty)
        assert float((lse - rl[keep])[~empty].abs().max()) <= 1e-4
        assert int(buf[: min(N.WORKSPACE_ZERO_BYTES, need)].count_nonzero()) == 0
        assert bool((buf[need:] == 0xA5).all())


@pytest.mark.parametrize("page,Hkv,chunk", [
    (16, 2, 0), (32, 2, 0), (16, 2, 128), (16, 2, 640), (8, 2, 0),  # chunked kernel
    (16, 32, 0), (64, 32, 0),                                       # stream-K kernel
])
@pytest.mark.parametrize("table", list(_TABLES))
def test_paged_tables_outside_the_contract_stay_inside_their_arrays(dev, table, page, Hkv, chunk):
    _check_table(dev, _TABLES[table], page, Hkv, chunk, 20, len(table) + page)


@pytest.mark.parametrize("page", [16, 8])
def test_paged_tables_outside_the_contract_past_1024_sequences(dev, page):
    g = torch.Generator().manual_seed(page)
    B = 1100
    indptr = [0] + torch.randint(0, 30, (B,), generator=g).cumsum(0).tolist()
    T = indptr[-1]
    indptr[3], indptr[500], indptr[700] = -9, indptr[400], _HIGH
    _check_table(dev, indptr, page, 2, 0, T, page)
