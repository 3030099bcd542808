"""Performance cases of the attention entry points, and the inputs, work and exact results of each.

A case is a dict of plain values.  Its "kind" names the call that a program makes:

  prefill       flash_attention_prefill, dense or (varlen) right-padded, with or without the LSE
  decode        flash_attention_decode over a dense cache
  paged         flash_attention_decode_paged over a paged cache
  append        one new token per sequence written by append_paged_kv, then the paged decode: a
                serving step of one layer
  sparse        select_kept on uniform draws, then sparsetoken_flash_attention_decode on its lists
  sparse_paged  sparsetoken_flash_attention_decode_paged, or with "magic" the MagicPIG form

Tensors are N(0, 1) in the layouts of the package's synthetic module: a pool
[P, 2, Hkv, page, D] behind a randomly permuted block table, sequence lengths spread over
[min_len, max_len].  Lengths follow from the case; everything else follows from the seed.
"""
from __future__ import annotations

import math
import random

import torch

from attention_kernel_triton_amd import (
    decode_flash_attention_redundant as dense_mod,
    decode_flash_attention_redundant_var_len_paged as paged_mod,
    kept_index,
    magicpig_sparsetoken_decode_flash_attention_redundant_var_len_paged_with_norm as magic_mod,
    paged_kv,
    prefill_flash_attention as prefill_mod,
    prefill_flash_attention_var_len_padding as varlen_mod,
    sparsetoken_decode_flash_attention_redundant as sparse_mod,
    sparsetoken_decode_flash_attention_redundant_var_len_paged as sparse_paged_mod,
)

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # A short prompt on its own, as an interactive request brings it: latency.
        {"name": "prefill_short_d128", "kind": "prefill", "B": 1, "Hq": 32, "Hkv": 8, "S": 333,
         "D": 128, "dtype": "fp16", "causal": True, "lse": False, "varlen": False},
        # The benchmark's batched causal prefill.
        {"name": "prefill_d64", "kind": "prefill", "B": 8, "Hq": 64, "Hkv": 16, "S": 1024,
         "D": 64, "dtype": "fp16", "causal": True, "lse": False, "varlen": False},
        # The same batch of unequal prompts, right-padded.
        {"name": "prefill_varlen_d64", "kind": "prefill", "B": 8, "Hq": 64, "Hkv": 16, "S": 1024,
         "D": 64, "dtype": "fp16", "causal": True, "lse": False, "varlen": True},
        # One long document in bf16, with the normaliser that a later merge needs.
        {"name": "prefill_long_d128_bf16", "kind": "prefill", "B": 1, "Hq": 32, "Hkv": 8,
         "S": 8192, "D": 128, "dtype": "bf16", "causal": True, "lse": True, "varlen": False},
        # A chunk against an earlier chunk of its context (no mask), wide heads, ragged size.
        {"name": "prefill_d256_full", "kind": "prefill", "B": 2, "Hq": 16, "Hkv": 4, "S": 1500,
         "D": 256, "dtype": "fp16", "causal": False, "lse": True, "varlen": False},
        # The benchmark's single-token decode over a dense cache.
        {"name": "decode_d64", "kind": "decode", "B": 8, "Hq": 64, "Hkv": 16, "S": 1024, "D": 64,
         "lse": False},
        # A large decode batch, eight query heads to a kv head, a length that fills no chunk.
        {"name": "decode_large_d128", "kind": "decode", "B": 32, "Hq": 64, "Hkv": 8, "S": 4100,
         "D": 128, "lse": False},
        # The benchmark's paged var-len decode batch.
        {"name": "paged_d128", "kind": "paged", "B": 32, "Hq": 32, "Hkv": 8, "D": 128, "page": 16,
         "min_len": 256, "max_len": 8192, "lse": False},
        # One long conversation decoding alone.
        {"name": "paged_single_long", "kind": "paged", "B": 1, "Hq": 32, "Hkv": 8, "D": 128,
         "page": 16, "min_len": 30001, "max_len": 30001, "lse": True},
        # A serving step of a small batch: write the new tokens, then decode.
        {"name": "append_decode_step", "kind": "append", "B": 16, "Hq": 32, "Hkv": 8, "D": 128,
         "page": 64, "min_len": 512, "max_len": 2048, "lse": False},
        # Kept-token selection and the sparse decode over a dense 32000-token cache.
        {"name": "sparse_select_d128", "kind": "sparse", "B": 1, "Hq": 32, "Hkv": 8, "S": 32000,
         "D": 128, "keep": 0.02, "lse": True},
        # The benchmark's MagicPIG decode over a paged var-len cache.
        {"name": "magicpig_paged_d256", "kind": "sparse_paged", "B": 3, "Hq": 32, "Hkv": 8,
         "D": 256, "page": 16, "min_len": 8192, "max_len": 32768, "keep": 0.02, "magic": True,
         "lse": True},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


# A drawn case moves or computes no more than the largest listed ones.
_MAX_FLOPS = 5.4e11
_MAX_BYTES = 5.3e8
_MAX_POOL = 2.4e8  # the append step returns its pool


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "prefill", "decode", "decode", "paged", "paged",
                       "append", "sparse", "sparse_paged"])
    while True:
        Hkv = rng.choice([1, 2, 4, 8, 16])
        case = {"kind": kind, "B": 1, "Hq": 0, "Hkv": Hkv}
        if kind == "prefill":
            G = rng.choice([1, 2, 4, 8])
            case.update(B=_log_int(rng, 1, 16), S=_log_int(rng, 17, 8192),
                        D=rng.choice([64, 64, 128, 128, 192, 256]),
                        dtype=rng.choice(["fp16", "fp16", "bf16"]), causal=rng.random() < 0.8,
                        lse=rng.random() < 0.3)
            case["varlen"] = case["B"] > 1 and case["causal"] and rng.random() < 0.4
        elif kind == "decode":
            G = rng.choice([1, 2, 4, 8, 16])
            case.update(B=_log_int(rng, 1, 64), S=_log_int(rng, 64, 32768),
                        D=rng.choice([64, 128, 128, 256]), lse=rng.random() < 0.3)
        elif kind in ("paged", "append"):
            G = rng.choice([1, 4, 4, 8])
            case.update(B=_log_int(rng, 1, 64), D=rng.choice([64, 128, 128, 256]),
                        page=rng.choice([16, 16, 32, 64, 128]))
            case["max_len"] = _log_int(rng, 64, 32768)
            case["min_len"] = max(1, round(case["max_len"] * rng.uniform(0.03, 1.0)))
            case["lse"] = rng.random() < 0.3
        elif kind == "sparse":
            G = rng.choice([1, 4, 4, 8])
            case.update(B=_log_int(rng, 1, 8), S=_log_int(rng, 2000, 32000),
                        D=rng.choice([64, 128, 128, 256]), keep=round(rng.uniform(0.01, 0.08), 4),
                        lse=True)
        else:
            G = rng.choice([1, 4, 4, 8])
            case.update(B=_log_int(rng, 1, 8), D=rng.choice([128, 256]), page=rng.choice([16, 16, 64]))
            case["max_len"] = _log_int(rng, 2000, 32768)
            case["min_len"] = max(1, round(case["max_len"] * rng.uniform(0.1, 1.0)))
            case.update(keep=round(rng.uniform(0.01, 0.08), 4), magic=rng.random() < 0.5, lse=True)
        case["Hq"] = Hkv * G
        if case["Hq"] > 64:
            continue
        w = work(case)
        if w["flops"] > _MAX_FLOPS or w["bytes"] > _MAX_BYTES:
            continue
        if kind == "append" and _pool_pages(case) * 2 * Hkv * case["page"] * case["D"] * 2 > _MAX_POOL:
            continue
        return case


# --------------------------------------------------------------------------- sizes
def _lens(case):
    """Sequence lengths of a case: spread over [min_len, max_len] (paged) or, right-padded
    prompts, the first of length S and the rest over [min(64, S), S]."""
    if case["kind"] == "prefill":
        lo, hi = min(64, case["S"]), case["S"]
    else:
        lo, hi = case["min_len"], case["max_len"]
    rng = random.Random(f"{case['B']} {lo} {hi}")
    lens = [rng.randint(lo, hi) for _ in range(case["B"])]
    if case["kind"] == "prefill":
        lens[0] = case["S"]
    return lens


def _pool_pages(case):
    return sum(-(-n // case["page"]) for n in _lens(case))


def work(case):
    """Bytes: every input element once and every output element once (K/V rows that the call
    has to read: valid tokens, kept tokens).  FLOPs: 4 D per (query head, visible key)."""
    kind, B, Hq, Hkv, D = case["kind"], case["B"], case["Hq"], case["Hkv"], case["D"]
    lse = 4 if case["lse"] else 0
    if kind == "prefill":
        S = case["S"]
        lens = _lens(case) if case["varlen"] else [S] * B
        rows = sum(lens)
        pairs = sum(n * (n + 1) // 2 if case["causal"] else n * n for n in lens)
        return {"bytes": rows * D * 2 * 2 * (Hq + Hkv) + rows * Hq * lse, "flops": 4 * D * Hq * pairs}
    qo = B * Hq * (D * 2 * 2 + lse)
    if kind == "decode":
        tokens = B * case["S"]
        return {"bytes": tokens * Hkv * D * 4 + qo, "flops": 4 * D * Hq * tokens}
    if kind in ("paged", "append"):
        tokens = sum(_lens(case))
        table = 4 * (_pool_pages(case) + 2 * B + 1)
        new = B * Hkv * D * 4 * 2 + 4 * (B + 1) if kind == "append" else 0
        return {"bytes": tokens * Hkv * D * 4 + qo + table + new, "flops": 4 * D * Hq * tokens}
    if kind == "sparse":
        S = case["S"]
        kept = round(B * Hq * S * case["keep"])
        l_max = int(S * (case["keep"] + 0.1))
        select = B * Hq * (S * 4 + l_max * 4 + 4)
        return {"bytes": select + kept * (D * 4 + 4) + qo, "flops": 4 * D * kept}
    kept = round(Hq * sum(_lens(case)) * case["keep"])
    return {"bytes": kept * (D * 4 + 4) + B * Hq * 4 + 4 * _pool_pages(case) + qo,
            "flops": 4 * D * kept}


# --------------------------------------------------------------------------- inputs
def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed) * 1000003 + 17)
    kind, B, Hq, Hkv, D = case["kind"], case["B"], case["Hq"], case["Hkv"], case["D"]

    def randn(*shape, dtype=torch.float16):
        return torch.randn(shape, generator=g, device=dev, dtype=torch.float32).to(dtype)

    x = {}
    if kind == "prefill":
        dt, S = DTYPES[case["dtype"]], case["S"]
        x["Q"], x["K"], x["V"] = (randn(B, h, S, D, dtype=dt) for h in (Hq, Hkv, Hkv))
        if case["varlen"]:
            x["lens"] = _lens(case)
            x["varlen"] = torch.tensor(x["lens"], dtype=torch.int64, device=dev)
        return x
    x["q"] = randn(B, Hq, 1, D)
    if kind in ("decode", "sparse"):
        x["K"], x["V"] = randn(B, Hkv, case["S"], D), randn(B, Hkv, case["S"], D)
        if kind == "sparse":
            x["uniform"] = torch.rand((B, Hq, case["S"]), generator=g, device=dev)
        return x
    page, lens = case["page"], _lens(case)
    counts = [-(-n // page) for n in lens]
    x["lens"] = lens
    x["indptr"] = torch.tensor([0] + counts, device=dev).cumsum(0).to(torch.int32)
    x["last"] = torch.tensor([(n - 1) % page + 1 for n in lens], dtype=torch.int32, device=dev)
    x["indices"] = torch.randperm(sum(counts), generator=g, device=dev).to(torch.int32)
    x["pool"] = randn(sum(counts), 2, Hkv, page, D)
    if kind == "append":
        x["k_new"], x["v_new"] = randn(B, Hkv, D), randn(B, Hkv, D)
        x["append_indptr"] = torch.arange(B + 1, dtype=torch.int32, device=dev)
    if kind == "sparse_paged":
        n = max(lens)
        uniform = torch.rand((B, Hq, n), generator=g, device=dev)
        valid = torch.arange(n, device=dev) < torch.tensor(lens, device=dev).view(B, 1, 1)
        keep = (uniform < case["keep"]) & valid
        keep[:, :, 0] |= ~keep.any(-1)
        l_max = max(counts) * page
        nnz = keep.sum(-1, dtype=torch.int32)
        pos = torch.arange(n, device=dev, dtype=torch.int32)
        rank = torch.where(keep, pos, n).sort(-1).values  # kept positions first, ascending
        ind = torch.full((B, Hq, l_max), -1, dtype=torch.int32, device=dev)
        ind[:, :, :n] = torch.where(rank < n, rank, -1)
        x["ind"], x["nnz"] = ind, nnz.unsqueeze(-1)
        if case["magic"]:
            x["lsh_k"] = torch.rand((B, Hq), generator=g, device=dev) * 5 + 1
            x["lsh_l"] = torch.rand((B, Hq), generator=g, device=dev) * 5 + 1
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    x["case"] = dict(case)
    x["scale"] = 1.0 / math.sqrt(case["D"])
    x["group"] = case["Hq"] // case["Hkv"]
    return x


def _paged_decode(x):
    return paged_mod.flash_attention_decode_paged(x["q"], x["pool"], x["indptr"], x["indices"],
                                                  x["last"], return_lse=x["case"]["lse"])


def run(x):
    case = x["case"]
    kind, lse = case["kind"], case["lse"]
    if kind == "prefill":
        if not case["varlen"]:
            return prefill_mod.flash_attention_prefill(x["Q"], x["K"], x["V"], case["causal"],
                                                       x["scale"], x["group"], return_lse=lse)
        out = varlen_mod.flash_attention_prefill(x["Q"], x["K"], x["V"], case["causal"],
                                                 x["scale"], x["group"], varlen=x["varlen"],
                                                 return_lse=lse)
        # Rows past a length are unspecified: the valid rows of each sequence, as views.
        parts = out if lse else (out,)
        return [t[b, :, :n] for t in parts for b, n in enumerate(x["lens"])]
    if kind == "decode":
        return dense_mod.flash_attention_decode(x["q"], x["K"], x["V"], x["scale"], x["group"],
                                                return_lse=lse)
    if kind == "paged":
        return _paged_decode(x)
    if kind == "append":
        paged_kv.append_paged_kv(x["k_new"], x["v_new"], x["append_indptr"], x["pool"],
                                 x["indptr"], x["indices"], x["last"])
        return {"out": _paged_decode(x), "pool": x["pool"]}
    if kind == "sparse":
        ind, nnz = kept_index.select_kept(int(case["S"] * (case["keep"] + 0.1)),
                                          uniform=x["uniform"], kept_ratio=case["keep"])
        out = sparse_mod.sparsetoken_flash_attention_decode(x["q"], x["K"], x["V"], ind, nnz,
                                                            x["scale"], x["group"],
                                                            return_lse=lse)
        return {"ind": ind, "nnz": nnz, "out": out}
    if case["magic"]:
        return magic_mod.magicpig_sparsetoken_flash_attention_decode_paged(
            x["q"], x["pool"], x["indptr"], x["indices"], x["ind"], x["nnz"], x["lsh_k"],
            x["lsh_l"], return_lse=lse)
    return sparse_paged_mod.sparsetoken_flash_attention_decode_paged(
        x["q"], x["pool"], x["indptr"], x["indices"], x["ind"], x["nnz"], return_lse=lse)


def tolerance(case):
    """P and the outputs are rounded to 16 bits (2^-11 in fp16, 2^-8 in bf16); the sums are
    32-bit.  Against exact() the outputs were 2.3e-4 to 2.9e-4 (fp16) and 2.1e-3 (bf16) off in
    the 2-norm: about four times that.  Index lists, counts and appended rows are the same."""
    if case.get("dtype") == "bf16":
        return {"rel": 1e-2, "differ": 0.0}
    return {"rel": 1e-3, "differ": 0.0}


# --------------------------------------------------------------------------- exact results
def _attend(q, k, v, scale, causal):
    """fp64 softmax(scale q k^T) v and its LSE for q [G, S, D], k and v [N, D]."""
    s = torch.matmul(q, k.t()) * scale
    if causal:
        n = torch.arange(k.shape[0], device=q.device)
        s.masked_fill_(n.view(1, 1, -1) > n[: q.shape[1]].view(1, -1, 1), -math.inf)
    lse = torch.logsumexp(s, -1)
    return torch.matmul(torch.exp_(s.sub_(lse.unsqueeze(-1))), v), lse


def _magic_scores(q, k, scale, K, L):
    """MagicPIG scores of one head in 64 bits: q.k scale - ln u (eq. 11)."""
    dot = torch.mv(k, q)
    cos = (dot / (q.norm() * k.norm(dim=-1) + 1e-8)).clamp(-1 + 1e-7, 1 - 1e-7)
    p = (1 - torch.acos(cos) / math.pi).clamp(0, 1) ** K
    u = 1 - (1 - p) ** L - L * p * (1 - p) ** (L - 1)
    return dot * scale - torch.log(u.clamp_min(1e-10))


def exact(case, seed):
    x = prepare(case, seed)
    kind, B, Hq, Hkv, D, G = (case["kind"], case["B"], case["Hq"], case["Hkv"], case["D"],
                              x["group"])
    scale, lse = x["scale"], case["lse"]
    f64 = torch.float64
    if kind == "prefill":
        S = case["S"]
        lens = x["lens"] if case["varlen"] else [S] * B
        O = torch.zeros((B, Hq, S, D), dtype=torch.float32, device="cuda")  # float: the arrays are large
        E = torch.zeros((B, Hq, S), dtype=f64, device="cuda")
        for b, n in enumerate(lens):
            for h in range(Hq):
                o, e = _attend(x["Q"][b, h : h + 1, :n].to(f64), x["K"][b, h // G, :n].to(f64),
                               x["V"][b, h // G, :n].to(f64), scale, case["causal"])
                O[b, h, :n], E[b, h, :n] = o[0].float(), e[0]
        if case["varlen"]:
            return [t[b, :, :n] for t in ((O, E) if lse else (O,)) for b, n in enumerate(lens)]
        return (O, E) if lse else O

    q = x["q"].to(f64)
    O = torch.zeros((B, Hq, D), dtype=f64, device="cuda")
    E = torch.zeros((B, Hq), dtype=f64, device="cuda")
    pool = None
    if kind in ("paged", "append", "sparse_paged"):
        pool = x["pool"].clone()
        page, ip = case["page"], x["indptr"].tolist()
        if kind == "append":
            for b, n in enumerate(x["lens"]):
                pg = int(x["indices"][ip[b] + (n - 1) // page])
                pool[pg, 0, :, (n - 1) % page] = x["k_new"][b]
                pool[pg, 1, :, (n - 1) % page] = x["v_new"][b]
    ind = nnz = None
    if kind == "sparse":
        l_max = int(case["S"] * (case["keep"] + 0.1))
        ind = torch.full((B, Hq, l_max), -1, dtype=torch.int32, device="cuda")
        nnz = torch.zeros((B, Hq, 1), dtype=torch.int32, device="cuda")
        keep = x["uniform"] < torch.tensor(case["keep"], dtype=torch.float32, device="cuda")
    for b in range(B):
        if pool is not None:
            rows = pool[x["indices"][ip[b] : ip[b + 1]].long()]  # [np, 2, Hkv, page, D]
            kv = rows.permute(1, 2, 0, 3, 4).reshape(2, Hkv, -1, D)[:, :, : x["lens"][b]]
        for kvh in range(Hkv):
            if pool is not None:
                k, v = kv[0, kvh].to(f64), kv[1, kvh].to(f64)
            else:
                k, v = x["K"][b, kvh].to(f64), x["V"][b, kvh].to(f64)
            if kind in ("decode", "paged", "append"):
                hs = slice(kvh * G, kvh * G + G)
                o, e = _attend(q[b, hs], k, v, scale, False)
                O[b, hs], E[b, hs] = o[:, 0], e[:, 0]
                continue
            for h in range(kvh * G, kvh * G + G):
                if kind == "sparse":
                    t = torch.nonzero(keep[b, h]).view(-1)
                    if t.numel() == 0:
                        t = torch.zeros(1, dtype=torch.int64, device="cuda")
                    ind[b, h, : t.numel()] = t[:l_max].to(torch.int32)
                    nnz[b, h, 0] = t.numel()
                else:
                    t = x["ind"][b, h, : int(x["nnz"][b, h, 0])].long()
                if kind == "sparse_paged" and case["magic"]:
                    s = _magic_scores(q[b, h, 0], k[t], scale, float(x["lsh_k"][b, h]),
                                      float(x["lsh_l"][b, h]))
                    e = torch.logsumexp(s, 0)
                    o = torch.mv(v[t].t(), torch.exp(s - e))
                else:
                    o, e = _attend(q[b, h : h + 1], k[t], v[t], scale, False)
                    o, e = o[0, 0], e[0, 0]
                O[b, h], E[b, h] = o, e
    if kind in ("decode", "sparse"):
        O = O.unsqueeze(2)
    out = (O, E) if lse else O
    if kind == "append":
        return {"out": out, "pool": pool}
    if kind == "sparse":
        return {"ind": ind, "nnz": nnz, "out": out}
    return out
