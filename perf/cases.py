"""The work that programs built on this library have it do, as measurable cases.

Each case is one call (or one short sequence of calls) through the public entry
points of ``opfoundry_amd.dsa``: sparse MLA decode over a paged latent cache
(bf16 and 656-byte fp8 rows, MTP, head shards), the cache write in front of it,
CSR-form decode, MXFP8 split streams, sparse prefill, DeepSeek-V4 prefill (bf16
and fp8 rows), the index scorer and the top-k selection.

``exact`` restates each path in 64-bit torch from its definition alone.
"""
from __future__ import annotations

import math

import torch

from opfoundry_amd import abi, dsa

D_QK, D_VO, D_ROPE = 576, 512, 64
FP8_ROW = 656
SM_SCALE = 1.0 / math.sqrt(192.0)
V4_SCALE = 1.0 / math.sqrt(512.0)
PAGE = 64                       # rows of a cache page, everywhere in this file
GOLDEN = 0.6180339887498949


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # One chat session, the smallest call there is: the new token's latent row goes into the
        # fp8 cache, then one query token attends a context shorter than top-k.  Latency.
        dict(name="decode_fp8_write_b1", kind="decode", rows="fp8", B=1, s_q=1, H=128, seq=1500,
             topk=2048, ragged=False, write=True, graph=False),
        # Two sessions at the usual top-k in a captured graph, as a serving loop replays a layer.
        dict(name="decode_bf16_b2_graph", kind="decode", rows="bf16", B=2, s_q=1, H=128, seq=8192,
             topk=2048, ragged=False, write=False, graph=True),
        # An ordinary serving batch on a bf16 cache.
        dict(name="decode_bf16_b64", kind="decode", rows="bf16", B=64, s_q=1, H=128, seq=32768,
             topk=2048, ragged=False, write=False, graph=False),
        # The headline: a full batch with one speculative token on the fp8 cache, long context.
        dict(name="decode_fp8_b128_mtp", kind="decode", rows="fp8", B=128, s_q=2, H=128, seq=65536,
             topk=2048, ragged=False, write=False, graph=False),
        # One rank of an 8-way head shard: 16 heads, an odd batch, ragged contexts.
        dict(name="decode_fp8_h16_ragged", kind="decode", rows="fp8", B=37, s_q=2, H=16, seq=20011,
             topk=2048, ragged=True, write=False, graph=False),
        # CSR lists of very different lengths; the call plans its own work split.
        dict(name="csr_bf16_varlen", kind="csr", rows="bf16", B=8, s_q=1, H=128, seq=65536,
             planned=False),
        # MXFP8 split streams at the full batch, one plan for all layers of a step.
        dict(name="mxfp8_b128_mtp", kind="mxfp8", B=128, s_q=2, H=128, seq=2048, planned=True),
        # A whole prompt's prefill, causal top-k lists over its own rows.
        dict(name="prefill_bf16_8192", kind="prefill", rows="bf16", N=8192, ctx=0, H=128, topk=2048),
        # DeepSeek-V4 prefill: scattered prefix pages plus a sliding window, with sinks.
        dict(name="v4_bf16_4096", kind="v4", rows="bf16", N=4096, H=128, topk=1024, pages=65536,
             window=128),
        # The same on fp8 rows for a ragged chunk on one rank of a 2-way head shard.
        dict(name="v4_fp8_1537_h64", kind="v4", rows="fp8", N=1537, H=64, topk=512, pages=16384,
             window=128),
        # Index scores of a decode step over ragged long contexts.
        dict(name="scores_b32_ragged", kind="scores", B=32, s_q=2, H_I=64, seq=100003, ragged=True),
        # The selection for a full decode batch (256 query tokens of 64 K positions).
        dict(name="topk_256x65536", kind="topk", T=256, n=65536, topk=2048, ragged=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "csr", "mxfp8", "prefill", "v4", "scores", "topk"])
    heads = rng.choice([16, 16, 32, 40, 64, 96, 128, 128, 128])
    rows = rng.choice(["bf16", "fp8"])
    if kind == "decode":
        B = _log(rng, 1, 128)
        seq = _log(rng, 512, min(131072, 4_000_000 // B))
        write = rows == "fp8" and B * seq <= 65536 and rng.random() < 0.5
        return dict(kind=kind, rows=rows, B=B, s_q=rng.randint(1, 3), H=heads, seq=seq,
                    topk=rng.choice([512, 1024, 2048, 2048, rng.randint(256, 2048)]),
                    ragged=rng.random() < 0.7, write=write,
                    graph=not write and B <= 8 and rng.random() < 0.5)
    if kind == "csr":
        B = _log(rng, 1, 128)
        return dict(kind=kind, rows=rows, B=B, s_q=rng.randint(1, 2), H=heads,
                    seq=_log(rng, 256, min(131072, 524288 // B)), planned=rng.random() < 0.5)
    if kind == "mxfp8":
        B = _log(rng, 1, 128)
        return dict(kind=kind, B=B, s_q=rng.randint(1, 2), H=heads,
                    seq=_log(rng, 256, min(65536, 300000 // B)), planned=rng.random() < 0.5)
    if kind == "prefill":
        N = _log(rng, 16, 8192 if rows == "bf16" else 6144)
        return dict(kind=kind, rows=rows, N=N, ctx=rng.choice([0, rng.randint(1, 8192)]), H=heads,
                    topk=rng.choice([512, 1024, 2048, rng.randint(256, 2048)]))
    if kind == "v4":
        return dict(kind=kind, rows=rows, N=_log(rng, 16, 4096), H=heads,
                    topk=rng.choice([512, 1024, rng.randint(128, 1536)]),
                    pages=_log(rng, 4096, 65536), window=128)
    if kind == "scores":
        if rng.random() < 0.3:          # a prefill chunk's scores: one sequence, many tokens
            return dict(kind=kind, B=1, s_q=_log(rng, 16, 512), H_I=rng.choice([32, 64]),
                        seq=_log(rng, 2048, 16384), ragged=False)
        B = _log(rng, 1, 128)
        return dict(kind=kind, B=B, s_q=rng.randint(1, 2), H_I=rng.choice([32, 64, 64]),
                    seq=_log(rng, 1024, min(131072, 4_000_000 // B)), ragged=rng.random() < 0.7)
    T = _log(rng, 1, 512)
    return dict(kind=kind, T=T, n=_log(rng, 1024, min(160000, 33_000_000 // T)),
                topk=rng.choice([512, 1024, 2048, 2048]), ragged=rng.random() < 0.7)


# ------------------------------------------------------------------ sizes that follow from a case

def _lens(count, lo, hi):
    """`count` lengths spread unevenly over [lo, hi]: the same ones for every seed."""
    return [lo + int((hi - lo + 1) * (((i + 1) * GOLDEN) % 1.0)) for i in range(count)]


def _decode_lens(c):
    return _lens(c["B"], max(c["s_q"], c["seq"] // 3), c["seq"]) if c["ragged"] else [c["seq"]] * c["B"]


def _csr_lens(c):
    """Row counts of each batch's list, from a handful up to the longest."""
    return _lens(c["B"], 5, c["seq"]) if c["kind"] == "csr" else [c["seq"]] * c["B"]


def _pairs(c):
    """(query token, row) pairs that a case attends, and the rows its pool holds of them."""
    k = c["kind"]
    if k == "decode":
        lens = _decode_lens(c)
        p = [min(c["topk"], n - t) for n in lens for t in range(c["s_q"])]
        return sum(p), min(sum(p), sum(lens))
    if k in ("csr", "mxfp8"):
        lens = _csr_lens(c)
        return sum(max(0, n - t) for n in lens for t in range(c["s_q"])), sum(lens)
    if k == "prefill":
        p = sum(min(c["topk"], c["ctx"] + t + 1) for t in range(c["N"]))
        return p, min(p, c["ctx"] + c["N"])
    p = c["N"] * min(c["topk"], c["pages"])
    w = sum(min(t + 1, c["window"]) for t in range(c["N"]))
    return p + w, min(p, c["pages"]) + c["N"]


def work(case):
    c = case
    if c["kind"] == "topk":
        lens = _lens(c["T"], max(1, c["n"] // 4), c["n"]) if c["ragged"] else [c["n"]] * c["T"]
        return {"bytes": 4 * sum(lens) + 4 * c["T"] * c["topk"] + 4 * c["T"], "flops": 0}
    if c["kind"] == "scores":
        lens = _decode_lens(c)
        cols = sum(max(0, n - (c["s_q"] - 1 - t)) for n in lens for t in range(c["s_q"]))
        T = c["B"] * c["s_q"]
        return {"bytes": sum(lens) * 256 + cols * 4 + T * c["H_I"] * (256 + 4),
                "flops": 2 * cols * c["H_I"] * 128}
    T = c["N"] if "N" in c else c["B"] * c["s_q"]
    H = c["H"]
    pairs, rows = _pairs(c)
    if c["kind"] == "v4":
        row, qrow, out, dims = (1024, 1024, 1024, 1024) if c["rows"] == "bf16" else (590, 590, 1024, 1024)
        lists = 4 * pairs
    elif c["kind"] == "mxfp8":
        row, qrow, out, dims = FP8_ROW, FP8_ROW, 1024, D_QK + D_VO
        lists = 4 * rows
    else:
        row, qrow, out, dims = (1152 if c["rows"] == "bf16" else FP8_ROW), 1152, 1024, D_QK + D_VO
        lists = 4 * (rows if c["kind"] == "csr" else pairs)
    moved = rows * row + lists + T * H * (qrow + out + 4)
    if c.get("write"):
        moved += T * (1152 + FP8_ROW)
    return {"bytes": moved, "flops": 2 * H * dims * pairs}


def tolerance(case):
    k = case["kind"]
    if k == "topk":
        return "exact"
    if k == "scores":
        return {"rel": 1e-5}            # bf16 products, 32-bit sums in any order
    # bf16 outputs with 16-bit probabilities round in two places: 0.0021 from exact(), times four
    return {"rel": 8e-3, "max": 5e-2}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _bf16(g, *shape):
    return _randn(g, *shape).to(torch.bfloat16)


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _positions(g, bounds, k):
    """Per entry of `bounds`: min(k, bound) distinct positions below it, ascending (the order the
    selection writes), then -1.  int32 [len(bounds), k]."""
    hi = torch.tensor(bounds, dtype=torch.int64, device="cuda")[:, None]
    n = torch.clamp(hi, max=k)
    j = torch.arange(k, device="cuda", dtype=torch.int64)[None, :]
    out = torch.empty((len(bounds), k), dtype=torch.int32, device="cuda")
    for r in range(0, len(bounds), 1024):
        h, m = hi[r:r + 1024], n[r:r + 1024].clamp(min=1)
        lo, up = j * h // m, (j + 1) * h // m
        u = torch.rand((h.shape[0], k), generator=g, device="cuda", dtype=torch.float64)
        pos = lo + ((up - lo) * u).long()
        out[r:r + 1024] = torch.where(j < n[r:r + 1024], pos, -1).to(torch.int32)
    return out


def _quantize_656(x):
    """bf16 rows [n, 576] as 656-byte rows: 512 e4m3 codes, 4 fp32 scales (amax / 448 per 128
    values), 64 bf16 values."""
    n = x.shape[0]
    v = x[:, :D_VO].float().view(n, 4, 128)
    scale = v.abs().amax(dim=2) / 448.0
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    codes = (v / scale[:, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    out = torch.empty((n, FP8_ROW), dtype=torch.uint8, device=x.device)
    out[:, :512] = codes.view(n, 512).view(torch.uint8)
    out[:, 512:528] = scale.contiguous().view(torch.uint8)
    out[:, 528:] = x[:, D_VO:].contiguous().view(torch.uint8)
    return out


def _pool(g, rows, n):
    """n latent rows: bf16 [n, 576], or uint8 [n, 656]."""
    if rows == "bf16":
        return _bf16(g, n, D_QK)
    out = torch.empty((n, FP8_ROW), dtype=torch.uint8, device="cuda")
    for r in range(0, n, 1 << 19):
        m = min(1 << 19, n - r)
        out[r:r + m] = _quantize_656(_bf16(g, m, D_QK))
    return out


def _mx_rows(g, n):
    """MXFP8 rows: 512 e4m3 codes, 16 E8M0 scale bytes (one per 32 values), 64 bf16 values."""
    e = torch.randint(0, 4, (n, 16), generator=g, device="cuda")
    x = _randn(g, n, 16, 32) * torch.exp2(-e.float())[:, :, None]
    nope = x.reshape(n, 512).to(torch.float8_e4m3fn).view(torch.uint8)
    return nope, (e + 127).to(torch.uint8), _bf16(g, n, D_ROPE)


def _v4_rows(g, rows, n):
    """V4 rows: bf16 [n, 512], or a 512-byte stream (448 e4m3 codes, 14 E8M0 bytes) and 64 bf16."""
    if rows == "bf16":
        return _bf16(g, n, 512)
    e = torch.randint(0, 4, (n, 14), generator=g, device="cuda")
    x = _randn(g, n, 14, 32) * torch.exp2(-e.float())[:, :, None]
    nope = torch.zeros((n, 512), dtype=torch.uint8, device="cuda")
    nope[:, :448] = x.reshape(n, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    nope[:, 448:462] = (e + 127).to(torch.uint8)
    return nope, _bf16(g, n, D_ROPE)


def _paged(g, c, lens):
    blocks = -(-max(lens) // PAGE)
    table = torch.randperm(c["B"] * blocks, generator=g, device="cuda").to(torch.int32)
    return table.view(c["B"], blocks)


def _prepare_decode(c, g):
    B, s_q, H, k = c["B"], c["s_q"], c["H"], c["topk"]
    lens = _decode_lens(c)
    table = _paged(g, c, lens)
    s = dict(c=c, table=table, lens=_int32(lens), kv=_pool(g, c["rows"], table.numel() * PAGE),
             q=_bf16(g, B, s_q, H, D_QK),
             idx=_positions(g, [n - (s_q - 1 - t) for n in lens for t in range(s_q)], k).view(B, s_q, k),
             out=torch.empty((B, s_q, H, D_VO), dtype=torch.bfloat16, device="cuda"),
             lse=torch.empty((B, s_q, H), dtype=torch.float32, device="cuda"))
    if c["write"]:      # the step's own tokens: their latent rows and the cache rows they go to
        s["new"] = _bf16(g, B * s_q, D_QK)
        b = torch.arange(B, device="cuda").repeat_interleave(s_q)
        pos = s["lens"].long()[b] - s_q + torch.arange(s_q, device="cuda").repeat(B)
        s["dst"] = table[b, pos // PAGE].long() * PAGE + pos % PAGE
    a = dsa.make_decode_args(s["q"], s["kv"], s["idx"], SM_SCALE, s["out"], s["lse"], seq_lens=s["lens"],
                             block_table=table, block_size=PAGE, causal=True)
    s["ws"] = torch.empty(max(16, dsa.decode_workspace_size(a)), dtype=torch.uint8, device="cuda")
    if c["graph"]:
        _decode(s)      # load the kernels before the capture
        torch.cuda.synchronize()
        s["captured"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["captured"]):
            _decode(s)
    return s


def _decode(s):
    if s["c"]["write"]:
        dsa.quantize_kv_fp8(s["new"], s["kv"], s["dst"])
    dsa.mla_decode(s["q"], s["kv"], s["idx"], SM_SCALE, s["out"], s["lse"], seq_lens=s["lens"],
                   block_table=s["table"], block_size=PAGE, causal=True, workspace=s["ws"])
    return (s["out"], s["lse"], s["kv"]) if s["c"]["write"] else (s["out"], s["lse"])


def _csr_lists(c, g):
    lens = _csr_lens(c)
    indptr = _int32([0] + list(torch.tensor(lens).cumsum(0).tolist()))
    return lens, indptr, torch.randperm(sum(lens), generator=g, device="cuda").to(torch.int32)


def _prepare_csr(c, g):
    lens, indptr, indices = _csr_lists(c, g)
    T = c["B"] * c["s_q"]
    s = dict(c=c, indptr=indptr, indices=indices, longest=max(lens), total=sum(lens),
             out=torch.empty((T, c["H"], D_VO), dtype=torch.bfloat16, device="cuda"),
             lse=torch.empty((T, c["H"]), dtype=torch.float32, device="cuda"))
    if c["kind"] == "csr":
        s["q"] = (_bf16(g, T, c["H"], D_QK),)
        s["kv"] = (_pool(g, c["rows"], sum(lens)),)
    else:
        q = _mx_rows(g, T * c["H"])
        s["q"] = tuple(x.view(T, c["H"], x.shape[-1]) for x in q)
        s["kv"] = _mx_rows(g, sum(lens))
    s["ws"] = dsa.csr_plan(indptr, c["B"], c["s_q"], c["H"], max(lens))
    return s


def _run_csr(s):
    c = s["c"]
    fn = dsa.mla_decode_csr if c["kind"] == "csr" else dsa.mla_decode_mxfp8
    return fn(*s["q"], *s["kv"], s["indptr"], s["indices"], SM_SCALE, s["out"], s["lse"], s_q=c["s_q"],
              max_kv_len=s["longest"], num_splits=abi.SPLITS_PLANNED if c["planned"] else 0,
              workspace=s["ws"])


def _prepare_prefill(c, g):
    return dict(c=c, q=_bf16(g, c["N"], c["H"], D_QK), kv=_pool(g, c["rows"], c["ctx"] + c["N"]),
                idx=_positions(g, [c["ctx"] + t + 1 for t in range(c["N"])], c["topk"]))


def _run_prefill(s):
    return dsa.mla_prefill(s["q"], s["kv"], s["idx"], SM_SCALE, causal=True, causal_offset=s["c"]["ctx"])


def _prepare_v4(c, g):
    N, H, window = c["N"], c["H"], c["window"]
    k = min(c["topk"], c["pages"])
    perm = torch.randperm(c["pages"], generator=g, device="cuda").to(torch.int32)
    pre = perm[_positions(g, [c["pages"]] * N, k).long()].view(-1)
    indptr_pre = torch.arange(N + 1, device="cuda", dtype=torch.int32) * k
    width = torch.clamp(torch.arange(N, device="cuda") + 1, max=window)
    indptr_ext = torch.zeros(N + 1, dtype=torch.int32, device="cuda")
    indptr_ext[1:] = torch.cumsum(width, 0).to(torch.int32)
    token = torch.repeat_interleave(torch.arange(N, device="cuda"), width)
    at = torch.arange(token.numel(), device="cuda") - indptr_ext[:-1].long()[token]
    ext = (token - (width[token] - 1) + at).to(torch.int32)
    q, pool, own = (_v4_rows(g, c["rows"], n) for n in (N * H, c["pages"], N))
    if c["rows"] == "bf16":
        q, pool, own = (q.view(N, H, 512),), (pool,), (own,)
    else:
        q = (q[0].view(N, H, 512), q[1].view(N, H, D_ROPE))
    return dict(c=c, q=q, pool=pool, own=own, sink=_randn(g, H), lists=(indptr_pre, pre, indptr_ext, ext),
                most=k + window)


def _run_v4(s):
    fn = dsa.mla_prefill_v4 if s["c"]["rows"] == "bf16" else dsa.mla_prefill_v4_fp8
    return fn(*s["q"], *s["pool"], *s["own"], s["sink"], *s["lists"], V4_SCALE, max_rows=s["most"])


def _prepare_scores(c, g):
    B, s_q = c["B"], c["s_q"]
    lens = _decode_lens(c)
    table = _paged(g, c, lens)
    width = -(-max(lens) // 64) * 64
    return dict(c=c, table=table, lens=_int32(lens), longest=max(lens),
                k=_bf16(g, table.numel(), PAGE, 128), q=_bf16(g, B, s_q, c["H_I"], 128),
                w=_randn(g, B, s_q, c["H_I"]) / math.sqrt(c["H_I"]),
                scores=torch.full((B, s_q, width), -math.inf, device="cuda"))


def _run_scores(s):
    return dsa.indexer_scores(s["q"], s["w"], s["k"], s["lens"], block_table=s["table"], block_size=PAGE,
                              causal=True, n_cols=s["longest"], scores=s["scores"])


def _prepare_topk(c, g):
    lens = _lens(c["T"], max(1, c["n"] // 4), c["n"]) if c["ragged"] else [c["n"]] * c["T"]
    return dict(c=c, lens=_int32(lens), scores=_randn(g, c["T"], -(-c["n"] // 4) * 4))


def _run_topk(s):
    return dsa.topk_indices(s["scores"], s["c"]["topk"], s["lens"])


PATHS = {
    "decode": (_prepare_decode, _decode), "csr": (_prepare_csr, _run_csr), "mxfp8": (_prepare_csr, _run_csr),
    "prefill": (_prepare_prefill, _run_prefill), "v4": (_prepare_v4, _run_v4),
    "scores": (_prepare_scores, _run_scores), "topk": (_prepare_topk, _run_topk),
}


def prepare(case, seed):
    return PATHS[case["kind"]][0](dict(case), _gen(seed))


def run(state):
    if "captured" in state:
        state["captured"].replay()
        return state["out"], state["lse"]
    return PATHS[state["c"]["kind"]][1](state)


# ------------------------------------------------------------------ the same in 64 bits

def _latent64(rows):
    """Cache rows [..., 576 bf16 | 656 bytes] as float64 [..., 576]."""
    if rows.dtype == torch.bfloat16:
        return rows.double()
    lead = rows.shape[:-1]
    codes = rows[..., :512].contiguous().view(torch.float8_e4m3fn).double()
    scale = rows[..., 512:528].contiguous().view(torch.float32).double()
    nope = codes.view(*lead, 4, 128) * scale[..., None]
    return torch.cat([nope.reshape(*lead, 512), rows[..., 528:].contiguous().view(torch.bfloat16).double()], -1)


def _mx64(nope, scale, rope):
    lead = nope.shape[:-1]
    codes = nope.view(torch.float8_e4m3fn).double().view(*lead, 16, 32)
    v = codes * torch.exp2(scale.double() - 127)[..., None]
    return torch.cat([v.reshape(*lead, 512), rope.double()], -1)


def _v464(parts):
    if len(parts) == 1:
        return parts[0].double()
    nope, rope = parts
    lead = nope.shape[:-1]
    codes = nope[..., :448].contiguous().view(torch.float8_e4m3fn).double().view(*lead, 14, 32)
    v = codes * torch.exp2(nope[..., 448:462].double() - 127)[..., None]
    return torch.cat([v.reshape(*lead, 448), rope.double()], -1)


def _attend64(q, k, valid, scale, sink=None):
    """q [c, H, D], k [c, n, D], valid [c, n] -> O [c, H, 512], LSE [c, H] (inf for no rows)."""
    s = torch.bmm(q, k.transpose(1, 2).contiguous()) * scale
    s.masked_fill_(~valid[:, None, :], -math.inf)
    lse = torch.logsumexp(s, dim=2)
    den = lse if sink is None else torch.logaddexp(lse, sink.double()[None, :].expand_as(lse))
    p = torch.exp(s - torch.where(torch.isinf(den), torch.zeros_like(den), den)[:, :, None])
    o = torch.bmm(p, k[:, :, :D_VO].contiguous())
    empty = ~valid.any(dim=1)
    return o, torch.where(empty[:, None], torch.full_like(den, math.inf), den)


def _attend_lists(T, width, queries, rows, scale, sink=None):
    """queries(a, b) -> [b-a, H, D]; rows(a, b) -> (k [b-a, width, D], valid [b-a, width])."""
    step = max(1, min(64, 400_000 // max(1, width)))
    got = []
    for a in range(0, T, step):
        b = min(T, a + step)
        k, valid = rows(a, b)
        got.append(_attend64(queries(a, b), k, valid, scale, sink))
    return torch.cat([x[0] for x in got]), torch.cat([x[1] for x in got])


def _exact_decode(s):
    c = s["c"]
    B, s_q, H, k = c["B"], c["s_q"], c["H"], c["topk"]
    kv = s["kv"]
    if c["write"]:
        kv = kv.clone()
        kv[s["dst"]] = _quantize_656(s["new"])
    idx = s["idx"].view(B * s_q, k).long()

    def rows(a, b):
        pos = idx[a:b].clamp(min=0)
        batch = torch.arange(a, b, device="cuda")[:, None] // s_q
        at = s["table"][batch, pos // PAGE].long() * PAGE + pos % PAGE
        return _latent64(kv[at]), idx[a:b] >= 0

    q = s["q"].view(B * s_q, H, D_QK)
    o, lse = _attend_lists(B * s_q, k, lambda a, b: q[a:b].double(), rows, SM_SCALE)
    o, lse = o.view(B, s_q, H, D_VO), lse.view(B, s_q, H)
    return (o, lse, None) if c["write"] else (o, lse)


def _exact_csr(s):
    c = s["c"]
    indptr, outs = s["indptr"].tolist(), []
    for b in range(c["B"]):
        at = s["indices"][indptr[b]:indptr[b + 1]].long()
        k = _latent64(s["kv"][0][at]) if c["kind"] == "csr" else _mx64(*(x[at] for x in s["kv"]))
        for t in range(c["s_q"]):
            row = b * c["s_q"] + t
            n = max(0, k.shape[0] - (c["s_q"] - 1 - t))
            q = s["q"][0][row].double() if c["kind"] == "csr" else _mx64(*(x[row] for x in s["q"]))
            valid = torch.ones((1, n), dtype=torch.bool, device="cuda")
            outs.append(_attend64(q[None], k[None, :n], valid, SM_SCALE))
    return torch.cat([o for o, _ in outs]), torch.cat([m for _, m in outs])


def _exact_prefill(s):
    idx = s["idx"].long()
    return _attend_lists(s["c"]["N"], s["c"]["topk"], lambda a, b: s["q"][a:b].double(),
                         lambda a, b: (_latent64(s["kv"][idx[a:b].clamp(min=0)]), idx[a:b] >= 0), SM_SCALE)


def _exact_v4(s):
    c = s["c"]
    N, window = c["N"], c["window"]
    k = min(c["topk"], c["pages"])
    pre = s["lists"][1].view(N, k).long()

    def rows(a, b):
        token = torch.arange(a, b, device="cuda")[:, None]
        own = token - torch.arange(window, device="cuda")[None, :]
        at = own.clamp(min=0)
        both = torch.cat([_v464([x[pre[a:b]] for x in s["pool"]]), _v464([x[at] for x in s["own"]])], 1)
        return both, torch.cat([torch.ones_like(pre[a:b], dtype=torch.bool), own >= 0], 1)

    return _attend_lists(N, k + window, lambda a, b: _v464([x[a:b] for x in s["q"]]), rows, V4_SCALE, s["sink"])


def _exact_scores(s):
    c = s["c"]
    flat = s["k"].view(-1, 128)
    out = torch.full(s["scores"].shape, -math.inf, dtype=torch.float64, device="cuda")
    at = torch.arange(s["longest"], device="cuda")
    for b, n in enumerate(s["lens"].tolist()):
        k = flat[s["table"][b, at[:n] // PAGE].long() * PAGE + at[:n] % PAGE].double()
        for t in range(c["s_q"]):
            m = n - (c["s_q"] - 1 - t)
            dots = torch.relu(k[:m] @ s["q"][b, t].double().t().contiguous())
            out[b, t, :m] = dots @ s["w"][b, t].double()
    return out


def exact(case, seed):
    if case["kind"] == "topk":
        return None
    s = prepare(dict(case, graph=False) if case["kind"] == "decode" else case, seed)
    return {"decode": _exact_decode, "csr": _exact_csr, "mxfp8": _exact_csr, "prefill": _exact_prefill,
            "v4": _exact_v4, "scores": _exact_scores}[case["kind"]](s)
