"""GPU parity of the 32- and 64-head kernels that run two workgroups per CU, against the CPU oracle
with the bar of every parity test: all row formats at the edges of its tiles (32 rows), its
row-list chunks (512, 768, 1024 and 2048 entries) and its head groups (16 and 40 heads), the
restart of the softmax reference from a late chunk, fp8 scales outside the fp16 path's range,
MTP lists, cut lists, work plans and a plan built for another call.
"""
import numpy as np
import pytest
import torch

import oracle
from _cases import SM_SCALE, assert_parity, bf16_rows, fp8_rows
from opfoundry_amd import abi, dsa
from test_csr_gpu import bits, t16
from test_mxfp8_gpu import dev_streams, mx_case, run_mx
from test_v4_gpu import v4_inputs
from test_v4fp8_gpu import run as run_v4fp8, to_dev as v4fp8_dev, v4fp8_inputs

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 2, 31, 32, 33, 63, 64, 65, 96, 511, 512, 513, 544, 767, 768, 769, 800, 1023, 1025, 1537, 2048]


def shared_case(seed, H, fp8, spike=False):
    """264 query tokens (more 32-head workgroups than CUs) over one flat cache, list lengths at
    the edges; spike: each token's last entry is a row far along its head 0's query."""
    rng = np.random.default_rng(seed)
    B, rows, k = 264, 4096, 2048
    q = oracle.normal_bf16(rng, (B, 1, H, 576))
    src = bf16_rows(rng, rows + B)
    if spike:
        src[rows:] = oracle.bf16_bits(3.0 * np.sign(oracle.bf16_to_f32(q[:, 0, 0])))
    kv = oracle.quantize_rows_656(oracle.bf16_to_f32(src)) if fp8 else src
    idx = np.full((B, 1, k), -1, np.int32)
    for b in range(B):
        n = EDGES[b % len(EDGES)]
        idx[b, 0, :n] = rng.permutation(rows)[:n]
        if n > 3:
            idx[b, 0, 2] = -1                       # a hole inside the list
        if spike and n:
            idx[b, 0, n - 1] = rows + b
    return q, kv, idx, np.full(B, rows + B, np.int32)


def decode(dev, q, kv, idx, sl):
    kvt = t16(kv, dev) if kv.dtype == np.uint16 else torch.from_numpy(kv).to(dev)
    out, lse = dsa.mla_decode(t16(q, dev), kvt, torch.from_numpy(idx).to(dev), SM_SCALE,
                              seq_lens=torch.from_numpy(sl).to(dev))
    torch.cuda.synchronize()
    return bits(out), lse.cpu().numpy()


@pytest.mark.parametrize("H,fp8,spike", [(16, False, False), (16, True, False), (40, False, True), (40, True, True),
                                         (64, False, False), (64, True, False)])
def test_decode_edges_and_restart(dev, H, fp8, spike):
    print(f"[case] pair decode H={H} fp8={fp8} spike={spike}", flush=True)
    c = shared_case(500 + H + 2 * fp8 + spike, H, fp8, spike)
    o, l = decode(dev, *c)
    o_ref, l_ref = oracle.mla_decode(c[0], c[1], c[2], c[3], SM_SCALE)
    n = (c[2] >= 0).sum(-1)                                                # [B, 1]
    assert np.isposinf(l[n == 0]).all() and (n == 0).any()
    if fp8:
        # lists of one or two rows: the LSE is off by at most a score's error.  The fp16 path
        # rounds a row's scale mantissa and then each value (2^-11 each), so a score is off by
        # at most 2^-10 sm_scale sum |q_i k_i| over the 512 dims (here 0.02; measured 0.0015,
        # with LSEs near 0).  The other lists, the empty ones too, have the common bar.
        few = (n == 1) | (n == 2)
        assert few.any()
        qa, ka = np.abs(oracle.bf16_to_f32(c[0]))[..., :512], np.abs(oracle.dequant_rows_656(c[1]))[:, :512]
        for b in np.flatnonzero(few[:, 0]):
            rows = c[2][b, 0][c[2][b, 0] >= 0]
            lim = 2.0 ** -10 * SM_SCALE * (qa[b, 0] @ ka[rows].T).max(-1) + 1e-5 * (1 + np.abs(l_ref[b, 0]))
            assert (np.abs(l[b, 0] - l_ref[b, 0]) <= lim).all()
        l = np.where(few[..., None], l_ref, l)
    assert_parity(o, l, o_ref, l_ref, f"pair decode H={H} fp8={fp8} spike={spike}")


@pytest.mark.parametrize("H,tokens,fp8", [(96, 7, False), (100, 5, True), (128, 5, False), (128, 6, True)])
def test_three_and_four_head_groups(dev, H, tokens, fp8):
    """Beyond 64 heads a split call of few tokens runs 32-head workgroups, two per CU where one
    round does not hold them (16 splits here: 320 workgroups and more)."""
    print(f"[case] pair decode of {tokens} tokens H={H} fp8={fp8}", flush=True)
    q, kv, idx, sl = (x[:tokens] if i != 1 else x for i, x in enumerate(shared_case(570 + H, H, fp8)))
    for b, n in enumerate([2048, 0, 1999, 33, 769, 16, 1537][:tokens]):
        idx[b, 0, :n] = np.random.default_rng(b).permutation(4096)[:n]
        idx[b, 0, n:] = -1
    kvt = torch.from_numpy(kv).to(dev) if fp8 else t16(kv, dev)
    out, lse = dsa.mla_decode(t16(q, dev), kvt, torch.from_numpy(idx).to(dev), SM_SCALE,
                              seq_lens=torch.from_numpy(sl).to(dev), num_splits=16)
    torch.cuda.synchronize()
    o_ref, l_ref = oracle.mla_decode(q, kv, idx, sl, SM_SCALE)
    assert_parity(bits(out), lse.cpu().numpy(), o_ref, l_ref, f"pair decode of {tokens} tokens H={H} fp8={fp8}")


def test_bad_scale_is_nan(dev):
    print("[case] pair fp8 bad scale", flush=True)
    q, kv, idx, sl = shared_case(520, 16, True)
    bad = int(idx[20, 0, 5])                        # a row of token 20 (1025 entries or more)
    for b in range(len(idx)):
        if b != 20:
            idx[b, 0][idx[b, 0] == bad] = -1
    kv[bad, 512:516] = np.frombuffer(np.float32(200.0).tobytes(), np.uint8)
    o, l = decode(dev, q, kv, idx, sl)
    f = oracle.bf16_to_f32(o)
    assert np.isnan(f[20]).all() and np.isnan(l[20]).all()
    keep = np.arange(len(idx)) != 20
    o_ref, l_ref = oracle.mla_decode(q[keep], kv, idx[keep], sl[keep], SM_SCALE)
    assert_parity(o[keep], l[keep], o_ref, l_ref, "pair fp8 bad scale: the other tokens")


@pytest.mark.parametrize("H,num_splits,reps", [(16, 0, 1), (40, 0, 1), (40, 3, 1), (40, 0, 22), (64, 2, 11)])
def test_mxfp8(dev, H, num_splits, reps):
    """(264 tokens, and 132 in two splits: 64-head workgroups.)"""
    lens, s_q = [2100, 0, 33, 700, 1, 513] * reps, 2
    print(f"[case] pair mxfp8 H={H} splits={num_splits} tokens={2 * len(lens)}", flush=True)
    q, kv, indptr, indices = mx_case(530 + H + num_splits, lens, s_q, 3000, bad=9)
    q = tuple(np.ascontiguousarray(x[:, :H]) for x in q)
    o, l = run_mx(*dev_streams(q, kv, dev), indptr, indices, s_q, dev, num_splits)
    o_ref, l_ref = oracle.mla_decode_mxfp8(*q, *kv, indptr, indices, s_q, SM_SCALE)
    assert_parity(o, l, o_ref, l_ref, f"pair mxfp8 H={H}")


@pytest.mark.parametrize("fp8,reps", [(False, 1), (True, 1), (False, 65), (True, 65)])
def test_csr_plan_and_cut_lists(dev, fp8, reps):
    """A work plan at 40 heads (two groups of 32 heads per item; 260 batches: one of 64), then
    the same workspace for a call of other lists: NaN for every row; and lists past max_kv_len:
    NaN for those rows alone."""
    rng = np.random.default_rng(540 + fp8 + reps)
    H, lens, rows = 40, [1500, 0, 64, 777] * reps, 3000
    kv = fp8_rows(rng, rows) if fp8 else bf16_rows(rng, rows)
    q = oracle.normal_bf16(rng, (len(lens), H, 576))
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    indices = rng.integers(0, rows, int(indptr[-1])).astype(np.int32)
    idx = np.full((len(lens), 1, max(lens)), -1, np.int32)
    for b, n in enumerate(lens):
        idx[b, 0, :n] = indices[indptr[b]:indptr[b + 1]]
    o_ref, l_ref = oracle.mla_decode(q[:, None], kv, idx, np.full(len(lens), rows, np.int32), SM_SCALE)
    o_ref, l_ref = o_ref[:, 0], l_ref[:, 0]
    kvt = torch.from_numpy(kv).to(dev) if fp8 else t16(kv, dev)
    ip, ix = torch.from_numpy(indptr).to(dev), torch.from_numpy(indices).to(dev)
    big = torch.empty(256 << 20, dtype=torch.uint8, device=dev)
    print(f"[case] pair csr plan fp8={fp8}", flush=True)
    run = lambda **kw: dsa.mla_decode_csr(t16(q, dev), kvt, ip, ix, SM_SCALE, **kw)  # noqa: E731
    out, lse = run(workspace=big)
    torch.cuda.synchronize()
    assert_parity(bits(out), lse.cpu().numpy(), o_ref, l_ref, "pair csr plan")
    dsa.csr_plan(ip, len(lens), 1, H, max(lens), workspace=big)
    out, lse = run(workspace=big, num_splits=abi.SPLITS_PLANNED, max_kv_len=max(lens) + 1)
    torch.cuda.synchronize()
    assert torch.isnan(out.float()).all() and torch.isnan(lse).all()
    out, lse = run(workspace=big, max_kv_len=1000)
    torch.cuda.synchronize()
    cut = np.array(lens) > 1000
    ct = torch.from_numpy(cut).to(dev)
    assert torch.isnan(out[ct].float()).all() and torch.isnan(lse[ct]).all()
    assert_parity(bits(out)[~cut], lse.cpu().numpy()[~cut], o_ref[~cut], l_ref[~cut], "pair csr cut list")


@pytest.mark.parametrize("H,topk,splits", [(16, 1100, 1), (40, 600, 1), (24, 2300, 3), (40, 2300, 2), (64, 1100, 1)])
def test_v4_bf16(dev, H, topk, splits):
    print(f"[case] pair V4 bf16 H={H} topk={topk}", flush=True)
    q, ukv, xkv, sink, *lists = v4_inputs(550 + H, N=280, total_pages=4096, topk=topk)
    q, sink = np.ascontiguousarray(q[:, :H]), sink[:H]
    scale = 1.0 / np.sqrt(512)
    o_ref, l_ref = oracle.mla_prefill_v4(q, ukv, xkv, sink, *lists, scale)
    ts = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    out, lse = dsa.mla_prefill_v4(t16(q, dev), t16(ukv, dev), t16(xkv, dev), ts(sink), *(ts(x) for x in lists), scale,
                                  num_splits=splits)
    torch.cuda.synchronize()
    assert_parity(bits(out), lse.cpu().numpy(), o_ref, l_ref, f"pair V4 bf16 H={H}")


@pytest.mark.parametrize("H,N,topk", [(16, 300, 1100), (32, 40, 300), (40, 260, 1100), (64, 140, 700), (33, 300, 20),
                                      (40, 256, 500)])      # the last: one round of 128-head workgroups
def test_v4_fp8(dev, H, N, topk):
    print(f"[case] pair V4 fp8 H={H} N={N}", flush=True)
    q, ukv, xkv, sink, lists = v4fp8_inputs(560 + H, N=N, total_pages=4096, topk=topk)
    q, sink = tuple(np.ascontiguousarray(x[:, :H]) for x in q), np.ascontiguousarray(sink[:H])
    scale = 1.0 / np.sqrt(512)
    o_ref, l_ref = oracle.mla_prefill_v4_fp8(*q, *ukv, *xkv, sink, *lists, scale)
    o, l = run_v4fp8(*v4fp8_dev(q, ukv, xkv, dev), sink, lists, scale, dev)
    assert_parity(o, l, o_ref, l_ref, f"pair V4 fp8 H={H}")
