"""GPU parity of the index scorer's row-block variants (one, two or four 32-row blocks of
(token, index head) rows per workgroup) at the edges of a wave's 32 positions, a chunk's 128
and a workgroup's 1024, against oracle.indexer_scores, with the bound of
test_indexer_gpu.check (bf16 products are exact in fp32; only the order of the sums differs).
"""
import numpy as np
import pytest
import torch

import oracle
from opfoundry_amd import dsa
from test_indexer_gpu import check, paged, t16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H_I,s_q", [(32, 1), (32, 2), (32, 3), (64, 1), (64, 3), (128, 2)])
def test_row_blocks(dev, H_I, s_q):
    rng = np.random.default_rng(430 + H_I + s_q)
    seq = np.array([3, 31, 32, 33, 127, 129, 160, 1023, 1024, 1025, 2080], np.int32)
    q, w, k, bt = paged(rng, len(seq), seq, 16, H_I, s_q, bad_blocks=5)
    n_cols = int(seq.max())
    print(f"[case] indexer blocks H_I={H_I} s_q={s_q}", flush=True)
    ref = oracle.indexer_scores(q, w, k, seq, block_table=bt, block_size=16, causal=True, n_cols=n_cols)
    got = dsa.indexer_scores(t16(q, dev), torch.from_numpy(w).to(dev), t16(k, dev), torch.from_numpy(seq).to(dev),
                             block_table=torch.from_numpy(bt).to(dev), block_size=16, causal=True, n_cols=n_cols)
    torch.cuda.synchronize()
    check(got, q, w, k, ref, f"indexer blocks H_I={H_I} s_q={s_q}")


@pytest.mark.parametrize("H_I,s_q,n", [(64, 1, 70001), (64, 9, 300), (32, 17, 4500), (64, 130, 1100), (128, 600, 260)])
def test_one_sequence(dev, H_I, s_q, n):
    """One sequence: whole workgroups per token group (one group; as many as chunks; parts that
    do not divide a list's chunks), and 600 groups, which are dealt out evenly."""
    rng = np.random.default_rng(440 + s_q)
    seq = np.array([n], np.int32)
    q, w, k, bt = paged(rng, 1, seq, 64, H_I, s_q)
    print(f"[case] indexer one sequence H_I={H_I} s_q={s_q} n={n}", flush=True)
    ref = oracle.indexer_scores(q, w, k, seq, block_table=bt, block_size=64, causal=True, n_cols=n)
    got = dsa.indexer_scores(t16(q, dev), torch.from_numpy(w).to(dev), t16(k, dev), torch.from_numpy(seq).to(dev),
                             block_table=torch.from_numpy(bt).to(dev), block_size=64, causal=True, n_cols=n)
    torch.cuda.synchronize()
    check(got, q, w, k, ref, f"indexer one sequence s_q={s_q}")


def test_nan_row_scores_zero(dev):
    """max(NaN, 0) is 0: a cache row of NaNs scores 0, its neighbours are untouched."""
    rng = np.random.default_rng(450)
    seq = np.array([200], np.int32)
    q, w, k, bt = paged(rng, 1, seq, 64, 64, 2)
    row = int(bt[0, 1]) * 64 + 7                        # position 71
    k[row] = 0x7FC0
    ref = oracle.indexer_scores(q, w, np.where(np.arange(len(k))[:, None] == row, np.uint16(0), k), seq,
                                block_table=bt, block_size=64, causal=True, n_cols=200)
    print("[case] indexer NaN row", flush=True)
    got = dsa.indexer_scores(t16(q, dev), torch.from_numpy(w).to(dev), t16(k, dev), torch.from_numpy(seq).to(dev),
                             block_table=torch.from_numpy(bt).to(dev), block_size=64, causal=True, n_cols=200)
    torch.cuda.synchronize()
    assert (got[0, :, 71].cpu().numpy() == 0.0).all()
    check(got, q, w, k, ref, "indexer NaN row")


@pytest.mark.parametrize("H_I,s_q,lens", [(64, 2, [500, 3, 128, 129] * 10), (64, 2, [2000, 700, 1, 1025] * 16),
                                          (128, 40, [700, 90, 513] * 10), (32, 2, [1] * 260 + [3001] * 11),
                                          (128, 3, [30] * 60 + [9000] * 3), (64, 5, [129] * 100 + [2500] * 12)])
def test_deals(dev, H_I, s_q, lens):
    """Whole workgroups per group (up to 4 chunks, up to 16, and 1200 groups in several rounds), and
    even deals whose runs count the groups' starts (chunks read once, and by several groups; more
    than 256 groups, in one block of the scan and two)."""
    rng = np.random.default_rng(460 + len(lens) + s_q)
    seq = np.array(lens, np.int32)
    q, w, k, bt = paged(rng, len(seq), seq, 64, H_I, s_q, bad_blocks=3)
    n = int(seq.max())
    print(f"[case] indexer deal H_I={H_I} s_q={s_q} B={len(seq)} n={n}", flush=True)
    ref = oracle.indexer_scores(q, w, k, seq, block_table=bt, block_size=64, causal=True, n_cols=n)
    got = dsa.indexer_scores(t16(q, dev), torch.from_numpy(w).to(dev), t16(k, dev), torch.from_numpy(seq).to(dev),
                             block_table=torch.from_numpy(bt).to(dev), block_size=64, causal=True, n_cols=n)
    torch.cuda.synchronize()
    check(got, q, w, k, ref, f"indexer deal H_I={H_I} s_q={s_q}")
