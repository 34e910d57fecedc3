"""The CSR work plan and its combine at their edges: row counts around a block of 512 and
around the rule's 256, lengths that put the chunk search on its bounds, rows of at most 4
items beside rows of more, rows of just as many items as one wave merges (16) and of one
more, and the plan's invariants (items in row order, each at most `chunk` long, the smallest
such chunk whose items fit 256 workgroups; the split rows and where their items' results
lie).  Outputs against one workgroup per row (num_splits = 1): the same sums in another order.
"""
import numpy as np
import pytest
import torch

import oracle
from opfoundry_amd import dsa

pytestmark = pytest.mark.gpu


def plan_of(dev, lens, s_q, H):
    indptr = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=dev)
    longest = int(max(lens))
    ws = dsa.csr_plan(indptr, len(lens), s_q, H, longest)
    torch.cuda.synchronize()
    hdr = ws[:28].cpu().numpy().view(np.int32)
    records = lambda at, n: ws[at:at + 16 * n].cpu().numpy().view(np.int32).reshape(-1, 4)  # noqa: E731
    items = records(256, int(hdr[0]))
    # the split rows follow room for rows + 256 items, on a multiple of 256 bytes
    split_rows = records(-(-(256 + 16 * (len(lens) * s_q + 256)) // 256) * 256, int(hdr[1]))
    return hdr, items, split_rows


@pytest.mark.parametrize("lens,s_q", [([1] * 255, 1), ([1] * 256, 1), ([1] * 257, 1), ([129] * 300, 2), ([4097], 1),
                                      ([128] * 5 + [70001], 1), ([65536, 5, 0, 33000], 2), ([200000], 3),
                                      (list(range(1, 250)), 1), ([2048] * 130, 1), ([100003] + [31] * 700, 1),
                                      ([600] * 200, 1), ([512, 513] * 3, 1), ([640, 641], 1), ([2048, 7], 1),
                                      ([2049, 7], 1), ([16384] * 2, 1), ([31] * 511, 1), ([300] * 512, 1),
                                      ([31] * 513 + [9000] * 3, 1), ([1, 20000, 2] * 400, 1), ([40] * 1023 + [5000], 1)])
def test_plan_rule(dev, lens, s_q):
    print(f"[case] plan of {len(lens)} lists, s_q={s_q}", flush=True)
    hdr, items, split_rows = plan_of(dev, lens, s_q, 16)
    L = np.maximum(np.repeat(np.array(lens, np.int64), s_q) - np.tile(np.arange(s_q)[::-1], len(lens)), 0)
    chunk = int(hdr[2])
    count = lambda c: int(np.maximum(1, -(-L // c)).sum())  # noqa: E731
    assert chunk % 32 == 0 and chunk >= 128
    if L.size < 256:
        assert count(chunk) <= 256 and (chunk == 128 or count(chunk - 32) > 256)
    assert int(hdr[0]) == count(chunk) == len(items)
    n = np.maximum(1, -(-L // chunk))
    row = np.repeat(np.arange(L.size), n)
    j = np.arange(len(items)) - np.repeat(np.cumsum(n) - n, n)
    assert (items[:, 0] == row).all() and (items[:, 1] == j * chunk).all()
    assert (items[:, 2] == np.minimum((j + 1) * chunk, L[row])).all()
    slot = (items[:, 3] & ((1 << 30) - 1)) - 1
    assert (slot[n[row] == 1] == -1).all() and (slot[n[row] > 1] == np.arange((n[row] > 1).sum())).all()
    assert ((items[:, 3] >> 30 & 1) == (j == n[row] - 1)).all()
    split = n > 1
    first = np.cumsum(np.where(split, n, 0)) - n
    want = np.stack([np.flatnonzero(split), first[split], n[split], np.zeros(split.sum(), np.int64)], 1)
    assert int(hdr[1]) == split.sum() and (split_rows == want).all()
    assert list(hdr[3:6]) == [len(lens), s_q, max(lens)]
    assert hdr[6] == int((n > 16).any())


@pytest.mark.parametrize("lens,counts", [([2048, 40], [16, 1]), ([2049, 40], [17, 1]), ([2048, 2049], [16, 17]),
                                         ([8000, 0, 130], [63, 1, 2]), ([16384, 16384], [128, 128])])
def test_combine_of_many_items(dev, lens, counts):
    """Rows of as many items as one wave merges (16), of one more, and up to the 128 that two
    rows can have, all of 128 entries but the last."""
    _, items, _ = plan_of(dev, lens, 1, 128)
    assert np.bincount(items[:, 0]).tolist() == counts
    rng = np.random.default_rng(sum(lens))
    B, H, rows = len(lens), 128, 4096
    t = lambda a: torch.from_numpy(a.view(np.int16)).view(torch.bfloat16).to(dev)  # noqa: E731
    q, kv = t(oracle.normal_bf16(rng, (B, H, 576))), t(oracle.normal_bf16(rng, (rows, 576)))
    idx = torch.from_numpy(rng.integers(0, rows, sum(lens)).astype(np.int32)).to(dev)
    indptr = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=dev)
    print(f"[case] plan combine lens={lens}", flush=True)
    o1, l1 = dsa.mla_decode_csr(q, kv, indptr, idx, 0.07, num_splits=1)
    o2, l2 = dsa.mla_decode_csr(q, kv, indptr, idx, 0.07, num_splits=0)
    torch.cuda.synchronize()
    # bf16 outputs of the same fp32 sums: within one bf16 step and the 16-bit probabilities' rounding
    # (2^-8 of the value, averaged over the row's entries); LSE within fp32 sums of 16400 terms
    assert torch.allclose(o1.float(), o2.float(), rtol=2.0 ** -7, atol=2e-3)
    assert torch.allclose(l1, l2, rtol=1e-5, atol=1e-5)
