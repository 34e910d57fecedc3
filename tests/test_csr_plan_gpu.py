"""The CSR work plan and its combine at their edges: row counts around a block of 256 and
around the rule's 256, lengths that put the chunk search on its bounds, rows of more items
than one wave merges at a time (16), and the plan's invariants (items in row order, each at
most `chunk` long, the smallest such chunk whose items fit 256 workgroups).  Outputs against
one workgroup per row (num_splits = 1): the same sums in another order.
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
    hdr = ws[:24].cpu().numpy().view(np.int32)
    items = ws[256:256 + 16 * int(hdr[0])].cpu().numpy().view(np.int32).reshape(-1, 4)
    return indptr, longest, ws, hdr, items


@pytest.mark.parametrize("lens,s_q", [([1] * 255, 1), ([1] * 256, 1), ([1] * 257, 1), ([129] * 300, 2), ([4097], 1),
                                      ([128] * 5 + [70001], 1), ([65536, 5, 0, 33000], 2), ([200000], 3),
                                      (list(range(1, 250)), 1), ([2048] * 130, 1), ([100003] + [31] * 700, 1)])
def test_plan_rule(dev, lens, s_q):
    print(f"[case] plan of {len(lens)} lists, s_q={s_q}", flush=True)
    _, _, _, hdr, items = plan_of(dev, lens, s_q, 16)
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


@pytest.mark.parametrize("lens", [[2100, 40], [2200, 40], [8000, 0, 130], [16400, 16400]])
def test_combine_of_many_items(dev, lens):
    """16, 17, ~60 and 128 items per row (chunks of 128)."""
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
