"""dsa_topk_indices at the edges of its row-length rules (pieces per lane, the register and
streaming kernels, the flags' LDS limit), against oracle.topk_indices: the same integers.
Rows shorter than n_max, ties at the threshold, crowded threshold bins (every refinement),
special values, and outputs past the staging buffer.
"""
import numpy as np
import pytest

from test_topk_gpu import run_case

import torch  # noqa: F401  (the GPU runtime, before the library)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 5, 4095, 4096, 4097, 8193, 16384, 16385, 32769, 65535, 65537, 70001, 131075])
@pytest.mark.parametrize("k", [1, 64, 2048])
def test_row_lengths(dev, n, k):
    print(f"[case] topk flags n={n} k={k}", flush=True)
    rng = np.random.default_rng(n * 7 + k)
    scores = rng.standard_normal((7, n)).astype(np.float32)
    scores[1] = np.round(scores[1] * 2)                       # ties at the threshold
    scores[2] = 3.25                                          # all equal
    scores[3] = 1.0 + rng.integers(0, 9000, n) * np.float32(2.0 ** -23)      # one 12-bit bin
    scores[4, rng.random(n) < 0.3] = np.nan
    scores[5] = rng.choice(np.array([0.0, -0.0, 1e-42, -1e-42, np.inf, -np.inf, -np.nan, np.nan, 1.0], np.float32), n)
    lengths = np.array([n, n, max(1, n - 1), n, n, n, max(1, n // 3)], np.int32)
    run_case(dev, scores, lengths, k)


@pytest.mark.parametrize("n,k", [(393216, 2048), (393217, 2048), (200000, 9000), (60000, 59990), (90000, 89999)])
def test_long_rows_and_outputs(dev, n, k):
    print(f"[case] topk flags long n={n} k={k}", flush=True)
    rng = np.random.default_rng(n + k)
    scores = rng.standard_normal((3, n)).astype(np.float32)
    scores[1] = 1.0 + rng.integers(0, 600, n) * np.float32(2.0 ** -23)       # crowded to the last bit
    run_case(dev, scores, np.array([n, n, n - 5], np.int32), k)
