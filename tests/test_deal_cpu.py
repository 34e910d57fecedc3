"""CPU unit test of how the index scorer deals its chunks to workgroups
(opfoundry_amd/csrc/dsa_deal.h, compiled here with g++: the kernel's own source).

Every chunk is taken exactly once, and no workgroup is kept much longer than an even share:
its chunks, and a fixed cost per group that it begins, stay within a bound of the average.
Causal scores of one prompt, whose first groups hold one chunk each, are the case where runs
of an equal number of chunks alone fail (a run of 64 groups against a run inside one).
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("deal") / "libdeal_check.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror",
                    os.path.join(HERE, "native", "deal_check.cpp"), "-o", so], check=True)
    L = ctypes.CDLL(so)
    L.deal_walk.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_uint32, ctypes.c_uint32] + 3 * [ctypes.c_void_p]
    L.deal_walk.restype = None
    return L


def walk(lib, chunks, G, parts=0):
    chunks = np.ascontiguousarray(chunks, np.uint32)
    n = int(chunks.sum())
    wgs = parts * len(chunks) if parts else G
    seen, taken, begun = np.zeros(max(1, n), np.uint32), np.zeros(wgs, np.int64).astype(np.uint32), np.zeros(wgs, np.uint32)
    lib.deal_walk(chunks.ctypes.data, len(chunks), G, parts, seen.ctypes.data, taken.ctypes.data, begun.ctypes.data)
    return seen[:n], taken.astype(np.int64), begun.astype(np.int64)


def causal(tokens, positions, per_group):
    """Chunks of 128 of one prompt's groups: the last tokens of `positions`, per_group to a group."""
    last = np.minimum(np.arange(per_group, tokens + per_group, per_group), tokens)
    return -(-(positions - tokens + last) // 128)


CASES = [([1], 1), ([3], 3), ([64] * 4, 256), ([16] * 32, 512), ([17] * 32, 512), ([1] * 1000, 512), ([8] * 300, 512),
         ([0, 5, 0, 0, 7], 12), ([0] * 300, 512), ([1] * 120 + [782] * 8, 512), ([1] * 400 + [32] * 100, 512),
         (causal(4096, 4096, 2), 512), (causal(2048, 2048, 4), 512), (causal(16384, 16384, 2), 512),
         (causal(1024, 1024, 1), 512), (causal(300, 500, 1), 512), (np.tile(causal(256, 300, 4), 8), 512),
         (np.tile(causal(512, 512, 4), 2), 512), ([2000], 512), ([3] * 511, 512), ([3] * 513, 512)]


@pytest.mark.parametrize("chunks,G", CASES)
def test_every_chunk_once_and_even(lib, chunks, G):
    chunks = np.asarray(chunks)
    G = max(1, min(G, len(chunks) * int(chunks.max())))      # as the launch sizes it
    seen, taken, begun = walk(lib, chunks, G)
    assert (seen == 1).all()
    start, some = lib.deal_start_units(), int((chunks > 0).sum())
    if chunks.sum() > G:
        # a run is an even share, and at most one more group's start when it begins inside one
        assert (taken + start * begun).max() <= -(-(chunks.sum() + start * some) // G) + start
    else:
        assert taken.max() <= -(-chunks.sum() // G)


@pytest.mark.parametrize("groups,chunks,G", [(4, 512, 512), (128, 128, 512), (128, 24, 512), (512, 17, 512), (1, 2048, 512)])
def test_equal_groups_in_equal_runs(lib, groups, chunks, G):
    """Equal groups that divide into as many equal runs each are cut that way, no run across two."""
    seen, taken, begun = walk(lib, [chunks] * groups, G)
    assert (seen == 1).all() and (taken == groups * chunks // G).all() and (begun == 1).all()


def test_random_deals(lib):
    rng = np.random.default_rng(5)
    for i in range(400):
        n, G = int(rng.integers(1, 700)), int(rng.integers(1, 513))
        chunks = rng.integers(0, rng.choice([2, 4, 9, 60, 400]), n)
        if rng.random() < 0.3:
            chunks[rng.random(n) < 0.9] = rng.integers(0, 3)
        seen, taken, _ = walk(lib, chunks, G, parts=int(rng.integers(1, 40)) if i % 4 == 0 else 0)
        assert (seen == 1).all() and taken.sum() == chunks.sum()
