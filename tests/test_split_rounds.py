"""Automatic split counts: the workgroups of a split call fit one round of the GPU (256 CUs,
each holding one 128-head workgroup or up to two smaller ones), the counts are among the fastest
measured, and neighbouring calls get neighbouring counts."""
import ctypes

import pytest

from opfoundry_amd import abi


def num_splits(fmt, B, H, topk):
    a = abi.DecodeArgs()
    for f in ("q", "kv_cache", "block_table", "seq_lens", "indices", "out", "lse"):
        setattr(a, f, 0x1000)
    a.kv_format, a.kv_total_rows, a.block_size, a.block_table_stride = fmt, 1 << 20, 64, 1024
    a.B, a.s_q, a.H, a.topk, a.sm_scale = B, 1, H, topk, 0.07
    ns = ctypes.c_int32(0)
    assert abi.load_library().dsa_mla_decode_num_splits(ctypes.byref(a), ctypes.byref(ns)) == 0
    return ns.value


@pytest.mark.parametrize("fmt", [abi.KV_BF16, abi.KV_FP8_656])
@pytest.mark.parametrize("B,H,topk", [(1, 128, 2048), (3, 16, 2048), (37, 16, 2048), (74, 16, 2048), (86, 128, 2048),
                                      (127, 128, 512), (128, 128, 2048), (129, 32, 2048), (130, 64, 2048),
                                      (170, 16, 2048), (171, 16, 2048), (255, 128, 4096), (255, 32, 4096),
                                      (256, 128, 4096), (256, 16, 4096), (300, 16, 100), (31, 40, 2048),
                                      (32, 40, 2048), (64, 64, 2048), (85, 64, 512), (86, 33, 1900), (86, 33, 2048),
                                      (255, 64, 2048), (256, 64, 2048), (100, 64, 1024), (64, 64, 2048), (65, 64, 2048),
                                      (65, 64, 1900), (213, 64, 1024), (214, 64, 1024), (214, 64, 2048),
                                      (100, 64, 512), (213, 16, 512), (214, 16, 512), (256, 16, 2048), (257, 16, 2048),
                                      (256, 64, 2048)])
def test_splits_fit_one_round(fmt, B, H, topk):
    """A split call's workgroups fit the GPU's places (256 CUs: one 128-head workgroup each, or two
    of 32 or 64 heads), and a split keeps at least four tiles of the list."""
    ns = num_splits(fmt, B, H, topk)
    wide = max(1, min(256 // min(256, B * ((H + 127) // 128)), -(-topk // 128)))
    small = H <= 64 or B * ((H + 127) // 128) * wide < 128       # 32- or 64-head workgroups
    wgs = B * ((H + 63) // 64 if 32 < H <= 64 else (H + 31) // 32 if small else (H + 127) // 128)
    assert ns == 1 or wgs * ns <= (512 if small else 256)
    assert 1 <= ns <= max(1, -(-topk // 128))


# the split counts within 6 % of the fastest measured kernel and count
@pytest.mark.parametrize("fmt,H,topk,B,fast", [
    (abi.KV_BF16, 40, 1920, 128, (2, 3, 4)), (abi.KV_BF16, 64, 1920, 128, (2, 3)), (abi.KV_BF16, 64, 1024, 128, (1,)),
    (abi.KV_BF16, 64, 2048, 100, (4, 5)), (abi.KV_BF16, 64, 1920, 100, (2, 4, 5)), (abi.KV_BF16, 40, 512, 43, (2, 4)),
    (abi.KV_BF16, 64, 1024, 213, (1,)), (abi.KV_BF16, 16, 2048, 75, (3, 4, 5, 6)), (abi.KV_BF16, 24, 256, 86, (1,)),
    (abi.KV_FP8_656, 32, 1024, 64, (4,)), (abi.KV_FP8_656, 32, 1536, 32, (7, 8)), (abi.KV_FP8_656, 32, 2048, 32, (8,)),
    (abi.KV_FP8_656, 32, 512, 128, (2,)), (abi.KV_FP8_656, 16, 2048, 75, (5, 6)), (abi.KV_FP8_656, 16, 2048, 256, (2,)),
    (abi.KV_FP8_656, 64, 2048, 150, (3,)), (abi.KV_FP8_656, 64, 1024, 150, (3,)), (abi.KV_FP8_656, 64, 512, 100, (1,)),
    (abi.KV_FP8_656, 128, 2048, 5, (8, 10, 12)), (abi.KV_FP8_656, 128, 2048, 6, (8, 10)),
    (abi.KV_FP8_656, 96, 2048, 7, (8, 10, 12))])
def test_counts_against_measured_times(fmt, H, topk, B, fast):
    assert num_splits(fmt, B, H, topk) in fast


@pytest.mark.parametrize("fmt,B,H", [(abi.KV_BF16, 100, 64), (abi.KV_FP8_656, 100, 64), (abi.KV_FP8_656, 74, 16)])
def test_no_cliff_between_neighbouring_lists(fmt, B, H):
    """One entry more, of lists that differ by little, does not unsplit a call or split it many ways."""
    ns = [num_splits(fmt, B, H, k) for k in range(1850, 2049)]
    assert max(ns) - min(ns) <= 1
