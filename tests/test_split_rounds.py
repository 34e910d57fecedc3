"""Automatic split counts: the workgroups of a split call fit one round of the 256 CUs."""
import ctypes

import pytest

from opfoundry_amd import abi


@pytest.mark.parametrize("B,H,topk", [(1, 128, 2048), (3, 16, 2048), (37, 16, 2048), (74, 16, 2048), (86, 128, 2048),
                                      (127, 128, 512), (128, 128, 2048), (129, 32, 2048), (255, 128, 4096),
                                      (256, 128, 4096), (300, 16, 100)])
def test_splits_fit_one_round(B, H, topk):
    a = abi.DecodeArgs()
    for f in ("q", "kv_cache", "block_table", "seq_lens", "indices", "out", "lse"):
        setattr(a, f, 0x1000)
    a.kv_format, a.kv_total_rows, a.block_size, a.block_table_stride = abi.KV_BF16, 1 << 20, 64, 1024
    a.B, a.s_q, a.H, a.topk, a.sm_scale = B, 1, H, topk, 0.07
    ns = ctypes.c_int32(0)
    assert abi.load_library().dsa_mla_decode_num_splits(ctypes.byref(a), ctypes.byref(ns)) == 0
    # 32-head workgroups for H <= 32 or a call whose 128-head ones would fill under half the GPU
    cap = max(1, (topk + 127) // 128)
    wide = max(1, min(256 // B, cap))
    wgs = B * ((H + 31) // 32 if H <= 32 or B * ((H + 127) // 128) * wide < 128 else (H + 127) // 128)
    assert ns.value == max(1, min(256 // wgs, cap, 64))
    assert wgs >= 256 or wgs * ns.value <= 256
