"""Automatic split counts: the workgroups of a split call fit one round of the GPU (256 CUs,
each holding one 128-head workgroup or up to two 32-head ones)."""
import ctypes

import pytest

from opfoundry_amd import abi


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
    a = abi.DecodeArgs()
    for f in ("q", "kv_cache", "block_table", "seq_lens", "indices", "out", "lse"):
        setattr(a, f, 0x1000)
    a.kv_format, a.kv_total_rows, a.block_size, a.block_table_stride = fmt, 1 << 20, 64, 1024
    a.B, a.s_q, a.H, a.topk, a.sm_scale = B, 1, H, topk, 0.07
    ns = ctypes.c_int32(0)
    assert abi.load_library().dsa_mla_decode_num_splits(ctypes.byref(a), ctypes.byref(ns)) == 0
    cap = max(1, (topk + 127) // 128)
    wide_wgs = B * ((H + 127) // 128)
    wide = 1 if wide_wgs >= 256 else min(256 // wide_wgs, cap, 64)
    if H <= 64 or wide_wgs * wide < 128:       # 32-head workgroups
        wgs = B * ((H + 31) // 32)
        two, longest = 32 < H <= 64, topk + 127
        if two and fmt == abi.KV_FP8_656 and (longest >= 2048 and wgs > 128 or longest >= 1024 and 170 < wgs <= 2 * 213):
            wgs, round_, cap = B, 512, longest // 225            # 64-head workgroups
        elif two and fmt == abi.KV_FP8_656 and wgs > 170:
            cap, round_ = 1, 512
        elif two and fmt == abi.KV_BF16 and wgs > 170 and B <= 213 and longest >= 2048:
            wgs, round_, cap = B, 512, longest // 400            # 64-head workgroups
        elif fmt == abi.KV_BF16 and (128 < wgs <= 170 or two and 64 <= wgs <= 170):
            one = max(1, min(256 // wgs, cap))
            round_, cap = 512, max(one, longest // 320)
        else:
            round_ = 512 if fmt == abi.KV_FP8_656 else 256
            if fmt == abi.KV_FP8_656 and wgs > 170:
                cap = longest // 400
    else:
        wgs, round_ = wide_wgs, 256
    assert ns.value == (1 if wgs >= round_ else max(1, min(round_ // wgs, cap, 64)))
    assert wgs >= round_ or wgs * ns.value <= round_
