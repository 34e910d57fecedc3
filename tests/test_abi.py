"""C ABI of libdsa_mla.so, checked without a GPU: the library loads, exports
every function include/dsa_mla.h declares, its argument structs have the
layout the ctypes mirror assumes (checked against the C compiler's own
sizeof / offsetof), and argument validation returns the documented error
codes before any launch (no device is touched on these paths)."""
from __future__ import annotations

import ctypes
import os
import re
import subprocess

import pytest

from opfoundry_amd import abi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADERS = [os.path.join(ROOT, "include", f) for f in sorted(os.listdir(os.path.join(ROOT, "include")))
           if f.endswith(".h")]


def declared_functions():
    names = []
    for h in HEADERS:
        text = open(h).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        for m in re.finditer(r"^\s*(?:const\s+)?[A-Za-z_][\w\s\*]*?\b([a-z_][a-z0-9_]*)\s*\(", text,
                             flags=re.M):
            if m.group(1) not in ("if", "while", "sizeof"):
                names.append(m.group(1))
    return names


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(abi.LIB_PATH):
        pytest.fail("libdsa_mla.so is not built (run __graft_entry__.build())")
    return abi.load_library()


def test_exports_every_declared_symbol(lib):
    names = declared_functions()
    assert set(names) == set(abi.EXPORTED_SYMBOLS), (names, abi.EXPORTED_SYMBOLS)
    for n in names:
        assert hasattr(lib, n), n
    out = subprocess.run(["nm", "-D", "--defined-only", abi.LIB_PATH], capture_output=True,
                         text=True, check=True).stdout
    exported = {line.split()[-1] for line in out.splitlines() if " T " in line}
    assert set(names) <= exported


def test_abi_version_and_strerror(lib):
    assert lib.dsa_mla_abi_version() == abi.ABI_VERSION
    for code in list(abi.ERRORS) + [0]:
        assert lib.dsa_mla_strerror(code)
    assert lib.dsa_mla_strerror(0) == b"success"


def _c_layout(struct: str, fields):
    src = "#include <stddef.h>\n#include <stdio.h>\n#include \"dsa_mla.h\"\n#include \"dsa_indexer.h\"\nint main(void){\n"
    src += f'printf("%zu\\n", sizeof({struct}));\n'
    for f in fields:
        src += f'printf("%zu\\n", offsetof({struct}, {f}));\n'
    src += "return 0;}\n"
    d = os.path.join(ROOT, "oracle", "_build")
    os.makedirs(d, exist_ok=True)
    c = os.path.join(d, f"layout_{struct}.c")
    exe = c[:-2]
    with open(c, "w") as fh:
        fh.write(src)
    subprocess.run(["gcc", "-std=c11", "-I", os.path.join(ROOT, "include"), c, "-o", exe], check=True)
    vals = [int(x) for x in subprocess.run([exe], capture_output=True, text=True,
                                           check=True).stdout.split()]
    return vals[0], vals[1:]


@pytest.mark.parametrize("cls,name", [(abi.DecodeArgs, "dsa_mla_decode_args"),
                                      (abi.IndexerArgs, "dsa_indexer_args"),
                                      (abi.CsrArgs, "dsa_mla_decode_csr_args"),
                                      (abi.MxArgs, "dsa_mla_decode_mxfp8_args"),
                                      (abi.PrefillV4Fp8Args, "dsa_mla_prefill_v4_fp8_args"),
                                      (abi.PrefillV4Args, "dsa_mla_prefill_v4_args"),
                                      (abi.PrefillArgs, "dsa_mla_prefill_args")])
def test_struct_layout_matches_c(cls, name):
    fields = [f for f, _ in cls._fields_]
    size, offs = _c_layout(name, fields)
    assert ctypes.sizeof(cls) == size
    assert [getattr(cls, f).offset for f in fields] == offs


def _decode_args(**kw):
    a = abi.DecodeArgs()
    a.q = 0x1000
    a.q_stride_b, a.q_stride_t, a.q_stride_h = 128 * 576, 128 * 576, 576
    a.kv_cache = 0x2000
    a.kv_total_rows = 1 << 20
    a.kv_format = abi.KV_BF16
    a.block_size = 64
    a.block_table = 0x3000
    a.block_table_stride = 1024
    a.seq_lens = 0x4000
    a.indices = 0x5000
    a.idx_stride_b, a.idx_stride_t = 2048, 2048
    a.out = 0x6000
    a.o_stride_b, a.o_stride_t, a.o_stride_h = 128 * 512, 128 * 512, 512
    a.lse = 0x7000
    a.B, a.s_q, a.H, a.topk = 8, 1, 128, 2048
    a.num_splits = 0
    a.causal = 0
    a.sm_scale = 0.07
    for k, v in kw.items():
        setattr(a, k, v)
    return a


def _ws(lib, a):
    n = ctypes.c_size_t(0)
    rc = lib.dsa_mla_decode_workspace_size(ctypes.byref(a), ctypes.byref(n))
    return rc, n.value


def _splits(lib, a):
    n = ctypes.c_int32(0)
    rc = lib.dsa_mla_decode_num_splits(ctypes.byref(a), ctypes.byref(n))
    return rc, n.value


def test_workspace_and_split_plan(lib):
    rc, ns = _splits(lib, _decode_args())
    assert rc == 0 and ns >= 1
    # few queries: the planner splits the top-k list to fill the chip
    rc, ns_small = _splits(lib, _decode_args(B=2))
    assert rc == 0 and ns_small > 1
    rc, ws = _ws(lib, _decode_args(B=2))
    assert rc == 0 and ws >= ns_small * 2 * 128 * 513 * 4
    rc, ws1 = _ws(lib, _decode_args(B=2, num_splits=1))
    assert rc == 0 and ws1 == 0
    # enough queries to fill the chip: a long list runs unsplit (the workgroup
    # walks it 2048 entries at a time)
    rc, ns_big = _splits(lib, _decode_args(B=512, topk=4096))
    assert rc == 0 and ns_big == 1
    assert _ws(lib, _decode_args(B=512, topk=4096))[1] == 0


@pytest.mark.parametrize("kw,code", [
    (dict(H=0), -2), (dict(H=-1), -2), (dict(B=-1), -2), (dict(s_q=0), -2), (dict(topk=-5), -2),
    (dict(kv_format=7), -4), (dict(num_splits=65), -6), (dict(num_splits=-1), -6),
    (dict(topk=2 ** 31 - 1), -2), (dict(block_size=0), -2),
    (dict(q=None), -1), (dict(indices=None), -1), (dict(seq_lens=None), -1), (dict(out=None), -1),
    (dict(q_stride_h=577), -7), (dict(o_stride_h=514), -7), (dict(q=0x1008), -7),
    (dict(kv_total_rows=-1), -2),
    # row stride (elements): shorter than a row, not 16-byte aligned, negative
    (dict(kv_stride_row=575), -7), (dict(kv_stride_row=580), -7), (dict(kv_stride_row=-576), -7),
    (dict(kv_format=abi.KV_FP8_656, kv_stride_row=600), -7),
    (dict(kv_format=abi.KV_FP8_656, kv_stride_row=664), -7),
    # row stride of 4 GiB or more (the kernels form row offsets as 32 x 32-bit products)
    (dict(kv_stride_row=2 ** 31), -7), (dict(kv_format=abi.KV_FP8_656, kv_stride_row=2 ** 32), -7),
])
def test_decode_rejects_bad_arguments(lib, kw, code):
    a = _decode_args(**kw)
    assert lib.dsa_mla_decode(ctypes.byref(a), None, 0, None) == code
    assert _ws(lib, a)[0] == code


def test_decode_rejects_missing_workspace(lib):
    a = _decode_args(B=2, num_splits=4)
    assert lib.dsa_mla_decode(ctypes.byref(a), None, 0, None) == -5
    assert lib.dsa_mla_decode(ctypes.byref(a), ctypes.c_void_p(0x10000), 16, None) == -5
    assert lib.dsa_mla_decode(ctypes.byref(a), ctypes.c_void_p(0x10008), 1 << 30, None) == -5


@pytest.mark.parametrize("kw,code", [
    (dict(H=0), -2), (dict(B=-1), -2), (dict(q=None), -1), (dict(kv_stride_row=575), -7),
    (dict(topk=2 ** 31 - 1), -2),
    # 64 splits of 2 x 128 rows: 33.6 MB of partials, beyond the 16 MiB scratch
    (dict(B=2, num_splits=64), -9),
    # automatic counts: 100 tokens of 32 heads (5 splits, 33 MB; at one workgroup per CU 3, 20 MB),
    # and 128-head workgroups (8 tokens of 72 heads, 16 splits, 19 MB)
    (dict(B=100, H=32, topk=2048, kv_format=abi.KV_FP8_656), -9), (dict(B=8, H=72, topk=2048), -9),
])
def test_decode_noalloc_rejects_before_launch(lib, kw, code):
    a = _decode_args(**kw)
    assert lib.dsa_mla_decode_noalloc(ctypes.byref(a), None) == code
    assert b"scratch" in lib.dsa_mla_strerror(-9)


def test_decode_noalloc_empty_batch_is_a_no_op(lib):
    assert lib.dsa_mla_decode_noalloc(ctypes.byref(_decode_args(B=0)), None) == 0


def test_decode_empty_batch_is_a_no_op(lib):
    a = _decode_args(B=0)
    assert lib.dsa_mla_decode(ctypes.byref(a), None, 0, None) == 0


def _csr_args(**kw):
    a = abi.CsrArgs()
    a.q, a.kv, a.out, a.lse = 0x1000, 0x2000, 0x3000, 0x4000
    a.kv_indptr, a.kv_indices = 0x5000, 0x6000
    a.B, a.s_q, a.H, a.total_tokens = 4, 2, 128, 100000
    a.stride_q_b, a.stride_q_h = 128 * 576, 576
    a.stride_o_b, a.stride_o_h = 128 * 512, 512
    a.kv_format = abi.KV_BF16
    a.max_kv_len = 3000
    a.num_splits = 0
    a.softmax_scale = 0.07
    for k, v in kw.items():
        setattr(a, k, v)
    return a


def _csr_ws(lib, a):
    n = ctypes.c_size_t(0)
    rc = lib.dsa_mla_decode_csr_workspace_size(ctypes.byref(a), ctypes.byref(n))
    return rc, n.value


def test_row_strides_accepted(lib):
    """Padded cache rows: any stride of at least one row in whole 16-byte steps."""
    for fmt, st in ((abi.KV_BF16, 0), (abi.KV_BF16, 576), (abi.KV_BF16, 584), (abi.KV_BF16, 640),
                    (abi.KV_FP8_656, 0), (abi.KV_FP8_656, 656), (abi.KV_FP8_656, 672)):
        assert _ws(lib, _decode_args(kv_format=fmt, kv_stride_row=st))[0] == 0
        assert _csr_ws(lib, _csr_args(kv_format=fmt, stride_kv_page=st))[0] == 0
    ok = _v4_args(total_pages=(1 << 30) - 1, total_tokens=(1 << 30) - 1, N=0)
    assert lib.dsa_mla_prefill_v4(ctypes.byref(ok), None, 0, None) == 0


def test_csr_split_plan():
    """Automatic splits of the CSR entry: a device work plan whose workspace holds the
    plan (header, item table, split-row map) and at most 512 partial rows."""
    lib = abi.load_library()
    row = 128 * 513 * 4                    # one partial row: H x (512 + 1) fp32
    # B = 4, s_q = 2, lists up to 3000: 8 rows x ceil(3000 / 128) items bound the partials
    rc, ws = _csr_ws(lib, _csr_args())
    assert rc == 0 and 8 * 24 * row <= ws < 8 * 24 * row + (1 << 16)
    # lists no longer than 128 entries are never split: no partial rows
    rc, ws_short = _csr_ws(lib, _csr_args(max_kv_len=128, B=512, s_q=1))
    assert rc == 0 and ws_short < (1 << 16)
    # however many rows, at most 2 x 256 partial rows
    rc, ws_big = _csr_ws(lib, _csr_args(max_kv_len=2048, B=100_000, s_q=1))
    assert rc == 0 and ws_big < 512 * row + (100_000 + 512) * 16 + (1 << 16)
    # one explicit split: no workspace
    assert _csr_ws(lib, _csr_args(num_splits=1)) == (0, 0)
    # the most rows a plan takes: rows + 256 items in a grid below 2^31 - 256
    assert _csr_ws(lib, _csr_args(B=2 ** 31 - 513, s_q=1, max_kv_len=128))[0] == 0
    assert _csr_ws(lib, _csr_args(B=2 ** 31 - 512, s_q=1, max_kv_len=128))[0] == -2


@pytest.mark.parametrize("kw,code", [
    (dict(H=0), -2), (dict(B=-1), -2), (dict(s_q=0), -2), (dict(max_kv_len=-1), -2),
    (dict(total_tokens=-1), -2), (dict(kv_format=9), -4), (dict(num_splits=65), -6),
    (dict(max_kv_len=2 ** 31 - 1), -2),
    (dict(q=None), -1), (dict(kv=None), -1), (dict(kv_indptr=None), -1), (dict(kv_indices=None), -1),
    (dict(out=None), -1), (dict(stride_q_h=577), -7), (dict(stride_o_b=-512), -7),
    (dict(q=0x1004), -7),
    (dict(stride_kv_page=500), -7), (dict(stride_kv_page=578), -7), (dict(stride_kv_page=-576), -7),
    (dict(kv_format=abi.KV_FP8_656, stride_kv_page=660), -7),
])
def test_csr_rejects_bad_arguments(lib, kw, code):
    a = _csr_args(**kw)
    assert lib.dsa_mla_decode_csr(ctypes.byref(a), None, 0, None) == code
    assert _csr_ws(lib, a)[0] == code


def test_empty_lists_still_need_q(lib):
    """The kernel reads Q before it knows a list is empty: q is required whenever B > 0."""
    assert lib.dsa_mla_decode(ctypes.byref(_decode_args(topk=0, q=None)), None, 0, None) == -1
    assert lib.dsa_mla_decode_csr(ctypes.byref(_csr_args(max_kv_len=0, q=None)), None, 0, None) == -1
    assert lib.dsa_mla_decode_mxfp8(ctypes.byref(_mx_args(max_kv_len=0, q_rope=None)), None, 0, None) == -1


def test_csr_missing_workspace_and_empty_batch(lib):
    assert lib.dsa_mla_decode_csr(ctypes.byref(_csr_args()), None, 0, None) == -5
    assert lib.dsa_mla_decode_csr(ctypes.byref(_csr_args(B=0)), None, 0, None) == 0


def _mx_args(**kw):
    a = abi.MxArgs()
    a.q_nope, a.q_scale, a.q_rope = 0x1000, 0x2000, 0x3000
    a.kv_nope, a.kv_scale, a.kv_rope = 0x4000, 0x5000, 0x6000
    a.out, a.lse, a.kv_indptr, a.kv_indices = 0x7000, 0x8000, 0x9000, 0xA000
    a.B, a.s_q, a.H, a.total_tokens = 4, 2, 128, 100000
    a.stride_q_nope_b, a.stride_q_nope_h = 128 * 512, 512
    a.stride_q_scale_b, a.stride_q_scale_h = 128 * 16, 16
    a.stride_q_rope_b, a.stride_q_rope_h = 128 * 64, 64
    a.stride_o_b, a.stride_o_h = 128 * 512, 512
    a.stride_kv_nope_page, a.stride_kv_scale_page, a.stride_kv_rope_page = 512, 16, 64
    a.max_kv_len = 3000
    a.num_splits = 0
    a.softmax_scale = 0.07
    for k, v in kw.items():
        setattr(a, k, v)
    return a


def _mx_ws(lib, a):
    n = ctypes.c_size_t(0)
    rc = lib.dsa_mla_decode_mxfp8_workspace_size(ctypes.byref(a), ctypes.byref(n))
    return rc, n.value


def test_mxfp8_split_plan(lib):
    rc, ws = _mx_ws(lib, _mx_args())
    assert rc == 0 and ws >= 2 * 4 * 2 * 128 * 513 * 4
    # automatic splits are the device work plan; one explicit split needs no workspace
    assert _mx_ws(lib, _mx_args(max_kv_len=1024, B=128, s_q=2, num_splits=1)) == (0, 0)
    rc, ws_plan = _mx_ws(lib, _mx_args(max_kv_len=1024, B=128, s_q=2))
    assert rc == 0 and ws_plan <= 512 * 128 * 513 * 4 + (1 << 16)
    # the reference harness pads the scale stream to 32 bytes per row: accepted
    assert _mx_ws(lib, _mx_args(stride_kv_scale_page=32))[0] == 0


@pytest.mark.parametrize("kw,code", [
    (dict(H=0), -2), (dict(B=-1), -2), (dict(s_q=0), -2), (dict(max_kv_len=-1), -2),
    (dict(total_tokens=-1), -2), (dict(num_splits=65), -6),
    (dict(max_kv_len=2 ** 31 - 1), -2),
    (dict(q_nope=None), -1), (dict(q_scale=None), -1), (dict(q_rope=None), -1),
    (dict(kv_nope=None), -1), (dict(kv_scale=None), -1), (dict(kv_rope=None), -1),
    (dict(kv_indptr=None), -1), (dict(kv_indices=None), -1), (dict(out=None), -1),
    (dict(stride_q_nope_h=520), -7), (dict(stride_q_scale_h=8), -7), (dict(stride_q_rope_h=68), -7),
    (dict(stride_kv_nope_page=520), -7), (dict(stride_kv_scale_page=20), -7),
    (dict(stride_kv_rope_page=-64), -7), (dict(stride_o_h=514), -7),
    (dict(kv_scale=0x5008), -7), (dict(q_nope=0x1004), -7),
])
def test_mxfp8_rejects_bad_arguments(lib, kw, code):
    a = _mx_args(**kw)
    assert lib.dsa_mla_decode_mxfp8(ctypes.byref(a), None, 0, None) == code
    assert _mx_ws(lib, a)[0] == code


def test_mxfp8_missing_workspace_and_empty_batch(lib):
    assert lib.dsa_mla_decode_mxfp8(ctypes.byref(_mx_args()), None, 0, None) == -5
    assert lib.dsa_mla_decode_mxfp8(ctypes.byref(_mx_args(B=0)), None, 0, None) == 0


def _v4_args(**kw):
    a = abi.PrefillV4Args()
    a.q, a.unified_kv, a.kv, a.attn_sink, a.out, a.lse = 0x1000, 0x2000, 0x3000, 0x4000, 0x5000, 0x6000
    a.kv_indptr_prefix, a.kv_indices_prefix = 0x7000, 0x8000
    a.kv_indptr_extend, a.kv_indices_extend = 0x9000, 0xA000
    a.N, a.H, a.D = 64, 128, 512
    a.total_pages, a.total_tokens = 65536, 4096
    a.stride_qo_n, a.stride_qo_h = 128 * 512, 512
    a.stride_kv_page = 512
    a.max_rows = 1152
    a.softmax_scale = 0.044
    for k, v in kw.items():
        setattr(a, k, v)
    return a


@pytest.mark.parametrize("kw,code", [
    (dict(H=0), -2), (dict(D=576), -3), (dict(max_rows=2 ** 31 - 1), -2), (dict(N=-1), -2),
    (dict(total_pages=-1), -2), (dict(max_rows=-1), -2),
    (dict(q=None), -1), (dict(out=None), -1), (dict(kv_indptr_prefix=None), -1),
    (dict(kv_indices_extend=None), -1), (dict(unified_kv=None), -1), (dict(kv=None), -1),
    (dict(stride_kv_page=500), -7), (dict(stride_kv_page=516), -7), (dict(stride_qo_h=513), -7),
    (dict(q=0x1008), -7), (dict(out=0x5004), -7),
    # row ids carry their pool in bit 30: each pool stays below 2^30 rows
    (dict(total_pages=1 << 30), -2), (dict(total_tokens=1 << 30), -2), (dict(total_pages=2 ** 31 - 1), -2),
])
def test_prefill_v4_rejects_bad_arguments(lib, kw, code):
    assert lib.dsa_mla_prefill_v4(ctypes.byref(_v4_args(**kw)), None, 0, None) == code


def test_prefill_v4_empty_is_a_no_op(lib):
    assert lib.dsa_mla_prefill_v4(ctypes.byref(_v4_args(N=0)), None, 0, None) == 0


def _prefill_args(**kw):
    a = abi.PrefillArgs()
    a.q = 0x1000
    a.q_stride_n, a.q_stride_h = 128 * 576, 576
    a.kv = 0x2000
    a.kv_rows = 8192
    a.kv_format = abi.KV_BF16
    a.indices = 0x3000
    a.idx_stride_n = 2048
    a.out = 0x4000
    a.o_stride_n, a.o_stride_h = 128 * 512, 512
    a.lse = 0x5000
    a.N, a.H, a.topk = 8192, 128, 2048
    a.causal = 1
    a.sm_scale = 0.07
    for k, v in kw.items():
        setattr(a, k, v)
    return a


@pytest.mark.parametrize("kw,code", [
    (dict(H=0), -2), (dict(N=-1), -2), (dict(topk=-1), -2), (dict(kv_format=3), -4),
    (dict(q=None), -1), (dict(kv=None), -1), (dict(out=None), -1), (dict(indices=None), -1),
    (dict(q_stride_h=100), -7), (dict(out=0x4002), -7), (dict(kv_rows=-3), -2),
    (dict(kv_stride_row=570), -7), (dict(kv_stride_row=590), -7), (dict(topk=2 ** 31 - 1), -2),
])
def test_prefill_rejects_bad_arguments(lib, kw, code):
    a = _prefill_args(**kw)
    assert lib.dsa_mla_prefill(ctypes.byref(a), None, 0, None) == code


def test_prefill_empty_is_a_no_op(lib):
    a = _prefill_args(N=0)
    assert lib.dsa_mla_prefill(ctypes.byref(a), None, 0, None) == 0


@pytest.mark.parametrize("args,code", [
    ((0x1000, 0x2000, 0, 4, 128, 0x3000, 512 * 128, 512, 0x4000, None), -6),
    ((0x1000, 0x2000, 65, 4, 128, 0x3000, 512 * 128, 512, 0x4000, None), -6),
    ((0x1000, 0x2000, 2, -1, 128, 0x3000, 512 * 128, 512, 0x4000, None), -2),
    ((None, 0x2000, 2, 4, 128, 0x3000, 512 * 128, 512, 0x4000, None), -1),
    ((0x1000, 0x2000, 2, 4, 128, 0x3002, 512 * 128, 512, 0x4000, None), -7),
    ((0x1000, 0x2000, 2, 0, 128, None, 0, 0, None, None), 0),
])
def test_combine_validation(lib, args, code):
    assert lib.dsa_mla_combine(*args) == code


@pytest.mark.parametrize("args,code", [
    ((0x1000, 576, -1, 0x2000, 10, None, None), -2),
    ((0x1000, 576, 0, 0x2000, 10, None, None), 0),
    ((None, 576, 5, 0x2000, 10, None, None), -1),
    ((0x1000, 577, 5, 0x2000, 10, None, None), -7),
    ((0x1000, 576, 11, 0x2000, 10, None, None), -2),
])
def test_quantize_validation(lib, args, code):
    assert lib.dsa_kv_quantize_fp8(*args) == code


def _v4fp8_args(**kw):
    a = abi.PrefillV4Fp8Args()
    a.q_nope, a.q_rope = 0x1000, 0x2000
    a.unified_kv_nope, a.unified_kv_rope, a.kv_nope, a.kv_rope = 0x3000, 0x4000, 0x5000, 0x6000
    a.attn_sink, a.out, a.lse = 0x7000, 0x8000, 0x9000
    a.kv_indptr_prefix, a.kv_indices_prefix = 0xA000, 0xB000
    a.kv_indptr_extend, a.kv_indices_extend = 0xC000, 0xD000
    a.N, a.H, a.total_pages, a.total_tokens = 16, 128, 1000, 100
    a.stride_q_nope_n, a.stride_q_nope_h = 128 * 512, 512
    a.stride_q_rope_n, a.stride_q_rope_h = 128 * 64, 64
    a.stride_o_n, a.stride_o_h = 128 * 512, 512
    a.stride_kv_nope_page, a.stride_kv_rope_page = 512, 64
    a.max_rows = 640
    a.softmax_scale = 0.04
    for k, v in kw.items():
        setattr(a, k, v)
    return a


@pytest.mark.parametrize("kw,code", [
    (dict(H=0), -2), (dict(N=-1), -2), (dict(max_rows=-1), -2), (dict(total_pages=-1), -2),
    (dict(max_rows=2 ** 31 - 1), -2),
    (dict(q_nope=None), -1), (dict(q_rope=None), -1), (dict(out=None), -1),
    (dict(unified_kv_nope=None), -1), (dict(kv_rope=None), -1), (dict(kv_indices_extend=None), -1),
    (dict(stride_q_nope_h=520), -7), (dict(stride_kv_nope_page=496), -7), (dict(stride_kv_rope_page=60), -7),
    (dict(stride_o_h=510), -7), (dict(kv_nope=0x5008), -7),
    (dict(total_pages=1 << 30), -2), (dict(total_tokens=1 << 30), -2),
])
def test_prefill_v4_fp8_rejects_bad_arguments(lib, kw, code):
    assert lib.dsa_mla_prefill_v4_fp8(ctypes.byref(_v4fp8_args(**kw)), None, 0, None) == code


def test_prefill_v4_fp8_empty_is_a_no_op(lib):
    assert lib.dsa_mla_prefill_v4_fp8(ctypes.byref(_v4fp8_args(N=0)), None, 0, None) == 0
    # empty pools need no pool pointers
    a = _v4fp8_args(N=0, total_pages=0, unified_kv_nope=None, unified_kv_rope=None)
    assert lib.dsa_mla_prefill_v4_fp8(ctypes.byref(a), None, 0, None) == 0


def test_long_lists_accepted_unsplit(lib):
    """Lists longer than one 2048-entry chunk run in one workgroup per query:
    every entry accepts them, unsplit, with no workspace."""
    rc, ws = _ws(lib, _decode_args(topk=4096, num_splits=1))
    assert rc == 0 and ws == 0
    rc, ws = _csr_ws(lib, _csr_args(max_kv_len=200_000, num_splits=1))
    assert rc == 0 and ws == 0
    # more than 64 x 2048 entries with automatic splits
    assert _csr_ws(lib, _csr_args(max_kv_len=200_000))[0] == 0
    n = ctypes.c_size_t(1)
    assert lib.dsa_mla_prefill_workspace_size(ctypes.byref(_prefill_args(topk=4096)), ctypes.byref(n)) == 0
    assert n.value == 0
    assert lib.dsa_mla_prefill_v4(ctypes.byref(_v4_args(max_rows=1 << 20, N=0)), None, 0, None) == 0
    assert lib.dsa_mla_prefill_v4_fp8(ctypes.byref(_v4fp8_args(max_rows=1 << 20, N=0)), None, 0, None) == 0


def test_max_list_bound(lib):
    """DSA_MLA_MAX_LIST (header) = abi.MAX_LIST: the longest list accepted; one more is a
    bad shape (entry positions plus one 2048-entry chunk stay within int32)."""
    hdr = open(os.path.join(os.path.dirname(abi.LIB_PATH), "..", "..", "include", "dsa_mla.h")).read()
    assert f"#define DSA_MLA_MAX_LIST {abi.MAX_LIST}" in hdr
    assert _ws(lib, _decode_args(topk=abi.MAX_LIST, num_splits=1))[0] == 0
    assert _ws(lib, _decode_args(topk=abi.MAX_LIST + 1, num_splits=1))[0] == -2
    assert _csr_ws(lib, _csr_args(max_kv_len=abi.MAX_LIST))[0] == 0
    assert _csr_ws(lib, _csr_args(max_kv_len=abi.MAX_LIST + 1))[0] == -2


@pytest.mark.parametrize("H", [1, 16, 40, 64, 96, 128, 200, 256])
def test_any_head_count_accepted(lib, H):
    """Any H >= 1: workgroups of 128 heads, the last masking heads past H.  Split
    workspaces scale with H."""
    rc, ws = _ws(lib, _decode_args(H=H, B=2))
    assert rc == 0 and ws >= 2 * 1 * H * 513 * 4
    assert _csr_ws(lib, _csr_args(H=H))[0] == 0
    n = ctypes.c_size_t(1)
    assert lib.dsa_mla_prefill_workspace_size(ctypes.byref(_prefill_args(H=H)), ctypes.byref(n)) == 0
    assert lib.dsa_mla_prefill_v4(ctypes.byref(_v4_args(H=H, N=0)), None, 0, None) == 0
    assert lib.dsa_mla_prefill_v4_fp8(ctypes.byref(_v4fp8_args(H=H, N=0)), None, 0, None) == 0


def test_head_groups_bound_the_grid(lib):
    """Query tokens x head groups (ceil(H / 128)) is the grid's x extent: beyond
    2^31 - 1 the call is a bad shape."""
    assert _ws(lib, _decode_args(H=1 << 20, B=1 << 24, num_splits=1))[0] == -2
    assert _ws(lib, _decode_args(H=1 << 7, B=1 << 24, num_splits=1))[0] == 0


def test_csr_plan_entry_validates(lib):
    """dsa_mla_csr_plan checks its shape, pointers and workspace before any launch;
    num_splits = DSA_MLA_SPLITS_PLANNED sizes the same workspace as num_splits = 0."""
    ws0 = _csr_ws(lib, _csr_args(num_splits=0))
    assert ws0[0] == 0 and _csr_ws(lib, _csr_args(num_splits=abi.SPLITS_PLANNED)) == ws0
    assert _csr_ws(lib, _csr_args(num_splits=-2))[0] == -6
    f = lib.dsa_mla_csr_plan
    assert f(None, 0, 1, 128, 100, None, 0, None) == 0                    # empty batch: a no-op
    assert f(None, 4, 2, 128, 3000, ctypes.c_void_p(0x10000), ws0[1], None) == -1
    assert f(ctypes.c_void_p(0x5000), 4, 2, 128, 3000, None, 0, None) == -5
    assert f(ctypes.c_void_p(0x5000), 4, 2, 128, 3000, ctypes.c_void_p(0x10000), ws0[1] - 1, None) == -5
    assert f(ctypes.c_void_p(0x5000), 4, 2, 128, 3000, ctypes.c_void_p(0x10008), ws0[1], None) == -5
    assert f(ctypes.c_void_p(0x5000), -1, 2, 128, 3000, None, 0, None) == -2
    assert f(ctypes.c_void_p(0x5000), 4, 0, 128, 3000, None, 0, None) == -2
    assert f(ctypes.c_void_p(0x5000), 4, 2, 0, 3000, None, 0, None) == -2
    assert f(ctypes.c_void_p(0x5000), 4, 2, 128, abi.MAX_LIST + 1, None, 0, None) == -2


def _ix_args(**kw):
    a = abi.IndexerArgs()
    a.q, a.weights, a.k_cache, a.seq_lens, a.scores = 0x1000, 0x2000, 0x3000, 0x4000, 0x5000
    a.q_stride_b, a.q_stride_t, a.q_stride_h = 2 * 64 * 128, 64 * 128, 128
    a.k_total_rows = 1 << 20
    a.block_table, a.block_table_stride, a.block_size = 0x6000, 1024, 64
    a.score_stride = 65536
    a.B, a.s_q, a.H_I, a.n_cols, a.causal = 4, 2, 64, 65536, 1
    for k, v in kw.items():
        setattr(a, k, v)
    return a


@pytest.mark.parametrize("kw,code", [
    (dict(B=-1), -2), (dict(s_q=0), -2), (dict(n_cols=-1), -2), (dict(k_total_rows=-1), -2),
    (dict(H_I=48), -3), (dict(H_I=256), -3), (dict(block_size=0), -2),
    (dict(k_stride_row=100), -7), (dict(k_stride_row=130), -7), (dict(score_stride=1000), -7),
    (dict(q=None), -1), (dict(weights=None), -1), (dict(seq_lens=None), -1), (dict(scores=None), -1),
    (dict(k_cache=None), -1), (dict(q_stride_h=100), -7), (dict(q=0x1008), -7), (dict(scores=0x5002), -7),
])
def test_indexer_rejects_bad_arguments(lib, kw, code):
    assert lib.dsa_indexer_scores(ctypes.byref(_ix_args(**kw)), None) == code


def test_indexer_empty_is_a_no_op(lib):
    for kw in (dict(B=0), dict(n_cols=0), dict(B=0, q=None)):
        assert lib.dsa_indexer_scores(ctypes.byref(_ix_args(**kw)), None) == 0
    # no k rows at all: accepted (every position scores -inf), k_cache may be NULL
    assert lib.dsa_indexer_scores(ctypes.byref(_ix_args(k_total_rows=0, k_cache=None, B=0)), None) == 0


def _prefill_ws(lib, fn, a):
    n = ctypes.c_size_t(0)
    rc = fn(ctypes.byref(a), ctypes.byref(n))
    return rc, n.value


def test_prefill_split_workspace(lib):
    """Split-K prefill: automatic splits only when fewer than 256 workgroups would run (at
    least 256 list entries per split), the workspace holding num_splits x N x H x 513 floats;
    explicit counts 1..64; a missing or short workspace is rejected before any launch.
    bf16 rows run 32-head workgroups (4 per query at H = 128) when the 128-head ones would
    number fewer than 128 even split, and then split for those."""
    per = 128 * 513 * 4
    # C5-sized: 8192 queries, unsplit, no workspace
    assert _prefill_ws(lib, lib.dsa_mla_prefill_workspace_size, _prefill_args()) == (0, 0)
    # 16 queries of a 65536-entry list: 16 splits (256 workgroups of 128 heads)
    rc, n = _prefill_ws(lib, lib.dsa_mla_prefill_workspace_size, _prefill_args(N=16, topk=65536))
    assert rc == 0 and n == 16 * 16 * per + 256
    # 16 queries of 2048-entry lists: 8 splits of 128 heads would be 128 workgroups: kept
    rc, n = _prefill_ws(lib, lib.dsa_mla_prefill_workspace_size, _prefill_args(N=16, topk=2048))
    assert rc == 0 and n == 8 * 16 * per + 256
    # 8 queries of 1024: 4 x 8 = 32 workgroups of 128 heads: 32-head groups, 4 splits
    rc, n = _prefill_ws(lib, lib.dsa_mla_prefill_workspace_size, _prefill_args(N=8, topk=1024))
    assert rc == 0 and n == 4 * 8 * per + 256
    # 64 queries: 128-head workgroups, 4 splits
    rc, n = _prefill_ws(lib, lib.dsa_mla_prefill_workspace_size, _prefill_args(N=64, topk=65536))
    assert rc == 0 and n == 4 * 64 * per + 256
    # short lists keep >= 256 entries per split
    rc, n = _prefill_ws(lib, lib.dsa_mla_prefill_workspace_size, _prefill_args(N=16, topk=600))
    assert rc == 0 and n == 2 * 16 * per + 256
    rc, n = _prefill_ws(lib, lib.dsa_mla_prefill_workspace_size, _prefill_args(N=8192, num_splits=3))
    assert rc == 0 and n == 3 * 8192 * per + 256
    for bad in (-1, 65):
        assert _prefill_ws(lib, lib.dsa_mla_prefill_workspace_size, _prefill_args(num_splits=bad))[0] == -6
    # V4 bf16 / fp8: the harness's -n 16 -topk 0 over 65536 pages
    rc, n = _prefill_ws(lib, lib.dsa_mla_prefill_v4_workspace_size, _v4_args(N=16, max_rows=65536 + 128))
    assert rc == 0 and n == 16 * 16 * per + 256
    rc, n = _prefill_ws(lib, lib.dsa_mla_prefill_v4_fp8_workspace_size, _v4fp8_args(N=16, max_rows=65536 + 128))
    assert rc == 0 and n == 16 * 16 * per + 256
    rc, n = _prefill_ws(lib, lib.dsa_mla_prefill_v4_workspace_size, _v4_args(N=4096))
    assert rc == 0 and n == 0
    assert _prefill_ws(lib, lib.dsa_mla_prefill_v4_workspace_size, _v4_args(num_splits=65))[0] == -6
    assert _prefill_ws(lib, lib.dsa_mla_prefill_v4_fp8_workspace_size, _v4fp8_args(num_splits=-2))[0] == -6
    # a split call without (or with too small) a workspace: DSA_ERR_WORKSPACE, nothing launched
    assert lib.dsa_mla_prefill_v4(ctypes.byref(_v4_args(num_splits=4)), None, 0, None) == -5
    assert lib.dsa_mla_prefill_v4_fp8(ctypes.byref(_v4fp8_args(num_splits=4)), 0x10000, 1024, None) == -5
    assert lib.dsa_mla_prefill(ctypes.byref(_prefill_args(num_splits=2)), None, 0, None) == -5
