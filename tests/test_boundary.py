"""CPU-side checks of the drop-in boundary: the C-ABI library loads, exports every symbol that
include/kvx.h declares, the ctypes structs match the C layout, argument validation answers without
a GPU, and the host classes keep the reference's error behaviour. No kernel is launched here."""
import ctypes
import os
import re
import subprocess
import tempfile

import pytest
import torch

from helpers import prefill_plan
from keys_values_amd import _lib
from keys_values_amd.attention import ops
from keys_values_amd.attention.sdpa import HipSDPA

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "kvx.h")


def _declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(kvx_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol(kvx):
    names = _declared_symbols()
    assert len(names) >= 15
    assert sorted(_lib.SYMBOLS) == names, "ctypes table and header disagree"
    for n in names:
        assert hasattr(kvx, n), f"libkvx.so does not export {n}"
    assert kvx.kvx_version() == 104


def test_struct_layouts_match_c(tmp_path):
    src = ['#include <stdio.h>', '#include <stddef.h>', f'#include "{HEADER}"', "int main(void){"]
    structs = {"kvx_sdpa_args": _lib.SdpaArgs, "kvx_cache_write_args": _lib.CacheWriteArgs, "kvx_h2o_args": _lib.H2OArgs,
               "kvx_prefill_plan": _lib.PrefillPlan}
    for cname, cls in structs.items():
        src.append(f'printf("{cname} %zu\\n", sizeof({cname}));')
        for fname, _ in cls._fields_:
            src.append(f'printf("{cname}.{fname} %zu\\n", offsetof({cname}, {fname}));')
    src.append("return 0;}")
    c = tmp_path / "layout.c"
    c.write_text("\n".join(src))
    exe = tmp_path / "layout"
    subprocess.check_call(["gcc", "-std=c11", str(c), "-o", str(exe)])
    got = dict(line.split() for line in subprocess.check_output([str(exe)], text=True).splitlines())
    for cname, cls in structs.items():
        assert int(got[cname]) == ctypes.sizeof(cls)
        for fname, _ in cls._fields_:
            assert int(got[f"{cname}.{fname}"]) == getattr(cls, fname).offset, f"{cname}.{fname}"


_OLD_CALLER = r"""
import ctypes, mmap, sys
from keys_values_amd import _lib
kvx = _lib.load()
libc = ctypes.CDLL(None, use_errno=True)
libc.mmap.restype, libc.mmap.argtypes = ctypes.c_void_p, [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_long]
libc.mprotect.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
page = mmap.PAGESIZE
base = libc.mmap(None, 2 * page, mmap.PROT_READ | mmap.PROT_WRITE, mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS, -1, 0)
assert libc.mprotect(base + page, page, 0) == 0
size = _lib.SdpaArgs.workspace_bytes.offset + 8  # the block as callers of the attention calls have written it from the start
a = ctypes.cast(base + page - size, ctypes.POINTER(_lib.SdpaArgs))
calls = (kvx.kvx_sdpa_prefill, kvx.kvx_sdpa_prefill_weights)
for kv_dtype in (0, 1, 2, 3, 4, 5):
    for D in (64, 128, 256):
        b = _lib.SdpaArgs()
        b.B, b.Hq, b.Hkv, b.q_len, b.kv_len, b.D, b.input_pos, b.kv_dtype, b.sm_scale, b.num_splits = 1, 32, 8, 1024, 65536, D, 64512, kv_dtype, 0.1, 4
        for name, ctype in b._fields_:
            if ctype is ctypes.c_void_p and name != "workspace":
                setattr(b, name, 0x10000)
        b.q_stride_t = b.k_stride_t = b.v_stride_t = b.o_stride_t = D
        ctypes.memmove(a, ctypes.byref(b), size)
        partials = 4 * 32 * 1024 * (D + 2) * 4  # of the four splits
        assert kvx.kvx_sdpa_prefill_workspace_bytes(a) == partials, (kv_dtype, D)
        for call in calls:  # no workspace: refused before anything is launched
            assert call(a, None) == _lib.KVX_ERR_WORKSPACE, kvx.kvx_last_error()
        b.lse = None
        ctypes.memmove(a, ctypes.byref(b), size)
        assert kvx.kvx_score_sum(a, None) == _lib.KVX_ERR_INVALID
print("read nothing behind the block")
"""


def test_prefill_reads_no_further_than_the_block_of_its_first_callers(kvx):
    """kvx_sdpa_args has grown behind workspace_bytes. The prefill and score-sum calls read nothing there, and ask for no
    more workspace than their partial results need: callers that end the block at workspace_bytes (here: at the end of
    their memory) get what they always got."""
    import sys

    r = subprocess.run([sys.executable, "-c", _OLD_CALLER], cwd=ROOT, capture_output=True, text=True)
    assert r.returncode == 0 and "read nothing" in r.stdout, (r.returncode, r.stderr[-2000:])


def test_validation_answers_without_a_gpu(kvx):
    # argument checks come before any HIP call
    rc = kvx.kvx_quantize_rows(None, 100, 4, 100, None, None, None, None)
    assert rc == _lib.KVX_ERR_UNSUPPORTED and b"row length 100" in kvx.kvx_last_error()
    with pytest.raises(NotImplementedError):
        _lib.check(rc)
    a = _lib.SdpaArgs()
    a.B, a.Hq, a.Hkv, a.q_len, a.kv_len, a.D = 1, 6, 4, 8, 16, 128
    a.sm_scale = 0.1
    rc = kvx.kvx_sdpa_prefill(ctypes.byref(a), None)
    assert rc == _lib.KVX_ERR_INVALID and b"multiple of Hkv" in kvx.kvx_last_error()
    with pytest.raises(ValueError):
        _lib.check(rc)
    a.Hq = 8
    a.D = 512
    assert kvx.kvx_sdpa_prefill(ctypes.byref(a), None) == _lib.KVX_ERR_UNSUPPORTED
    a.D, a.kv_dtype = 128, 17  # not a store type
    assert kvx.kvx_sdpa_prefill(ctypes.byref(a), None) == _lib.KVX_ERR_UNSUPPORTED and b"kv_dtype" in kvx.kvx_last_error()
    a.kv_dtype = _lib.KVX_KV_BF16
    h = _lib.H2OArgs()
    h.B, h.Hkv, h.kv_len, h.limit, h.k = 1, 1, 16, 16, 17
    assert kvx.kvx_h2o_update_select(ctypes.byref(h), None) == _lib.KVX_ERR_INVALID
    assert kvx.kvx_device_count() >= 0


def test_random_arguments_are_answered_not_trusted(kvx):
    """Seeded random argument blocks (sizes from a set of edge values, pointers NULL / aligned /
    misaligned, strides zero / negative / odd) through every entry point that takes one: each call must
    come back with a status (no division by a zero size, no walk over a NULL pointer on the host).
    Only where no device is visible: a block that happens to pass every check would be launched."""
    import random

    if kvx.kvx_device_count() > 0:
        pytest.skip("a device is visible: random pointers must not reach a kernel")
    rnd = random.Random(2024)
    ints = [-1, 0, 1, 2, 3, 7, 8, 64, 100, 128, 256, 4096, 4097, 2**31 - 1]
    ptrs = [0, 0, 0x10000, 0x10008, 0x10001]
    strides = [-8, 0, 1, 8, 64, 128, 1024, 2**40]
    codes = {_lib.KVX_OK, _lib.KVX_ERR_INVALID, _lib.KVX_ERR_UNSUPPORTED, _lib.KVX_ERR_WORKSPACE, _lib.KVX_ERR_HIP}

    def fill(obj):
        for name, ctype in obj._fields_:
            if ctype is ctypes.c_void_p:
                v = rnd.choice(ptrs)
            elif ctype is ctypes.c_int64 or ctype is ctypes.c_size_t:
                v = rnd.choice(strides)
                if ctype is ctypes.c_size_t:
                    v = abs(v)
            elif ctype is ctypes.c_int32:
                v = rnd.choice(ints)
            else:
                v = rnd.choice([-1.0, 0.0, 0.125, 0.5, 2.0])
            setattr(obj, name, v)
        return obj

    def valid_sdpa():
        a = _lib.SdpaArgs()
        a.B, a.Hkv, a.D, a.kv_dtype = rnd.choice([1, 2]), rnd.choice([1, 2]), rnd.choice([64, 128]), rnd.choice([0, 1, 2])
        a.Hq = a.Hkv * rnd.choice([1, 2, 4])
        a.kv_len = rnd.choice([1, 63, 64, 1000, 70000])
        a.q_len = rnd.choice([1, min(a.kv_len, 100)])
        a.input_pos, a.sm_scale = a.kv_len - a.q_len, 0.125
        for name, ctype in a._fields_:
            if ctype is ctypes.c_void_p:
                setattr(a, name, 0x10000)
        a.q_stride_t = a.k_stride_t = a.v_stride_t = a.o_stride_h = a.D
        a.q_stride_h, a.k_stride_h = a.q_len * a.D, a.kv_len * a.D
        a.v_stride_h, a.o_stride_t = a.k_stride_h, a.Hq * a.D
        a.q_stride_b, a.k_stride_b = a.Hq * a.q_stride_h, a.Hkv * a.k_stride_h
        a.v_stride_b, a.o_stride_b = a.k_stride_b, a.q_len * a.o_stride_t
        a.qs_stride_h = a.tp_stride_h = a.kv_len
        a.qs_stride_b = a.tp_stride_b = a.Hkv * a.kv_len
        a.workspace_bytes = 1 << 40
        return a

    def mutate(obj, times):
        for _ in range(times):
            name, ctype = rnd.choice(obj._fields_)
            if ctype is ctypes.c_void_p:
                setattr(obj, name, rnd.choice(ptrs))
            elif ctype is ctypes.c_int64 or ctype is ctypes.c_size_t:
                setattr(obj, name, abs(rnd.choice(strides)) if ctype is ctypes.c_size_t else rnd.choice(strides))
            elif ctype is ctypes.c_int32:
                setattr(obj, name, rnd.choice(ints))
            else:
                setattr(obj, name, rnd.choice([-1.0, 0.0, 0.125, 0.5, 2.0]))
        return obj

    for it in range(600):
        # half of the blocks are random throughout, half are valid ones with up to two fields replaced
        a = fill(_lib.SdpaArgs()) if it % 2 else mutate(valid_sdpa(), rnd.choice([0, 1, 1, 2]))
        h = fill(_lib.H2OArgs())
        for fn in (kvx.kvx_sdpa_prefill, kvx.kvx_sdpa_prefill_copying, kvx.kvx_score_sum, kvx.kvx_sdpa_decode):
            assert fn(ctypes.byref(a), None) in codes
        assert kvx.kvx_sdpa_decode_h2o(ctypes.byref(a), ctypes.byref(h), None) in codes
        for fn in (kvx.kvx_sdpa_prefill_workspace_bytes, kvx.kvx_sdpa_prefill_copying_workspace_bytes, kvx.kvx_sdpa_decode_workspace_bytes, kvx.kvx_sdpa_decode_h2o_workspace_bytes):
            assert fn(ctypes.byref(a)) >= 0
        assert kvx.kvx_sdpa_prefill_block_rows(ctypes.byref(a), it & 4) in (0, 16, 32, 128, 256)
        assert kvx.kvx_sdpa_prefill_plan(ctypes.byref(a), it & 4, ctypes.byref(_lib.PrefillPlan())) in codes
        assert kvx.kvx_h2o_update_select(ctypes.byref(h), None) in codes
        assert kvx.kvx_h2o_workspace_bytes(ctypes.byref(h)) >= 0
        assert kvx.kvx_cache_write(ctypes.byref(fill(_lib.CacheWriteArgs())), None) in codes
        q = fill(_lib.BlockQuantArgs())
        assert kvx.kvx_quantize_blocks(ctypes.byref(q), None) in codes
        assert kvx.kvx_dequantize_blocks(ctypes.byref(q), None) in codes
        r = lambda: rnd.choice(ptrs)  # noqa: E731
        n, d, st = rnd.choice(ints), rnd.choice(ints), rnd.choice(strides)
        assert kvx.kvx_quantize_rows(r(), st, n, d, r(), r(), r(), None) in codes
        assert kvx.kvx_dequantize_rows(r(), r(), r(), n, d, r(), st, None) in codes
        assert kvx.kvx_quantize_rows4(r(), st, n, d, r(), r(), r(), None) in codes
        assert kvx.kvx_dequantize_rows4(r(), r(), r(), n, d, r(), st, None) in codes
        assert kvx.kvx_rmsnorm_rows(r(), st, r(), st, r(), n, d, 1e-6, None) in codes
        assert kvx.kvx_add_rmsnorm_rows(r(), st, r(), st, r(), st, r(), st, r(), n, d, 1e-6, None) in codes
        assert kvx.kvx_swiglu_rows(r(), st, r(), st, n, d, None) in codes
        assert kvx.kvx_qk_norm_rope(r(), st, st, rnd.choice(ints), n, rnd.choice(ints), rnd.choice(ints), d, r(), r(), 1e-6, r(), r(),
                                    rnd.choice(ints), rnd.choice(ints), None) in codes


def test_no_cpu_fallback():
    q = torch.zeros(1, 4, 2, 64, dtype=torch.bfloat16)
    k = torch.zeros(1, 2, 8, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        ops.prefill_core(q, k, k, 0.125, 6)
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        ops.decode_core(q[:, :, :1], k, k, 0.125)


def test_load_error_is_reported(monkeypatch, tmp_path):
    # keys_values/attention/flashinfer_ops.py:86-147: a failed load leaves a message, a good one None
    from keys_values_amd import attention

    _lib.load()
    assert attention.get_load_error() is None
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "_load_error", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libkvx.so"))
    with pytest.raises(ImportError):
        _lib.load()
    assert "not found" in attention.get_load_error()
    assert not attention.is_available()
    monkeypatch.undo()
    _lib.load()
    assert attention.get_load_error() is None


def test_hip_sdpa_keeps_reference_errors():
    # keys_values/attention/flashinfer_wrapper.py:406-432, keys_values/attention/sdpa_wrapper.py:24-47
    s = HipSDPA.__new__(HipSDPA)
    q = torch.zeros(1, 4, 2, 64, dtype=torch.bfloat16)
    k = torch.zeros(1, 2, 8, 64, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="input_pos must be positive"):
        s.scaled_dot_product_attention(q, k, k, None, 0, None)
    with pytest.raises(ValueError, match="int scalar"):
        s.scaled_dot_product_attention(q, k, k, None, 1.0, None)
    with pytest.raises(ValueError, match="same shape"):
        s.scaled_dot_product_attention(q, k, k[:, :, :4], None, 6, None)
    with pytest.raises(ValueError, match="q_len"):
        s.scaled_dot_product_attention(torch.zeros(1, 4, 9, 64, dtype=torch.bfloat16), k, k, None, 6, None)
    with pytest.raises(ValueError, match="multiple of n_query_groups"):
        s.scaled_dot_product_attention(torch.zeros(1, 3, 2, 64, dtype=torch.bfloat16), k, k, None, 6, None)
    with pytest.raises(ValueError, match="Not compatible"):
        s.scaled_dot_product_attention(q, k, k, None, 6, torch.zeros(1, 2, 7, dtype=torch.int32))
    with pytest.raises(NotImplementedError):  # float32 is not served (float16 and bfloat16 are, as in the reference)
        s.scaled_dot_product_attention(q.float(), k.float(), k.float(), None, 6, None)
    with pytest.raises(NotImplementedError, match="head_size <= 256"):
        s.scaled_dot_product_attention(torch.zeros(1, 4, 2, 264, dtype=torch.bfloat16), torch.zeros(1, 2, 8, 264, dtype=torch.bfloat16),
                                       torch.zeros(1, 2, 8, 264, dtype=torch.bfloat16), None, 6, None)
    with pytest.raises(NotImplementedError, match="q_len=1, kv_len=1"):
        s.scaled_dot_product_attention(q[:, :, :1], k[:, :, :1], k[:, :, :1], None, 6, None)


def test_bench_refuses_more_than_one_gpu_and_runs_nothing_without_one():
    import sys

    bench = os.path.join(ROOT, "bench.py")
    r = subprocess.run([sys.executable, bench, "--gpus", "2"], capture_output=True, text=True)
    assert r.returncode != 0 and "one GPU" in r.stderr and r.stdout.strip() == ""
    if not torch.cuda.is_available():  # no device: it must say so, not fall back to the CPU
        r = subprocess.run([sys.executable, bench, "--steps", "1", "--warmup", "0"], capture_output=True, text=True)
        assert r.returncode != 0 and "no CPU fallback" in r.stderr and r.stdout.strip() == ""


def test_c_oracle_builds():
    from oracle import c_oracle

    assert os.path.exists(c_oracle.build())


def test_libraries_without_the_first_chunk_write_bind(kvx, tmp_path):
    src, so = tmp_path / "stub.c", tmp_path / "libstub.so"
    names = [n for n in _declared_symbols() if n != "kvx_cache_write_first"]
    src.write_text("".join(f"int {n}(void) {{ return 1; }}\n" for n in names))
    subprocess.check_call(["gcc", "-shared", "-fPIC", str(src), "-o", str(so)])
    host = _lib.host()
    try:
        host.bind(str(so), _lib.KvxError, torch.OutOfMemoryError)
        with pytest.raises(ImportError):
            host.cache_write_first(None, None, None, None)
    finally:
        host.bind(_lib.LIB_PATH, _lib.KvxError, torch.OutOfMemoryError)


@pytest.mark.skipif(torch.cuda.is_available(), reason="the pointers are made up: where nothing can be launched")
def test_first_chunk_write_refuses(kvx):
    def call(**fields):
        a = _lib.CacheWriteArgs()
        a.B, a.Hkv, a.num, a.D, a.cache_len = 1, 8, 4, 64, 4096
        a.index = a.key = a.value = a.k_cache = a.v_cache = a.token_pos = 4096
        a.key_stride_t = a.value_stride_t = a.kc_stride_t = a.vc_stride_t = 64
        for name, value in fields.items():
            setattr(a, name, value)
        return kvx.kvx_cache_write_first(ctypes.byref(a), None)

    assert call() == _lib.KVX_ERR_HIP  # a call like any other: no device
    assert call(input_pos=4) == _lib.KVX_ERR_INVALID  # not the first chunk
    assert call(replay_log=4096, log_blocksize=64) == _lib.KVX_ERR_INVALID
    assert call(grace_num=1, grace_period=1, grace_slots=4096, input_pos=1) == _lib.KVX_ERR_INVALID
    assert call(Hkv=65536, cache_len=32767) == _lib.KVX_ERR_HIP
    assert call(Hkv=65536, cache_len=32768) == _lib.KVX_ERR_UNSUPPORTED  # 2^31 slots
    assert call(Hkv=65536, cache_len=65536) == _lib.KVX_ERR_UNSUPPORTED
    assert call(Hkv=65536, cache_len=32767, num=2047, D=256) == _lib.KVX_ERR_UNSUPPORTED  # 2^24 workgroups


@pytest.mark.parametrize("rows,kv_len,k,keys", [
    (32, 256, 200, 0),           # one list: its sort is the choice, no keys are handed on
    (32, 257, 8, 0),
    (32, 1024, 1000, 0),
    (32, 1025, 8, 5 * 256),      # sorted lists of 256 keys
    (24, 7936, 16, 31 * 256),    # three workgroups to each of 256 units
    (25, 7936, 16, 8 * 1024),    # more of them: lists of 512, the same room
    (8, 7936, 1057, 31 * 256),
    (8, 7936, 1058, 8 * 1024),   # too many look-ups for a row
    (32, 3840, 1092, 15 * 256),
    (32, 3840, 1093, 4 * 1024),  # for all rows
    (16, 24000, 500, 47 * 512),  # lists of 512: three workgroups to each of 256 units
    (17, 24000, 500, 24 * 1024),
    (21, 24000, 65, 24 * 1024),  # 987 workgroups: those of 1024 keys fit at once
    (22, 24000, 65, 47 * 512),   # neither do: 3055 look-ups a row
    (22, 24000, 66, 24 * 1024),
    (8, 36300, 20, 71 * 512),    # up to 72 of them
    (4, 36865, 20, 37 * 1024),
])
def test_workspace_of_a_choice_is_its_lists(kvx, rows, kv_len, k, keys):
    """Which lists a row is sorted in, by the workspace that a choice asks for (on 256 compute units, what is assumed without a device):
    the keys, 20 bytes of statistics for 1024 slots, rounded up to 16."""
    a = _lib.H2OArgs()
    a.B, a.Hkv, a.kv_len, a.limit, a.k = 1, rows, kv_len, kv_len, k
    parts = rows * ((kv_len + 1023) // 1024)
    assert kvx.kvx_h2o_workspace_bytes(ctypes.byref(a)) == rows * keys * 8 + (parts * 4 + 15) // 16 * 16 + parts * 16


def _prefill_block(B, heads, kv_heads, q_len, kv_len, D, splits):
    a = _lib.SdpaArgs()
    a.B, a.Hq, a.Hkv, a.q_len, a.kv_len, a.D, a.num_splits = B, heads, kv_heads, q_len, kv_len, D, splits
    a.kv_dtype, a.sm_scale = _lib.elem_kv_dtype(torch.bfloat16), 1.0
    a.q = a.k = a.v = a.o = 4096
    a.q_stride_b, a.q_stride_h, a.q_stride_t = heads * q_len * D, q_len * D, D
    a.k_stride_b, a.k_stride_h, a.k_stride_t = kv_heads * kv_len * D, kv_len * D, D
    a.v_stride_b, a.v_stride_h, a.v_stride_t = kv_heads * kv_len * D, kv_len * D, D
    return a


@pytest.mark.skipif(torch.cuda.is_available(), reason="the pointers are made up: where nothing can be launched")
def test_slot_write_that_asks_for_a_first_chunk_is_refused(kvx):
    a = _lib.CacheWriteArgs()
    a.B, a.Hkv, a.num, a.D, a.cache_len = 1, 8, 4, 64, 4096
    a.index = a.key = a.value = a.k_cache = a.v_cache = a.token_pos = 4096
    a.key_stride_t = a.value_stride_t = a.kc_stride_t = a.vc_stride_t = 64
    assert kvx.kvx_cache_write(ctypes.byref(a), None) == _lib.KVX_ERR_HIP  # no device
    a.clear_behind = 0
    assert kvx.kvx_cache_write(ctypes.byref(a), None) == _lib.KVX_ERR_HIP
    a.clear_behind = 1
    assert kvx.kvx_cache_write(ctypes.byref(a), None) == _lib.KVX_ERR_UNSUPPORTED


@pytest.mark.skipif(torch.cuda.is_available(), reason="the pointers are made up: where nothing can be launched")
@pytest.mark.parametrize("q_len,kv_len", [(4, 100), (300, 9000)])  # one launch, two
def test_weights_refuse_query_rows_of_4_gib(kvx, q_len, kv_len):
    for call in (kvx.kvx_sdpa_prefill_weights, kvx.kvx_sdpa_prefill_copying):
        a = _prefill_block(1, 8, 2, q_len, kv_len, 64, 0)
        a.lse = a.w = a.workspace = 4096
        a.workspace_bytes = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
        assert call(ctypes.byref(a), None) == _lib.KVX_ERR_HIP  # no device
        for name, stride in (("q_stride_h", 2**30), ("q_stride_t", 2**30), ("q_stride_h", -64)):
            b = _lib.SdpaArgs.from_buffer_copy(a)
            setattr(b, name, stride)
            assert call(ctypes.byref(b), None) == _lib.KVX_ERR_UNSUPPORTED


@pytest.mark.skipif(torch.cuda.is_available(), reason="the pointers are made up: where nothing can be launched")
def test_copy_of_a_store_is_refused_beyond_the_blocks_of_a_launch(kvx):
    for kv_len, status in ((2**30 - 64, _lib.KVX_ERR_HIP), (2**30, _lib.KVX_ERR_UNSUPPORTED)):  # 2^24 - 1 workgroups of 64 rows (no device), 2^24
        a = _prefill_block(1, 16, 1, 128, kv_len, 128, 0)
        a.kv_dtype, a.k_scale, a.k_zp, a.v_scale, a.v_zp = _lib.KVX_KV_U8, 4096, 4096, 4096, 4096
        a.workspace, a.workspace_bytes = 4096, 2**50
        assert kvx.kvx_sdpa_prefill_copying(ctypes.byref(a), None) == status


@pytest.mark.parametrize("B,heads,kv_heads,q_len,kv_len,D,input_pos,combined", [
    (1, 32, 8, 101, 3013, 128, 2912, 1),   # the sums lie behind the partials that the same launches combine
    (1, 8, 2, 152, 11212, 64, 11060, 0),   # 44 pairs a row: combined in a launch of their own, the sums take their place
    (1, 8, 2, 596, 14030, 64, 0, 0),       # a causal first chunk in splits
    (1, 16, 8, 809, 36679, 64, 0, 0),      # one split
    (1, 28, 4, 703, 6646, 256, 5943, 0),   # 40 tiles of rows
])
def test_workspace_of_weights_holds_partials_and_sums_where_both_are_read(kvx, B, heads, kv_heads, q_len, kv_len, D, input_pos, combined):
    a = _prefill_block(B, heads, kv_heads, q_len, kv_len, D, 0)
    a.input_pos = input_pos
    without = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))  # the larger of partials and sums
    a.lse = a.w = 4096
    plan = prefill_plan(a)
    assert (plan.one_launch, plan.score_sum, plan.combined) == (0, _lib.KVX_SCORE_SUM_TILED, combined)
    need = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    assert need > without if combined else need == without


@pytest.mark.parametrize("heads,kv_heads,q_len,D,kv_len,pairs", [
    (16, 4, 488, 128, 50688, 8),   # eight wavefronts
    (28, 4, 110, 128, 30208, 18),  # likewise, over 16 pairs a row
    (28, 4, 340, 128, 19968, 6),   # a split of the query rows
    (28, 4, 73, 256, 43520, 16),
    (8, 2, 262, 128, 23040, 28),
    (32, 8, 422, 64, 28672, 6),
])
def test_weights_over_long_stores_leave_the_splits_to_a_launch_of_their_own(kvx, heads, kv_heads, q_len, D, kv_len, pairs):
    """The line lies where all workgroups of the score-sums together would read 24 K (maximum, sum) pairs a compute unit."""
    for more in (0, 1):  # one more block of keys
        a = _prefill_block(1, heads, kv_heads, q_len, kv_len + more, D, 0)
        a.input_pos, a.lse, a.w = kv_len + more - q_len, 4096, 4096
        plan = prefill_plan(a)
        assert (plan.score_sum, plan.splits * plan.teams, plan.combined) == (_lib.KVX_SCORE_SUM_TILED, pairs, 1 - more)


def _first_chunk_blocks(heads, kv_heads, tokens, **fields):
    """Argument blocks of a first chunk: fields of the slot write, or of the attention with a leading ``a_``."""
    a, w = _prefill_block(1, heads, kv_heads, tokens, tokens, 128, 0), _lib.CacheWriteArgs()
    a.workspace, a.workspace_bytes = 4096, 2**40
    w.B, w.Hkv, w.num, w.D, w.cache_len, w.kv_dtype = 1, kv_heads, tokens, 128, 4096, _lib.KVX_KV_U8
    w.index = w.key = w.value = w.k_cache = w.v_cache = w.token_pos = w.k_scale = w.k_zp = w.v_scale = w.v_zp = 4096
    w.key_stride_t = w.value_stride_t = w.kc_stride_t = w.vc_stride_t = 128
    for name, value in fields.items():
        setattr(*((a, name[2:]) if name.startswith("a_") else (w, name)), value)
    return ctypes.byref(a), ctypes.byref(w)


def test_first_chunks_in_one_launch(kvx):
    """Which first chunks are one launch (on 256 compute units, what is assumed without a device)."""
    def one(heads=32, kv_heads=8, tokens=1000, **fields):
        return kvx.kvx_sdpa_prefill_first_in_one_launch(*_first_chunk_blocks(heads, kv_heads, tokens, **fields))

    assert one() == 1
    for fields in ({"num": 999}, {"kv_dtype": _lib.KVX_KV_U8_F16}, {"D": 64}, {"B": 2}, {"a_input_pos": 1}, {"a_token_positions": 4096}, {"a_kv_len": 1001},
                   {"a_kv_dtype": _lib.KVX_KV_F16}):
        assert one(**fields) == 0  # other rows than those attended over, or not a first chunk
    assert one(tokens=3072) == 1 and one(tokens=3073) == 0  # three blocks of rows a unit
    assert one(kv_heads=16, tokens=1024) == 1 and one(kv_heads=16, tokens=1025) == 0  # two heads a KV head
    assert one(kv_heads=16, tokens=641) == 1 and one(kv_heads=16, tokens=640) == 0  # 176 and 160 blocks of rows, 64 tokens of 128 codes to write each
    plain = {"kv_dtype": _lib.KVX_KV_BF16, "heads": 16, "kv_heads": 16}  # 128 and 112, 128 tokens each
    assert one(tokens=897, **plain) == 1 and one(tokens=896, **plain) == 0 and one(16, 16, 897) == 0
    assert one(input_pos=1) == 0  # refused


@pytest.mark.skipif(torch.cuda.is_available(), reason="the pointers are made up: where nothing can be launched")
@pytest.mark.parametrize("heads,kv_heads,tokens,one", [(32, 8, 1000, 1), (8, 8, 137, 0)])
def test_first_chunk_with_its_attention_refuses(kvx, heads, kv_heads, tokens, one):
    def call(**fields):
        return kvx.kvx_sdpa_prefill_first(*_first_chunk_blocks(heads, kv_heads, tokens, **fields), None)

    assert kvx.kvx_sdpa_prefill_first_in_one_launch(*_first_chunk_blocks(heads, kv_heads, tokens)) == one
    assert call() == _lib.KVX_ERR_HIP  # a call like any other: no device
    assert call(num=tokens - 1) == call(a_input_pos=5) == call(a_token_positions=4096) == call(kv_dtype=_lib.KVX_KV_U8_F16) == _lib.KVX_ERR_HIP  # two launches
    assert call(input_pos=4) == _lib.KVX_ERR_INVALID  # not the first chunk
    assert call(replay_log=4096, log_blocksize=64) == _lib.KVX_ERR_INVALID
    assert call(grace_num=1, grace_period=1, grace_slots=4096, input_pos=1) == _lib.KVX_ERR_INVALID
    assert call(key=0) == call(key=4100) == call(cache_len=tokens - 1) == call(k_scale=0) == _lib.KVX_ERR_INVALID
    assert call(Hkv=65536, cache_len=32768) == _lib.KVX_ERR_UNSUPPORTED  # 2^31 slots
    assert call(Hkv=65536, cache_len=32767, num=4096) == _lib.KVX_ERR_UNSUPPORTED  # 2^24 workgroups
    assert call(a_kv_len=tokens - 1) == call(a_q=0) == _lib.KVX_ERR_INVALID
    assert call(a_workspace=4100) == _lib.KVX_ERR_WORKSPACE


@pytest.mark.parametrize("B,heads,kv_heads,q_len,kv_len,D", [(1, 4, 1, 3, 64, 64), (1, 8, 2, 128, 1024, 64), (1, 16, 4, 128, 1500, 64), (1, 2, 1, 8, 8000, 128)])
def test_a_chunk_waits_for_a_few_times_its_own_time(kvx, B, heads, kv_heads, q_len, kv_len, D):
    # a poll is 1.5 to 2 us, these calls take 10 to 20; the single-token step waits for 2^15 polls
    a = _prefill_block(B, heads, kv_heads, q_len, kv_len, D, 0)
    a.lse = a.w = 4096
    plan = prefill_plan(a)
    assert plan.one_launch and 40 <= plan.polls <= 200


@pytest.mark.parametrize("B,heads,kv_heads,q_len,kv_len,D,kv_dtype,one_launch", [
    (2, 56, 8, 15, 756, 128, _lib.KVX_KV_BF16, 0),    # 105 rows: several splits and blocks of rows
    (1, 16, 4, 46, 3428, 64, _lib.KVX_KV_U8, 0),      # 184
    (1, 28, 2, 2, 15221, 64, _lib.KVX_KV_F16, 0),     # 28 rows, streamed
    (1, 24, 8, 12, 14390, 128, _lib.KVX_KV_BF16, 0),  # 36 rows, tiled
    (1, 8, 2, 128, 1024, 64, _lib.KVX_KV_BF16, 1),
    (1, 28, 4, 30, 400, 128, _lib.KVX_KV_U4, 1),
    (1, 4, 2, 8, 4000, 64, _lib.KVX_KV_BF16, 1),      # one block of rows
    (1, 32, 8, 20, 200, 64, _lib.KVX_KV_BF16, 1),     # one split
])
def test_weights_in_one_launch_or_two(kvx, B, heads, kv_heads, q_len, kv_len, D, kv_dtype, one_launch):
    # the launches that measured faster (on 256 compute units)
    a = _prefill_block(B, heads, kv_heads, q_len, kv_len, D, 0)
    a.lse = a.w = 4096
    a.kv_dtype = kv_dtype
    a.k_scale = a.k_zp = a.v_scale = a.v_zp = 4096
    assert bool(prefill_plan(a).one_launch) == bool(one_launch)


@pytest.mark.parametrize("B,heads,kv_heads,q_len,splits", [(1, 4, 2, 100, 2), (4, 64, 16, 1446, 6), (8, 64, 16, 4096, 3)])
def test_workspace_of_splits_of_any_size(kvx, B, heads, kv_heads, q_len, splits):
    # the second and third beyond 2^31 and 2^32 bytes
    a = _prefill_block(B, heads, kv_heads, q_len, 8192, 256, splits)
    assert kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a)) == splits * B * heads * q_len * (256 + 2) * 4


@pytest.mark.parametrize("q_len", [400000, 600000, 700000, 1000000])
def test_long_first_chunks_are_not_split(kvx, q_len):
    # 32 heads fill the device: one split and no workspace, also where the estimates pass 2^31 ns
    a = _prefill_block(1, 32, 8, q_len, q_len, 128, 0)
    assert kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a)) == 0


@pytest.mark.parametrize("heads,kv_heads,q_len,splits", [
    (1, 1, 380, 6),    # a unit has one job at most: a tile a split, whatever the bounds of row blocks
    (6, 2, 209, 4),
])
def test_splits_of_short_first_chunks(kvx, heads, kv_heads, q_len, splits):
    """By the workspace that the partial results ask for (on 256 compute units, what is assumed without a device)."""
    a = _prefill_block(1, heads, kv_heads, q_len, q_len, 256, 0)
    assert kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a)) == splits * heads * q_len * (256 + 2) * 4
