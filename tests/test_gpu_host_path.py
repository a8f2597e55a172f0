"""The native host path (csrc/host.cpp): other Python threads run while a call allocates and launches, the arguments it
takes, and what a call over a quantised store allocates."""
import ctypes
import os
import subprocess
import threading
import time
from types import SimpleNamespace

import pytest
import torch

from helpers import rel_err
from keys_values_amd import _lib
from keys_values_amd.attention import ops
from keys_values_amd.attention.sdpa import HipMultiHeadSelfAttention, HipSDPA
from keys_values_amd.kvcache.buffers import QuantizedKeysAndValues
from keys_values_amd.kvcache.h2o import H2OKVCache, KVCacheParams, create_kv_cache
from keys_values_amd.kvcache.quantize import RowQuantizer
from keys_values_amd.longctx import ops as lops

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# A library with the kernels' entry points and no kernels: a call that would launch returns once another thread has
# acknowledged it, or with an error after two seconds without.
_STUB = r"""
#include <time.h>
#include "kvx.h"
volatile int calls, acknowledged;
static int meet(void) {
  struct timespec a, b;
  const int mine = ++calls;
  clock_gettime(CLOCK_MONOTONIC, &a);
  do {
    if (acknowledged >= mine) return KVX_OK;
    clock_gettime(CLOCK_MONOTONIC, &b);
  } while ((b.tv_sec - a.tv_sec) * 1000000000L + (b.tv_nsec - a.tv_nsec) < 2000000000L);
  return KVX_ERR_HIP;
}
const char* kvx_last_error(void) { return "no other thread ran during the call"; }
#define SIZE1(name) size_t name(const kvx_sdpa_args* a) { (void)a; return 4096; }
SIZE1(kvx_sdpa_prefill_workspace_bytes) SIZE1(kvx_sdpa_prefill_copying_workspace_bytes) SIZE1(kvx_sdpa_decode_workspace_bytes)
size_t kvx_h2o_workspace_bytes(const kvx_h2o_args* a) { (void)a; return 4096; }
size_t kvx_h2o_decode_step_workspace_bytes(const kvx_sdpa_args* a, const kvx_h2o_args* h) { (void)a; (void)h; return 4096; }
#define CALL(name, ...) int name(__VA_ARGS__) { return meet(); }
CALL(kvx_sdpa_prefill, const kvx_sdpa_args* a, void* s)
CALL(kvx_sdpa_prefill_copying, const kvx_sdpa_args* a, void* s)
CALL(kvx_score_sum, const kvx_sdpa_args* a, void* s)
CALL(kvx_sdpa_prefill_weights, const kvx_sdpa_args* a, void* s)
CALL(kvx_sdpa_decode, const kvx_sdpa_args* a, void* s)
CALL(kvx_h2o_decode_step, const kvx_cache_write_args* w, const kvx_sdpa_args* a, const kvx_h2o_args* h, void* s)
CALL(kvx_quantize_blocks, const kvx_block_quant_args* a, void* s)
CALL(kvx_dequantize_blocks, const kvx_block_quant_args* a, void* s)
CALL(kvx_dequantize_rows_typed, const uint8_t* c, const float* sc, const int32_t* z, int64_t n, int32_t d, int32_t b, int32_t e, void* o, int64_t os, void* s)
CALL(kvx_cache_write, const kvx_cache_write_args* a, void* s)
CALL(kvx_h2o_update_select, const kvx_h2o_args* a, void* s)
CALL(kvx_rmsnorm_rows, const void* x, int64_t xs, void* o, int64_t os, const float* w, int64_t n, int32_t d, float e, void* s)
CALL(kvx_add_rmsnorm_rows, const void* x, int64_t xs, const void* dl, int64_t ds, void* xo, int64_t xos, void* o, int64_t os, const float* w, int64_t n,
     int32_t d, float e, void* s)
CALL(kvx_swiglu_rows, const void* g, int64_t gs, void* o, int64_t os, int64_t n, int32_t d, void* s)
CALL(kvx_qk_norm_rope, void* x, int64_t sb, int64_t st, int32_t B, int32_t n, int32_t hq, int32_t hkv, int32_t D, const float* qw, const float* kw, float e,
     const float* c, const float* sn, int32_t tr, int32_t ip, void* s)
"""


@pytest.fixture
def stub(tmp_path, gpu):
    """The host path bound to the library above, and a thread that acknowledges its calls."""
    src, so = tmp_path / "stub.c", tmp_path / "libstub.so"
    src.write_text(_STUB)
    subprocess.check_call(["gcc", "-std=gnu11", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "include"), str(src), "-o", str(so)])
    lib = ctypes.CDLL(str(so))
    calls, acknowledged = ctypes.c_int.in_dll(lib, "calls"), ctypes.c_int.in_dll(lib, "acknowledged")
    stop = threading.Event()

    def acknowledge():
        while not stop.is_set():
            acknowledged.value = calls.value
            time.sleep(0)

    host = _lib.host()
    thread = threading.Thread(target=acknowledge, daemon=True)
    host.bind(str(so), _lib.KvxError, torch.OutOfMemoryError)
    thread.start()
    try:
        yield calls
    finally:
        stop.set()
        thread.join()
        host.bind(_lib.LIB_PATH, _lib.KvxError, torch.OutOfMemoryError)


def test_other_threads_run_during_a_call(gpu, stub):
    """Every function that launches lets other Python threads run meanwhile: a launch can wait for room in a hardware
    queue, and for work whose end needs Python (a host function in a stream)."""

    def rows(*shape):
        return torch.zeros(shape, dtype=torch.bfloat16, device=gpu)

    q, k = rows(1, 4, 8, 64), rows(1, 2, 32, 64)
    lse = torch.zeros(1, 8, 4, device=gpu)
    codes, sc, zp = (torch.zeros(s, dtype=t, device=gpu) for s, t in (((1, 2, 32, 64), torch.uint8), ((1, 2, 32), torch.float32), ((1, 2, 32), torch.int32)))
    qz = RowQuantizer((1, 2, 32, 64), device=gpu, allocate_buffers=True)
    weight, table = torch.ones(64, device=gpu), torch.zeros(64, 32, device=gpu)
    state = ops.QuantState(sc, zp, sc, zp)
    runs = [
        lambda: ops.prefill_core(q, k, k, 0.125, 24),
        lambda: ops.prefill_core(q, k, k, 0.125, 24, return_weights=True),
        lambda: ops.prefill_core(q, codes, codes, 0.125, 24, return_weights=True, quant=state),
        lambda: ops.score_sum_core(q, k, lse, 0.125, 24),
        lambda: ops.decode_core(q[:, :, :1], k, k, 0.125, return_weights=True),
        lambda: qz.quantize(0, 32, k),
        lambda: qz.dequantize(0, 32),
        lambda: _lib.host().dequantize_rows(codes, sc, zp, 8, rows(64, 64)),
        lambda: lops.rmsnorm(rows(3, 64), weight, 1e-6),
        lambda: lops.add_rmsnorm_(rows(3, 64), rows(3, 64), weight, 1e-6),
        lambda: lops.swiglu(rows(3, 64)),
        lambda: lops.qk_norm_rope_(rows(1, 4, 8 * 64), 4, 2, 64, weight, weight, 1e-6, table, table, 0),
    ]
    for run in runs:
        before = stub.value
        run()
        assert stub.value == before + 1
    cache = H2OKVCache(KVCacheParams(1, 2, 64, 64, 4), max_chunk_size=8, device=gpu)
    for num, launches in ((64, 2), (8, 3), (1, 1)):  # first chunk: write, attention; chunk: and the choice; one token: one call
        before = stub.value
        cache.forward(rows(1, 4, num, 64), rows(1, 2, num, 64), rows(1, 2, num, 64))
        assert stub.value == before + launches


def test_first_chunks_with_libraries_from_before_the_one_call(gpu, tmp_path):
    """The two calls that it stands for, in their order: the write of a chunk that fills the cache is an ordinary one."""
    names = {"kvx_cache_write": 1, "kvx_cache_write_first": 2, "kvx_sdpa_prefill": 3}
    host = _lib.host()
    try:
        for without in ((), ("kvx_cache_write_first",)):
            src, so = tmp_path / f"stub{len(without)}.c", tmp_path / f"libstub{len(without)}.so"
            calls = "".join(f"int {n}(const void* a) {{ order[n++] = {i}; return 0; }}\n" for n, i in names.items() if n not in without)
            others = "".join(f"size_t {n}(void) {{ return 0; }}\n" for n in _lib.SYMBOLS if n not in names and n not in ("kvx_sdpa_prefill_first",))
            src.write_text("#include <stddef.h>\nint order[16], n;\n" + calls + others)
            subprocess.check_call(["gcc", "-shared", "-fPIC", str(src), "-o", str(so)])
            host.bind(str(so), _lib.KvxError, torch.OutOfMemoryError)
            lib = ctypes.CDLL(str(so))
            n, order = ctypes.c_int.in_dll(lib, "n"), (ctypes.c_int * 16).in_dll(lib, "order")
            for num, want in ((64, [1, 3]), (40, [2, 3])):
                cache = H2OKVCache(KVCacheParams(1, 2, 64, 64, 4), device=gpu)
                q, k = (torch.zeros(1, h, num, 64, dtype=torch.bfloat16, device=gpu) for h in (4, 2))
                n.value = 0
                if num < 64 and without:
                    with pytest.raises(ImportError):
                        cache.forward(q, k, k)
                    assert n.value == 0
                else:
                    assert cache.forward(q, k, k).shape == (1, num, 256)
                    assert order[:n.value] == want
    finally:
        host.bind(_lib.LIB_PATH, _lib.KvxError, torch.OutOfMemoryError)


def test_two_threads_on_two_streams(gpu):
    """Caches stepped by two threads at once, each on its stream: the bits of the same steps one after the other."""

    def steps(seed, quantized):
        gen = torch.Generator(device=gpu).manual_seed(seed)
        cache = H2OKVCache(KVCacheParams(2, 2, 512, 64, 8), max_chunk_size=32, quantized=quantized, device=gpu)
        got = []
        for num in [512] + [1, 1, 32, 1, 20] * 8:
            got.append(cache.forward(*(torch.randn(2, h, num, 64, generator=gen, device=gpu).to(torch.bfloat16) for h in (8, 2, 2))))
        return got + [cache.scores, cache.token_pos, cache.k, cache.v]

    want = [steps(seed, quantized) for seed, quantized in ((1, False), (2, True))]
    torch.cuda.synchronize()
    got, errors = [None, None], []

    def work(i, seed, quantized):
        try:
            stream = torch.cuda.Stream(gpu)
            with torch.cuda.stream(stream):
                got[i] = steps(seed, quantized)
            stream.synchronize()
        except Exception as ex:  # noqa: BLE001 -- reported by the test's own thread
            errors.append(ex)

    threads = [threading.Thread(target=work, args=(0, 1, False)), threading.Thread(target=work, args=(1, 2, True))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for one, other in zip(want, got):
        assert all(torch.equal(x, y) for x, y in zip(one, other))


def _store(gpu, B, Hkv, T, D, bits=8, dtype=torch.bfloat16, seed=0):
    gen = torch.Generator(device=gpu).manual_seed(seed)
    codes, state, rows = [], [], []
    for _ in range(2):
        qz = RowQuantizer((B, Hkv, T, D), dtype, bits, allocate_buffers=True, device=gpu)
        qz.quantize(0, T, torch.randn(B, Hkv, T, D, generator=gen, device=gpu).to(dtype))
        codes.append(qz.quant_buffer.view(B, Hkv, T, -1))
        state += [qz.quant_scales.view(B, Hkv, T), qz.quant_zero_points.view(B, Hkv, T)]
        rows.append(qz.dequantize(0, T))
    return codes, ops.QuantState(*state), rows


def test_score_sums_need_the_state_of_the_keys_only(gpu):
    B, Hq, Hkv, q_len, T, D = 2, 8, 2, 40, 300, 64
    (kc, _), state, (kd, _) = _store(gpu, B, Hkv, T, D)
    q = torch.randn(B, Hq, q_len, D, device=gpu).to(torch.bfloat16)
    _, _, lse = ops.prefill_core(q, kd, kd, 0.125, T - q_len, return_lse=True)
    want = ops.score_sum_core(q, kc, lse, 0.125, T - q_len, quant=state)
    for given in (state._replace(v_scale=None, v_zp=None), SimpleNamespace(k_scale=state.k_scale, k_zp=state.k_zp)):
        assert torch.equal(ops.score_sum_core(q, kc, lse, 0.125, T - q_len, quant=given), want)


def test_state_objects_of_other_types(gpu):
    """Any object with the four arrays is a quantiser state, and so is a bare tuple of them."""
    B, Hq, Hkv, T, D = 1, 4, 2, 200, 64
    (kc, vc), state, _ = _store(gpu, B, Hkv, T, D)

    class State:
        def __init__(self, s):
            self.k_scale, self.k_zp, self.v_scale, self.v_zp = s

        def __iter__(self):
            return iter((self.k_scale, self.k_zp, self.v_scale, self.v_zp))

    q = torch.randn(B, Hq, 16, D, device=gpu).to(torch.bfloat16)
    out, _, _ = ops.prefill_core(q, kc, vc, 0.125, T - 16, quant=state)
    assert torch.equal(ops.prefill_core(q, kc, vc, 0.125, T - 16, quant=State(state))[0], out)
    one, _, _ = ops.decode_core(q[:, :, :1], kc, vc, 0.125, quant=state)
    assert torch.equal(ops.decode_core(q[:, :, :1], kc, vc, 0.125, quant=State(state))[0], one)
    assert torch.equal(ops.prefill_core(q, kc, vc, 0.125, T - 16, quant=tuple(state))[0], out)
    with pytest.raises(ValueError, match="QuantState"):
        ops.prefill_core(q, kc, vc, 0.125, T - 16, quant=tuple(state)[:3])
    with pytest.raises(TypeError, match="v_zp"):
        ops.prefill_core(q, kc, vc, 0.125, T - 16, quant=state._replace(v_zp=None))


def test_positions_and_counts_of_other_types(gpu):
    """They are converted as int() does."""
    q, k = (torch.randn(1, h, n, 64, device=gpu).to(torch.bfloat16) for h, n in ((4, 16), (2, 200)))
    out, w, lse = ops.prefill_core(q, k, k, 0.125, 184, return_weights=True, return_lse=True, num_splits=2)
    for pos, splits in ((184.0, 2.0), (torch.tensor(184), torch.tensor(2.0)), ("184", "2")):
        got = ops.prefill_core(q, k, k, 0.125, pos, return_weights=True, return_lse=True, num_splits=splits)
        assert all(torch.equal(x, y) for x, y in zip(got, (out, w, lse)))
        assert torch.equal(ops.score_sum_core(q, k, lse, 0.125, pos), ops.score_sum_core(q, k, lse, 0.125, 184))
        one = ops.decode_core(q[:, :, :1], k, k, 0.125, num_splits=splits)[0]
        assert torch.equal(one, ops.decode_core(q[:, :, :1], k, k, 0.125, num_splits=2)[0])
    x, weight, table = torch.randn(1, 4, 8 * 64, device=gpu).to(torch.bfloat16), torch.ones(64, device=gpu), torch.rand(64, 32, device=gpu)
    assert torch.equal(lops.qk_norm_rope_(x.clone(), 4, 2, 64, weight, weight, 1e-6, table, table, 3.0),
                       lops.qk_norm_rope_(x.clone(), 4, 2, 64, weight, weight, 1e-6, table, table, 3))
    with pytest.raises(TypeError):
        ops.prefill_core(q, k, k, 0.125, None)


# A long chunk over 8 x 16384 8-bit rows of 128: the copy of the store in 16-bit rows is 64 MiB
_LONG = dict(B=1, Hkv=8, T=16384, D=128, Hq=32, q_len=512)
_COPY = 2 * 8 * 16384 * 128 * 2


def _long_call(gpu):
    c = _LONG
    codes, state, rows = _store(gpu, c["B"], c["Hkv"], c["T"], c["D"])
    q = torch.randn(c["B"], c["Hq"], c["q_len"], c["D"], device=gpu).to(torch.bfloat16)
    return q, codes, state, rows, (c["D"] ** -0.5, c["T"] - c["q_len"], None)


def _extra_bytes(gpu, run):
    """Largest amount of memory in use during run() beyond what was in use before."""
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats(gpu)
    before = torch.cuda.memory_allocated(gpu)
    out = run()
    torch.cuda.synchronize()
    return torch.cuda.max_memory_allocated(gpu) - before, out


def test_the_caller_decides_on_the_copy_of_a_quantised_store(gpu):
    q, codes, state, rows, args = _long_call(gpu)
    want, w_want, _ = ops.prefill_core(q, *rows, *args, return_weights=True)
    scale, pos, _ = args
    mine = QuantizedKeysAndValues(*codes, state, _LONG["D"], 8, torch.bfloat16)
    every = torch.arange(_LONG["T"], device=gpu).expand(1, 8, -1)
    calls = {
        "prefill_core": lambda **kw: ops.prefill_core(q, *codes, *args, return_weights=True, num_splits=1, quant=state, **kw)[:2],
        "HipSDPA": lambda **kw: HipSDPA(**kw).scaled_dot_product_attention(q, *codes, scale, pos, None, True, output_transposed=True, quant=state),
        "HipMultiHeadSelfAttention": lambda **kw: HipMultiHeadSelfAttention(**kw)(q, mine, 0, pos, True, every),
    }
    for name, call in calls.items():
        copied, (out, w) = _extra_bytes(gpu, call)
        fused, (out_f, w_f) = _extra_bytes(gpu, lambda: call(fused_dequant=True))
        print(name, copied, fused, flush=True)
        assert copied >= _COPY, name
        assert fused <= copied - _COPY // 2, name
        for o, x in ((out, w), (out_f, w_f)):
            assert rel_err(o.float().view(want.shape), want.float()) < 1e-2
            torch.testing.assert_close(x, w_want, rtol=1e-4, atol=1e-7)


def test_no_room_for_the_copy(gpu):
    """Where the memory for the copy is not there the call runs without one, and does not make the allocator empty its
    cache to find out."""
    q, codes, state, rows, args = _long_call(gpu)
    want, _, _ = ops.prefill_core(q, *rows, *args)
    del rows
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(gpu).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_allocated(gpu) + _COPY // 2) / total, gpu)
        torch.cuda.reset_peak_memory_stats(gpu)
        retries = torch.cuda.memory_stats(gpu)["num_alloc_retries"]
        outs = [ops.prefill_core(q, *codes, *args, quant=state, num_splits=1)[0] for _ in range(3)]
        torch.cuda.synchronize()
        stats = torch.cuda.memory_stats(gpu)
        assert stats["num_alloc_retries"] == retries and stats["num_ooms"] == 0
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, gpu)
    for out in outs:
        assert rel_err(out.float(), want.float()) < 1e-2
    assert _extra_bytes(gpu, lambda: ops.prefill_core(q, *codes, *args, quant=state, num_splits=1))[0] >= _COPY  # room again: the copy


def test_an_allocation_for_the_copy_that_fails_all_the_same(gpu):
    """Memory that the allocator's account shows as free and that it cannot use (here: a graph's own) is found out by asking."""
    q, codes, state, rows, args = _long_call(gpu)
    want, _, _ = ops.prefill_core(q, *rows, *args)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        torch.empty(2 * _COPY, dtype=torch.uint8, device=gpu)[:1].add_(1)
    try:
        limit = torch.cuda.memory_reserved(gpu) + _COPY // 4
        torch.cuda.set_per_process_memory_fraction(limit / torch.cuda.get_device_properties(gpu).total_memory, gpu)
        failed = torch.cuda.memory_stats(gpu)["num_ooms"]
        out, _, _ = ops.prefill_core(q, *codes, *args, quant=state, num_splits=1)
        torch.cuda.synchronize()
        assert torch.cuda.memory_stats(gpu)["num_ooms"] == failed + 1
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, gpu)
    assert rel_err(out.float(), want.float()) < 1e-2


def test_a_long_chunk_over_a_quantised_store_in_a_graph(gpu):
    """Recorded with its copy, replayed between other work: the eager call's results each time."""
    q, codes, state, _, args = _long_call(gpu)
    q0, q1 = q.clone(), torch.randn_like(q)
    run = lambda: ops.prefill_core(q, *codes, *args, return_weights=True, quant=state)[:2]  # noqa: E731
    run()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()  # the recorded call's memory comes from the device
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, w = run()
    for query in (q0, q1, q0, q1):
        q.copy_(query)
        want, w_want = run()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(w, w_want)


def test_a_chosen_threshold_is_kept_to(gpu):
    """dequantize_chunk_rows given by the caller, or set later, holds, also where it is the default's number: chunks below it
    never take a copy. Left at its default the call decides."""
    Hkv, L, D, Hq, chunk = 8, 8192, 128, 32, 400  # 1600 query rows
    extra = {}
    for name, kw in (("default", {}), ("chosen", {"dequantize_chunk_rows": 2048}), ("never", {"dequantize_chunk_rows": None})):
        for make in (lambda c: c, lambda c: c.clone()):
            cache = make(create_kv_cache("h2o-torch-quantized8", KVCacheParams(1, Hkv, L, D, Hq), max_chunk_size=chunk, device=gpu, **kw))
            first = [torch.randn(1, h, L, D, device=gpu).to(torch.bfloat16) for h in (Hq, Hkv, Hkv)]
            cache.forward(*first)
            step = [t[:, :, :chunk].contiguous() for t in first]
            cache.forward(*step)
            extra[name], _ = _extra_bytes(gpu, lambda: cache.forward(*step))
        if name == "default":
            cache.dequantize_chunk_rows = None
            extra["set later"], _ = _extra_bytes(gpu, lambda: cache.forward(*step))
    print(extra, flush=True)
    copy = 2 * Hkv * L * D * 2
    assert extra["default"] >= copy
    assert extra["chosen"] == extra["never"] == extra["set later"] <= extra["default"] - copy // 2
    p256 = KVCacheParams(1, 2, 256, 256, 4)
    assert H2OKVCache(p256, quantized=True, device=gpu).dequantize_chunk_rows == 129
    assert H2OKVCache(p256, quantized=True, device=gpu, dequantize_chunk_rows=2048).dequantize_chunk_rows == 2048
    assert H2OKVCache(p256, quantized=True, device=gpu, dequantize_chunk_rows=None).dequantize_chunk_rows is None
