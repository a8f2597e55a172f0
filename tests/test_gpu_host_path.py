"""The native host path (csrc/host.cpp): other Python threads run while a call allocates and launches, and the
arguments it takes."""
import ctypes
import os
import subprocess
import threading
import time
from types import SimpleNamespace

import pytest
import torch

from keys_values_amd import _lib
from keys_values_amd.attention import ops
from keys_values_amd.kvcache.h2o import H2OKVCache, KVCacheParams
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
