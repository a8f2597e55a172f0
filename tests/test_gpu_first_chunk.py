"""The first chunk of a sequence into a cache that was in use: scores, norms and errors of the slots behind it are zero, by the launch that
writes its rows (csrc/quantize.hip)."""
import ctypes

import pytest
import torch

from helpers import randn
from keys_values_amd import _lib
from keys_values_amd.kvcache.h2o import KVCacheParams, create_kv_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,B,Hkv,T,D,lengths", [
    ("h2o-default", 1, 2, 300, 64, (1, 255, 299, 300)),
    ("h2o-vlen-torch-quantized8", 2, 3, 1025, 128, (7, 1024, 1025)),
    ("qh2o-vlen-torch-quantized4", 3, 1, 129, 64, (2, 128)),
    ("qh2o-torch-quantized8", 1, 8, 2000, 256, (976,)),  # 8192 slots to clear: whole workgroups
])
@pytest.mark.parametrize("spare", [0, 1])  # batch elements that the chunk does not write
def test_slots_behind_the_first_chunk(kvx, gpu, name, B, Hkv, T, D, lengths, spare):
    gen = torch.Generator().manual_seed(T)
    cache = create_kv_cache(name, KVCacheParams(B + spare, Hkv, T, D, 2 * Hkv))
    state = [t for t in (cache.scores, cache.v_norm, cache.q_errors) if t is not None]
    for num in lengths:
        for t in state:
            t.fill_(float("nan"))
        q, k, v = (randn(gen, B, h, num, D).to(gpu) for h in (2 * Hkv, Hkv, Hkv))
        cache.reset()
        cache.forward(q, k, v)
        assert all(torch.equal(t[..., num:], torch.zeros_like(t[..., num:])) for t in state)
        assert all(torch.equal(t[B:], torch.zeros_like(t[B:])) for t in state)
        assert torch.equal(cache.scores, torch.zeros_like(cache.scores))
        if cache.v_norm is not None:
            torch.testing.assert_close(cache.v_norm[:B, :, :num], v.float().norm(dim=-1), rtol=1e-5, atol=0)
        if cache.q_errors is not None:
            assert torch.isfinite(cache.q_errors).all() and (cache.q_errors[:B, :, :num] > 0).all()


def test_refusals(kvx):
    a = _lib.CacheWriteArgs()
    a.B, a.Hkv, a.num, a.D, a.cache_len = 1, 65536, 1, 64, 65536
    a.index = a.key = a.value = a.k_cache = a.v_cache = 4096
    a.key_stride_t = a.value_stride_t = a.kc_stride_t = a.vc_stride_t = 64
    a.clear_behind = 1
    assert kvx.kvx_cache_write(ctypes.byref(a), None) != 0  # 2^32 slots
    a.Hkv, a.token_pos, a.grace_num, a.grace_period, a.grace_slots, a.input_pos = 1, 4096, 1, 1, 4096, 1
    assert kvx.kvx_cache_write(ctypes.byref(a), None) != 0
