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


@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("name,dtype,spare", [("h2o-default", torch.bfloat16, 0), ("h2o-torch-quantized8", torch.float32, 0), ("h2o-default", torch.bfloat16, 1)])
def test_rows_with_a_strided_head_dimension_are_refused(kvx, gpu, name, dtype, spare, which):
    gen = torch.Generator().manual_seed(5)
    q, k, v = (randn(gen, 1, h, 40, 64).to(gpu) for h in (4, 2, 2))
    kv = [k.to(dtype), v.to(dtype)]
    kv[which] = kv[which].transpose(2, 3).contiguous().transpose(2, 3)
    cache = create_kv_cache(name, KVCacheParams(1 + spare, 2, 300, 64, 4))
    with pytest.raises(ValueError, match="head dimension must be contiguous"):
        cache.forward(q, *kv)
    assert cache.forward(q, k, v).shape == (1, 40, 256)


def test_refusals(kvx):
    a = _lib.CacheWriteArgs()
    a.B, a.Hkv, a.num, a.D, a.cache_len = 1, 65536, 1, 64, 65536
    a.index = a.key = a.value = a.k_cache = a.v_cache = 4096
    a.key_stride_t = a.value_stride_t = a.kc_stride_t = a.vc_stride_t = 64
    a.clear_behind = 1
    assert kvx.kvx_cache_write(ctypes.byref(a), None) != 0  # 2^32 slots
    a.Hkv, a.token_pos, a.grace_num, a.grace_period, a.grace_slots, a.input_pos = 1, 4096, 1, 1, 4096, 1
    assert kvx.kvx_cache_write(ctypes.byref(a), None) != 0


def test_padding_means_nothing(kvx, gpu):
    # a caller that sets every field and leaves the bytes between them as they are
    B, Hkv, T, D, num = 1, 2, 64, 64, 3
    gen = torch.Generator().manual_seed(1)
    key, value = (randn(gen, B, Hkv, num, D).to(gpu) for _ in range(2))
    k, v = (torch.zeros(B, Hkv, T, D, dtype=key.dtype, device=gpu) for _ in range(2))
    scores = torch.full((B, Hkv, T), 5.0, device=gpu)
    token_pos = torch.arange(T, dtype=torch.int32, device=gpu).expand(B, Hkv, T).contiguous()
    index = torch.tensor([7, 9, 11], dtype=torch.int32, device=gpu)
    ring = torch.tensor([60], dtype=torch.int32, device=gpu)
    for grace in (0, 1):
        a = _lib.CacheWriteArgs()
        ctypes.memset(ctypes.byref(a), 0xFF, ctypes.sizeof(a))
        for name, _ in a._fields_:
            setattr(a, name, 0)
        a.B, a.Hkv, a.num, a.D, a.cache_len, a.input_pos, a.kv_dtype = B, Hkv, num, D, T, T, _lib.KVX_KV_BF16
        a.index, a.key, a.value, a.k_cache, a.v_cache = (t.data_ptr() for t in (index, key, value, k, v))
        a.key_stride_b, a.key_stride_h, a.key_stride_t = key.stride()[:3]
        a.value_stride_b, a.value_stride_h, a.value_stride_t = value.stride()[:3]
        a.kc_stride_b, a.kc_stride_h, a.kc_stride_t = k.stride()[:3]
        a.vc_stride_b, a.vc_stride_h, a.vc_stride_t = v.stride()[:3]
        a.token_pos, a.tp_stride_b, a.tp_stride_h = token_pos.data_ptr(), *token_pos.stride()[:2]
        a.scores, a.sc_stride_b, a.sc_stride_h = scores.data_ptr(), *scores.stride()[:2]
        a.grace_num, a.grace_period, a.grace_slots = grace, grace, ring.data_ptr()
        _lib.check(kvx.kvx_cache_write(ctypes.byref(a), _lib.stream_ptr(gpu)))
    want = torch.full((B, Hkv, T), 5.0)
    want[:, :, [7, 9, 11, 60]] = 0.0  # the ring's slot holds a new token, its former one moved to slot 7 with a score of 5 or 0
    got = scores.cpu()
    got[:, :, 7] = 0.0
    assert torch.equal(got, want)
