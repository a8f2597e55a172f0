"""The first chunk's rows written by the attention launch (csrc/sdpa_prefill.hip) against the slot write and the attention as two launches: the same bits. Every
case asserts how the library takes it (on 256 compute units)."""
import ctypes

import pytest
import torch

from helpers import prefill_plan, randn
from keys_values_amd import _lib
from keys_values_amd.attention import ops
from keys_values_amd.kvcache.h2o import KVCacheParams, create_kv_cache

pytestmark = pytest.mark.gpu


def route(kvx, cache, q, k, v):
    """Whether the first chunk is one launch, and the KV splits of its attention."""
    a, w = _lib.SdpaArgs(), _lib.CacheWriteArgs()
    ops._fill_common(a, q, k, v, cache.scale_factor, 0, None, None, 0)
    a.o = q.data_ptr()  # nothing is launched: any aligned address
    w.B, w.Hkv, w.num, w.D, w.cache_len, w.kv_dtype = k.shape[0], k.shape[1], k.shape[2], k.shape[3], cache.cache_length, cache._store_dtype
    for name in ("index", "key", "value", "k_cache", "v_cache", "k_scale", "k_zp", "v_scale", "v_zp"):
        setattr(w, name, q.data_ptr())
    return kvx.kvx_sdpa_prefill_first_in_one_launch(ctypes.byref(a), ctypes.byref(w)), prefill_plan(a).splits


@pytest.mark.parametrize("name,dtype,B,Hq,Hkv,T,num,D,one,splits", [
    ("h2o-default", torch.bfloat16, 2, 32, 4, 300, 253, 128, 1, 1),             # the last block has 13 of 16 tokens
    ("h2o-vlen-default", torch.float16, 1, 8, 2, 2000, 1001, 128, 1, 4),        # in splits that end at bounds of blocks: the first ones write
    ("h2o-default", torch.bfloat16, 1, 8, 2, 3000, 2111, 64, 1, 4),
    ("h2o-vlen-torch-quantized8", torch.float16, 2, 28, 4, 517, 517, 128, 1, 1),  # tokens whose heads lie in two blocks; no slot behind the chunk
    ("qh2o-vlen-torch-quantized8", torch.bfloat16, 2, 16, 8, 1100, 1000, 128, 1, 1),
    ("qh2o-vlen-torch-quantized8", torch.bfloat16, 1, 8, 2, 2500, 2001, 128, 1, 4),
    ("h2o-vlen-default", torch.bfloat16, 2, 8, 8, 4200, 900, 128, 1, 4),        # 128 tokens a workgroup; many slots to clear
    ("qh2o-vlen-torch-quantized4", torch.bfloat16, 4, 8, 8, 1500, 1001, 64, 1, 1),
    ("h2o-torch-quantized4", torch.float16, 1, 16, 2, 1500, 1100, 128, 1, 3),
    ("qh2o-torch-quantized8", torch.bfloat16, 1, 24, 8, 700, 650, 64, 1, 1),
    ("h2o-torch-quantized4", torch.float16, 2, 32, 4, 1300, 1001, 64, 1, 1),
    ("qh2o-vlen-torch-quantized4", torch.float16, 1, 16, 4, 1500, 1201, 64, 1, 3),
    # two launches: the kernel for few rows, workgroups with many rows to write and no others beside them, two heads with more than 1024 tokens, heads of 256
    ("h2o-default", torch.bfloat16, 1, 32, 8, 300, 253, 128, 0, 1),
    ("qh2o-vlen-torch-quantized4", torch.bfloat16, 1, 8, 8, 2000, 137, 128, 0, 1),
    ("h2o-vlen-default", torch.float16, 1, 6, 2, 900, 641, 128, 0, 1),
    ("qh2o-vlen-torch-quantized4", torch.bfloat16, 1, 8, 8, 1200, 900, 128, 0, 4),
    ("qh2o-vlen-torch-quantized8", torch.bfloat16, 1, 16, 8, 1100, 1030, 128, 0, 4),
    ("qh2o-vlen-torch-quantized8", torch.bfloat16, 1, 8, 2, 400, 300, 256, 0, 5),
])
def test_first_chunk_in_one_launch(kvx, gpu, name, dtype, B, Hq, Hkv, T, num, D, one, splits):
    gen = torch.Generator().manual_seed(num)
    q, k, v = (randn(gen, B, h, num, D, dtype=dtype).to(gpu) for h in (Hq, Hkv, Hkv))
    k, v = k.transpose(1, 2).contiguous().transpose(1, 2), v  # a token's heads side by side, and rows side by side
    got = []
    for fused in (True, False):
        cache = create_kv_cache(name, KVCacheParams(B, Hkv, T, D, Hq, dtype))
        assert route(kvx, cache, q, k, v) == (one, splits)
        tensors = [getattr(cache, n, None) for n in ("k", "v", "k_scale", "k_zp", "v_scale", "v_zp", "token_pos", "scores", "v_norm", "q_errors")]
        tensors = [t for t in tensors if t is not None]
        for t in tensors:
            t.fill_(7)
        if fused:
            out = cache.forward(q, k, v)
        else:  # what the one launch stands for
            cache.batch_size = B
            index = cache._run_of_slots(0, num)
            _lib.host().cache_write_first(cache, index, k, v) if num < T else cache._write(index, k, v, 0)
            out = _lib.host().prefill(q, k, v, cache.scale_factor, 0, None, False, False, True, None, 0, False)[0].view(B, num, Hq * D)
        got.append([out] + tensors)
    assert all(torch.equal(x, y) for x, y in zip(*got))


def test_refusals(kvx):
    a, w = _lib.SdpaArgs(), _lib.CacheWriteArgs()
    assert kvx.kvx_sdpa_prefill_first(ctypes.byref(a), ctypes.byref(w), None) == _lib.KVX_ERR_INVALID  # nothing set
