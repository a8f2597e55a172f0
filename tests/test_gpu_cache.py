"""GPU parity of the cache kernels (quantiser, slot write, H2O update/selection, the H2O cache step)
against the CPU oracle, through the C ABI."""
import ctypes
import math

import pytest
import torch

from helpers import make_qkv, rel_err, scattered_positions
from keys_values_amd import _lib
from keys_values_amd.attention import ops
from keys_values_amd.kvcache.h2o import H2OKVCache, KVCacheParams
from keys_values_amd.kvcache.quantize import RowQuantizer8
from oracle import kvx_oracle as O

pytestmark = pytest.mark.gpu


def outlier_rows(seed, rows, D):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, D, generator=gen)
    mask = torch.rand(rows, D, generator=gen) < 0.01
    return torch.where(mask, torch.randn(rows, D, generator=gen) * 8, x).to(torch.bfloat16)


def gpu_quantize(lib, x_gpu):
    rows, D = x_gpu.shape
    codes = torch.empty((rows, D), dtype=torch.uint8, device=x_gpu.device)
    sc = torch.empty(rows, dtype=torch.float32, device=x_gpu.device)
    zp = torch.empty(rows, dtype=torch.int32, device=x_gpu.device)
    _lib.check(lib.kvx_quantize_rows(x_gpu.data_ptr(), x_gpu.stride(0), rows, D, codes.data_ptr(), sc.data_ptr(), zp.data_ptr(),
                                      _lib.stream_ptr(x_gpu.device)))
    return codes, sc, zp


@pytest.mark.parametrize("rows,D", [(1, 128), (7, 64), (1000, 128), (4099, 64), (65536, 128), (8 * 65536, 128)])
def test_quantize_rows_bit_exact(kvx, gpu, rows, D):
    x = outlier_rows(2, rows, D)
    if rows >= 7:  # edge rows: constant, all negative, tiny range, extremes of bf16 dynamics
        x[0] = 0.0
        x[1] = -3.5
        x[2] = torch.linspace(-1e-3, 1e-3, D).to(torch.bfloat16)
        x[3] = torch.linspace(100.0, 101.0, D).to(torch.bfloat16)
        x[4] = 7.0
        x[5, ::2] = -1e4
    c_ref, s_ref, z_ref = O.quantize_rows(x)
    codes, sc, zp = gpu_quantize(kvx, x.to(gpu))
    torch.cuda.synchronize()
    assert torch.equal(sc.cpu(), s_ref), "scales differ"
    assert torch.equal(zp.cpu(), z_ref), "zero points differ"
    assert torch.equal(codes.cpu(), c_ref), "codes differ"
    out = torch.empty((rows, D), dtype=torch.bfloat16, device=gpu)
    _lib.check(kvx.kvx_dequantize_rows(codes.data_ptr(), sc.data_ptr(), zp.data_ptr(), rows, D, out.data_ptr(), D, _lib.stream_ptr(gpu)))
    torch.cuda.synchronize()
    assert torch.equal(out.cpu(), O.dequantize_rows(c_ref, s_ref, z_ref, torch.bfloat16)), "dequantised rows differ"


@pytest.mark.parametrize("bits,rows,D", [(8, 1000, 128), (8, 77, 64), (4, 1000, 128), (4, 5, 64)])
def test_quantize_rows_of_float16_bit_exact(kvx, gpu, bits, rows, D):
    """The typed entry points on float16 rows (a float16 model's store): the quantiser upcasts to fp32 and casts the
    dequantised values back to the rows' type (keys_values/kvcache/quantize/pytorch.py:333,478)."""
    x = outlier_rows(5, rows, D).to(torch.float16)
    x[0] = 0.0
    x[1] = -3.5
    x[2] = torch.linspace(100.0, 101.0, D).to(torch.float16)
    c_ref, s_ref, z_ref = O.quantize_rows(x, bits)
    xg = x.to(gpu)
    st = _lib.stream_ptr(gpu)
    codes = torch.empty((rows, D * bits // 8), dtype=torch.uint8, device=gpu)
    sc = torch.empty(rows, dtype=torch.float32, device=gpu)
    zp = torch.empty(rows, dtype=torch.int32, device=gpu)
    _lib.check(kvx.kvx_quantize_rows_typed(xg.data_ptr(), D, rows, D, bits, _lib.KVX_KV_F16, codes.data_ptr(), sc.data_ptr(), zp.data_ptr(), st))
    out = torch.empty((rows, D), dtype=torch.float16, device=gpu)
    _lib.check(kvx.kvx_dequantize_rows_typed(codes.data_ptr(), sc.data_ptr(), zp.data_ptr(), rows, D, bits, _lib.KVX_KV_F16, out.data_ptr(), D, st))
    torch.cuda.synchronize()
    assert torch.equal(sc.cpu(), s_ref) and torch.equal(zp.cpu(), z_ref), "row state differs"
    assert torch.equal(codes.cpu(), O.compress4(c_ref) if bits == 4 else c_ref), "codes differ"
    assert torch.equal(out.cpu(), O.dequantize_rows(c_ref, s_ref, z_ref, torch.float16)), "dequantised rows differ"
    with pytest.raises(NotImplementedError):
        _lib.check(kvx.kvx_quantize_rows_typed(xg.data_ptr(), D, rows, D, bits, _lib.KVX_KV_U8, codes.data_ptr(), sc.data_ptr(), zp.data_ptr(), st))


@pytest.mark.parametrize("bits", [8, 4])
def test_quantize_row_with_nan(kvx, gpu, bits):
    """torch.aminmax gives NaN extremes for a row that holds a NaN (keys_values/kvcache/quantize/pytorch.py:90),
    so the row's scale is NaN and the row dequantises to NaN throughout; what its zero point and codes are
    is a float-to-integer conversion of NaN, which the reference leaves to the platform: not compared.
    Rows without a NaN are untouched by their neighbours."""
    rows, D = 64, 128
    x = outlier_rows(5, rows, D)
    x[3, 17] = float("nan")
    x[40, 0] = float("nan")
    x[41, D - 1] = -float("nan")
    bad = torch.tensor([3, 40, 41])
    good = torch.tensor([r for r in range(rows) if r not in (3, 40, 41)])
    c_ref, s_ref, z_ref = O.quantize_rows(x, bits)
    assert torch.isnan(s_ref[bad]).all() and not torch.isnan(s_ref[good]).any()
    xg = x.to(gpu)
    codes = torch.empty((rows, D if bits == 8 else D // 2), dtype=torch.uint8, device=gpu)
    sc = torch.empty(rows, dtype=torch.float32, device=gpu)
    zp = torch.empty(rows, dtype=torch.int32, device=gpu)
    fn = kvx.kvx_quantize_rows if bits == 8 else kvx.kvx_quantize_rows4
    _lib.check(fn(xg.data_ptr(), D, rows, D, codes.data_ptr(), sc.data_ptr(), zp.data_ptr(), _lib.stream_ptr(gpu)))
    out = torch.empty((rows, D), dtype=torch.bfloat16, device=gpu)
    dq = kvx.kvx_dequantize_rows if bits == 8 else kvx.kvx_dequantize_rows4
    _lib.check(dq(codes.data_ptr(), sc.data_ptr(), zp.data_ptr(), rows, D, out.data_ptr(), D, _lib.stream_ptr(gpu)))
    torch.cuda.synchronize()
    assert torch.isnan(sc.cpu()[bad]).all()
    assert torch.isnan(out.cpu()[bad].float()).all()
    want_codes = O.compress4(c_ref) if bits == 4 else c_ref
    assert torch.equal(sc.cpu()[good], s_ref[good]) and torch.equal(zp.cpu()[good], z_ref[good])
    assert torch.equal(codes.cpu()[good], want_codes[good])
    assert torch.equal(out.cpu()[good], O.dequantize_rows(c_ref, s_ref, z_ref)[good])


def test_quantize_empty_and_strided(kvx, gpu):
    assert kvx.kvx_quantize_rows(None, 128, 0, 128, None, None, None, None) == 0
    x = outlier_rows(4, 300, 256).to(gpu)  # rows of 128 inside rows of 256
    codes, sc, zp = gpu_quantize(kvx, x[:, :128])
    c_ref, s_ref, z_ref = O.quantize_rows(x[:, :128].cpu())
    assert torch.equal(codes.cpu(), c_ref) and torch.equal(sc.cpu(), s_ref) and torch.equal(zp.cpu(), z_ref)


def test_row_quantizer_class_known_answer(gpu):
    # test/kvcache/test_quantization.py:647-766 through the Quantizer surface: integers 0..255 with
    # both extremes in every row survive a round trip exactly (bf16 holds them exactly)
    gen = torch.Generator().manual_seed(31415927)
    shape = (3, 4, 32, 64)
    data = torch.randint(0, 256, shape, generator=gen)
    i0 = torch.randint(0, 64, shape[:-1], generator=gen)
    i1 = (i0 + 1 + torch.randint(0, 63, shape[:-1], generator=gen)) % 64
    data.scatter_(-1, i0.unsqueeze(-1), 0)
    data.scatter_(-1, i1.unsqueeze(-1), 255)
    qz = RowQuantizer8(shape, torch.bfloat16, 8, allocate_buffers=True, device=gpu)
    assert qz.quant_buffer.shape == (12, 32, 64) and qz.quant_buffer.dtype == torch.uint8
    assert qz.quant_scales.dtype == torch.float32 and qz.quant_zero_points.dtype == torch.int32
    x = data.to(torch.bfloat16).to(gpu)
    qz.quantize(0, 32, x)
    assert torch.equal(qz.dequantize(0, 32), x)
    assert torch.equal(qz.quant_buffer.view(shape).cpu().long(), data)
    # partial range write keeps the other slots
    x2 = (data[:, :, 5:9] // 2).to(torch.bfloat16).to(gpu)
    qz.quantize(5, 9, x2)
    back = qz.dequantize(0, 32)
    c_ref, s_ref, z_ref = O.quantize_rows(x2.cpu())
    assert torch.equal(back[:, :, 5:9].cpu(), O.dequantize_rows(c_ref, s_ref, z_ref))
    assert torch.equal(back[:, :, :5], x[:, :, :5]) and torch.equal(back[:, :, 9:], x[:, :, 9:])
    err = qz.quantization_error(x2)
    torch.testing.assert_close(err.cpu(), O.quantization_error(x2.cpu()), rtol=1e-5, atol=1e-6)
    with pytest.raises(ValueError):
        qz.quantize(0, 4, x)
    with pytest.raises(NotImplementedError):
        RowQuantizer8(shape, torch.bfloat16, 4)


def run_cache_write(kvx, gpu, quantized):
    B, Hkv, L, D, num, input_pos = 2, 3, 50, 128, 7, 90
    gen = torch.Generator().manual_seed(17)
    kc = torch.randn(B, Hkv, L, D, generator=gen).to(torch.bfloat16)
    vc = torch.randn(B, Hkv, L, D, generator=gen).to(torch.bfloat16)
    key = torch.randn(B, Hkv, num, D, generator=gen).to(torch.bfloat16)
    val = torch.randn(B, Hkv, num, D, generator=gen).to(torch.bfloat16)
    tp = torch.randint(0, 90, (B, Hkv, L), generator=gen, dtype=torch.int32)
    sc = torch.rand(B, Hkv, L, generator=gen)
    index = torch.stack([torch.randperm(L, generator=gen)[:num] for _ in range(B * Hkv)]).view(B, Hkv, num)
    k_ref, v_ref, tp_ref, sc_ref = kc.clone(), vc.clone(), tp.clone(), sc.clone()
    O.cache_write(k_ref, v_ref, tp_ref, sc_ref, index, key, val, input_pos)
    a = _lib.CacheWriteArgs()
    a.B, a.Hkv, a.num, a.D, a.cache_len, a.input_pos = B, Hkv, num, D, L, input_pos
    idx32 = index.to(torch.int32).to(gpu)
    key_g, val_g, tp_g, sc_g = key.to(gpu), val.to(gpu), tp.to(gpu), sc.to(gpu)
    a.index, a.index_stride_b, a.index_stride_h = idx32.data_ptr(), idx32.stride(0), idx32.stride(1)
    a.key, a.key_stride_b, a.key_stride_h, a.key_stride_t = key_g.data_ptr(), *key_g.stride()[:3]
    a.value, a.value_stride_b, a.value_stride_h, a.value_stride_t = val_g.data_ptr(), *val_g.stride()[:3]
    a.token_pos, a.tp_stride_b, a.tp_stride_h = tp_g.data_ptr(), tp_g.stride(0), tp_g.stride(1)
    a.scores, a.sc_stride_b, a.sc_stride_h = sc_g.data_ptr(), sc_g.stride(0), sc_g.stride(1)
    if not quantized:
        a.kv_dtype = _lib.KVX_KV_BF16
        kc_g, vc_g = kc.to(gpu), vc.to(gpu)
    else:
        a.kv_dtype = _lib.KVX_KV_U8
        qk, qv = O.quantize_rows(kc), O.quantize_rows(vc)
        kc_g, vc_g = qk[0].to(gpu), qv[0].to(gpu)
        ks_g, kz_g, vs_g, vz_g = qk[1].to(gpu), qk[2].to(gpu), qv[1].to(gpu), qv[2].to(gpu)
        a.k_scale, a.k_zp, a.v_scale, a.v_zp = ks_g.data_ptr(), kz_g.data_ptr(), vs_g.data_ptr(), vz_g.data_ptr()
        a.qs_stride_b, a.qs_stride_h = ks_g.stride(0), ks_g.stride(1)
    a.k_cache, a.kc_stride_b, a.kc_stride_h, a.kc_stride_t = kc_g.data_ptr(), *kc_g.stride()[:3]
    a.v_cache, a.vc_stride_b, a.vc_stride_h, a.vc_stride_t = vc_g.data_ptr(), *vc_g.stride()[:3]
    _lib.check(kvx.kvx_cache_write(ctypes.byref(a), _lib.stream_ptr(gpu)))
    torch.cuda.synchronize()
    assert torch.equal(tp_g.cpu(), tp_ref) and torch.equal(sc_g.cpu(), sc_ref)
    if not quantized:
        assert torch.equal(kc_g.cpu(), k_ref) and torch.equal(vc_g.cpu(), v_ref)
    else:
        for got, ref in (((kc_g, ks_g, kz_g), k_ref), ((vc_g, vs_g, vz_g), v_ref)):
            c_ref, s_ref, z_ref = O.quantize_rows(ref)  # rows not written keep their old codes
            assert torch.equal(got[0].cpu(), c_ref) and torch.equal(got[1].cpu(), s_ref) and torch.equal(got[2].cpu(), z_ref)


def test_cache_write_bf16(kvx, gpu):
    run_cache_write(kvx, gpu, False)


def test_cache_write_uint8(kvx, gpu):
    run_cache_write(kvx, gpu, True)


def gpu_h2o(kvx, gpu, scores, w, kv_len, limit, k, normalize=False, token_pos=None, input_pos=0, prefill_len=0):
    B, Hkv, L = scores.shape
    sc_g = scores.to(gpu)
    w_g = None if w is None else w.contiguous().to(gpu)
    tp_g = None if token_pos is None else token_pos.to(torch.int32).to(gpu)
    nxt = torch.empty((B, Hkv, k), dtype=torch.int32, device=gpu)
    a = _lib.H2OArgs()
    a.B, a.Hkv, a.kv_len, a.limit, a.k = B, Hkv, kv_len, limit, k
    a.normalize, a.input_pos, a.prefill_len = int(normalize), input_pos, prefill_len
    a.scores, a.sc_stride_b, a.sc_stride_h = sc_g.data_ptr(), sc_g.stride(0), sc_g.stride(1)
    a.w = _lib.ptr(w_g)
    if tp_g is not None:
        a.token_pos, a.tp_stride_b, a.tp_stride_h = tp_g.data_ptr(), tp_g.stride(0), tp_g.stride(1)
    a.next_index = nxt.data_ptr()
    nb = kvx.kvx_h2o_workspace_bytes(ctypes.byref(a))
    ws = torch.empty(max(nb, 8), dtype=torch.uint8, device=gpu)
    a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
    _lib.check(kvx.kvx_h2o_update_select(ctypes.byref(a), _lib.stream_ptr(gpu)))
    torch.cuda.synchronize()
    return sc_g.cpu(), nxt.cpu()


@pytest.mark.parametrize("B,Hkv,L,kv_len,limit,k", [
    (2, 3, 300, 300, 300, 1), (8, 8, 5000, 5000, 5000, 1), (1, 2, 1024, 1024, 1024, 128), (2, 2, 4097, 4000, 3999, 1000),
    (1, 8, 16384, 16384, 16384, 1024), (1, 1, 64, 64, 64, 64), (1, 2, 131072, 131072, 131072, 4096), (2, 2, 10001, 10001, 10001, 1),
    # more than one launch of 4096 slots, up to the whole argsort (keys_values/kvcache/attn_weights.py:773-774)
    (1, 2, 20000, 20000, 20000, 9000), (2, 1, 8192, 8192, 8192, 8192), (1, 2, 131072, 131072, 131000, 131000), (1, 1, 5000, 4999, 4500, 4097),
])
def test_h2o_update_select(kvx, gpu, B, Hkv, L, kv_len, limit, k):
    gen = torch.Generator().manual_seed(L + k)
    scores = torch.rand(B, Hkv, L, generator=gen) * 3
    w = torch.rand(B, Hkv, kv_len, generator=gen)
    s_ref = scores.clone()
    n_ref = O.h2o_update_select(s_ref, w, kv_len, limit, k)
    s_gpu, n_gpu = gpu_h2o(kvx, gpu, scores, w, kv_len, limit, k)
    assert torch.equal(s_gpu, s_ref), "scores += w differs"
    assert torch.equal(n_gpu.long(), n_ref), "selected slots differ"


def test_h2o_select_ties_and_no_weights(kvx, gpu):
    # many exact ties (quantised scores), zeros and negative zeros: lower slot first, like a stable argsort
    gen = torch.Generator().manual_seed(3)
    scores = torch.randint(0, 6, (2, 2, 999), generator=gen).float() * 0.25
    scores[0, 0, 100:140] = 0.0
    scores[0, 0, 120] = -0.0
    for k in (1, 50, 333):
        s_ref = scores.clone()
        n_ref = O.h2o_update_select(s_ref, None, 999, 999, k)
        s_gpu, n_gpu = gpu_h2o(kvx, gpu, scores, None, 999, 999, k)
        assert torch.equal(n_gpu.long(), n_ref)
        assert torch.equal(s_gpu, scores)


def test_h2o_select_ties_across_launches(kvx, gpu):
    # a selection of several launches whose cuts fall inside long runs of equal scores: the order within a
    # run is by slot, and a run is continued, not repeated, by the next launch
    gen = torch.Generator().manual_seed(8)
    scores = torch.randint(0, 4, (2, 2, 12000), generator=gen).float()
    for k in (4096, 4097, 9000, 12000):
        s_ref = scores.clone()
        n_ref = O.h2o_update_select(s_ref, None, 12000, 12000, k)
        _, n_gpu = gpu_h2o(kvx, gpu, scores, None, 12000, 12000, k)
        assert torch.equal(n_gpu.long(), n_ref), k


def test_cache_selects_again_when_asked_for_more(gpu):
    """No max_chunk_size: the reference keeps the whole argsort and serves any chunk up to the cache length
    (keys_values/kvcache/attn_weights.py:501-508,773-774). The cache chooses one slot after a single-token
    step and selects again when a longer chunk follows."""
    B, Hq, Hkv, L, D = 1, 2, 1, 10000, 64
    gen = torch.Generator().manual_seed(12)
    total = L + 1 + 1 + 6000 + 1
    qs = torch.randn(B, Hq, total, D, generator=gen).to(torch.bfloat16)
    ks = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16)
    vs = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16)
    ref = O.H2OCacheOracle(B, Hq, Hkv, L, D, dtype=torch.bfloat16, max_chunk_size=None)
    cache = H2OKVCache(KVCacheParams(B, Hkv, L, D, Hq), max_chunk_size=None, device=gpu)
    ref.prefill(qs[:, :, :L], ks[:, :, :L], vs[:, :, :L])
    cache.forward(qs[:, :, :L].to(gpu), ks[:, :, :L].to(gpu), vs[:, :, :L].to(gpu))
    pos = L
    for num in (1, 1, 6000, 1):
        assert cache.max_forward_length() == L
        sl = slice(pos, pos + num)
        had = ref.next_index is not None
        if had:
            want = ref.next_index[:, :, :num]
            got = cache.next_positions(num).cpu()
            assert got.shape == want.shape
            _sets_equal_away_from_ties(got, want, ref.scores, num)
            cache.set_next_positions(want)  # stay on the oracle's slots
        o_ref, _, _ = ref.forward(qs[:, :, sl], ks[:, :, sl], vs[:, :, sl])
        o = cache.forward(qs[:, :, sl].to(gpu), ks[:, :, sl].to(gpu), vs[:, :, sl].to(gpu))
        torch.cuda.synchronize()
        assert rel_err(o.float().cpu().view(B, num, Hq, D).transpose(1, 2), o_ref.float()) < 2e-2
        assert torch.equal(cache.token_pos.cpu(), ref.token_pos)
        torch.testing.assert_close(cache.scores.cpu(), ref.scores, rtol=2e-3, atol=1e-5)
        pos += num


def test_h2o_select_normalized(kvx, gpu):
    # keys_values/kvcache/h2o.py:183-196
    gen = torch.Generator().manual_seed(4)
    B, Hkv, L = 2, 2, 777
    scores = torch.rand(B, Hkv, L, generator=gen) * 5
    w = torch.rand(B, Hkv, L, generator=gen)
    tp = torch.stack([torch.randperm(2000, generator=gen)[:L] for _ in range(B * Hkv)]).view(B, Hkv, L).to(torch.int32)
    for k in (1, 64):
        s_ref = scores.clone()
        n_ref = O.h2o_update_select(s_ref, w, L, L, k, normalize=True, token_pos=tp, input_pos=2100, prefill_len=512)
        s_gpu, n_gpu = gpu_h2o(kvx, gpu, scores, w, L, L, k, True, tp, 2100, 512)
        assert torch.equal(s_gpu, s_ref)
        assert torch.equal(n_gpu.long(), n_ref)


def _sets_equal_away_from_ties(n_gpu, n_ref, scores_ref, k):
    """Selected sets must agree unless the cut falls between numerically indistinguishable scores
    (GPU and CPU scores differ in the last bits)."""
    for b in range(n_ref.shape[0]):
        for h in range(n_ref.shape[1]):
            a, r = set(n_gpu[b, h, :k].tolist()), set(n_ref[b, h, :k].tolist())
            if a != r:
                srt = torch.sort(scores_ref[b, h]).values
                gap = (srt[k] - srt[k - 1]).item()
                diff = a ^ r
                assert gap < 1e-3 * max(srt[k].item(), 1e-6) or all(
                    abs(scores_ref[b, h, i].item() - srt[k - 1].item()) < 2e-3 * max(srt[k].item(), 1e-6) for i in diff
                ), f"selection differs away from a tie at ({b},{h}): {sorted(diff)}"


@pytest.mark.parametrize("quantized,dtype,bits,D", [(False, torch.bfloat16, 8, 64), (True, torch.bfloat16, 8, 64), (True, torch.float16, 8, 64),
                                                     (True, torch.float16, 4, 64), (True, torch.bfloat16, 8, 256), (True, torch.float16, 4, 256)])
def test_h2o_cache_steps_vs_oracle(gpu, quantized, dtype, bits, D):
    """Prefill that fills the cache, then chunked steps: initial rule, evict-write, attention with
    scattered positions, score accumulation, selection (configuration 1 shapes: 8/2 heads, D 64,
    1024 slots, 128-token chunks). With the uint8 store every row is quantised once, when written,
    so the oracle is fed the dequantised rows: what the reference's attention reads from its
    dequantised working buffer (keys_values/kvcache/quant_buffers.py:776-793)."""
    B, Hq, Hkv, L, chunk = 1, 8, 2, 1024, 128
    gen = torch.Generator().manual_seed(0)
    total = L + 4 * chunk
    qs = torch.randn(B, Hq, total, D, generator=gen).to(dtype)
    ks = torch.randn(B, Hkv, total, D, generator=gen).to(dtype)
    vs = torch.randn(B, Hkv, total, D, generator=gen).to(dtype)
    ks_o = O.dequantize_rows(*O.quantize_rows(ks, bits), dtype) if quantized else ks
    vs_o = O.dequantize_rows(*O.quantize_rows(vs, bits), dtype) if quantized else vs
    ref = O.H2OCacheOracle(B, Hq, Hkv, L, D, dtype=dtype, max_chunk_size=chunk)
    cache = H2OKVCache(KVCacheParams(B, Hkv, L, D, Hq, dtype), max_chunk_size=chunk, quantized=quantized, num_bits=bits, device=gpu)
    codes_of = O.uncompress4 if bits == 4 else (lambda c: c)
    ref.prefill(qs[:, :, :L], ks_o[:, :, :L], vs_o[:, :, :L])
    # the first chunk attends over the keys/values as given, not over the store (kvcache/base.py:567-571)
    o_ref, _ = O.sdpa_in_blocks(qs[:, :, :L], ks[:, :, :L], vs[:, :, :L], 1 / math.sqrt(D), 0, None, return_attn_weights=False)
    o = cache.forward(qs[:, :, :L].to(gpu), ks[:, :, :L].to(gpu), vs[:, :, :L].to(gpu))
    assert rel_err(o.float().cpu().view(B, L, Hq, D).transpose(1, 2), o_ref.float()) < 2e-2
    assert cache.next_positions(chunk)[0, 0].tolist() == list(range(51, 51 + chunk))  # int(0.05 * 1024) = 51
    pos = L
    for step in range(4):
        sl = slice(pos, pos + chunk)
        o_ref, w_ref, index = ref.forward(qs[:, :, sl], ks_o[:, :, sl], vs_o[:, :, sl])
        if step > 0:
            # write to the oracle's slots so that the two caches stay comparable step after step
            # (the GPU's own choice is checked below)
            cache.set_next_positions(index)
        o = cache.forward(qs[:, :, sl].to(gpu), ks[:, :, sl].to(gpu), vs[:, :, sl].to(gpu))
        torch.cuda.synchronize()
        assert cache.input_pos == ref.input_pos
        assert torch.equal(cache.token_pos.cpu(), ref.token_pos)
        assert rel_err(o.float().cpu().view(B, chunk, Hq, D).transpose(1, 2), o_ref.float()) < 2e-2
        torch.testing.assert_close(cache.scores.cpu(), ref.scores, rtol=2e-3, atol=1e-5)
        if quantized:
            assert torch.equal(O.dequantize_rows(codes_of(cache.k.cpu()), cache.k_scale.cpu(), cache.k_zp.cpu(), dtype), ref.k)
            assert torch.equal(O.dequantize_rows(codes_of(cache.v.cpu()), cache.v_scale.cpu(), cache.v_zp.cpu(), dtype), ref.v)
        else:
            assert torch.equal(cache.k.cpu(), ref.k) and torch.equal(cache.v.cpu(), ref.v)
        _sets_equal_away_from_ties(cache._next_index[:B].cpu().long(), ref.next_index, ref.scores, chunk)
        pos += chunk
    if quantized:  # single-token steps over the quantised store (the fused decode + H2O call)
        extra = torch.Generator().manual_seed(99)
        for _ in range(3):
            q1 = torch.randn(B, Hq, 1, D, generator=extra).to(dtype)
            k1 = torch.randn(B, Hkv, 1, D, generator=extra).to(dtype)
            v1 = torch.randn(B, Hkv, 1, D, generator=extra).to(dtype)
            k1o, v1o = O.dequantize_rows(*O.quantize_rows(k1, bits), dtype), O.dequantize_rows(*O.quantize_rows(v1, bits), dtype)
            o_ref, w_ref, index = ref.forward(q1, k1o, v1o)
            cache.set_next_positions(index)
            o = cache.forward(q1.to(gpu), k1.to(gpu), v1.to(gpu))
            assert o.dtype == dtype
            assert rel_err(o.float().cpu().view(B, 1, Hq, D).transpose(1, 2), o_ref.float()) < 2e-2
            torch.testing.assert_close(cache.scores.cpu(), ref.scores, rtol=2e-3, atol=1e-5)


@pytest.mark.parametrize("Hq,Hkv", [(8, 2), (6, 2), (7, 1)])
def test_h2o_cache_decode_steps(gpu, Hq, Hkv):
    # single-token steps: argmin selection, slot reuse, scores = running sum (test/kvcache/test_h2o.py:109-137);
    # group sizes 4, 3 and 7 (the fused decode step pads the last two to 4 and 8 heads inside the kernel)
    B, L, D = 2, 256, 128
    gen = torch.Generator().manual_seed(3)
    total = L + 6
    qs = torch.randn(B, Hq, total, D, generator=gen).to(torch.bfloat16)
    ks = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16)
    vs = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16)
    ref = O.H2OCacheOracle(B, Hq, Hkv, L, D, dtype=torch.bfloat16, max_chunk_size=1)
    cache = H2OKVCache(KVCacheParams(B, Hkv, L, D, Hq), max_chunk_size=1, device=gpu)
    ref.prefill(qs[:, :, :L], ks[:, :, :L], vs[:, :, :L])
    cache.forward(qs[:, :, :L].to(gpu), ks[:, :, :L].to(gpu), vs[:, :, :L].to(gpu))
    for t in range(L, total):
        sl = slice(t, t + 1)
        o_ref, w_ref, index = ref.forward(qs[:, :, sl], ks[:, :, sl], vs[:, :, sl])
        if t > L:
            assert torch.equal(cache.next_positions(1).cpu(), index), "evicted slot differs"
        o = cache.forward(qs[:, :, sl].to(gpu), ks[:, :, sl].to(gpu), vs[:, :, sl].to(gpu))
        torch.cuda.synchronize()
        assert rel_err(o.float().cpu().view(B, 1, Hq, D).transpose(1, 2), o_ref.float()) < 2e-2
        torch.testing.assert_close(cache.scores.cpu(), ref.scores, rtol=2e-3, atol=1e-5)
        assert torch.equal(cache.token_pos.cpu(), ref.token_pos)


def test_attention_over_uint8_cache(kvx, gpu):
    """Configuration 3 semantics at a reduced size: K with 1% outliers, quantised on the GPU,
    attention + score-sums with dequantisation fused into the loads, against the oracle run on the
    dequantised bf16 cache."""
    B, Hq, Hkv, q_len, T, D = 1, 8, 2, 96, 2048 + 40, 128
    gen = torch.Generator().manual_seed(2)
    k = outlier_rows(2, B * Hkv * T, D).view(B, Hkv, T, D)
    v = torch.randn(B, Hkv, T, D, generator=gen).to(torch.bfloat16)
    q = torch.randn(B, Hq, q_len, D, generator=gen).to(torch.bfloat16)
    input_pos = T - q_len
    kc, ks, kz = gpu_quantize(kvx, k.view(-1, D).to(gpu))
    vc, vs, vz = gpu_quantize(kvx, v.view(-1, D).to(gpu))
    quant = ops.QuantState(ks.view(B, Hkv, T), kz.view(B, Hkv, T), vs.view(B, Hkv, T), vz.view(B, Hkv, T))
    kd = O.dequantize_rows(*O.quantize_rows(k))
    vd = O.dequantize_rows(*O.quantize_rows(v))
    scale = 1 / math.sqrt(D)
    o_ref, w_ref = O.sdpa_in_blocks(q, kd, vd, scale, input_pos, None)
    out, w, _ = ops.prefill_core(q.to(gpu), kc.view(B, Hkv, T, D), vc.view(B, Hkv, T, D), scale, input_pos, None,
                                 return_weights=True, quant=quant, output_transposed=False)
    torch.cuda.synchronize()
    assert rel_err(out.float().cpu(), o_ref.float()) < 2e-2
    torch.testing.assert_close(w.cpu(), w_ref, rtol=1e-3, atol=1e-6)
    # decode over the same store
    o1_ref, w1_ref = O.sdpa_in_blocks(q[:, :, :1], kd, vd, scale, T - 1, None)
    out1, w1, _ = ops.decode_core(q[:, :, :1].to(gpu), kc.view(B, Hkv, T, D), vc.view(B, Hkv, T, D), scale, return_weights=True, quant=quant)
    torch.cuda.synchronize()
    assert rel_err(out1.float().cpu().unsqueeze(2), o1_ref.float()) < 2e-2
    torch.testing.assert_close(w1.cpu(), w1_ref, rtol=1e-3, atol=1e-6)


@pytest.mark.parametrize("B,Hq,Hkv,T,D,limit,normalize,quantized", [
    (2, 8, 2, 1000, 128, 1000, False, False),
    (1, 4, 4, 777, 64, 700, True, False),
    (2, 8, 1, 4096 + 33, 128, 4096, True, True),
    (1, 2, 1, 17, 64, 17, False, True),
    (2, 6, 2, 600, 128, 600, False, False),
    (1, 5, 1, 300, 64, 256, True, True),
    (1, 8, 2, 12000, 128, 11000, True, False),
    (1, 16, 1, 2100, 128, 2000, False, True),   # 16 heads per KV head over the 8-bit store
    (1, 12, 1, 900, 64, 900, True, False),
    (2, 32, 4, 5000, 128, 5000, False, True),   # 8 heads per KV head, 8-bit store, several splits per row
    (16, 16, 16, 2500, 64, 2400, True, False),  # one split a row
    (8, 16, 8, 4500, 64, 4500, False, True),    # splits of more keys than four a thread
])
def test_fused_decode_h2o_matches_separate_calls(kvx, gpu, decode_route, B, Hq, Hkv, T, D, limit, normalize, quantized):
    """kvx_sdpa_decode_h2o == kvx_sdpa_decode (with weights) followed by kvx_h2o_update_select(k=1),
    and both match the oracle."""
    q, k, v, _ = make_qkv(50 + T, B, Hq, Hkv, 1, T, D)
    gen = torch.Generator().manual_seed(T)
    scores = torch.rand(B, Hkv, T, generator=gen) * 2
    tp = torch.stack([torch.randperm(3 * T, generator=gen)[:T] for _ in range(B * Hkv)]).view(B, Hkv, T).to(torch.int32)
    input_pos, prefill_len = 3 * T + 5, T // 2
    scale = 1.0 / math.sqrt(D)
    quant = None
    kg, vg = k.to(gpu), v.to(gpu)
    if quantized:
        kc, ks, kz = O.quantize_rows(k.reshape(-1, D))
        vc, vs, vz = O.quantize_rows(v.reshape(-1, D))
        k = O.dequantize_rows(kc, ks, kz).view(B, Hkv, T, D)
        v = O.dequantize_rows(vc, vs, vz).view(B, Hkv, T, D)
        kg, vg = kc.view(B, Hkv, T, D).to(gpu), vc.view(B, Hkv, T, D).to(gpu)
        quant = ops.QuantState(ks.view(B, Hkv, T).to(gpu), kz.view(B, Hkv, T).to(gpu), vs.view(B, Hkv, T).to(gpu), vz.view(B, Hkv, T).to(gpu))
    # separate calls
    out_a, w_a, _ = ops.decode_core(q.to(gpu), kg, vg, scale, return_weights=True, quant=quant)
    s_a, n_a = gpu_h2o(kvx, gpu, scores, w_a.cpu(), T, limit, 1, normalize, tp, input_pos, prefill_len)
    # fused call
    qg = q.to(gpu)
    out_b = torch.empty((B, Hq, D), dtype=torch.bfloat16, device=gpu)
    ov = out_b.unsqueeze(2)
    sc_g, tp_g = scores.to(gpu), tp.to(gpu)
    nxt = torch.full((B, Hkv, 1), -1, dtype=torch.int32, device=gpu)
    a = _lib.SdpaArgs()
    ops._fill_common(a, qg, kg, vg, scale, T - 1, None, quant, 0)
    a.o, a.o_stride_b, a.o_stride_h, a.o_stride_t = ov.data_ptr(), ov.stride(0), ov.stride(1), ov.stride(2)
    h = _lib.H2OArgs()
    h.B, h.Hkv, h.kv_len, h.limit, h.k = B, Hkv, T, limit, 1
    h.normalize, h.input_pos, h.prefill_len = int(normalize), input_pos, prefill_len
    h.scores, h.sc_stride_b, h.sc_stride_h = sc_g.data_ptr(), sc_g.stride(0), sc_g.stride(1)
    h.token_pos, h.tp_stride_b, h.tp_stride_h = tp_g.data_ptr(), tp_g.stride(0), tp_g.stride(1)
    h.next_index = nxt.data_ptr()
    nb_h = (kvx.kvx_h2o_workspace_bytes(ctypes.byref(h)) + 255) // 256 * 256
    nb_a = kvx.kvx_sdpa_decode_h2o_workspace_bytes(ctypes.byref(a))
    ws = torch.empty(nb_h + nb_a + 256, dtype=torch.uint8, device=gpu)
    h.workspace, h.workspace_bytes = ws.data_ptr(), nb_h
    a.workspace, a.workspace_bytes = ws.data_ptr() + nb_h, nb_a
    _lib.check(kvx.kvx_sdpa_decode_h2o(ctypes.byref(a), ctypes.byref(h), _lib.stream_ptr(gpu)))
    torch.cuda.synchronize()
    assert torch.equal(out_b, out_a)
    assert torch.equal(sc_g.cpu(), s_a)
    assert torch.equal(nxt.cpu(), n_a)
    # oracle
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, T - 1, None)
    assert rel_err(out_b.float().cpu().unsqueeze(2), o_ref.float()) < 2e-2
    s_ref = scores.clone()
    n_ref = O.h2o_update_select(s_ref, w_ref, T, limit, 1, normalize=normalize, token_pos=tp, input_pos=input_pos, prefill_len=prefill_len)
    torch.testing.assert_close(sc_g.cpu(), s_ref, rtol=1e-3, atol=1e-6)
    _sets_equal_away_from_ties(nxt.cpu().long(), n_ref, (s_ref[..., :limit] / (input_pos - torch.maximum(tp, torch.tensor(prefill_len - 1)))[..., :limit].float()) if normalize else s_ref[..., :limit], 1)


def test_full_size_decode_h2o_properties(kvx, gpu):
    """Configuration 4 at its real shape (B8, 32/8 heads, D128, 131072 slots, 4.3 GB of bf16 K/V, byte
    offsets beyond 2^31): the fused decode + H2O step against the separate calls, the weights of a
    token sum to one, the scores grow by exactly the weights, the evicted slot holds the minimum, and
    the last (batch, KV head) pair — the largest offsets — against the oracle."""
    B, Hq, Hkv, T, D = 8, 32, 8, 131072, 128
    G = Hq // Hkv
    torch.manual_seed(3)
    k = torch.randn(B, Hkv, T, D, device=gpu, dtype=torch.bfloat16)
    v = torch.randn(B, Hkv, T, D, device=gpu, dtype=torch.bfloat16)
    q = torch.randn(B, Hq, 1, D, device=gpu, dtype=torch.bfloat16)
    scores0 = torch.rand(B, Hkv, T, device=gpu) * 0.01
    scale = 1.0 / math.sqrt(D)
    out_a, w_a, _ = ops.decode_core(q, k, v, scale, return_weights=True)
    out_b = torch.empty((B, Hq, D), dtype=torch.bfloat16, device=gpu)
    ov = out_b.unsqueeze(2)
    sc_g = scores0.clone()
    nxt = torch.full((B, Hkv, 1), -1, dtype=torch.int32, device=gpu)
    a = _lib.SdpaArgs()
    ops._fill_common(a, q, k, v, scale, T - 1, None, None, 0)
    a.o, a.o_stride_b, a.o_stride_h, a.o_stride_t = ov.data_ptr(), ov.stride(0), ov.stride(1), ov.stride(2)
    h = _lib.H2OArgs()
    h.B, h.Hkv, h.kv_len, h.limit, h.k = B, Hkv, T, T, 1
    h.scores, h.sc_stride_b, h.sc_stride_h = sc_g.data_ptr(), sc_g.stride(0), sc_g.stride(1)
    h.next_index = nxt.data_ptr()
    nb_h = (kvx.kvx_h2o_workspace_bytes(ctypes.byref(h)) + 255) // 256 * 256
    nb_a = kvx.kvx_sdpa_decode_h2o_workspace_bytes(ctypes.byref(a))
    ws = torch.empty(nb_h + nb_a + 256, dtype=torch.uint8, device=gpu)
    h.workspace, h.workspace_bytes = ws.data_ptr(), nb_h
    a.workspace, a.workspace_bytes = ws.data_ptr() + nb_h, nb_a
    _lib.check(kvx.kvx_sdpa_decode_h2o(ctypes.byref(a), ctypes.byref(h), _lib.stream_ptr(gpu)))
    torch.cuda.synchronize()
    assert torch.equal(out_b, out_a)
    assert (w_a >= 0).all()
    torch.testing.assert_close(w_a.sum(-1), torch.ones(B, Hkv, device=gpu), rtol=2e-5, atol=0)
    assert torch.equal(sc_g, scores0 + w_a)
    chosen = sc_g.gather(-1, nxt.long())
    assert torch.equal(chosen.squeeze(-1), sc_g.min(-1).values)
    b, kh = B - 1, Hkv - 1
    o_ref, w_ref = O.sdpa_in_blocks(q[b : b + 1, G * kh : G * kh + G].cpu(), k[b : b + 1, kh : kh + 1].cpu(), v[b : b + 1, kh : kh + 1].cpu(),
                                    scale, T - 1, None)
    assert rel_err(out_b[b, G * kh : G * kh + G].float().cpu(), o_ref[0, :, 0].float()) < 2e-2
    torch.testing.assert_close(w_a[b : b + 1, kh : kh + 1].cpu(), w_ref, rtol=1e-3, atol=1e-9)


@pytest.mark.parametrize("bits", [8, 4])
def test_chunk_over_dequantised_copy_equals_fused_dequantisation(gpu, bits):
    """Long chunks attend over a bf16 copy of the quantised store made once per chunk, short ones
    dequantise inside the kernels: same values either way, so outputs, scores and evicted slots agree
    (to summation order) and the store itself is bit-identical."""
    B, Hq, Hkv, L, D, chunk = 2, 8, 2, 1024, 128, 96
    steps = (96, 50, 96, 7, 96)
    gen = torch.Generator().manual_seed(77)
    total = L - 96 + sum(steps)
    q = torch.randn(B, Hq, total, D, generator=gen).to(torch.bfloat16).to(gpu)
    k = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16).to(gpu)
    v = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16).to(gpu)
    params = KVCacheParams(B, Hkv, L, D, Hq)
    copy = H2OKVCache(params, max_chunk_size=chunk, quantized=True, num_bits=bits, device=gpu, dequantize_chunk_rows=1)
    fused = H2OKVCache(params, max_chunk_size=chunk, quantized=True, num_bits=bits, device=gpu, dequantize_chunk_rows=None)
    n0 = L - 96  # the first step fills the cache exactly
    for c in (copy, fused):
        c.forward(q[:, :, :n0], k[:, :, :n0], v[:, :, :n0])
    pos = n0
    for num in steps:
        sl = slice(pos, pos + num)
        o1 = copy.forward(q[:, :, sl], k[:, :, sl], v[:, :, sl])
        o2 = fused.forward(q[:, :, sl], k[:, :, sl], v[:, :, sl])
        torch.cuda.synchronize()
        assert rel_err(o1.float().cpu(), o2.float().cpu()) < 1e-2
        torch.testing.assert_close(copy.scores, fused.scores, rtol=1e-3, atol=1e-6)
        assert torch.equal(copy.k, fused.k) and torch.equal(copy.v, fused.v) and torch.equal(copy.token_pos, fused.token_pos)
        if copy._have_next:
            fused.set_next_positions(copy._next_index)  # keep the two in step where scores tie in the last bits
        pos += num


def test_overlapped_selection_equals_in_order_selection(gpu):
    """overlap_select=True runs the score update + eviction choice on a second stream beside the
    caller's next launches; every result must equal the in-order cache's bit for bit."""
    B, Hq, Hkv, L, D, chunk = 1, 8, 2, 2048, 128, 128
    gen = torch.Generator().manual_seed(5)
    total = L + 6 * chunk
    qs = torch.randn(B, Hq, total, D, generator=gen).to(torch.bfloat16).to(gpu)
    ks = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16).to(gpu)
    vs = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16).to(gpu)
    a = H2OKVCache(KVCacheParams(B, Hkv, L, D, Hq), max_chunk_size=chunk, quantized=True, device=gpu)
    b = H2OKVCache(KVCacheParams(B, Hkv, L, D, Hq), max_chunk_size=chunk, quantized=True, device=gpu, overlap_select=True)
    busy = torch.randn(2048, 2048, device=gpu)
    for cache in (a, b):
        cache.forward(qs[:, :, :L], ks[:, :, :L], vs[:, :, :L])
    pos = L
    for step in range(6):
        sl = slice(pos, pos + chunk)
        oa = a.forward(qs[:, :, sl], ks[:, :, sl], vs[:, :, sl])
        ob = b.forward(qs[:, :, sl], ks[:, :, sl], vs[:, :, sl])
        for _ in range(3):  # the caller's own work, enqueued while the choice may still be running
            busy = (busy @ busy).clamp_(-1, 1)
        assert torch.equal(a.next_positions(chunk), b.next_positions(chunk))  # waits for the second stream
        torch.cuda.synchronize()
        assert torch.equal(oa, ob)
        assert torch.equal(a.scores, b.scores) and torch.equal(a.token_pos, b.token_pos)
        assert torch.equal(a.k, b.k) and torch.equal(a.v, b.v)
        pos += chunk


@pytest.mark.parametrize("bits,grace", [(8, 0), (4, 0), (8, 40)])
def test_overlapped_score_sum_pass_equals_in_order_pass(gpu, bits, grace):
    """Long chunks over a quantised store with overlap_select: the score-sum pass, the score update and the
    eviction choice all run on the second stream. Outputs, scores, stores and choices equal the in-order
    cache's bit for bit, also when the ring of recent tokens moves."""
    B, Hq, Hkv, L, D, chunk = 2, 8, 2, 1024, 128, 64
    gen = torch.Generator().manual_seed(123 + bits + grace)
    total = L + 6 * chunk
    qs = torch.randn(B, Hq, total, D, generator=gen).to(torch.bfloat16).to(gpu)
    ks = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16).to(gpu)
    vs = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16).to(gpu)
    params = KVCacheParams(B, Hkv, L, D, Hq)
    kw = dict(max_chunk_size=chunk, quantized=True, num_bits=bits, device=gpu, dequantize_chunk_rows=1, grace_period=grace)
    plain = H2OKVCache(params, **kw)
    beside = H2OKVCache(params, overlap_select=True, **kw)
    busy = torch.randn(1024, 1024, device=gpu)
    for cache in (plain, beside):
        cache.forward(qs[:, :, :L], ks[:, :, :L], vs[:, :, :L])
    pos = L
    for step in range(6):
        sl = slice(pos, pos + chunk)
        o1 = plain.forward(qs[:, :, sl], ks[:, :, sl], vs[:, :, sl])
        o2 = beside.forward(qs[:, :, sl], ks[:, :, sl], vs[:, :, sl])
        for _ in range(3):  # the caller's own work, enqueued while the second stream may still be running
            busy = (busy @ busy).clamp_(-1, 1)
        assert torch.equal(plain.next_positions(chunk), beside.next_positions(chunk))  # waits for the second stream
        torch.cuda.synchronize()
        assert torch.equal(o1, o2)
        assert torch.equal(plain.scores, beside.scores) and torch.equal(plain.token_pos, beside.token_pos)
        assert torch.equal(plain.k, beside.k) and torch.equal(plain.v, beside.v)
        pos += chunk


def _requantise_slots(ref, slots, bits, dtype):
    """What a write-back does to the oracle's rows: the slots ``slots`` (batch, n) of ref.k / ref.v, each a block
    over all heads, are quantised and dequantised (keys_values/kvcache/quant_buffers.py:732-775 with blocks over
    the heads, keys_values/kvcache/quantize/pytorch.py:235-245,334-337)."""
    B, Hkv, L, D = ref.k.shape
    n = slots.shape[1]
    gi = slots.view(B, 1, n, 1).expand(B, Hkv, n, D)
    for store in (ref.k, ref.v):
        rows = store.gather(2, gi)
        c, sc, z = O.quantize_store(rows, bits, True)
        store.scatter_(2, gi, O.dequantize_store(c, sc, z, (B, Hkv, n, D), bits, True, dtype).contiguous())


@pytest.mark.parametrize("bits,dtype,grace", [(8, torch.bfloat16, 0), (4, torch.bfloat16, 0), (8, torch.float16, 0)])
def test_h2o_cache_with_blocks_over_heads_vs_oracle(gpu, bits, dtype, grace):
    """The cache over a store whose quantisation blocks run over the heads: prefill that fills it, chunk steps with
    slots that differ per head, single-token steps (the fused decode + H2O call). The oracle is the plain cache with
    the write-back applied to the slots of every write before attention reads them; rows, positions and scores are
    compared after every step, the block stores' codes must dequantise to the working rows."""
    B, Hq, Hkv, L, D, chunk = 2, 8, 2, 512, 64, 64
    gen = torch.Generator().manual_seed(bits)
    total = L + 3 * chunk + 3
    qs = torch.randn(B, Hq, total, D, generator=gen).to(dtype)
    ks = torch.randn(B, Hkv, total, D, generator=gen).to(dtype)
    vs = (torch.randn(B, Hkv, total, D, generator=gen) * 2).to(dtype)
    ref = O.H2OCacheOracle(B, Hq, Hkv, L, D, dtype=dtype, max_chunk_size=chunk)
    cache = H2OKVCache(KVCacheParams(B, Hkv, L, D, Hq, dtype), max_chunk_size=chunk, quantized=True, num_bits=bits, blocks_over_heads=True,
                       grace_period=grace, device=gpu)
    assert cache.blocks_over_heads
    # another cache of the same kind takes the working buffer in between: each must find its own rows again
    other = H2OKVCache(KVCacheParams(B, Hkv, L, D, Hq, dtype), max_chunk_size=chunk, quantized=True, num_bits=bits, blocks_over_heads=True, device=gpu)

    def check_rows():
        b, T = cache.batch_size, cache.current_length  # the shared working buffer is undefined beyond the slots in use
        assert torch.equal(cache.k[:b, :, :T].cpu(), ref.k[:, :, :T]) and torch.equal(cache.v[:b, :, :T].cpu(), ref.v[:, :, :T])
        back = cache.block_store_k.dequantize(0, T)
        assert torch.equal(back.cpu(), ref.k[:, :, :T])

    first = L - chunk  # prefill leaves room for one chunk: the filling branch
    ref.prefill(qs[:, :, :first], ks[:, :, :first], vs[:, :, :first])
    _requantise_slots(ref, torch.arange(first).view(1, -1).expand(B, -1), bits, dtype)
    o = cache.forward(qs[:, :, :first].to(gpu), ks[:, :, :first].to(gpu), vs[:, :, :first].to(gpu))
    o_ref, _ = O.sdpa_in_blocks(qs[:, :, :first], ks[:, :, :first], vs[:, :, :first], 1 / math.sqrt(D), 0, None, return_attn_weights=False)
    assert rel_err(o.float().cpu().view(B, first, Hq, D).transpose(1, 2), o_ref.float()) < 2e-2
    check_rows()
    other.forward(qs[:, :, :first].to(gpu) * 0.5, vs[:, :, :first].to(gpu), ks[:, :, :first].to(gpu))
    pos = first
    for step, num in enumerate([chunk, chunk, chunk, 1, 1, 1]):
        sl = slice(pos, pos + num)
        # the oracle's step with the write-back between the slot write and the attention
        if ref.current_length < L:
            index = torch.arange(ref.current_length, ref.current_length + num).view(1, 1, -1).expand(B, Hkv, -1)
            ref.current_length += num
        elif ref.use_initial_rule:
            n0 = min(int(0.05 * L), L - num)
            index = torch.arange(n0, n0 + num).view(1, 1, -1).expand(B, Hkv, -1)
            ref.use_initial_rule = False
        else:
            index = ref.next_index[:, :, :num]
        index = index.contiguous().to(torch.int64)
        if step > 0 and cache._have_next:
            cache.set_next_positions(index)  # keep the two caches on the same slots; the GPU's own choice is checked below
        O.cache_write(ref.k, ref.v, ref.token_pos, ref.scores, index, ks[:, :, sl], vs[:, :, sl], ref.input_pos)
        _requantise_slots(ref, index.reshape(B, -1), bits, dtype)
        T = ref.current_length
        o_ref, w = O.sdpa_in_blocks(qs[:, :, sl], ref.k[:, :, :T], ref.v[:, :, :T], ref.scale, ref.input_pos, ref.token_pos[:, :, :T].to(torch.int64))
        ref.input_pos += num
        if T == L:
            ref.next_index = O.h2o_update_select(ref.scores, w, T, L, chunk)
        else:
            ref.scores[:, :, :T] += w
        o = cache.forward(qs[:, :, sl].to(gpu), ks[:, :, sl].to(gpu), vs[:, :, sl].to(gpu))
        torch.cuda.synchronize()
        assert cache.input_pos == ref.input_pos and torch.equal(cache.token_pos.cpu(), ref.token_pos)
        assert rel_err(o.float().cpu().view(B, num, Hq, D).transpose(1, 2), o_ref.float()) < 2e-2
        torch.testing.assert_close(cache.scores.cpu(), ref.scores, rtol=2e-3, atol=1e-5)
        check_rows()
        if T == L and num > 1:
            _sets_equal_away_from_ties(cache._next_index[:B].cpu().long(), ref.next_index, ref.scores, chunk)
        if step % 2 == 0:  # the working buffer changes hands
            other.forward(qs[:, :, sl].to(gpu), vs[:, :, sl].to(gpu), ks[:, :, sl].to(gpu))
        pos += num


def test_h2o_cache_blocks_over_heads_with_grace_period(gpu):
    """With a grace period the ring rows move between slots: both ends of every move are written back. The block
    stores' codes must dequantise to the working rows after every step, and the cache must stay close to the
    unquantised one (8-bit blocks: a small relative error)."""
    B, Hq, Hkv, L, D, chunk, grace = 1, 4, 2, 256, 64, 32, 48
    gen = torch.Generator().manual_seed(7)
    total = L + 4 * chunk
    qs = torch.randn(B, Hq, total, D, generator=gen).to(torch.bfloat16)
    ks = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16)
    vs = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16)
    params = KVCacheParams(B, Hkv, L, D, Hq)
    cache = H2OKVCache(params, max_chunk_size=chunk, quantized=True, num_bits=8, blocks_over_heads=True, grace_period=grace, device=gpu)
    plain = H2OKVCache(params, max_chunk_size=chunk, grace_period=grace, device=gpu)
    pos = 0
    for num in [L] + [chunk] * 4:
        sl = slice(pos, pos + num)
        args = (qs[:, :, sl].to(gpu), ks[:, :, sl].to(gpu), vs[:, :, sl].to(gpu))
        if plain._have_next and cache._have_next:  # both on the slots the plain cache chose for this step
            cache.set_next_positions(plain.next_positions(num))
        o_plain = plain.forward(*args)
        o = cache.forward(*args)
        torch.cuda.synchronize()
        assert torch.equal(cache.token_pos.cpu(), plain.token_pos.cpu())
        assert rel_err(o.float().cpu(), o_plain.float().cpu()) < 5e-2
        assert torch.equal(cache.block_store_k.dequantize(0, L).cpu(), cache.k[:B].cpu())
        assert torch.equal(cache.block_store_v.dequantize(0, L).cpu(), cache.v[:B].cpu())
        assert rel_err(cache.k[:B].float().cpu(), plain.k[:B].float().cpu()) < 2e-2
        pos += num


def test_q_hitter_over_blocks_over_heads(gpu):
    """The Q-Hitter policy on a store with blocks over the heads: the error buffer holds, at every written slot,
    |k - dq(q(k))| + |v - dq(q(v))| of the token's row inside the block of that token over all heads
    (keys_values/kvcache/quant_buffers.py:306-331, keys_values/kvcache/qh2o.py:130-160), and the ring slots' errors
    move with their rows."""
    B, Hq, Hkv, L, D, chunk, grace, bits = 1, 4, 2, 128, 64, 16, 24, 8
    gen = torch.Generator().manual_seed(11)
    total = L + 3 * chunk
    qs = torch.randn(B, Hq, total, D, generator=gen).to(torch.bfloat16)
    ks = torch.randn(B, Hkv, total, D, generator=gen).to(torch.bfloat16)
    vs = (torch.randn(B, Hkv, total, D, generator=gen) * 3).to(torch.bfloat16)

    def block_error(x):  # (B, Hkv, n, D) -> (B, Hkv, n)
        c, sc, z = O.quantize_store(x, bits, True)
        back = O.dequantize_store(c, sc, z, tuple(x.shape), bits, True, x.dtype)
        return torch.linalg.vector_norm(x - back, dim=-1, dtype=torch.float32)

    token_err = block_error(ks) + block_error(vs)  # per token position, as if written alone
    cache = H2OKVCache(KVCacheParams(B, Hkv, L, D, Hq), max_chunk_size=chunk, quantized=True, num_bits=bits, blocks_over_heads=True,
                       q_hitter=True, grace_period=grace, device=gpu)
    pos = 0
    for num in [L, chunk, chunk, chunk]:
        sl = slice(pos, pos + num)
        cache.forward(qs[:, :, sl].to(gpu), ks[:, :, sl].to(gpu), vs[:, :, sl].to(gpu))
        torch.cuda.synchronize()
        # every slot holds the error of the token whose position it carries
        tp = cache.token_pos[:B].cpu().long()
        want = token_err.gather(2, tp)
        torch.testing.assert_close(cache.q_errors[:B].cpu(), want, rtol=1e-5, atol=1e-6)
        pos += num


@pytest.mark.parametrize("name,kw", [("h2o-default", {}), ("h2o-torch-quantized8", {}), ("qh2o-vlen-torch-quantized4", {}),
                                     ("h2o-torch-quantized8", {"blocks_over_heads": True})])
def test_cache_surface_beyond_forward(gpu, name, kw):
    """reset, get_keys_values, get_params, size_estimate (= size_estimate_apriori), update_requires_attn_weights,
    clone, get_v_norm as the reference's caches have them (keys_values/kvcache/base.py:249-377,669-712,
    keys_values/kvcache/attn_weights.py:900-937, keys_values/kvcache/h2o.py:235-283)."""
    from keys_values_amd.kvcache import create_kv_cache

    B, Hq, Hkv, L, D, chunk = 2, 4, 2, 128, 64, 16
    params = KVCacheParams(B, Hkv, L, D, Hq)
    cache = create_kv_cache(name, params, max_chunk_size=chunk, device=gpu, **kw)
    assert cache.update_requires_attn_weights() and cache.get_params() == params
    assert cache.get_keys_values() is None
    gen = torch.Generator().manual_seed(5)
    q = torch.randn(B, Hq, L + chunk, D, generator=gen).to(torch.bfloat16).to(gpu)
    k = torch.randn(B, Hkv, L + chunk, D, generator=gen).to(torch.bfloat16).to(gpu)
    v = torch.randn(B, Hkv, L + chunk, D, generator=gen).to(torch.bfloat16).to(gpu)
    cache.forward(q[:, :, :L], k[:, :, :L], v[:, :, :L])
    cache.forward(q[:, :, L:], k[:, :, L:], v[:, :, L:])
    kv = cache.get_keys_values()
    keys, values = kv.keys(), kv.values()
    assert keys.shape == (B, Hkv, L, D) and values.dtype == torch.bfloat16
    tp = cache.token_positions().long()
    gi = tp.unsqueeze(-1).expand(-1, -1, -1, D)
    err = rel_err(keys.float().cpu(), k.gather(2, gi).float().cpu())  # slot s holds the row of the token at position tp[s]
    assert err < (1e-6 if cache.num_bits is None else 2e-2 if cache.num_bits == 8 else 2e-1), err
    total, parts = cache.size_estimate()
    quantized, bits = cache.quantized, cache.num_bits or 8
    total_a, parts_a = type(cache).size_estimate_apriori(params, quantized=quantized, num_bits=bits, v_length=cache.v_length, q_hitter=cache.q_hitter, **kw)
    assert (total, parts) == (total_a, parts_a)
    rows = B * Hkv * L
    assert parts["token_pos"] == rows * 32 and parts["buffers"] == 2 * rows * D * (bits if quantized else 16)
    if cache.v_length:
        vn = cache.get_v_norm()
        torch.testing.assert_close(vn.cpu(), torch.linalg.vector_norm(v.gather(2, gi).float(), dim=-1).cpu(), rtol=1e-2, atol=1e-3)
    twin = cache.clone()
    assert type(twin) is type(cache) and twin.get_keys_values() is None and twin.quantized == cache.quantized
    # a new sequence after reset gives what a new cache gives
    cache.reset()
    assert cache.input_pos == 0
    o1 = cache.forward(q[:, :, :L], k[:, :, :L], v[:, :, :L])
    o2 = twin.forward(q[:, :, :L], k[:, :, :L], v[:, :, :L])
    assert torch.equal(o1, o2) and torch.equal(cache.token_pos, twin.token_pos) and torch.equal(cache.scores, twin.scores)
