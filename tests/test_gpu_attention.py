"""GPU parity of the attention kernels against the CPU oracle, through the C ABI (ctypes)."""
import ctypes
import math

import pytest
import torch

from helpers import make_qkv, rel_err, scattered_positions
from keys_values_amd import _lib
from keys_values_amd.attention import ops
from keys_values_amd.attention.sdpa import HipSDPA
from keys_values_amd.kvcache.quantize import RowQuantizer
from oracle import kvx_oracle as O

pytestmark = pytest.mark.gpu

# tolerances of the path: outputs 2e-2 relative (bf16), score-sums 1e-3 relative (fp32 accumulation)
O_RTOL = 2e-2
W_RTOL = 1e-3


def check_o(o_gpu, o_ref):
    o_gpu = o_gpu.float().cpu()
    o_ref = o_ref.float()
    assert rel_err(o_gpu, o_ref) < O_RTOL
    torch.testing.assert_close(o_gpu, o_ref, rtol=O_RTOL, atol=2e-2)


def check_w(w_gpu, w_ref, q_len):
    w_gpu = w_gpu.cpu()
    assert w_gpu.dtype == torch.float32
    assert (w_gpu >= 0).all()
    torch.testing.assert_close(w_gpu, w_ref, rtol=W_RTOL, atol=1e-6)
    torch.testing.assert_close(w_gpu.sum(-1), torch.full(w_gpu.shape[:2], float(q_len)), rtol=5e-5, atol=3e-4)


CASES = [
    # B, Hq, Hkv, q_len, T, D, input_pos, scattered, splits
    (1, 8, 2, 128, 1024, 64, 896, False, 0),     # configuration 1 shapes
    (1, 8, 2, 128, 1024, 64, 896, True, 2),
    (2, 4, 4, 16, 200, 128, 300, True, 1),       # G = 1, ragged T
    (1, 8, 2, 100, 333, 128, 233, False, 3),     # ragged rows and keys, 3 splits
    (2, 8, 1, 37, 700, 128, 1000, True, 0),      # G = 8
    (1, 32, 8, 64, 192, 128, 128, False, 1),     # the reference's fused-prefill test shape
    (1, 4, 2, 2, 64, 64, 62, False, 1),
    (1, 4, 2, 300, 300, 128, 0, False, 2),       # square causal prefill (input_pos = 0)
]


@pytest.mark.parametrize("B,Hq,Hkv,q_len,T,D,input_pos,scattered,splits", CASES)
def test_prefill_with_weights(gpu, B, Hq, Hkv, q_len, T, D, input_pos, scattered, splits):
    q, k, v, gen = make_qkv(100 + T + q_len, B, Hq, Hkv, q_len, T, D)
    tp = scattered_positions(gen, B, Hkv, T, input_pos, q_len) if scattered else None
    if tp is None and input_pos != T - q_len:
        tp = (torch.arange(T, dtype=torch.int32) + (input_pos - (T - q_len))).view(1, 1, T).expand(B, Hkv, T).contiguous()
    scale = 1.0 / math.sqrt(D)
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, input_pos, None if tp is None else tp.to(torch.int64))
    l_ref = O.lse2(q, k, scale, input_pos, tp)
    out, w, lse = ops.prefill_core(
        q.to(gpu), k.to(gpu), v.to(gpu), scale, input_pos, None if tp is None else tp.to(gpu),
        return_weights=True, return_lse=True, output_transposed=False, num_splits=splits,
    )
    torch.cuda.synchronize()
    check_o(out, o_ref)
    torch.testing.assert_close(lse.cpu(), l_ref, rtol=1e-4, atol=1e-3)
    check_w(w, w_ref, q_len)


def test_prefill_strided_cache_views_and_layouts(gpu):
    # K/V as views k[:B, :, :T] of a larger (Bmax, Hkv, L, D) allocation
    # (keys_values/kvcache/buffers.py:538-541) and the extension's [B, len, H, D] layout
    B, Hq, Hkv, q_len, T, D, L = 2, 8, 2, 48, 160, 128, 256
    q, k, v, gen = make_qkv(5, B, Hq, Hkv, q_len, T, D)
    tp = scattered_positions(gen, B, Hkv, T, 400, q_len)
    scale = 0.09
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, 400, tp.to(torch.int64))
    kbuf = torch.zeros(3, Hkv, L, D, dtype=torch.bfloat16, device=gpu)
    vbuf = torch.zeros(3, Hkv, L, D, dtype=torch.bfloat16, device=gpu)
    tpbuf = torch.zeros(3, Hkv, L, dtype=torch.int32, device=gpu)
    kbuf[:B, :, :T] = k.to(gpu)
    vbuf[:B, :, :T] = v.to(gpu)
    tpbuf[:B, :, :T] = tp.to(gpu)
    out, w, _ = ops.prefill_core(q.to(gpu), kbuf[:B, :, :T], vbuf[:B, :, :T], scale, 400, tpbuf[:B, :, :T], return_weights=True)
    assert out.shape == (B, q_len, Hq, D)
    check_o(out.permute(0, 2, 1, 3), o_ref)
    check_w(w, w_ref, q_len)
    # reference extension layout, right-aligned causal
    o2_ref, w2_ref = O.sdpa_in_blocks(q, k, v, scale, T - q_len, None)
    out2, w2, lse2 = ops.sdpa_prefill(
        q.to(gpu).transpose(1, 2).contiguous(), k.to(gpu).transpose(1, 2).contiguous(), v.to(gpu).transpose(1, 2).contiguous(),
        scale, return_weights=True, return_lse=True,
    )
    check_o(out2.permute(0, 2, 1, 3), o2_ref)
    check_w(w2, w2_ref, q_len)
    torch.testing.assert_close(lse2.cpu(), O.lse2(q, k, scale, T - q_len, None), rtol=1e-4, atol=1e-3)


def test_score_sum_from_given_lse(gpu):
    # the score-sum kernel alone, fed the oracle's LSE (as the reference tests its Triton kernel,
    # test/attention/test_flashinfer_wrapper.py:1207-1307)
    B, Hq, Hkv, q_len, T, D = 1, 8, 2, 70, 530, 128
    q, k, v, gen = make_qkv(77, B, Hq, Hkv, q_len, T, D)
    tp = scattered_positions(gen, B, Hkv, T, 600, q_len)
    scale = 1.0 / math.sqrt(D)
    _, w_ref = O.sdpa_in_blocks(q, k, v, scale, 600, tp.to(torch.int64))
    lse = O.lse2(q, k, scale, 600, tp)
    w = ops.score_sum_core(q.to(gpu), k.to(gpu), lse.to(gpu), scale, 600, tp.to(gpu))
    check_w(w, w_ref, q_len)


@pytest.mark.parametrize("store", ["bf16", "u8"])
def test_score_sum_with_eight_wavefront_workgroups(gpu, store):
    # enough keys for the launch to take workgroups of 512 keys (8 KV heads x 32 workgroups), the last one
    # ragged, causal inside the chunk, scattered slots
    B, Hq, Hkv, q_len, T, D = 1, 16, 8, 40, 16000, 64
    q, k, v, gen = make_qkv(78, B, Hq, Hkv, q_len, T, D)
    input_pos = T + 11
    tp = scattered_positions(gen, B, Hkv, T, input_pos, q_len)
    scale = 1.0 / math.sqrt(D)
    quant, kg = None, k.to(gpu)
    if store == "u8":
        kc, ks, kz = O.quantize_rows(k)
        k = O.dequantize_rows(kc, ks, kz)
        kg = kc.to(gpu)
        quant = ops.QuantState(ks.to(gpu), kz.to(gpu), ks.to(gpu), kz.to(gpu))
    _, w_ref = O.sdpa_in_blocks(q, k, v, scale, input_pos, tp.to(torch.int64))
    lse = O.lse2(q, k, scale, input_pos, tp)
    w = ops.score_sum_core(q.to(gpu), kg, lse.to(gpu), scale, input_pos, tp.to(gpu), quant=quant)
    check_w(w, w_ref, q_len)
    torch.testing.assert_close(w.sum(-1).cpu(), torch.full((B, Hkv), float(q_len)), rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("store", ["bf16", "u8", "u4"])
@pytest.mark.parametrize("B,Hq,Hkv,q_len,T,D,splits", [
    (1, 1, 1, 2, 2, 64, 0),          # less than a block of rows, a handful of keys
    (1, 7, 1, 9, 65, 128, 0),        # 63 rows, one key beyond a workgroup's 64
    (2, 6, 2, 43, 190, 128, 3),      # 129 rows of 3 heads
    (1, 8, 2, 256, 1087, 64, 17),    # 1024 rows, the most; one split more than a pass over the partials takes
    (1, 2, 1, 16, 2200, 64, 33),     # the partials in three passes
    (1, 12, 1, 85, 700, 256, 2),     # 1020 rows of 12 heads
    (1, 5, 1, 205, 640, 128, 2),     # 1025 rows: the long kernel
])
def test_score_sums_of_few_rows_over_few_keys(gpu, store, B, Hq, Hkv, q_len, T, D, splits):
    # score-sums and the combination of the KV splits in one launch; tolerances of the path
    q, k, v, gen = make_qkv(310 + T, B, Hq, Hkv, q_len, T, D)
    quant = None
    kd, vd = k.to(gpu), v.to(gpu)
    if store != "bf16":
        bits = 8 if store == "u8" else 4
        (kc, ks, kz), (vc, vs, vz) = ([t.view(B, Hkv, T, -1) if t.dim() > 1 else t.view(B, Hkv, T) for t in O.quantize_rows(x.reshape(-1, D), bits)] for x in (k, v))
        k, v = ((O.dequantize_rows(c.reshape(-1, D), s.reshape(-1), z.reshape(-1), torch.bfloat16)).view(B, Hkv, T, D) for c, s, z in ((kc, ks, kz), (vc, vs, vz)))
        if bits == 4:
            kc, vc = (O.compress4(c.reshape(-1, D)).view(B, Hkv, T, D // 2) for c in (kc, vc))
        kd, vd = kc.to(gpu), vc.to(gpu)
        quant = ops.QuantState(*(t.to(gpu) for t in (ks, kz, vs, vz)))
    tp = scattered_positions(gen, B, Hkv, T, 2 * T, q_len)
    scale = 1.0 / math.sqrt(D)
    for pos, tpos in ((2 * T, tp), (T - q_len, None)):
        o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, pos, None if tpos is None else tpos.to(torch.int64))
        out, w, lse = ops.prefill_core(q.to(gpu), kd, vd, scale, pos, None if tpos is None else tpos.to(gpu), return_weights=True, return_lse=True,
                                       output_transposed=False, quant=quant, num_splits=splits)
        check_o(out, o_ref)
        check_w(w, w_ref, q_len)
        torch.testing.assert_close(lse.cpu(), O.lse2(q, k, scale, pos, tpos), rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("store", ["bf16", "u8", "u4"])
@pytest.mark.parametrize("B,Hq,Hkv,q_len,T,D,splits", [
    (2, 8, 8, 2, 1100, 128, 2),       # 2 rows, 17.2 blocks of keys
    (2, 24, 8, 10, 1090, 256, 5),     # 30 rows of 3 heads
    (1, 32, 8, 8, 2112, 128, 17),     # a full block of rows; the partials in two passes
    (5, 4, 4, 32, 5000, 64, 0),       # several blocks of keys a wavefront
    (4, 28, 4, 18, 1030, 64, 3),      # 126 rows
])
def test_score_sums_with_streamed_keys(gpu, store, B, Hq, Hkv, q_len, T, D, splits):
    # few rows over more keys than the short kernel takes, alone and with the combination of the KV splits
    test_score_sums_of_few_rows_over_few_keys(gpu, store, B, Hq, Hkv, q_len, T, D, splits)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("store", ["plain", "u8", "u4"])
@pytest.mark.parametrize("B,Hq,Hkv,q_len,T,D,splits", [
    (1, 1, 1, 2, 2, 128, 0),         # two rows and keys
    (2, 4, 2, 8, 31, 64, 0),         # a full tile of 16 rows, a key short of a block
    (1, 17, 1, 2, 129, 128, 0),      # 34 rows, one key beyond a round of the four wavefronts
    (1, 3, 1, 11, 385, 256, 2),      # 33 rows; codes: 256 columns of V over two tiles of rows
    (1, 6, 2, 43, 1535, 64, 0),      # 129 rows of 3 heads, the last block short
    (3, 8, 8, 5, 4097, 128, 0),      # 5 rows, many splits, the last one of a single key
    (1, 8, 2, 4, 700, 128, 11),      # a split a tile
    (2, 16, 2, 16, 640, 256, 0),     # 128 rows of 256, the most over codes
    (1, 32, 8, 75, 1000, 128, 0),    # 300 rows in splits
    (1, 8, 2, 384, 640, 128, 0),     # 1536 rows, as many as keys of them are new: most blocks are masked
    (2, 16, 4, 260, 640, 128, 0),    # 1040 rows: over plain rows above the line to the tiled kernel, over codes below it
    (2, 16, 4, 260, 900, 128, 0),    # above it in every store
])
def test_attention_of_few_rows(kvx, gpu, dtype, store, B, Hq, Hkv, q_len, T, D, splits):
    # plain rows of 256 values always take the tiled kernel
    few = T != 900 and not (store == "plain" and (D == 256 or T == 640 and q_len == 260))
    check_attention(kvx, gpu, dtype, store, B, Hq, Hkv, q_len, T, D, splits, few, False)


def block_rows(kvx, q, k, v, input_pos, tp=None, quant=None, copying=False):
    """query rows of a workgroup of the attention kernel: up to 32 in the one for few rows"""
    a = _lib.SdpaArgs()
    ops._fill_common(a, q, k, v, 1.0, input_pos, tp, quant, 0)
    rows = kvx.kvx_sdpa_prefill_block_rows(ctypes.byref(a), copying)
    assert rows in (16, 32, 128, 256)
    return rows


def check_attention(kvx, gpu, dtype, store, B, Hq, Hkv, q_len, T, D, splits, few_rows, fused_dequant):
    # dense, offset and scattered positions; rows, positions and row state on 4-element bounds and off them
    # tolerances of the path
    q, k, v, gen = make_qkv(510 + T, B, Hq, Hkv, q_len, T, D, dtype=dtype)
    state = None
    if store != "plain":
        bits = 8 if store == "u8" else 4
        (kc, ks, kz), (vc, vs, vz) = (O.quantize_rows(x.reshape(-1, D), bits) for x in (k, v))
        k, v = (O.dequantize_rows(*t, dtype).view(B, Hkv, T, D) for t in ((kc, ks, kz), (vc, vs, vz)))
        if bits == 4:
            kc, vc = O.compress4(kc), O.compress4(vc)
        kd, vd = kc.view(B, Hkv, T, -1), vc.view(B, Hkv, T, -1)
        state = [t.view(B, Hkv, T) for t in (ks, kz, vs, vz)]
    else:
        kd, vd = k, v
    scale = 1.0 / math.sqrt(D)

    def shifted(x, by):
        """``x`` on the device in a buffer whose rows are 3 longer and begin ``by`` in"""
        buf = torch.zeros(B, Hkv, T + 3, *x.shape[3:], dtype=x.dtype, device=gpu)
        buf[:, :, by : by + T] = x.to(gpu)
        return buf[:, :, by : by + T]

    for pos, tp, by in ((T - q_len, None, 0), (2 * T, scattered_positions(gen, B, Hkv, T, 2 * T, q_len), 0), (T, scattered_positions(gen, B, Hkv, T, T, q_len), 1)):
        move = (lambda x: x.to(gpu)) if by == 0 else (lambda x: shifted(x, by))
        o_ref, _ = O.sdpa_in_blocks(q, k, v, scale, pos, None if tp is None else tp.to(torch.int64))
        qg, kg, vg, tpg, quant = q.to(gpu), move(kd), move(vd), None if tp is None else move(tp), None if state is None else ops.QuantState(*(move(t) for t in state))
        assert (block_rows(kvx, qg, kg, vg, pos, tpg, quant, not fused_dequant) <= 32) == few_rows
        out, _, lse = ops.prefill_core(qg, kg, vg, scale, pos, tpg, return_lse=True, output_transposed=False, quant=quant, num_splits=splits, fused_dequant=fused_dequant)
        check_o(out, o_ref)
        torch.testing.assert_close(lse.cpu(), O.lse2(q, k, scale, pos, tp), rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("store", ["plain", "u8", "u4"])
@pytest.mark.parametrize("dtype,B,Hq,Hkv,q_len,T,D,splits", [
    (torch.bfloat16, 8, 48, 16, 27, 961, 64, 0),    # 81 rows of 3 heads; the last tile a single key
    (torch.float16, 8, 48, 16, 27, 1023, 128, 0),   # one key short of whole tiles
    (torch.bfloat16, 12, 128, 16, 60, 60, 64, 0),   # less than a tile of keys, all of them new
    (torch.float16, 12, 128, 16, 50, 63, 128, 2),   # more splits than tiles
    (torch.bfloat16, 4, 56, 8, 33, 1300, 128, 3),   # 231 rows of 7 heads, 21 tiles
    (torch.float16, 4, 36, 4, 60, 1345, 64, 2),     # 540 rows of 9 heads, 22 tiles, the last one a single key
    (torch.bfloat16, 8, 32, 32, 65, 511, 128, 3),   # 65 rows; the last split one tile shorter
    (torch.float16, 1, 6, 2, 45, 700, 256, 0),      # 135 rows of 256, over codes the fewest
])
def test_attention_of_many_rows(kvx, gpu, store, dtype, B, Hq, Hkv, q_len, T, D, splits):
    """The tiled kernel, over codes the form that dequantises for itself, above every line to the kernel for few rows."""
    check_attention(kvx, gpu, dtype, store, B, Hq, Hkv, q_len, T, D, splits, False, True)


@pytest.mark.parametrize("scattered", [False, True])
@pytest.mark.parametrize("store,B,Hkv,T,D,most", [
    # the most queries of 2 heads per KV head that take the kernel for few rows
    ("plain", 2, 8, 1000, 128, 160), ("plain", 2, 8, 1000, 64, 256), ("plain", 16, 16, 40, 128, 8),
    ("u8", 2, 8, 1000, 64, 320), ("u4", 2, 8, 1000, 64, 224), ("u8", 2, 8, 1000, 128, 192), ("u4", 2, 8, 1000, 128, 192),
    ("u8", 4, 8, 8000, 128, 32), ("u4", 4, 8, 8000, 64, 32), ("u8", 2, 8, 1000, 256, 64), ("u4", 2, 8, 1000, 256, 64),
    # and few keys: as many workgroups as the units hold; over a tile of keys, one for each unit
    ("plain", 4, 16, 250, 128, 64), ("plain", 4, 16, 250, 64, 128), ("u8", 8, 8, 250, 128, 64), ("u4", 8, 8, 250, 128, 128), ("plain", 8, 16, 64, 128, 16),
])
def test_both_sides_of_the_lines_between_the_attention_kernels(kvx, gpu, store, B, Hkv, T, D, most, scattered):
    """Just below a line, and the same queries in a call with one more just above it. On each side the outputs are rounded to 8 bits and the
    probabilities before, by up to 2^-9 either way: 2^-9 / sqrt(3) each in the mean square, four of them 2.3e-3 in the norm."""
    gen = torch.Generator().manual_seed(T + D)
    q = torch.randn(B, 2 * Hkv, most + 1, D, generator=gen).to(torch.bfloat16).to(gpu)
    rows = [torch.randn(B, Hkv, T, D, generator=gen).to(torch.bfloat16).to(gpu) for _ in range(2)]
    quant = None
    if store != "plain":
        bits, state = 8 if store == "u8" else 4, []
        for i, x in enumerate(rows):
            qz = RowQuantizer((B, Hkv, T, D), torch.bfloat16, bits, allocate_buffers=True, device=gpu)
            qz.quantize(0, T, x)
            rows[i] = qz.quant_buffer.view(B, Hkv, T, -1)
            state += [qz.quant_scales.view(B, Hkv, T), qz.quant_zero_points.view(B, Hkv, T)]
        quant = ops.QuantState(*state)
    pos, tp = T - most - 1, None
    if scattered:
        pos, tp = 2 * T, scattered_positions(gen, B, Hkv, T, 2 * T, most + 1).to(gpu)
    got = []
    for n in (most, most + 1):
        qn = q[:, :, :n]
        assert (block_rows(kvx, qn, *rows, pos, tp, quant) <= 32) == (n == most)
        got.append(ops.prefill_core(qn, *rows, D ** -0.5, pos, tp, return_lse=True, output_transposed=False, quant=quant, fused_dequant=True))
    (below, _, lse), (above, _, lse_above) = got
    assert rel_err(below.float(), above[:, :, :most].float()) < 4 * 2.3e-3
    torch.testing.assert_close(lse, lse_above[:, :most], rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("q_len", [1, 9])
@pytest.mark.parametrize("bits,D", [(8, 64), (8, 128), (8, 256), (4, 64), (4, 128), (4, 256)])
def test_rows_of_codes_that_begin_on_8_bytes(gpu, bits, D, q_len):
    # strides of whole 8 bytes are what the calls ask for: every other row of codes is not 16-byte aligned. The same bits as over
    # adjacent rows.
    B, Hq, Hkv, T = 1, 8, 2, 333
    q, k, v, _ = make_qkv(60 + D, B, Hq, Hkv, q_len, T, D)
    row = D * bits // 8
    codes, wide, state = [], [], []
    for x in (k, v):
        c, s, z = O.quantize_rows(x.reshape(-1, D), bits)
        c = (O.compress4(c) if bits == 4 else c).view(B, Hkv, T, row).to(gpu)
        buf = torch.full((B, Hkv, T, row + 8), 255, dtype=torch.uint8, device=gpu)
        buf[..., :row] = c
        codes.append(c)
        wide.append(buf[..., :row])
        state += [s.view(B, Hkv, T).to(gpu), z.view(B, Hkv, T).to(gpu)]
    quant = ops.QuantState(*state)
    assert wide[0].stride(2) == row + 8
    got = []
    for kd, vd in (codes, wide):
        if q_len == 1:
            got.append(ops.decode_core(q.to(gpu), kd, vd, 0.1, return_weights=True, quant=quant))
        else:
            got.append(ops.prefill_core(q.to(gpu), kd, vd, 0.1, T - q_len, return_weights=True, quant=quant))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("B,Hq,Hkv,q_len,T,D,splits", [(1, 4, 2, 9, 200, 64, 0), (2, 4, 1, 20, 333, 128, 3)])
def test_attention_of_few_rows_whose_logits_lie_far_below_zero(gpu, B, Hq, Hkv, q_len, T, D, splits):
    """Finite logits are weighed however low they are: all keys alike, q.k = -2^112 or so (a power of two, so that its scaling is
    exact), the outputs are means of V. A mean of fewer than 2^9 rows in 16 bits: 2^-8 of the largest value."""
    gen = torch.Generator().manual_seed(T)
    v = torch.randn(B, Hkv, T, D, generator=gen).to(torch.bfloat16)
    q, k = torch.full((B, Hq, q_len, D), 2.0 ** 53, dtype=torch.bfloat16), torch.full((B, Hkv, T, D), -(2.0 ** 53), dtype=torch.bfloat16)
    out, _, lse = ops.prefill_core(q.to(gpu), k.to(gpu), v.to(gpu), 0.125, T - q_len, return_lse=True, output_transposed=False, num_splits=splits)
    ref = torch.stack([v[:, :, : T - q_len + i + 1].double().mean(2) for i in range(q_len)], 2).repeat_interleave(Hq // Hkv, 1)
    torch.testing.assert_close(out.double().cpu(), ref, rtol=2.0 ** -8, atol=2.0 ** -8)
    torch.testing.assert_close(lse.double().cpu(), torch.full((B, q_len, Hq), -(2.0 ** 106) * D * 0.125 * math.log2(math.e), dtype=torch.float64), rtol=1e-6, atol=0)


@pytest.mark.parametrize("scattered", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,q_len,T,D", [
    (1, 7, 1, 297, 600, 128),    # 2079 rows: 33 tiles of 63, all full
    (1, 7, 1, 298, 4500, 64),    # one query more
    (2, 6, 2, 460, 900, 128),    # 21 queries of 3 heads a tile
    (1, 12, 1, 171, 400, 128),   # tiles of 60 rows
    (1, 9, 1, 190, 700, 64),     # 63 rows of 9 heads
    (1, 24, 1, 90, 300, 128),    # 48 of 64 rows would be used: full tiles, the general step
    (1, 5, 1, 420, 1200, 256),
])
def test_score_sums_of_tiles_of_whole_queries(gpu, B, Hq, Hkv, q_len, T, D, scattered):
    # group sizes that do not divide the 64 rows of a query tile, more than the 1024 rows the short kernel takes
    q, k, v, gen = make_qkv(610 + T, B, Hq, Hkv, q_len, T, D)
    pos = 2 * T if scattered else T - q_len
    tp = scattered_positions(gen, B, Hkv, T, pos, q_len) if scattered else None
    scale = 1.0 / math.sqrt(D)
    _, w_ref = O.sdpa_in_blocks(q, k, v, scale, pos, None if tp is None else tp.to(torch.int64))
    _, w, _ = ops.prefill_core(q.to(gpu), k.to(gpu), v.to(gpu), scale, pos, None if tp is None else tp.to(gpu), return_weights=True)
    check_w(w, w_ref, q_len)


@pytest.mark.parametrize("B,Hq,Hkv,q_len,T,D", [(1, 8, 2, 700, 900, 128), (2, 4, 1, 1100, 1100, 64), (1, 16, 2, 300, 2048, 128)])
def test_score_sum_over_split_query_rows(kvx, gpu, B, Hq, Hkv, q_len, T, D):
    # a short cache: with a workspace the query rows are split over several workgroups and the partial sums
    # added by a second launch; without one the kernel walks all rows. Both against the oracle, and each other.
    q, k, v, gen = make_qkv(79 + T, B, Hq, Hkv, q_len, T, D)
    input_pos = T - q_len + 3
    tp = scattered_positions(gen, B, Hkv, T, input_pos, q_len)
    scale = 1.0 / math.sqrt(D)
    _, w_ref = O.sdpa_in_blocks(q, k, v, scale, input_pos, tp.to(torch.int64))
    lse = O.lse2(q, k, scale, input_pos, tp).to(gpu)
    qg, kg, tpg = q.to(gpu), k.to(gpu), tp.to(gpu)
    w_split = ops.score_sum_core(qg, kg, lse, scale, input_pos, tpg)
    check_w(w_split, w_ref, q_len)
    a = _lib.SdpaArgs()
    ops._fill_common(a, qg, kg, None, scale, input_pos, tpg, None, 0)
    assert kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a)) > 0  # the shape does split
    w_whole = torch.empty_like(w_split)
    a.lse, a.w = lse.data_ptr(), w_whole.data_ptr()
    _lib.check(kvx.kvx_score_sum(ctypes.byref(a), _lib.stream_ptr(gpu)))  # no workspace: no split
    torch.cuda.synchronize()
    check_w(w_whole, w_ref, q_len)
    torch.testing.assert_close(w_split, w_whole, rtol=1e-5, atol=1e-7)
    assert torch.equal(w_split, ops.score_sum_core(qg, kg, lse, scale, input_pos, tpg))  # the same bits every time


def test_causal_weights_decay(gpu):
    # test/attention/test_flashinfer_wrapper.py:1074-1124: early keys collect far more weight
    q, k, v, _ = make_qkv(3, 1, 8, 2, 64, 64, 64)
    _, w, _ = ops.prefill_core(q.to(gpu), k.to(gpu), v.to(gpu), 0.125, 0, None, return_weights=True)
    w = w.cpu()
    assert (w[:, :, 0] > 2 * w[:, :, -1]).all()


def test_hip_sdpa_dropin(gpu):
    # FlashInferSDPA surface incl. head-size padding (keys_values/attention/flashinfer_wrapper.py:276-308)
    B, Hq, Hkv, q_len, T, D = 1, 4, 2, 20, 90, 48
    q, k, v, gen = make_qkv(42, B, Hq, Hkv, q_len, T, D)
    tp = scattered_positions(gen, B, Hkv, T, 111, q_len)
    sdpa = HipSDPA()
    assert sdpa.available
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, 1 / math.sqrt(D), 111, tp.to(torch.int64))
    out, w = sdpa.scaled_dot_product_attention(q.to(gpu), k.to(gpu), v.to(gpu), None, 111, tp.to(gpu), return_attn_weights=True)
    assert out.shape == (B, Hq, q_len, D) and w.shape == (B, Hkv, T)
    check_o(out, o_ref)
    check_w(w, w_ref, q_len)
    out_t, w_none = sdpa.scaled_dot_product_attention(q.to(gpu), k.to(gpu), v.to(gpu), None, 111, tp.to(gpu), output_transposed=True)
    assert w_none is None and out_t.shape == (B, q_len, Hq, D)
    check_o(out_t.transpose(1, 2), o_ref)
    # q_len == 1 routes to the decode kernel and ignores positions
    o1_ref, w1_ref = O.sdpa_in_blocks(q[:, :, :1], k, v, 1 / math.sqrt(D), 10**6, None)
    out1, w1 = sdpa.scaled_dot_product_attention(q[:, :, :1].to(gpu), k.to(gpu), v.to(gpu), None, 500, tp.to(gpu), return_attn_weights=True)
    check_o(out1, o1_ref)
    check_w(w1, w1_ref, 1)


DECODE_CASES = [
    # B, Hq, Hkv, T, D, splits
    (2, 8, 2, 1000, 128, 0),
    (1, 32, 8, 4096 + 77, 128, 0),
    (3, 4, 4, 130, 64, 1),
    (1, 8, 1, 5000, 128, 3),
    (2, 4, 2, 17, 64, 0),
    (1, 8, 2, 9000, 64, 2),
    (2, 6, 2, 700, 128, 0),        # group sizes that are not powers of two: 3, 7 (Qwen2-7B: 28 / 4), 5, 6
    (1, 28, 4, 3000, 128, 2),
    (1, 5, 1, 513, 64, 1),
    (2, 12, 2, 260, 128, 0),
    (1, 32, 2, 3000, 128, 0),      # 16 and 12 heads per KV head: both products on the matrix cores, 16 head columns
    (2, 24, 2, 700, 64, 0),
    (1, 16, 1, 1100, 64, 2),
]


@pytest.mark.parametrize("B,Hq,Hkv,T,D,splits", DECODE_CASES + [(2, 8, 2, 20000, 128, 0), (1, 8, 1, 9000, 64, 0), (1, 4, 2, 5000, 256, 0), (1, 16, 2, 4100, 128, 0),
                                                           # more splits than a wavefront and two have lanes; splits of more keys than four a thread
                                                           (1, 4, 1, 8300, 64, 130), (1, 2, 1, 4481, 256, 70), (1, 4, 2, 4500, 128, 2)])
def test_decode_with_weights(gpu, decode_route, B, Hq, Hkv, T, D, splits):
    q, k, v, _ = make_qkv(900 + T, B, Hq, Hkv, 1, T, D)
    scale = 1.0 / math.sqrt(D)
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, T - 1, None)
    l_ref = O.lse2(q, k, scale, T - 1, None)
    out, w, lse = ops.decode_core(q.to(gpu), k.to(gpu), v.to(gpu), scale, return_weights=True, return_lse=True, num_splits=splits)
    torch.cuda.synchronize()
    check_o(out.unsqueeze(2), o_ref)
    torch.testing.assert_close(lse.cpu(), l_ref, rtol=1e-4, atol=1e-3)
    check_w(w, w_ref, 1)
    # reference extension layout
    out2, w2 = ops.sdpa_decode(q[:, :, 0].to(gpu), k.to(gpu).transpose(1, 2).contiguous(), v.to(gpu).transpose(1, 2).contiguous(), scale, return_weights=True)
    check_o(out2.unsqueeze(2), o_ref)
    check_w(w2, w_ref, 1)
    out3, w3 = ops.sdpa_decode(q[:, :, 0].to(gpu), k.to(gpu).transpose(1, 2).contiguous(), v.to(gpu).transpose(1, 2).contiguous(), scale)
    assert w3 is None
    check_o(out3.unsqueeze(2), o_ref)


def test_decode_reports_the_splits_that_took_the_scratch_route(kvx, gpu):
    """The optional counter of a decode call: 0 when every split turned its own logits into weights, every split
    when that form is switched off or no split waits, and nothing written without score-sums."""
    B, Hq, Hkv, T, D = 2, 8, 2, 20000, 128
    q, k, v, _ = make_qkv(77, B, Hq, Hkv, 1, T, D)
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    scale = 1.0 / math.sqrt(D)
    counts, ws = {}, {}
    try:
        for name, setting in (("resident", (-1, -1, -1)), ("scratch", (0, -1, -1)), ("no-wait", (-1, 0, -1))):
            kvx.kvx_decode_tuning(*setting)
            n = torch.full((1,), -5, dtype=torch.int32, device=gpu)
            _, ws[name], _ = ops.decode_core(qg, kg, vg, scale, return_weights=True, scratch_splits=n)
            counts[name] = int(n.item())
    finally:
        kvx.kvx_decode_tuning(-1, -1, -1)
    assert counts["resident"] == 0
    assert counts["scratch"] == counts["no-wait"] and counts["scratch"] >= B * Hkv and counts["scratch"] % (B * Hkv) == 0
    assert torch.equal(ws["resident"], ws["scratch"]) and torch.equal(ws["resident"], ws["no-wait"])
    n = torch.full((1,), -5, dtype=torch.int32, device=gpu)
    ops.decode_core(qg, kg, vg, scale, return_weights=False, scratch_splits=n)
    assert int(n.item()) == 0  # no logits, nothing through the scratch


@pytest.mark.parametrize("B,Hq,Hkv,T,store,splits,on_chip", [
    (1, 16, 1, 196608, "plain", 0, True),   # 256 splits of 768 keys or fewer: their weights fit beside the logits
    (1, 16, 1, 196609, "plain", 0, True),   # more: they take the logits' place
    (1, 12, 1, 262144, "plain", 0, True),   # 12 heads padded to 16
    (1, 24, 2, 262144, "plain", 0, False),  # two rows of them: not all side by side, through the scratch
    (1, 16, 1, 393216, "u8", 0, True),      # 512 full splits, the most that stays on the chip
    (1, 8, 1, 32769, "u4", 512, True),      # asked for: 257 splits, the last one of a single key
    (2, 4, 1, 32768, "plain", 512, True),   # 512 splits of 64 keys, the kernel without matrix instructions
    (1, 2, 2, 33000, "plain", 400, True),
])
def test_decode_at_head_size_64_in_more_than_256_splits(gpu, decode_route, B, Hq, Hkv, T, store, splits, on_chip):
    """A row of up to 512 splits can be one launch with the logits on the chip. Tolerances of the path."""
    D, scale = 64, 0.125
    q, k, v, _ = make_qkv(T + Hq, B, Hq, Hkv, 1, T, D)
    quant, kd, vd = None, k.to(gpu), v.to(gpu)
    if store != "plain":
        bits, codes, state, rows = 8 if store == "u8" else 4, [], [], []
        for x in (kd, vd):
            qz = RowQuantizer((B, Hkv, T, D), torch.bfloat16, bits, allocate_buffers=True, device=gpu)
            qz.quantize(0, T, x)
            codes.append(qz.quant_buffer.view(B, Hkv, T, -1))
            state += [qz.quant_scales.view(B, Hkv, T), qz.quant_zero_points.view(B, Hkv, T)]
            rows.append(qz.dequantize(0, T).cpu())
        (kd, vd), (k, v), quant = codes, rows, ops.QuantState(*state)
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, T - 1, None)
    n = torch.full((1,), -5, dtype=torch.int32, device=gpu)
    out, w, lse = ops.decode_core(q.to(gpu), kd, vd, scale, return_weights=True, return_lse=True, quant=quant, num_splits=splits, scratch_splits=n)
    if decode_route == "resident":
        assert (int(n.item()) == 0) == on_chip
    check_o(out.unsqueeze(2), o_ref)
    torch.testing.assert_close(lse.cpu(), O.lse2(q, k, scale, T - 1, None), rtol=1e-4, atol=1e-3)
    check_w(w, w_ref, 1)
    out2, _, lse2 = ops.decode_core(q.to(gpu), kd, vd, scale, return_lse=True, quant=quant, num_splits=splits or 300)
    check_o(out2.unsqueeze(2), o_ref)
    torch.testing.assert_close(lse2, lse, rtol=1e-4, atol=1e-3)


def test_decode_workspace_counts_the_splits_asked_for(kvx, gpu):
    """Up to 512 splits a row at every head size: 512 partial outputs of fp32 values, and no more for a larger number."""
    for D in (64, 128, 256):
        q, k, v, _ = make_qkv(D, 1, 1, 1, 1, 32768, D)
        a = _lib.SdpaArgs()
        need = []
        for splits in (511, 512, 600):
            ops._fill_common(a, q, k, v, 1.0, 32767, None, None, splits)
            need.append(kvx.kvx_sdpa_decode_workspace_bytes(ctypes.byref(a)))
        # splits are whole multiples of 64 keys: 511 are 256 of 128
        assert need[1] == need[2] and need[1] - need[0] >= 256 * D * 4, need


def test_decode_splits_of_long_rows_through_the_scratch(kvx, gpu):
    """Logits that fit the chip in no 512 splits: as many splits as give every compute unit one workgroup, whatever the number of rows."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for Hq, Hkv, T, D in ((16, 1, 600000, 64), (16, 1, 270000, 128), (8, 1, 950000, 128), (32, 2, 600000, 64), (32, 2, 300000, 128)):
        a = _lib.SdpaArgs()
        need = []
        for splits in (0, cus // Hkv):
            a.B, a.Hq, a.Hkv, a.q_len, a.kv_len, a.D, a.input_pos, a.sm_scale, a.num_splits = 1, Hq, Hkv, 1, T, D, T - 1, 1.0, splits
            a.q = a.k = a.v = a.w = 16  # for the size alone
            a.q_stride_h = a.q_stride_t = a.k_stride_t = a.v_stride_t = D
            need.append(kvx.kvx_sdpa_decode_workspace_bytes(ctypes.byref(a)))
        assert need[0] == need[1] > 0, (Hq, Hkv, T, D)


def test_full_size_prefill_properties(gpu):
    """Configuration 2 at its real shape (B1, 32/8 heads, D128, 32768 slots, 1024 queries, RoPE):
    one KV head against the oracle, row sums, and layout independence (scattered slots give the
    same O and, after un-permuting, the same W as the contiguous layout)."""
    B, Hq, Hkv, q_len, T, D, input_pos = 1, 32, 8, 1024, 32768, 128, 31744
    gen = torch.Generator().manual_seed(1)
    q = torch.randn(B, Hq, q_len, D, generator=gen)
    k = torch.randn(B, Hkv, T, D, generator=gen)
    v = torch.randn(B, Hkv, T, D, generator=gen).to(torch.bfloat16)
    q = O.apply_rope(q, torch.arange(input_pos, input_pos + q_len)).to(torch.bfloat16)
    k = O.apply_rope(k, torch.arange(T)).to(torch.bfloat16)
    scale = D ** -0.5
    out, w, lse = ops.prefill_core(q.to(gpu), k.to(gpu), v.to(gpu), scale, input_pos, None, return_weights=True, return_lse=True)
    torch.cuda.synchronize()
    w_c = w.cpu()
    assert (w_c >= 0).all()
    torch.testing.assert_close(w_c.sum(-1), torch.full((B, Hkv), float(q_len)), rtol=5e-5, atol=3e-2)
    # oracle on KV head 3 (4 query heads)
    h = 3
    o_ref, w_ref = O.sdpa_in_blocks(q[:, 4 * h : 4 * h + 4], k[:, h : h + 1], v[:, h : h + 1], scale, input_pos, None)
    check_o(out.permute(0, 2, 1, 3)[:, 4 * h : 4 * h + 4], o_ref)
    torch.testing.assert_close(w_c[:, h : h + 1], w_ref, rtol=W_RTOL, atol=1e-6)
    # scattered layout: permute slots independently per head
    perm = torch.stack([torch.randperm(T, generator=gen) for _ in range(Hkv)]).view(B, Hkv, T)
    gi = perm.unsqueeze(-1).expand(-1, -1, -1, D)
    out_s, w_s, _ = ops.prefill_core(q.to(gpu), k.gather(2, gi).to(gpu), v.gather(2, gi).to(gpu), scale, input_pos,
                                     perm.to(torch.int32).to(gpu), return_weights=True)
    torch.cuda.synchronize()
    # same values, other summation order and other running maxima: equal up to bf16 rounding
    assert rel_err(out_s.float().cpu(), out.float().cpu()) < 1e-2
    w_back = torch.zeros_like(w_c).scatter_(-1, perm, w_s.cpu())
    torch.testing.assert_close(w_back, w_c, rtol=W_RTOL, atol=1e-6)


def _random_cases(n, seed):
    """Seeded shapes that mix what the fixed cases vary one at a time: group size, head size, ragged
    query and key counts, forced splits, position layout, store."""
    import random

    rnd = random.Random(seed)
    cases = []
    for _ in range(n):
        G = rnd.choice([1, 2, 3, 4, 5, 6, 7, 8])
        Hkv = rnd.choice([1, 2, 3])
        D = rnd.choice([64, 128])
        T = rnd.choice([1, 2, 63, 64, 65, 127, 200, 333, 512, 777, 1025, 2049])
        q_len = rnd.randint(1, min(T, 150))
        cases.append((len(cases), rnd.choice([1, 2]), G * Hkv, Hkv, q_len, T, D, rnd.choice([0, 0, 1, 2, 3, 5]), rnd.choice(["contig", "scattered"]),
                      rnd.choice(["bf16", "bf16", "u8", "u4"])))
    return cases


@pytest.mark.parametrize("case", _random_cases(28, 20240607), ids=lambda c: "-".join(str(x) for x in c))
def test_prefill_and_decode_random_shapes(gpu, case):
    n, B, Hq, Hkv, q_len, T, D, splits, layout, store = case
    q, k, v, gen = make_qkv(5000 + n, B, Hq, Hkv, q_len, T, D)
    scale = 1.0 / math.sqrt(D)
    if layout == "contig":
        input_pos, tp = T - q_len, None
    else:
        input_pos = T + 37
        tp = scattered_positions(gen, B, Hkv, T, input_pos, q_len)
    quant = None
    kg, vg = k.to(gpu), v.to(gpu)
    if store != "bf16":
        bits = 8 if store == "u8" else 4
        (kc, ks, kz), (vc, vs, vz) = O.quantize_rows(k, bits), O.quantize_rows(v, bits)
        k, v = O.dequantize_rows(kc, ks, kz), O.dequantize_rows(vc, vs, vz)
        if bits == 4:
            kc, vc = O.compress4(kc), O.compress4(vc)
        kg, vg = kc.to(gpu), vc.to(gpu)
        quant = ops.QuantState(ks.to(gpu), kz.to(gpu), vs.to(gpu), vz.to(gpu))
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, input_pos, None if tp is None else tp.long())
    out, w, lse = ops.prefill_core(q.to(gpu), kg, vg, scale, input_pos, None if tp is None else tp.to(gpu), return_weights=True,
                                   return_lse=True, output_transposed=False, quant=quant, num_splits=splits)
    torch.cuda.synchronize()
    assert rel_err(out.float().cpu(), o_ref.float()) < 2e-2
    torch.testing.assert_close(w.cpu(), w_ref, rtol=1e-3, atol=1e-6)
    torch.testing.assert_close(lse.cpu(), O.lse2(q, k, scale, input_pos, None if tp is None else tp.long()), rtol=0, atol=2e-3)
    # single-token decode over the same store (unmasked: the new token is the newest)
    o1_ref, w1_ref = O.sdpa_in_blocks(q[:, :, :1], k, v, scale, 10 * T + 100, None)
    out1, w1, _ = ops.decode_core(q[:, :, :1].to(gpu), kg, vg, scale, return_weights=True, quant=quant)
    torch.cuda.synchronize()
    assert rel_err(out1.float().cpu().unsqueeze(2), o1_ref.float()) < 2e-2
    torch.testing.assert_close(w1.cpu(), w1_ref, rtol=1e-3, atol=1e-6)


def _random_cases_wide(n, seed):
    """A second seeded mix over what later builds added: up to 16 heads per KV head, head size 256, float16 rows,
    quantised stores of every one of them."""
    import random

    rnd = random.Random(seed)
    cases = []
    for _ in range(n):
        D = rnd.choice([64, 128, 256])
        G = rnd.choice([1, 2, 4, 6, 8] if D == 256 else [1, 3, 4, 8, 9, 12, 16])
        Hkv = rnd.choice([1, 2])
        T = rnd.choice([3, 64, 97, 256, 511, 1000, 1537])
        q_len = rnd.randint(1, min(T, 100))
        cases.append((len(cases), rnd.choice([1, 2]), G * Hkv, Hkv, q_len, T, D, rnd.choice([0, 0, 2]), rnd.choice(["contig", "scattered"]),
                      rnd.choice(["plain", "u8", "u8", "u4"]), rnd.choice(["bf16", "f16"])))
    return cases


@pytest.mark.parametrize("case", _random_cases_wide(24, 77), ids=lambda c: "-".join(str(x) for x in c))
def test_prefill_and_decode_random_shapes_wide(gpu, case):
    n, B, Hq, Hkv, q_len, T, D, splits, layout, store, dt = case
    dtype = torch.bfloat16 if dt == "bf16" else torch.float16
    q, k, v, gen = make_qkv(9000 + n, B, Hq, Hkv, q_len, T, D, dtype=dtype)
    scale = 1.0 / math.sqrt(D)
    if layout == "contig":
        input_pos, tp = T - q_len, None
    else:
        input_pos = T + 37
        tp = scattered_positions(gen, B, Hkv, T, input_pos, q_len)
    quant = None
    kg, vg = k.to(gpu), v.to(gpu)
    if store != "plain":
        bits = 8 if store == "u8" else 4
        (kc, ks, kz), (vc, vs, vz) = O.quantize_rows(k, bits), O.quantize_rows(v, bits)
        k, v = O.dequantize_rows(kc, ks, kz, dtype), O.dequantize_rows(vc, vs, vz, dtype)
        if bits == 4:
            kc, vc = O.compress4(kc), O.compress4(vc)
        kg, vg = kc.to(gpu), vc.to(gpu)
        quant = ops.QuantState(ks.to(gpu), kz.to(gpu), vs.to(gpu), vz.to(gpu))
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, input_pos, None if tp is None else tp.long())
    out, w, lse = ops.prefill_core(q.to(gpu), kg, vg, scale, input_pos, None if tp is None else tp.to(gpu), return_weights=True,
                                   return_lse=True, output_transposed=False, quant=quant, num_splits=splits)
    torch.cuda.synchronize()
    assert out.dtype == dtype
    assert rel_err(out.float().cpu(), o_ref.float()) < 2e-2
    torch.testing.assert_close(w.cpu(), w_ref, rtol=1e-3, atol=1e-6)
    torch.testing.assert_close(lse.cpu(), O.lse2(q, k, scale, input_pos, None if tp is None else tp.long()), rtol=0, atol=2e-3)
    o1_ref, w1_ref = O.sdpa_in_blocks(q[:, :, :1], k, v, scale, 10 * T + 100, None)
    out1, w1, _ = ops.decode_core(q[:, :, :1].to(gpu), kg, vg, scale, return_weights=True, quant=quant)
    torch.cuda.synchronize()
    assert rel_err(out1.float().cpu().unsqueeze(2), o1_ref.float()) < 2e-2
    torch.testing.assert_close(w1.cpu(), w1_ref, rtol=1e-3, atol=1e-6)


# ---- float16 queries / keys / values and head size 256 (keys_values/attention/flashinfer_wrapper.py:276,311-319) ----

TYPED_CASES = [
    # dtype, B, Hq, Hkv, q_len, T, D, input_pos, scattered, splits
    (torch.float16, 1, 8, 2, 128, 1024, 64, 896, True, 2),
    (torch.float16, 2, 8, 2, 100, 333, 128, 233, False, 3),
    (torch.float16, 1, 4, 4, 37, 700, 128, 1000, True, 0),
    (torch.float16, 1, 4, 2, 70, 300, 256, 400, True, 2),
    (torch.bfloat16, 1, 8, 2, 128, 1024, 256, 896, True, 0),
    (torch.bfloat16, 2, 4, 1, 33, 200, 256, 167, False, 1),
    (torch.bfloat16, 1, 4, 2, 300, 300, 256, 0, False, 2),  # square causal prefill
    (torch.float16, 1, 16, 2, 40, 900, 128, 1000, True, 0),  # 8 heads per KV head: the decode step multiplies on the matrix cores
    (torch.float16, 1, 16, 1, 20, 450, 64, 500, False, 0),
]


@pytest.mark.parametrize("dtype,B,Hq,Hkv,q_len,T,D,input_pos,scattered,splits", TYPED_CASES)
def test_prefill_decode_fp16_and_head_size_256(gpu, dtype, B, Hq, Hkv, q_len, T, D, input_pos, scattered, splits):
    q, k, v, gen = make_qkv(200 + T + q_len + D, B, Hq, Hkv, q_len, T, D, dtype=dtype)
    tp = scattered_positions(gen, B, Hkv, T, input_pos, q_len) if scattered else None
    if tp is None and input_pos != T - q_len:
        tp = (torch.arange(T, dtype=torch.int32) + (input_pos - (T - q_len))).view(1, 1, T).expand(B, Hkv, T).contiguous()
    scale = 1.0 / math.sqrt(D)
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, input_pos, None if tp is None else tp.to(torch.int64))
    l_ref = O.lse2(q, k, scale, input_pos, tp)
    out, w, lse = ops.prefill_core(q.to(gpu), k.to(gpu), v.to(gpu), scale, input_pos, None if tp is None else tp.to(gpu),
                                   return_weights=True, return_lse=True, output_transposed=False, num_splits=splits)
    torch.cuda.synchronize()
    assert out.dtype == dtype
    check_o(out, o_ref)
    torch.testing.assert_close(lse.cpu(), l_ref, rtol=1e-4, atol=1e-3)
    check_w(w, w_ref, q_len)
    # the score-sum kernel alone, fed the oracle's log-sum-exp
    w2 = ops.score_sum_core(q.to(gpu), k.to(gpu), l_ref.to(gpu), scale, input_pos, None if tp is None else tp.to(gpu))
    check_w(w2, w_ref, q_len)
    # one new token over the same cache
    o1_ref, w1_ref = O.sdpa_in_blocks(q[:, :, :1], k, v, scale, 10 * T, None)
    out1, w1, lse1 = ops.decode_core(q[:, :, :1].to(gpu), k.to(gpu), v.to(gpu), scale, return_weights=True, return_lse=True)
    torch.cuda.synchronize()
    assert out1.dtype == dtype
    check_o(out1.unsqueeze(2), o1_ref)
    check_w(w1, w1_ref, 1)
    torch.testing.assert_close(lse1.cpu(), O.lse2(q[:, :, :1], k, scale, 10 * T, None), rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("dtype,D", [(torch.float16, 128), (torch.bfloat16, 256), (torch.float16, 256)])
def test_h2o_cache_steps_fp16_and_head_size_256(gpu, dtype, D):
    """The cache object with float16 rows / heads of 256: prefill, chunk steps and a single-token step
    against the oracle (the slot write is a copy of 16-bit rows, the V-norm policy reads them as float16)."""
    from keys_values_amd.kvcache.h2o import H2OKVCache, KVCacheParams

    B, Hq, Hkv, L, chunk = 1, 4, 2, 256, 32
    gen = torch.Generator().manual_seed(D)
    total = L + 2 * chunk + 1
    qs = torch.randn(B, Hq, total, D, generator=gen).to(dtype)
    ks = torch.randn(B, Hkv, total, D, generator=gen).to(dtype)
    vs = torch.randn(B, Hkv, total, D, generator=gen).to(dtype)
    ref = O.H2OCacheOracle(B, Hq, Hkv, L, D, dtype=dtype, max_chunk_size=chunk)
    cache = H2OKVCache(KVCacheParams(B, Hkv, L, D, Hq, dtype), max_chunk_size=chunk, device=gpu)
    ref.prefill(qs[:, :, :L], ks[:, :, :L], vs[:, :, :L])
    cache.forward(qs[:, :, :L].to(gpu), ks[:, :, :L].to(gpu), vs[:, :, :L].to(gpu))
    pos = L
    for num in (chunk, chunk, 1):
        sl = slice(pos, pos + num)
        had = ref.next_index is not None
        o_ref, _, index = ref.forward(qs[:, :, sl], ks[:, :, sl], vs[:, :, sl])
        if had:
            cache.set_next_positions(index)
        o = cache.forward(qs[:, :, sl].to(gpu), ks[:, :, sl].to(gpu), vs[:, :, sl].to(gpu))
        torch.cuda.synchronize()
        assert o.dtype == dtype
        assert rel_err(o.float().cpu().view(B, num, Hq, D).transpose(1, 2), o_ref.float()) < 2e-2
        assert torch.equal(cache.k.cpu(), ref.k) and torch.equal(cache.v.cpu(), ref.v)
        assert torch.equal(cache.token_pos.cpu(), ref.token_pos)
        torch.testing.assert_close(cache.scores.cpu(), ref.scores, rtol=2e-3, atol=1e-5)
        pos += num


def test_gate_mirrors_the_reference(gpu):
    from keys_values_amd.attention.sdpa import can_do_hip_sdpa

    # keys_values/attention/flashinfer_wrapper.py:311-319: float16 or bfloat16, head sizes up to 256
    for dtype in (torch.float16, torch.bfloat16):
        for hs in (1, 48, 64, 100, 128, 200, 256):
            assert can_do_hip_sdpa(hs, dtype, True) and can_do_hip_sdpa(hs, dtype, False)
        assert not can_do_hip_sdpa(257, dtype)
    assert not can_do_hip_sdpa(128, torch.float32)
    # zero-padding from 129..255 to 256
    B, Hq, Hkv, q_len, T, D = 1, 4, 2, 9, 70, 200
    q, k, v, gen = make_qkv(43, B, Hq, Hkv, q_len, T, D, dtype=torch.float16)
    tp = scattered_positions(gen, B, Hkv, T, 100, q_len)
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, 1 / math.sqrt(D), 100, tp.to(torch.int64))
    out, w = HipSDPA().scaled_dot_product_attention(q.to(gpu), k.to(gpu), v.to(gpu), None, 100, tp.to(gpu), return_attn_weights=True)
    assert out.shape == (B, Hq, q_len, D) and out.dtype == torch.float16
    check_o(out, o_ref)
    check_w(w, w_ref, q_len)


def test_decode_with_weights_beside_other_work(gpu):
    """The split kernel's wait for its row's other splits while another stream keeps the compute units busy
    (its workgroups then start at scattered times): same bits as on an idle device."""
    B, Hq, Hkv, T, D = 2, 8, 2, 30000, 128
    q, k, v, _ = make_qkv(4242, B, Hq, Hkv, 1, T, D)
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    scale = 1.0 / math.sqrt(D)
    out0, w0, lse0 = ops.decode_core(qg, kg, vg, scale, return_weights=True, return_lse=True)
    torch.cuda.synchronize()
    side = torch.cuda.Stream(gpu)
    busy = torch.randn(4096, 4096, device=gpu, dtype=torch.bfloat16)
    side.wait_stream(torch.cuda.current_stream(gpu))  # `busy` was made on the current stream
    for _ in range(3):
        with torch.cuda.stream(side):
            for _ in range(20):
                busy = (busy @ busy).clamp_(-1, 1)
        out1, w1, lse1 = ops.decode_core(qg, kg, vg, scale, return_weights=True, return_lse=True)
        torch.cuda.synchronize()
        assert torch.equal(out0, out1) and torch.equal(w0, w1) and torch.equal(lse0, lse1)
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, T - 1, None)
    check_o(out0.unsqueeze(2), o_ref)
    check_w(w0, w_ref, 1)


@pytest.mark.parametrize("T", [777, 5000, 9001])
@pytest.mark.parametrize("D,G,store", [(128, 4, "plain"), (64, 1, "plain"), (128, 8, "plain"), (128, 4, "u8"), (256, 2, "u4")])
def test_decode_output_at_large_logits(gpu, decode_route, D, G, store, T):
    """Every key the same row, the logits around 10^6: all weights are equal and the output is the mean of the V rows,
    whatever the logits round to. Outputs are float16 (each within 2^-11 of its value) and sums run in float32, so 1e-3
    covers both; a normaliser taken from a log-sum-exp in float32 is off by up to 2^-5 here."""
    Hkv = 2
    gen = torch.Generator(device=gpu).manual_seed(T + D + G)

    def uniform(*shape):
        return (200 + 100 * torch.rand(*shape, generator=gen, device=gpu)).to(torch.float16)

    q = uniform(1, Hkv * G, 1, D)
    k = uniform(1, Hkv, 1, D).expand(1, Hkv, T, D).contiguous()
    v = (torch.randn(1, Hkv, T, D, generator=gen, device=gpu) + 1).to(torch.float16)
    quant, kd, vd = None, k, v
    if store != "plain":
        codes, state, rows = [], [], []
        for x in (k, v):
            qz = RowQuantizer((1, Hkv, T, D), torch.float16, 8 if store == "u8" else 4, allocate_buffers=True, device=gpu)
            qz.quantize(0, T, x)
            codes.append(qz.quant_buffer.view(1, Hkv, T, -1))
            state += [qz.quant_scales.view(1, Hkv, T), qz.quant_zero_points.view(1, Hkv, T)]
            rows.append(qz.dequantize(0, T))
        (kd, vd), (k, v), quant = codes, rows, ops.QuantState(*state)
    want = v.double().mean(2).repeat_interleave(G, 1)
    for weights in (True, False):
        out, _, lse = ops.decode_core(q, kd, vd, D ** -0.5, return_weights=weights, return_lse=True, quant=quant)
        assert lse.min() > 2.0 ** 17
        assert rel_err(out, want) < 1e-3, (weights, rel_err(out, want))


def test_decode_without_weights_beside_other_work(gpu, decode_route):
    """Without weights the splits of a row wait for each other too, before each writes its share of the outputs; where the
    wait runs out the last one makes up for it. The same bits whoever does."""
    B, Hq, Hkv, T, D = 2, 8, 2, 30000, 128
    q, k, v, _ = make_qkv(4243, B, Hq, Hkv, 1, T, D)
    qg, kg, vg = q.to(gpu), k.to(gpu), v.to(gpu)
    scale = 1.0 / math.sqrt(D)
    out0, _, lse0 = ops.decode_core(qg, kg, vg, scale, return_lse=True)
    torch.cuda.synchronize()
    side = torch.cuda.Stream(gpu)
    busy = torch.randn(4096, 4096, device=gpu, dtype=torch.bfloat16)
    side.wait_stream(torch.cuda.current_stream(gpu))
    for _ in range(3):
        with torch.cuda.stream(side):
            for _ in range(20):
                busy = (busy @ busy).clamp_(-1, 1)
        out1, _, lse1 = ops.decode_core(qg, kg, vg, scale, return_lse=True)
        torch.cuda.synchronize()
        assert torch.equal(out0, out1) and torch.equal(lse0, lse1)
    o_ref, _ = O.sdpa_in_blocks(q, k, v, scale, T - 1, None)
    check_o(out0.unsqueeze(2), o_ref)
    torch.testing.assert_close(lse0.cpu(), O.lse2(q, k, scale, T - 1, None), rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("store", ["bf16", "u8", "u4"])
@pytest.mark.parametrize("B,Hq,Hkv,q_len,T,D,splits", [
    (1, 24, 8, 11, 32769, 128, 0),    # 33 rows: two blocks over 8 x 32769 keys, their combination in a launch of its own
    (1, 24, 8, 10, 32769, 128, 0),    # 30 rows, their combination in the same launch
    (2, 28, 4, 36, 32800, 128, 3),    # 252 rows, more than the launch combines: a launch of its own
    (1, 16, 8, 128, 32768, 128, 2),   # 256 rows, the most
    (1, 8, 8, 257, 32768, 128, 2),    # one more: the tiled kernel
    (2, 10, 2, 26, 65536, 256, 2),    # 130 rows of 256: the tiled kernel
    (2, 8, 2, 32, 65540, 256, 5),     # 128 rows of 256, the most
    (1, 16, 4, 10, 65600, 256, 0),    # 40 rows of 256
])
def test_score_sums_with_streamed_keys_of_long_rows(gpu, store, B, Hq, Hkv, q_len, T, D, splits):
    """Several blocks of rows over 256 K keys and more. The oracle takes one KV head of each batch element (its heads do not
    meet); the others are checked by the sum of their weights."""
    _check_some_heads(gpu, store, torch.bfloat16, B, Hq, Hkv, q_len, T, D, splits)


@pytest.mark.parametrize("store", ["plain", "u8", "u4"])
@pytest.mark.parametrize("B,Hq,Hkv,q_len,T,D,splits", [
    (2, 6, 2, 43, 190, 128, 3),       # few rows over few keys
    (1, 12, 1, 85, 700, 256, 2),
    (2, 8, 8, 4, 1100, 64, 2),        # streamed keys
    (2, 24, 8, 10, 1090, 256, 5),
    (1, 16, 8, 20, 32768, 128, 0),
    (1, 7, 1, 298, 4500, 64, 0),      # tiles of whole queries
    (2, 6, 2, 460, 900, 128, 0),
])
def test_score_sums_over_float16_stores(gpu, store, B, Hq, Hkv, q_len, T, D, splits):
    """The three score-sum kernels on float16 rows and on codes that dequantise to them."""
    _check_some_heads(gpu, store, torch.float16, B, Hq, Hkv, q_len, T, D, splits)


def _check_some_heads(gpu, store, dtype, B, Hq, Hkv, q_len, T, D, splits):
    G = Hq // Hkv
    gen = torch.Generator(device=gpu).manual_seed(T + q_len)
    q, k, v = (torch.randn(B, h, n, D, generator=gen, device=gpu).to(dtype) for h, n in ((Hq, q_len), (Hkv, T), (Hkv, T)))
    quant, kd, vd = None, k, v
    if store in ("u8", "u4"):
        codes, state, rows = [], [], []
        for x in (k, v):
            qz = RowQuantizer((B, Hkv, T, D), dtype, 8 if store == "u8" else 4, allocate_buffers=True, device=gpu)
            qz.quantize(0, T, x)
            codes.append(qz.quant_buffer.view(B, Hkv, T, -1))
            state += [qz.quant_scales.view(B, Hkv, T), qz.quant_zero_points.view(B, Hkv, T)]
            rows.append(qz.dequantize(0, T))
        (kd, vd), (k, v), quant = codes, rows, ops.QuantState(*state)
    scale, pos = D ** -0.5, T - q_len
    # every position in a slot of another KV head's order: the newest ones are spread over the row
    tp = torch.rand(B, Hkv, T, generator=gen, device=gpu).argsort(-1).to(torch.int32)
    out, w, lse = ops.prefill_core(q, kd, vd, scale, pos, tp, return_weights=True, return_lse=True, output_transposed=False, quant=quant, num_splits=splits)
    torch.testing.assert_close(w.sum(-1).cpu(), torch.full((B, Hkv), float(q_len)), rtol=5e-5, atol=3e-4)
    for b in range(B):
        h = (Hkv - 1 + b) % Hkv
        one, heads = slice(b, b + 1), slice(G * h, G * h + G)
        qc, kc, vc, tc = q[one, heads].cpu(), k[one, h : h + 1].cpu(), v[one, h : h + 1].cpu(), tp[one, h : h + 1].cpu()
        o_ref, w_ref = O.sdpa_in_blocks(qc, kc, vc, scale, pos, tc.to(torch.int64))
        assert rel_err(out[one, heads].float().cpu(), o_ref.float()) < O_RTOL
        torch.testing.assert_close(w[one, h : h + 1].cpu(), w_ref, rtol=W_RTOL, atol=1e-6)
        torch.testing.assert_close(lse[one, :, heads].cpu(), O.lse2(qc, kc, scale, pos, tc), rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("dtype,B,Hq,Hkv,q_len,behind,D", [
    (torch.bfloat16, 1, 8, 2, 2048, 0, 128),   # whole periods of blocks
    (torch.float16, 1, 7, 1, 2311, 0, 128),    # 7 heads: splits of an even number of tiles; the last period short, its last block ragged
    (torch.bfloat16, 1, 2, 1, 4000, 77, 128),  # keys that nobody sees behind the chunk
    (torch.bfloat16, 1, 12, 2, 1921, 0, 64),   # one token beyond 30 tiles
    (torch.float16, 1, 4, 2, 1500, 1, 256),
    (torch.bfloat16, 1, 1, 1, 9000, 0, 64),    # one head, many splits
])
def test_causal_first_chunk_in_splits(gpu, dtype, B, Hq, Hkv, q_len, behind, D):
    # tolerances of the path; and against the same call in one split and in three of all rows alike
    T, scale = q_len + behind, D ** -0.5
    q, k, v, _ = make_qkv(17 + T, B, Hq, Hkv, q_len, T, D, dtype=dtype)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    out, _, lse = ops.prefill_core(qd, kd, vd, scale, 0, return_lse=True, output_transposed=False)
    for splits in (1, 3):
        o2, _, l2 = ops.prefill_core(qd, kd, vd, scale, 0, return_lse=True, output_transposed=False, num_splits=splits)
        check_o(out, o2.cpu())
        torch.testing.assert_close(lse, l2, rtol=1e-4, atol=1e-3)
    heads = slice(0, Hq // Hkv)  # one KV head against the oracle
    qc, kc, vc = q[:1, heads], k[:1, :1], v[:1, :1]
    check_o(out[:1, heads], O.sdpa_in_blocks(qc, kc, vc, scale, 0, None)[0])
    torch.testing.assert_close(lse[:1, :, heads].cpu(), O.lse2(qc, kc, scale, 0, None), rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("B,Hq,Hkv,q_len,T,D", [
    (1, 4, 1, 256, 256, 256),
    (1, 16, 16, 1024, 1024, 128),
    (1, 16, 16, 1000, 1024, 64),   # keys that nobody sees behind the chunk
    (1, 16, 8, 511, 1024, 128),    # 1022 rows
])
def test_causal_first_chunk_in_splits_with_weights(kvx, gpu, B, Hq, Hkv, q_len, T, D):
    """Splits that the score-sum launch combines, in a workspace of NaN: what the attention kernel leaves unwritten is not used.
    Tolerances of the path."""
    q, k, v, _ = make_qkv(27 + T, B, Hq, Hkv, q_len, T, D)
    scale = D ** -0.5
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    assert block_rows(kvx, qd, kd, vd, 0) >= 128
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, 0, None)
    l_ref = O.lse2(q, k, scale, 0, None)
    a = _lib.SdpaArgs()
    ops._fill_common(a, qd, kd, vd, scale, 0, None, None, 0)
    n = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    rows = B * Hq * q_len * (D + 2) * 4
    assert n >= 2 * rows and n % rows == 0  # splits, and no sums of the score-sum pass: it combines them
    for call in (kvx.kvx_sdpa_prefill_weights, kvx.kvx_sdpa_prefill):
        ws = torch.full((n // 4,), math.nan, device=gpu)
        out, lse = torch.full_like(qd, math.nan), torch.full((B, q_len, Hq), math.nan, device=gpu)
        w = torch.full((B, Hkv, T), math.nan, device=gpu)
        a.o, a.lse, a.w, a.workspace, a.workspace_bytes = out.data_ptr(), lse.data_ptr(), w.data_ptr(), ws.data_ptr(), n
        a.o_stride_b, a.o_stride_h, a.o_stride_t = out.stride(0), out.stride(1), out.stride(2)
        _lib.check(call(ctypes.byref(a), _lib.stream_ptr(gpu)))
        check_o(out, o_ref)
        torch.testing.assert_close(lse.cpu(), l_ref, rtol=1e-4, atol=1e-3)
        if call is kvx.kvx_sdpa_prefill_weights:
            check_w(w, w_ref, q_len)


@pytest.mark.parametrize("Hq,Hkv,q_len,splits", [
    (1, 1, 380, 6),    # splits of a tile, for all rows alike
    (24, 8, 353, 1),   # a merge that costs more than splits save
    (24, 8, 196, 1),
])
def test_splits_of_short_first_chunks_without_weights(kvx, gpu, Hq, Hkv, q_len, splits):
    # what is written of a workspace of NaN tells the splits: a maximum and a sum for every row in each. Tolerances of the path.
    D, scale = 256, 0.0625
    q, k, v, _ = make_qkv(q_len, 1, Hq, Hkv, q_len, q_len, D)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    a = _lib.SdpaArgs()
    ops._fill_common(a, qd, kd, vd, scale, 0, None, None, 0)
    n = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    ws, out = torch.full((n // 4,), math.nan, device=gpu), torch.full_like(qd, math.nan)
    a.o, a.workspace, a.workspace_bytes = out.data_ptr(), ws.data_ptr(), n
    a.o_stride_b, a.o_stride_h, a.o_stride_t = out.stride(0), out.stride(1), out.stride(2)
    _lib.check(kvx.kvx_sdpa_prefill(ctypes.byref(a), _lib.stream_ptr(gpu)))
    check_o(out, O.sdpa_in_blocks(q, k, v, scale, 0, None)[0])
    rows = Hq * q_len
    if splits == 1:
        assert torch.isnan(ws).all()
    else:
        assert ws.numel() == splits * rows * (D + 2) and not torch.isnan(ws[splits * rows * D:]).any()


@pytest.mark.parametrize("room", [False, True])
@pytest.mark.parametrize("store,Hq,Hkv,q_len,T,D", [
    ("plain", 32, 2, 2, 384, 128),   # with room one split a step of keys, without it one split
    ("plain", 16, 8, 72, 571, 64),
    ("u8", 64, 8, 2, 235, 128),
])
def test_weights_of_few_rows_with_and_without_a_workspace(kvx, gpu, store, Hq, Hkv, q_len, T, D, room):
    """Splits are nearly free where the score-sum launch combines them, and a call takes more of them if the workspace has room. Tolerances
    of the path."""
    q, k, v, _ = make_qkv(31 + T, 1, Hq, Hkv, q_len, T, D)
    kd, vd, quant = k.to(gpu), v.to(gpu), None
    if store == "u8":
        (kc, ks, kz), (vc, vs, vz) = (O.quantize_rows(x.reshape(-1, D), 8) for x in (k, v))
        k, v = (O.dequantize_rows(*t, torch.bfloat16).view(1, Hkv, T, D) for t in ((kc, ks, kz), (vc, vs, vz)))
        kd, vd = kc.view(1, Hkv, T, D).to(gpu), vc.view(1, Hkv, T, D).to(gpu)
        quant = ops.QuantState(*(t.view(1, Hkv, T).to(gpu) for t in (ks, kz, vs, vz)))
    scale, pos, qd = D ** -0.5, T - q_len, q.to(gpu)
    o_ref, w_ref = O.sdpa_in_blocks(q, k, v, scale, pos, None)
    a = _lib.SdpaArgs()
    ops._fill_common(a, qd, kd, vd, scale, pos, None, quant, 0)
    n = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    assert n > 0 and block_rows(kvx, qd, kd, vd, pos, None, quant) <= 32
    ws = torch.full((n // 4,), math.nan, device=gpu)
    out, lse = torch.full_like(qd, math.nan), torch.full((1, q_len, Hq), math.nan, device=gpu)
    w = torch.full((1, Hkv, T), math.nan, device=gpu)
    a.o, a.lse, a.w = out.data_ptr(), lse.data_ptr(), w.data_ptr()
    a.o_stride_b, a.o_stride_h, a.o_stride_t = out.stride(0), out.stride(1), out.stride(2)
    if room:
        a.workspace, a.workspace_bytes = ws.data_ptr(), n
    _lib.check(kvx.kvx_sdpa_prefill_weights(ctypes.byref(a), _lib.stream_ptr(gpu)))
    check_o(out, o_ref)
    check_w(w, w_ref, q_len)
    torch.testing.assert_close(lse.cpu(), O.lse2(q, k, scale, pos, None), rtol=1e-4, atol=1e-3)
    assert torch.isnan(ws).all().item() != room  # the splits' results lie there
