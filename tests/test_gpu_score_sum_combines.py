"""Attention with weights where the launches of the tiled score-sum kernel combine the attention's KV splits (csrc/score_sum.hip): workgroups beside the score
jobs, or the launch that adds the sums of a split of the query rows. Against the CPU oracle, and bit for bit against the attention alone, which combines the
splits in a launch of their own, and the score-sums from its log-sum-exps; where the query rows are split also against the same call without the workspace for
both. Every case asserts that the library takes it that way (on 256 compute units)."""
import ctypes

import pytest
import torch

from helpers import make_qkv, prefill_plan, scattered_positions
from keys_values_amd import _lib
from keys_values_amd.attention import ops
from keys_values_amd.kvcache.quantize import RowQuantizer
from oracle import kvx_oracle as O
from test_gpu_pairs import check_out, prepare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,B,Hq,Hkv,q_len,T,D,where,teams,splits", [
    (torch.bfloat16, 1, 32, 8, 101, 3013, 128, "end", 2, 6),          # a last block of 20 rows, twelve pairs of the splits a row
    (torch.float16, 1, 28, 4, 150, 1343, 128, "scattered", 2, 4),     # seven heads a KV head: tiles of 63 rows
    (torch.bfloat16, 2, 32, 8, 35, 2443, 128, "start", 2, 7),         # splits that no row sees
    (torch.float16, 1, 24, 8, 110, 2129, 256, "end", 1, 9),           # more than eight pairs a row, one team
    (torch.bfloat16, 1, 16, 8, 858, 1800, 64, "scattered", 2, 2),
    (torch.float16, 1, 64, 4, 170, 4161, 64, "end", 1, 5),            # a key in the last tile
    (torch.bfloat16, 2, 24, 8, 200, 4100, 128, "scattered", 2, 3),    # beside workgroups of eight wavefronts
])
def test_launches_of_the_weights_combine_the_splits(kvx, gpu, dtype, B, Hq, Hkv, q_len, T, D, where, teams, splits):
    a, _tensors, out, lse, ref = prepare(gpu, dtype, B, Hq, Hkv, q_len, T, D, where)
    w = torch.full((B, Hkv, T), float("nan"), device=gpu)
    without = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))  # of the call without weights: the partials alone
    a.w = w.data_ptr()
    plan = prefill_plan(a)
    assert (plan.one_launch, plan.teams, plan.splits, plan.score_sum, plan.combined) == (0, teams, splits, _lib.KVX_SCORE_SUM_TILED, 1)
    need = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    bits = []
    for n in (need, need, without):
        ws = torch.full((n,), 255, dtype=torch.uint8, device=gpu)
        a.workspace, a.workspace_bytes = ws.data_ptr(), n
        for t in (out, lse, w):
            t.fill_(float("nan"))
        _lib.check(kvx.kvx_sdpa_prefill_weights(ctypes.byref(a), _lib.stream_ptr(gpu)))
        check_out(out, lse, ref)
        torch.testing.assert_close(w.cpu(), ref[1], rtol=1e-3, atol=1e-6)
        bits.append([t.clone() for t in (out, lse)])
    for other in bits[1:]:
        assert all(torch.equal(x, y) for x, y in zip(bits[0], other))


@pytest.mark.parametrize("dtype,bits,copying,B,Hq,Hkv,q_len,T,D,where,block,teams,splits,rows_split", [
    # workgroups beside the score jobs
    (torch.bfloat16, 16, 0, 2, 32, 8, 35, 2443, 128, "start", 128, 2, 7, 0),
    (torch.bfloat16, 16, 0, 2, 24, 8, 200, 4100, 128, "scattered", 128, 2, 3, 0),  # of eight wavefronts
    (torch.bfloat16, 8, 0, 2, 16, 8, 402, 2972, 64, "end", 256, 1, 4, 0),          # likewise, over codes
    (torch.bfloat16, 16, 0, 1, 8, 8, 307, 3086, 128, "end", 128, 2, 9, 0),         # 18 pairs a row, of two lanes
    (torch.float16, 16, 0, 1, 32, 8, 64, 3314, 128, "scattered", 128, 2, 9, 0),
    (torch.float16, 8, 0, 1, 32, 8, 64, 7425, 128, "scattered", 256, 1, 30, 0),
    (torch.float16, 4, 0, 2, 16, 4, 44, 2360, 256, "end", 128, 1, 13, 0),
    (torch.bfloat16, 4, 0, 1, 16, 8, 256, 2899, 64, "scattered", 256, 1, 16, 0),
    # the launch that adds the sums of a split of the query rows
    (torch.bfloat16, 16, 0, 1, 6, 2, 343, 3768, 128, "end", 128, 2, 10, 1),
    (torch.float16, 16, 0, 2, 6, 2, 99, 5327, 256, "start", 128, 1, 21, 1),        # an odd number of pairs over two lanes
    (torch.bfloat16, 8, 0, 1, 8, 2, 277, 2928, 128, "end", 256, 1, 23, 1),
    (torch.bfloat16, 8, 0, 1, 32, 4, 34, 4285, 256, "start", 128, 1, 17, 1),
    # partials of the kernel for few rows
    (torch.bfloat16, 16, 0, 2, 16, 4, 51, 4003, 64, "end", 32, 1, 4, 0),
    (torch.bfloat16, 16, 0, 1, 8, 2, 426, 1973, 64, "scattered", 32, 1, 2, 1),
    (torch.bfloat16, 4, 0, 2, 16, 8, 81, 1886, 128, "start", 32, 1, 5, 0),
    (torch.float16, 4, 0, 1, 8, 2, 259, 2567, 128, "scattered", 32, 1, 7, 1),
    # over the dequantised copy: the rows' sums take its place
    (torch.bfloat16, 8, 1, 1, 8, 2, 575, 1227, 128, "end", 128, 2, 5, 1),
    (torch.float16, 4, 1, 1, 16, 4, 144, 5890, 128, "scattered", 128, 2, 12, 1),
    (torch.float16, 8, 1, 2, 8, 2, 67, 4471, 256, "end", 128, 1, 18, 1),
    (torch.bfloat16, 4, 1, 1, 8, 2, 523, 1501, 64, "start", 32, 1, 3, 1),
])
def test_same_bits_as_launches_of_their_own(kvx, gpu, dtype, bits, copying, B, Hq, Hkv, q_len, T, D, where, block, teams, splits, rows_split):
    q, k, v, gen = make_qkv(700 + T + q_len, B, Hq, Hkv, q_len, T, D, dtype=dtype)
    pos, tp = {"end": T - q_len, "start": 1, "scattered": 2 * T}[where], None
    if where == "scattered":
        tp = scattered_positions(gen, B, Hkv, T, pos, q_len)
    stores, quant = [k.to(gpu), v.to(gpu)], None
    if bits < 16:
        stores, states = [], []
        for x in (k, v):
            qz = RowQuantizer((B, Hkv, T, D), dtype, bits, allocate_buffers=True, device=gpu)
            qz.quantize(0, T, x.to(gpu))
            x.copy_(qz.dequantize(0, T).view(x.shape))
            stores.append(qz.quant_buffer.view(B, Hkv, T, -1))
            states += [qz.quant_scales.view(B, Hkv, T), qz.quant_zero_points.view(B, Hkv, T)]
        quant = ops.QuantState(*states)
    scale = D ** -0.5
    ref = *O.sdpa_in_blocks(q, k, v, scale, pos, None if tp is None else tp.to(torch.int64)), O.lse2(q, k, scale, pos, tp)
    q, tp = q.to(gpu), None if tp is None else tp.to(gpu)
    a = _lib.SdpaArgs()
    ops._fill_common(a, q, *stores, scale, pos, tp, quant, 0)
    out = torch.empty(B, Hq, q_len, D, dtype=dtype, device=gpu)
    lse, w = torch.empty(B, q_len, Hq, device=gpu), torch.empty(B, Hkv, T, device=gpu)
    a.o, a.lse = out.data_ptr(), lse.data_ptr()
    a.o_stride_b, a.o_stride_h, a.o_stride_t = out.stride()[:3]
    size = kvx.kvx_sdpa_prefill_copying_workspace_bytes if copying else kvx.kvx_sdpa_prefill_workspace_bytes
    attend = kvx.kvx_sdpa_prefill_copying if copying else kvx.kvx_sdpa_prefill
    one = _lib.SdpaArgs.from_buffer_copy(a)
    one.num_splits = 1
    assert (kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(one)) > 0) == rows_split  # without partials: the sums of a split of the query rows

    def run(call, n):
        ws = torch.full((max(n, 16),), 255, dtype=torch.uint8, device=gpu)
        a.workspace, a.workspace_bytes = ws.data_ptr(), n
        _lib.check(call(ctypes.byref(a), _lib.stream_ptr(gpu)))
        return [t.clone() for t in (out, lse, w)]

    for t in (out, lse, w):
        t.fill_(float("nan"))
    run(attend, size(ctypes.byref(a)))  # the attention alone, its splits combined in a launch of their own
    sums = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    a.w = w.data_ptr()
    plan = prefill_plan(a, copying)
    assert (plan.one_launch, plan.copied, plan.block_rows, plan.teams, plan.splits, plan.score_sum, plan.combined) == (
        0, copying, block, teams, splits, _lib.KVX_SCORE_SUM_TILED, 1)
    want = run(kvx.kvx_score_sum, sums)
    for t in (out, lse, w):
        t.fill_(float("nan"))
    for _ in range(2):
        got = run(attend if copying else kvx.kvx_sdpa_prefill_weights, size(ctypes.byref(a)))
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        if teams * splits <= 16:
            assert torch.equal(got[2], want[2])
        else:
            # the sums of 32 terms 32 roundings apart, log-sum-exps below 32 rounded twice: exponents 2.8e-6 + 2e-6 apart, times ln 2
            torch.testing.assert_close(got[2], want[2], rtol=4e-6, atol=0)
    check_out(out, lse, ref)
    torch.testing.assert_close(w.cpu(), ref[1], rtol=1e-3, atol=1e-6)


@pytest.mark.parametrize("kv_len,combined", [(19968, 1), (19969, 0)])
def test_on_both_sides_of_the_line_of_long_stores(kvx, gpu, kv_len, combined):
    q, k, v, _ = make_qkv(41, 1, 28, 4, 340, kv_len, 128)
    q, k, v = q.to(gpu), k.to(gpu), v.to(gpu)
    scale, pos = 128 ** -0.5, kv_len - 340
    a = _lib.SdpaArgs()
    ops._fill_common(a, q, k, v, scale, pos, None, None, 0)
    a.o = a.lse = a.w = q.data_ptr()  # nothing is launched: any aligned address
    assert prefill_plan(a).combined == combined
    out, w, lse = ops.prefill_core(q, k, v, scale, pos, return_weights=True, return_lse=True)
    out1, _, lse1 = ops.prefill_core(q, k, v, scale, pos, return_lse=True)
    assert torch.equal(out, out1) and torch.equal(lse, lse1)
    assert torch.equal(w, ops.score_sum_core(q, k, lse, scale, pos))
