"""The tiled attention kernel (csrc/sdpa_prefill.hip) where wavefronts of a workgroup lie behind the last row: they bring tiles and multiply nothing. Against
the CPU oracle (over a quantised store: of its dequantised rows). Every case asserts its blocks of rows."""
import ctypes

import pytest
import torch

from helpers import make_qkv, prefill_plan, scattered_positions
from keys_values_amd import _lib
from keys_values_amd.attention import ops
from keys_values_amd.kvcache.quantize import RowQuantizer
from oracle import kvx_oracle as O
from test_gpu_pairs import check_out

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,bits,B,Hq,Hkv,q_len,T,D,where,block,teams", [
    (torch.bfloat16, 8, 1, 32, 8, 32, 12801, 128, "scattered", 256, 1),  # 128 rows: four of eight wavefronts; a last tile of one key
    (torch.float16, 4, 1, 28, 4, 15, 15000, 128, "end", 256, 1),         # 105 rows
    (torch.bfloat16, 8, 2, 8, 8, 67, 9090, 128, "start", 256, 1),        # three rows in the third wavefront; splits that no row sees
    (torch.float16, 8, 1, 16, 4, 31, 40000, 64, "end", 256, 1),
    (torch.bfloat16, 4, 1, 32, 4, 16, 33153, 64, "scattered", 256, 1),
    (torch.bfloat16, 8, 16, 32, 8, 72, 600, 128, "end", 256, 1),        # a whole block of rows ahead of one wavefront's
    (torch.bfloat16, 16, 1, 32, 8, 33, 5000, 128, "scattered", 128, 2), # plain rows, two teams: a block of four rows
    (torch.float16, 16, 1, 8, 2, 1001, 1001, 128, "first", 128, 1),     # a first chunk in splits that end at bounds of blocks
    (torch.float16, 16, 2, 24, 8, 43, 4000, 64, "end", 128, 2),
])
def test_wavefronts_without_rows(kvx, gpu, dtype, bits, B, Hq, Hkv, q_len, T, D, where, block, teams):
    q, k, v, gen = make_qkv(500 + T + q_len, B, Hq, Hkv, q_len, T, D, dtype=dtype)
    pos, tp = {"end": T - q_len, "start": 1, "scattered": 2 * T, "first": 0}[where], None
    if where == "scattered":
        tp = scattered_positions(gen, B, Hkv, T, pos, q_len)
    a = _lib.SdpaArgs()
    rows, quant = [], None
    if bits < 16:
        for x in (k, v):
            qz = RowQuantizer((B, Hkv, T, D), dtype, bits, allocate_buffers=True, device=gpu)
            qz.quantize(0, T, x.to(gpu))
            x.copy_(qz.dequantize(0, T).view(x.shape))
            rows.append((qz.quant_buffer.view(B, Hkv, T, -1), qz.quant_scales.view(B, Hkv, T), qz.quant_zero_points.view(B, Hkv, T)))
        quant = ops.QuantState(rows[0][1], rows[0][2], rows[1][1], rows[1][2])
    scale = D ** -0.5
    ref = *O.sdpa_in_blocks(q, k, v, scale, pos, None if tp is None else tp.to(torch.int64)), O.lse2(q, k, scale, pos, tp)
    tensors = [q.to(gpu), rows[0][0] if rows else k.to(gpu), rows[1][0] if rows else v.to(gpu), None if tp is None else tp.to(gpu)]
    ops._fill_common(a, *tensors[:3], scale, pos, tensors[3], quant, 0)
    out = torch.full((B, Hq, q_len, D), float("nan"), dtype=dtype, device=gpu)
    lse = torch.full((B, q_len, Hq), float("nan"), device=gpu)
    a.o, a.lse = out.data_ptr(), lse.data_ptr()
    a.o_stride_b, a.o_stride_h, a.o_stride_t = out.stride(0), out.stride(1), out.stride(2)
    plan = prefill_plan(a)
    assert (plan.block_rows, plan.teams) == (block, teams) and q_len * (Hq // Hkv) % block <= block - 32
    n = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    ws = torch.full((max(n, 16),), 255, dtype=torch.uint8, device=gpu)
    a.workspace, a.workspace_bytes = ws.data_ptr(), n
    _lib.check(kvx.kvx_sdpa_prefill(ctypes.byref(a), _lib.stream_ptr(gpu)))
    check_out(out, lse, ref)
