"""The dequantised copy that an attention call over codes takes first (csrc/quantize.hip, ``dequantize_kv_kernel``), in both orders of its workgroups, at the
line between them: the rows in the workspace have the bits of the row quantiser's own."""
import ctypes

import pytest
import torch

from helpers import prefill_plan, randn
from keys_values_amd import _lib
from keys_values_amd.attention import ops
from keys_values_amd.kvcache.quantize import RowQuantizer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,bits,B,Hkv,T,D", [
    (torch.bfloat16, 8, 1, 8, 8192, 128),  # 2^23 values of K: pairs are the fastest index
    (torch.bfloat16, 8, 1, 8, 8193, 128),  # one row a pair more: rows are
    (torch.float16, 4, 2, 3, 21845, 64),   # 128 values below the line
    (torch.float16, 4, 2, 3, 21846, 64),
    (torch.float16, 8, 3, 1, 10923, 256),  # just beyond it
    (torch.bfloat16, 4, 1, 5, 513, 256),
])
def test_rows_of_the_copy(kvx, gpu, dtype, bits, B, Hkv, T, D):
    gen = torch.Generator().manual_seed(T)
    G, q_len = 8, 256
    q = randn(gen, B, Hkv * G, q_len, D, dtype=dtype).to(gpu)
    stores, want = [], []
    for _ in range(2):
        qz = RowQuantizer((B, Hkv, T + 3, D), dtype, bits, allocate_buffers=True, device=gpu)  # three slots more than the call looks at
        qz.quantize(0, T + 3, randn(gen, B, Hkv, T + 3, D, dtype=dtype).to(gpu))
        stores.append([t.view(B, Hkv, T + 3, -1)[:, :, :T] for t in (qz.quant_buffer, qz.quant_scales, qz.quant_zero_points)])
        want.append(qz.dequantize(0, T + 3).view(B, Hkv, T + 3, D)[:, :, :T])
    (k, ks, kz), (v, vs, vz) = stores
    a = _lib.SdpaArgs()
    ops._fill_common(a, q, k, v, D ** -0.5, T - q_len, None, ops.QuantState(*(t.squeeze(-1) for t in (ks, kz, vs, vz))), 0)
    out = torch.empty(B, Hkv * G, q_len, D, dtype=dtype, device=gpu)
    a.o, a.o_stride_b, a.o_stride_h, a.o_stride_t = out.data_ptr(), *out.stride()[:3]
    assert prefill_plan(a, 1).copied
    n = kvx.kvx_sdpa_prefill_copying_workspace_bytes(ctypes.byref(a))
    ws = torch.full((n,), 255, dtype=torch.uint8, device=gpu)
    a.workspace, a.workspace_bytes = ws.data_ptr(), n
    _lib.check(kvx.kvx_sdpa_prefill_copying(ctypes.byref(a), _lib.stream_ptr(gpu)))
    rows = ws[:4 * B * Hkv * T * D].view(dtype).view(2, B, Hkv, T, D)
    assert all(torch.equal(rows[i].view(torch.int16), want[i].contiguous().view(torch.int16)) for i in range(2))
    plain = ops.prefill_core(q, want[0].contiguous(), want[1].contiguous(), D ** -0.5, T - q_len, output_transposed=False)[0]
    assert torch.equal(out, plain)
