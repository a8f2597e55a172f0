"""The tiled attention kernel where two teams of a workgroup walk the halves of a split (csrc/sdpa_prefill.hip) against the CPU oracle, at the
sizes where the halves differ: odd numbers of tiles, last splits of one tile, rows that see the first tile only."""
import ctypes

import pytest
import torch

from helpers import make_qkv, rel_err, scattered_positions
from keys_values_amd import _lib
from keys_values_amd.attention import ops
from oracle import kvx_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,B,Hq,Hkv,q_len,T,D,where", [
    (torch.bfloat16, 2, 32, 8, 130, 700, 128, "end"),         # one split of 11 tiles, 520 rows: a last block of 8
    (torch.float16, 2, 28, 4, 150, 1153, 128, "scattered"),   # 19 tiles, the last one of a single key; 7 heads a KV head
    (torch.bfloat16, 2, 32, 8, 130, 704, 128, "start"),       # blocks that see one tile: the second team has none
    (torch.bfloat16, 1, 32, 8, 100, 3000, 128, "scattered"),  # several splits
    (torch.float16, 1, 32, 8, 100, 3013, 128, "start"),       # several splits, most of them seen by no row
    (torch.bfloat16, 2, 32, 8, 130, 1000, 64, "end"),
    (torch.float16, 1, 24, 8, 300, 2050, 64, "scattered"),
    (torch.bfloat16, 1, 64, 8, 256, 385, 128, "end"),         # full blocks of rows, a last tile of one key
    (torch.bfloat16, 2, 128, 8, 60, 65, 64, "end"),           # two tiles: one a team
])
def test_two_teams(kvx, gpu, dtype, B, Hq, Hkv, q_len, T, D, where):
    q, k, v, gen = make_qkv(300 + T + q_len, B, Hq, Hkv, q_len, T, D, dtype=dtype)
    pos, tp = {"end": T - q_len, "start": 1, "scattered": 2 * T}[where], None
    if where == "scattered":
        tp = scattered_positions(gen, B, Hkv, T, pos, q_len)
    scale = D ** -0.5
    o_ref, _ = O.sdpa_in_blocks(q, k, v, scale, pos, None if tp is None else tp.to(torch.int64))
    qd, kd, vd, tpd = q.to(gpu), k.to(gpu), v.to(gpu), None if tp is None else tp.to(gpu)
    a = _lib.SdpaArgs()
    ops._fill_common(a, qd, kd, vd, scale, pos, tpd, None, 0)
    if q_len > 60:
        assert kvx.kvx_sdpa_prefill_block_rows(ctypes.byref(a), 0) == 128
    out, lse = torch.full_like(qd, float("nan")), torch.full((B, q_len, Hq), float("nan"), device=gpu)
    a.o, a.lse = out.data_ptr(), lse.data_ptr()
    a.o_stride_b, a.o_stride_h, a.o_stride_t = out.stride(0), out.stride(1), out.stride(2)
    n = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    ws = torch.full((max(n, 16),), 255, dtype=torch.uint8, device=gpu)
    a.workspace, a.workspace_bytes = ws.data_ptr(), n
    first = None
    for _ in range(10):  # the teams run at paces of their own: every run gives the same bits
        _lib.check(kvx.kvx_sdpa_prefill(ctypes.byref(a), _lib.stream_ptr(gpu)))
        if first is None:
            first = (out.clone(), lse.clone())
            # tolerances of the path
            assert rel_err(out.float().cpu(), o_ref.float()) < 2e-2
            torch.testing.assert_close(out.float().cpu(), o_ref.float(), rtol=2e-2, atol=2e-2)
            torch.testing.assert_close(lse.cpu(), O.lse2(q, k, scale, pos, tp), rtol=1e-4, atol=1e-3)
        assert torch.equal(out, first[0]) and torch.equal(lse, first[1])
        out.fill_(float("nan"))
        lse.fill_(float("nan"))
