"""The tiled attention kernel where two teams of a workgroup walk the halves of a split (csrc/sdpa_prefill.hip) against the CPU oracle, at the
sizes where the halves differ: odd numbers of tiles, last splits of one tile, rows that see the first tile only. Every case asserts that
the library takes it that way (on 256 compute units)."""
import ctypes

import pytest
import torch

from helpers import make_qkv, prefill_plan, rel_err, scattered_positions
from keys_values_amd import _lib
from keys_values_amd.attention import ops
from oracle import kvx_oracle as O

pytestmark = pytest.mark.gpu


def prepare(gpu, dtype, B, Hq, Hkv, q_len, T, D, where):
    """The call's tensors on the device, its oracle, and its argument block without outputs."""
    q, k, v, gen = make_qkv(300 + T + q_len, B, Hq, Hkv, q_len, T, D, dtype=dtype)
    pos, tp = {"end": T - q_len, "start": 1, "scattered": 2 * T}[where], None
    if where == "scattered":
        tp = scattered_positions(gen, B, Hkv, T, pos, q_len)
    scale = D ** -0.5
    ref = *O.sdpa_in_blocks(q, k, v, scale, pos, None if tp is None else tp.to(torch.int64)), O.lse2(q, k, scale, pos, tp)
    tensors = [t if t is None else t.to(gpu) for t in (q, k, v, tp)]
    a = _lib.SdpaArgs()
    ops._fill_common(a, *tensors[:3], scale, pos, tensors[3], None, 0)
    out = torch.full((B, Hq, q_len, D), float("nan"), dtype=dtype, device=gpu)
    lse = torch.full((B, q_len, Hq), float("nan"), device=gpu)
    a.o, a.lse = out.data_ptr(), lse.data_ptr()
    a.o_stride_b, a.o_stride_h, a.o_stride_t = out.stride(0), out.stride(1), out.stride(2)
    return a, tensors, out, lse, ref


def check_out(out, lse, ref):
    # tolerances of the path
    assert rel_err(out.float().cpu(), ref[0].float()) < 2e-2
    torch.testing.assert_close(out.float().cpu(), ref[0].float(), rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(lse.cpu(), ref[2], rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("dtype,B,Hq,Hkv,q_len,T,D,where,splits", [
    (torch.bfloat16, 2, 32, 8, 130, 700, 128, "end", 1),         # one split of 11 tiles, 520 rows: a last block of 8
    (torch.float16, 2, 28, 4, 150, 1153, 128, "scattered", 2),   # 19 tiles, the last one of a single key; 7 heads a KV head
    (torch.bfloat16, 2, 32, 8, 130, 704, 128, "start", 1),       # blocks that see one tile: the second team has none
    (torch.bfloat16, 1, 32, 8, 100, 3000, 128, "scattered", 6),  # several splits
    (torch.float16, 1, 32, 8, 100, 3013, 128, "start", 6),       # several splits, most of them seen by no row
    (torch.bfloat16, 2, 32, 8, 130, 1000, 64, "end", 1),
    (torch.float16, 1, 24, 8, 300, 2050, 64, "scattered", 4),
    (torch.bfloat16, 1, 64, 8, 256, 385, 128, "end", 1),         # full blocks of rows, a last tile of one key
    (torch.bfloat16, 2, 128, 8, 100, 101, 128, "end", 1),        # two tiles: one a team
    (torch.float16, 2, 128, 8, 100, 116, 128, "scattered", 1),
])
def test_two_teams(kvx, gpu, dtype, B, Hq, Hkv, q_len, T, D, where, splits):
    a, _tensors, out, lse, ref = prepare(gpu, dtype, B, Hq, Hkv, q_len, T, D, where)
    plan = prefill_plan(a)
    assert (plan.block_rows, plan.teams, plan.splits) == (128, 2, splits)
    n = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    ws = torch.full((max(n, 16),), 255, dtype=torch.uint8, device=gpu)
    a.workspace, a.workspace_bytes = ws.data_ptr(), n
    first = None
    for _ in range(10):  # the teams run at paces of their own: every run gives the same bits
        _lib.check(kvx.kvx_sdpa_prefill(ctypes.byref(a), _lib.stream_ptr(gpu)))
        if first is None:
            first = (out.clone(), lse.clone())
            check_out(out, lse, ref)
        assert torch.equal(out, first[0]) and torch.equal(lse, first[1])
        out.fill_(float("nan"))
        lse.fill_(float("nan"))


@pytest.mark.parametrize("dtype,B,Hq,Hkv,q_len,T,D,where,kind,splits", [
    (torch.bfloat16, 4, 8, 8, 6, 15775, 128, "scattered", _lib.KVX_SCORE_SUM_STREAMED, 8),
    (torch.float16, 2, 8, 2, 31, 36382, 64, "end", _lib.KVX_SCORE_SUM_STREAMED, 57),
    (torch.bfloat16, 1, 8, 8, 18, 23745, 128, "start", _lib.KVX_SCORE_SUM_STREAMED, 31),  # splits that no row sees
    (torch.bfloat16, 1, 16, 4, 250, 4001, 128, "scattered", _lib.KVX_SCORE_SUM_SHORT, 8),  # a last tile of 33 keys
    (torch.float16, 1, 8, 2, 256, 8000, 64, "end", _lib.KVX_SCORE_SUM_SHORT, 16),
    (torch.bfloat16, 1, 8, 8, 1000, 2000, 128, "scattered", _lib.KVX_SCORE_SUM_SHORT, 4),  # four splits: all maxima in a thread
])
def test_two_teams_of_several_splits_combined_with_the_weights(kvx, gpu, dtype, B, Hq, Hkv, q_len, T, D, where, kind, splits):
    """The launch that forms the weights takes the rows' log-sum-exps from the maxima and sums of both teams of every split, and combines the outputs."""
    a, _tensors, out, lse, ref = prepare(gpu, dtype, B, Hq, Hkv, q_len, T, D, where)
    w = torch.full((B, Hkv, T), float("nan"), device=gpu)
    a.w = w.data_ptr()
    plan = prefill_plan(a)
    assert (plan.one_launch, plan.teams, plan.splits, plan.score_sum, plan.combined) == (0, 2, splits, kind, 1)
    n = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    ws = torch.full((n,), 255, dtype=torch.uint8, device=gpu)
    a.workspace, a.workspace_bytes = ws.data_ptr(), n
    for _ in range(2):
        _lib.check(kvx.kvx_sdpa_prefill_weights(ctypes.byref(a), _lib.stream_ptr(gpu)))
        check_out(out, lse, ref)
        torch.testing.assert_close(w.cpu(), ref[1], rtol=1e-3, atol=1e-6)
        torch.testing.assert_close(w.sum(-1).cpu(), torch.full((B, Hkv), float(q_len)), rtol=5e-5, atol=3e-4)
        for t in (out, lse, w):
            t.fill_(float("nan"))
