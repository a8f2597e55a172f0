"""Attention with weights where the launches of the tiled score-sum kernel combine the attention's KV splits (csrc/score_sum.hip): workgroups beside the score
jobs, or the launch that adds the sums of a split of the query rows. Against the CPU oracle, and bit for bit against the same call without the
workspace for it, which combines the splits in a launch of their own. Every case asserts that the library takes it that way (on 256 compute units)."""
import ctypes

import pytest
import torch

from helpers import prefill_plan
from keys_values_amd import _lib
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
