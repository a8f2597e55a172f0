"""Attention with weights of few rows or keys in one launch (csrc/sdpa_rows.hip) against the CPU oracle, with its waits as they are and
with waits that run out; recorded in a graph; on two streams at once. Every case asserts that the library takes it that way (on 256 compute units)."""
import ctypes

import pytest
import torch

from helpers import make_qkv, prefill_plan, rel_err, scattered_positions
from keys_values_amd import _lib
from keys_values_amd.attention import ops
from oracle import kvx_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[(-1, -1), (0, -1), (1, 0)], ids=["wait", "no-wait", "one-poll"])
def waits(request, kvx):
    kvx.kvx_decode_tuning(-1, *request.param)
    yield request.param
    kvx.kvx_decode_tuning(-1, -1, -1)


def stored(k, v, store, dtype):
    """what the oracle attends over, what the kernels get, the state of the codes"""
    if store == "plain":
        return (k, v), (k, v), None
    B, H, T, D = k.shape
    bits = 8 if store == "u8" else 4
    rows = [O.quantize_rows(x.reshape(-1, D), bits) for x in (k, v)]
    seen = tuple(O.dequantize_rows(*t, dtype).view(B, H, T, D) for t in rows)
    codes = tuple((O.compress4(t[0]) if bits == 4 else t[0]).view(B, H, T, -1) for t in rows)
    return seen, codes, [t.view(B, H, T) for r in rows for t in r[1:]]


# plan: rows of a workgroup, blocks of rows of a KV head, splits of the keys
@pytest.mark.parametrize("dtype,store,B,Hq,Hkv,q_len,T,D,where,plan", [
    (torch.bfloat16, "plain", 1, 8, 2, 128, 1024, 64, "end", (32, 16, 8)),      # blocks of rows and splits of keys
    (torch.float16, "plain", 2, 6, 2, 11, 999, 128, "scattered", (16, 3, 16)),  # 33 rows: a block of one; an odd number of keys
    (torch.bfloat16, "plain", 1, 4, 1, 3, 64, 64, "end", (16, 1, 1)),           # one block, one split: no workspace
    (torch.bfloat16, "plain", 1, 16, 8, 130, 130, 128, "first", (16, 17, 1)),   # as many queries as keys
    (torch.float16, "u8", 1, 8, 2, 200, 257, 64, "end", (16, 50, 1)),           # many blocks, a last tile of one key
    (torch.float16, "u8", 1, 8, 2, 3, 257, 64, "end", (16, 1, 5)),              # a last split of one key
    (torch.bfloat16, "u8", 1, 16, 2, 10, 321, 128, "scattered", (16, 5, 6)),    # and several blocks
    (torch.bfloat16, "u4", 2, 8, 4, 40, 1500, 128, "scattered", (16, 5, 6)),
    (torch.bfloat16, "u8", 1, 7, 1, 5, 700, 256, "scattered", (16, 3, 11)),
    (torch.bfloat16, "plain", 1, 4, 2, 100, 700, 128, "first", (16, 13, 6)),    # splits of which some rows see no key
    (torch.bfloat16, "u8", 1, 2, 1, 8, 8000, 128, "end", (16, 1, 63)),
])
def test_weights_in_one_launch(kvx, gpu, waits, dtype, store, B, Hq, Hkv, q_len, T, D, where, plan):
    q, k, v, gen = make_qkv(900 + T + q_len, B, Hq, Hkv, q_len, T, D, dtype=dtype)
    (ks, vs), (kd, vd), state = stored(k, v, store, dtype)
    pos, tp = {"end": T - q_len, "first": 0, "scattered": 2 * T}[where], None
    if where == "scattered":
        tp = scattered_positions(gen, B, Hkv, T, pos, q_len)
    scale = D ** -0.5
    o_ref, w_ref = O.sdpa_in_blocks(q, ks, vs, scale, pos, None if tp is None else tp.to(torch.int64))
    quant = None if state is None else ops.QuantState(*(t.to(gpu) for t in state))
    qd, kd, vd, tpd = q.to(gpu), kd.to(gpu), vd.to(gpu), None if tp is None else tp.to(gpu)
    a = _lib.SdpaArgs()
    ops._fill_common(a, qd, kd, vd, scale, pos, tpd, quant, 0)
    out, lse = torch.full_like(qd, float("nan")), torch.full((B, q_len, Hq), float("nan"), device=gpu)
    w = torch.full((B, Hkv, T), float("nan"), device=gpu)
    a.o, a.lse, a.w = out.data_ptr(), lse.data_ptr(), w.data_ptr()
    taken = prefill_plan(a)
    assert taken.one_launch and (taken.block_rows, taken.row_blocks, taken.splits) == plan
    n = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    ws = torch.full((n,), 255, dtype=torch.uint8, device=gpu)
    a.o_stride_b, a.o_stride_h, a.o_stride_t = out.stride(0), out.stride(1), out.stride(2)
    a.workspace, a.workspace_bytes = ws.data_ptr(), n
    for _ in range(2):  # the second call finds what the first one left
        _lib.check(kvx.kvx_sdpa_prefill_weights(ctypes.byref(a), _lib.stream_ptr(gpu)))
        # tolerances of the path
        assert rel_err(out.float().cpu(), o_ref.float()) < 2e-2
        torch.testing.assert_close(out.float().cpu(), o_ref.float(), rtol=2e-2, atol=2e-2)
        torch.testing.assert_close(lse.cpu(), O.lse2(q, ks, scale, pos, tp), rtol=1e-4, atol=1e-3)
        torch.testing.assert_close(w.cpu(), w_ref, rtol=1e-3, atol=1e-6)
        torch.testing.assert_close(w.sum(-1).cpu(), torch.full((B, Hkv), float(q_len)), rtol=5e-5, atol=3e-4)
        for t in (out, lse, w):
            t.fill_(float("nan"))


def test_what_is_handed_on_carries_its_token_in_every_8_bytes(kvx, gpu):
    # the heads of the workspace: maxima and sums of rows and splits, then weights of pairs of keys of every block of rows; of two words each half as
    # wide as what is performed whole, each beside half of the call's token
    B, Hq, Hkv, q_len, T, D = 1, 12, 2, 17, 999, 128  # 102 rows of a KV head: 7 blocks of 16
    q, k, v, _ = make_qkv(4, B, Hq, Hkv, q_len, T, D)
    qd, kd, vd = (t.to(gpu) for t in (q, k, v))
    a = _lib.SdpaArgs()
    ops._fill_common(a, qd, kd, vd, 0.09, T - q_len, None, None, 0)
    out, lse, w = torch.empty_like(qd), torch.empty(B, q_len, Hq, device=gpu), torch.empty(B, Hkv, T, device=gpu)
    a.o, a.lse, a.w = out.data_ptr(), lse.data_ptr(), w.data_ptr()
    a.o_stride_b, a.o_stride_h, a.o_stride_t = out.stride(0), out.stride(1), out.stride(2)
    plan = prefill_plan(a)
    assert plan.one_launch and plan.block_rows == 16 and plan.row_blocks == 7 and plan.splits > 1
    n = kvx.kvx_sdpa_prefill_workspace_bytes(ctypes.byref(a))
    ws = torch.full((n,), 255, dtype=torch.uint8, device=gpu)
    a.workspace, a.workspace_bytes = ws.data_ptr(), n
    tokens = []
    for _ in range(2):
        _lib.check(kvx.kvx_sdpa_prefill_weights(ctypes.byref(a), _lib.stream_ptr(gpu)))
        words = ws[: n // 16 * 16].view(torch.int32).view(-1, 4).cpu()
        blocks = B * Hkv * plan.row_blocks
        pairs, sums = words[: blocks * 16 * plan.splits], words[blocks * 16 * plan.splits :][: blocks * ((T + 1) // 2)]
        for part in (pairs, sums):
            assert (part[:, 1::2] == pairs[0, 1::2]).all()
        tokens.append(tuple(pairs[0, 1::2].tolist()))
        m, s = pairs[:, ::2].contiguous().view(torch.float32).view(Hkv, -1, plan.splits, 2)[:, : q_len * Hq // Hkv].unbind(-1)
        rows = torch.logsumexp(m.double() * 0.6931471805599453 + s.double().log(), -1) / 0.6931471805599453
        torch.testing.assert_close(rows.view(Hkv, q_len, Hq // Hkv).transpose(0, 1).reshape(1, q_len, Hq).float(), lse.cpu(), rtol=1e-5, atol=1e-4)
        of_keys = sums[:, ::2].contiguous().view(torch.float32).view(Hkv, plan.row_blocks, -1).sum(1)[:, :T] / (Hq // Hkv)
        torch.testing.assert_close(of_keys, w[0].cpu(), rtol=1e-5, atol=1e-7)
    assert tokens[0] != tokens[1]


def test_repeats_itself_and_the_call_without_weights(gpu):
    # 16-bit outputs of other splits: 2^-9 / sqrt(3) in the mean square, probabilities and outputs on either side
    q, k, v, _ = (t.to(gpu) if isinstance(t, torch.Tensor) else t for t in make_qkv(5, 1, 16, 4, 60, 1200, 128))
    first = ops.prefill_core(q, k, v, 0.09, 1140, None, return_weights=True, return_lse=True)
    for _ in range(20):
        again = ops.prefill_core(q, k, v, 0.09, 1140, None, return_weights=True, return_lse=True)
        assert all(torch.equal(x, y) for x, y in zip(first, again))
    alone = ops.prefill_core(q, k, v, 0.09, 1140, None, return_lse=True)
    assert rel_err(first[0].float(), alone[0].float()) < 4 * 2.3e-3
    torch.testing.assert_close(first[2], alone[2], rtol=1e-5, atol=1e-4)


def test_replayed_from_a_graph(gpu):
    # a repeated call repeats its token: the recorded launches clear what it marks
    B, Hq, Hkv, q_len, T, D = 1, 8, 2, 64, 1024, 64
    inputs = [[t.to(gpu) for t in make_qkv(70 + i, B, Hq, Hkv, q_len, T, D)[:3]] for i in range(4)]
    q, k, v = (t.clone() for t in inputs[0])

    def call():
        return ops.prefill_core(q, k, v, 0.125, T - q_len, None, return_weights=True, return_lse=True)

    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream(gpu)):
        got = call()
    busy = torch.randn(512, 512, device=gpu)
    for tensors in inputs + inputs[:2]:
        for to, x in zip((q, k, v), tensors):
            to.copy_(x)
        want = call()
        graph.replay()
        busy = (busy @ busy).clamp_(-1, 1)  # the program's own work between the replays
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(want, got))


def test_two_streams_at_once(gpu):
    tensors = [[t.to(gpu) for t in make_qkv(80 + i, 1, 8, 2, 128, 1024, 64)[:3]] for i in range(2)]
    want = [ops.prefill_core(*t, 0.125, 896, None, return_weights=True) for t in tensors]
    streams = [torch.cuda.Stream(gpu) for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(20):
        got = []
        for s, t in zip(streams, tensors):
            with torch.cuda.stream(s):
                got.append(ops.prefill_core(*t, 0.125, 896, None, return_weights=True))
        torch.cuda.synchronize()
        for x, y in zip(want, got):
            assert torch.equal(x[0], y[0]) and torch.equal(x[1], y[1])


@pytest.mark.parametrize("Hq,Hkv,q_len,T,D", [(16, 4, 128, 1500, 64), (32, 8, 256, 512, 64)])  # splits and blocks of rows; blocks of rows alone
def test_two_streams_that_fill_the_device_each(kvx, gpu, Hq, Hkv, q_len, T, D):
    # more workgroups than units hold of both calls: those that wait take places of those that are waited for
    tensors = [[t.to(gpu) for t in make_qkv(90 + i, 1, Hq, Hkv, q_len, T, D)[:3]] for i in range(2)]
    a = _lib.SdpaArgs()
    ops._fill_common(a, *tensors[0], 0.125, T - q_len, None, None, 0)
    a.o, a.lse, a.w = (tensors[0][0].data_ptr(),) * 3  # (nothing is launched with them)
    a.o_stride_b, a.o_stride_h, a.o_stride_t = tensors[0][0].stride()[:3]
    plan = prefill_plan(a)
    lds = plan.block_rows * (4 * 4 * (D + 4) + 4 * plan.split_keys)  # of a workgroup, without the smaller parts
    assert plan.one_launch and plan.row_blocks > 1 and lds > 80 * 1024 and plan.row_blocks * Hkv * plan.splits > 128
    want = [ops.prefill_core(*t, 0.125, T - q_len, None, return_weights=True) for t in tensors]
    streams = [torch.cuda.Stream(gpu) for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(10):
        got = []
        for s, t in zip(streams, tensors):
            with torch.cuda.stream(s):
                got.append(ops.prefill_core(*t, 0.125, T - q_len, None, return_weights=True))
        torch.cuda.synchronize()
        for x, y in zip(want, got):
            assert torch.equal(x[0], y[0]) and torch.equal(x[1], y[1])
