"""Normalisation, activation and rotary rows (csrc/norm_rope.hip) where their arithmetic or their split of a row changes: every 16-bit gate,
norms beyond the range of the shared reciprocal, row lengths and head counts on both sides of a workgroup's sizes."""
import pytest
import torch
import torch.nn.functional as F

from keys_values_amd.longctx import ops
from oracle import longctx_oracle as LO

pytestmark = pytest.mark.gpu


def test_swiglu_of_every_gate(gpu):
    # neighbours share a wavefront with the extremes, and once without them
    gates = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    for g in (gates, gates[(gates.float() > -79) & (gates.float() < 1e30)]):
        g = g[: g.numel() // 16 * 16].view(1, -1)
        out = ops.swiglu(torch.cat((g, torch.ones_like(g)), 1).to(gpu)).cpu()
        g64 = g.double()
        exact = torch.where(g64 == -float("inf"), torch.nan, g64 / (1 + torch.exp(-g64)))  # -inf / inf
        seen = exact.abs() > 2.7e-37  # exp(88.73) is infinite in 32 bits, as it is in torch: gates from there on, of -2.6e-37, give 0
        assert torch.equal(out.isnan(), exact.isnan())
        torch.testing.assert_close(out.double()[seen], exact[seen], rtol=2**-8 + 1e-6, atol=0)  # half a unit of 8 bits, and 32-bit arithmetic
        assert (out.double()[~seen & ~exact.isnan()].abs() < 2.8e-37).all()
        ref = F.silu(g)
        assert ((out != ref) & ~ref.isnan()).float().mean().item() < 1e-3


@pytest.mark.parametrize("dim", [8, 520, 2040, 2048, 2560, 4104, 8192])
def test_norms_out_of_range(gpu, dim):
    gen = torch.Generator().manual_seed(dim)
    x = torch.randn(9, dim, generator=gen).to(torch.bfloat16)
    x[1] = 0.0  # with eps = 0: 0 / 0
    x[2] *= 1e30  # the sum of squares is infinite
    x[3] *= 1e-15  # norm below the range
    x[4] *= 1e14  # above
    x[5, 0] = float("inf")
    x[6, 0] = float("nan")
    x[7, ::3] *= 2.0 ** -100  # tiny values among ordinary ones: remainders and quotients below the normal range
    x[8, 1::2] = x[8, 1::2].sign() * x[8, 1::2].abs().clamp_min(1.0) * 2.0 ** -125  # (whose halves, below, are exact)
    weight = torch.rand(dim, generator=gen) + 0.5
    for eps in (0.0, 1e-6):
        ref = LO.rmsnorm(x, weight, eps)
        ref[2] = 0.0  # the row's norm overflows in 32 bits
        assert torch.equal(ref[1].isnan(), torch.full((dim,), eps == 0.0))
        out = ops.rmsnorm(x.to(gpu), weight.to(gpu), eps).cpu()
        half = (x.float() / 2).to(torch.bfloat16)
        added = ops.add_rmsnorm_(half.to(gpu), half.to(gpu), weight.to(gpu), eps).cpu()
        for got in (out, added):
            torch.testing.assert_close(got.float(), ref.float(), rtol=2**-7, atol=2**-133, equal_nan=True)  # (2^-133: a unit of 16-bit denormals)


# the longest row of 4, 5, 6, 7 and 8 wavefronts, and one chunk more; sums beyond the last-level cache, and rows of a wavefront each
@pytest.mark.parametrize("rows,dim", [(3, 2048), (2, 3584), (3, 3592), (2, 4096), (3, 4104), (2, 5120), (3, 5128), (2, 6144), (3, 6152), (2, 7168), (3, 7176), (2, 8192),
                                      (16384, 3592), (16385, 2056)])
def test_norms_at_the_ends_of_a_split(gpu, rows, dim):
    gen = torch.Generator().manual_seed(rows + dim)
    half = (torch.randn(rows, dim, generator=gen) * 2).to(torch.bfloat16)
    x, weight = half * 2, torch.rand(dim, generator=gen) + 0.5
    ref = LO.rmsnorm(x, weight, 1e-6)
    added = half.to(gpu)
    for got in (ops.rmsnorm(x.to(gpu), weight.to(gpu), 1e-6), ops.add_rmsnorm_(added, half.to(gpu), weight.to(gpu), 1e-6)):
        torch.testing.assert_close(got.cpu().float(), ref.float(), rtol=2**-7, atol=0)  # a unit of the 8 bits kept
    assert torch.equal(added.cpu(), x)


def test_zeros_keep_their_sign(gpu):
    gen = torch.Generator().manual_seed(3)
    x = torch.randn(5, 2048, generator=gen).to(torch.bfloat16)
    x[:, ::7], x[:, 3::7] = -0.0, 0.0
    weight = torch.rand(2048, generator=gen) + 0.5
    ref = LO.rmsnorm(x, weight, 1e-6)
    half = (x.float() / 2).to(torch.bfloat16).to(gpu)
    for got in (ops.rmsnorm(x.to(gpu), weight.to(gpu), 1e-6), ops.add_rmsnorm_(half.clone(), half, weight.to(gpu), 1e-6)):
        assert torch.equal(got.cpu().signbit(), ref.signbit())
    up = torch.randn(5, 2048, generator=gen).to(torch.bfloat16)
    assert torch.equal(ops.swiglu(torch.cat((x, up), 1).to(gpu)).cpu().signbit(), (F.silu(x) * up).signbit())
    # rotated by the angles of position 0, whose sines are zero: a head's value and minus its partner times zero
    qkv = x.view(1, 5, 2048)[:, :1].clone()
    cos, sin = LO.rope_tables(4, 128, 1e6)
    w = torch.ones(128)
    q, k, _ = LO.qk_norm_rope(qkv, 8, 4, 128, w, w, 1e-6, cos, sin, 0)
    g = qkv.to(gpu)
    ops.qk_norm_rope_(g, 8, 4, 128, w.to(gpu), w.to(gpu), 1e-6, cos.to(gpu), sin.to(gpu), 0)
    got = g.cpu().view(1, 1, 16, 128).transpose(1, 2)
    assert torch.equal(got[:, :12].signbit(), torch.cat((q, k), 1).signbit())


@pytest.mark.parametrize("Hq,Hkv,D", [(1, 1, 64), (8, 2, 64), (28, 4, 64), (29, 4, 64), (12, 4, 128), (13, 4, 128), (32, 8, 128), (64, 8, 128), (32, 8, 256)])
def test_rope_head_counts(gpu, Hq, Hkv, D):
    gen = torch.Generator().manual_seed(Hq)
    B, num, pos = 2, 5, 11
    qkv = (torch.randn(B, num, (Hq + 2 * Hkv) * D, generator=gen) * 2).to(torch.bfloat16)
    qkv[0, 0, :D] = 0.0
    qw, kw = (torch.rand(D, generator=gen) + 0.5 for _ in range(2))
    cos, sin = LO.rope_tables(64, D, 1e6)
    for w in ((qw, kw), (None, None)):
        refs = LO.qk_norm_rope(qkv, Hq, Hkv, D, *w, 1e-6, cos, sin, pos)
        g = qkv.to(gpu)
        ops.qk_norm_rope_(g, Hq, Hkv, D, *(None if t is None else t.to(gpu) for t in w), 1e-6, cos.to(gpu), sin.to(gpu), pos)
        out = g.cpu().view(B, num, Hq + 2 * Hkv, D).transpose(1, 2)
        for got, ref in zip(out.split((Hq, Hkv, Hkv), 1), refs):
            # one rounding to 16 bits may go the other way before the rotation and one after it
            torch.testing.assert_close(got.float(), ref.float(), rtol=2**-6, atol=2**-6)
            assert (got != ref).float().mean().item() < 5e-3


# tokens for two workgroups a unit and more: one workgroup of two rows a lane up to 640 lanes of rows, several of one row a lane above
@pytest.mark.parametrize("num,Hq,Hkv,D", [(512, 32, 8, 64), (513, 32, 8, 64), (700, 35, 5, 128), (600, 36, 5, 128), (513, 33, 4, 64), (520, 28, 4, 256), (530, 9, 2, 256)])
def test_rope_of_many_tokens(gpu, num, Hq, Hkv, D):
    gen = torch.Generator().manual_seed(num + Hq)
    qkv = torch.randn(1, num, (Hq + 2 * Hkv) * D, generator=gen).to(torch.bfloat16)
    qw, kw = (torch.rand(D, generator=gen) + 0.5 for _ in range(2))
    cos, sin = LO.rope_tables(num, D, 1e6)
    refs = LO.qk_norm_rope(qkv, Hq, Hkv, D, qw, kw, 1e-6, cos, sin, 0)
    g = qkv.to(gpu)
    ops.qk_norm_rope_(g, Hq, Hkv, D, qw.to(gpu), kw.to(gpu), 1e-6, cos.to(gpu), sin.to(gpu), 0)
    out = g.cpu().view(1, num, Hq + 2 * Hkv, D).transpose(1, 2)
    for got, ref in zip(out.split((Hq, Hkv, Hkv), 1), refs):
        torch.testing.assert_close(got.float(), ref.float(), rtol=2**-6, atol=2**-6)  # (as above)
        assert (got != ref).float().mean().item() < 5e-3


def in_turn(x):
    """Sum over the last axis, one after the other, in the type of x."""
    total = torch.zeros_like(x[..., 0])
    for i in range(x.shape[-1]):
        total = total + x[..., i]
    return total


def rounded_root(x):
    return x.double().sqrt().float()  # (the root of 32-bit tensors on the CPU may be a unit off)


@pytest.mark.parametrize("dim", [2048, 2560, 3592, 4096])
def test_norms_add_their_squares_in_this_order(gpu, dim):
    # 256 lanes: a lane's chunks of eight values one after the other, the lanes of a wavefront in pairs that lie 32, 16, ... 1 apart, four wavefronts in turn
    gen = torch.Generator().manual_seed(dim)
    x = torch.randn(400, dim, generator=gen).to(torch.bfloat16)
    weight = torch.rand(dim, generator=gen) + 0.5
    squares = F.pad(x.float(), (0, 4096 - dim)) ** 2
    lanes = in_turn(squares.view(-1, 2, 4, 64, 8).permute(0, 2, 3, 1, 4).reshape(-1, 4, 64, 16))
    while lanes.shape[-1] > 1:
        half = lanes.shape[-1] // 2
        lanes = lanes[..., :half] + lanes[..., half:]
    norm = rounded_root(in_turn(lanes[..., 0])) * (1.0 / rounded_root(torch.tensor(float(dim)))) + 1e-6
    ref = (x.float() / norm[:, None] * weight).to(torch.bfloat16)
    assert torch.equal(ops.rmsnorm(x.to(gpu), weight.to(gpu), 1e-6).cpu(), ref)


@pytest.mark.parametrize("D", [64, 128, 256])
def test_heads_add_their_squares_in_this_order(gpu, D):
    # runs of eight values one after the other, then the runs in pairs of neighbours
    gen = torch.Generator().manual_seed(D)
    num, Hq, Hkv = 300, 8, 4
    qkv = torch.randn(1, num, (Hq + 2 * Hkv) * D, generator=gen).to(torch.bfloat16)
    w = torch.rand(D, generator=gen) + 0.5
    cos, sin = LO.rope_tables(num, D, 1e6)
    x = qkv.float().view(num, Hq + 2 * Hkv, D)[:, : Hq + Hkv]
    runs = in_turn((x * x).view(num, Hq + Hkv, D // 8, 8))
    while runs.shape[-1] > 1:
        runs = runs[..., 0::2] + runs[..., 1::2]
    y = (x / (rounded_root(runs) * (1.0 / rounded_root(torch.tensor(float(D)))) + 1e-6) * w).to(torch.bfloat16).float()
    lo, hi, c, s = y[..., : D // 2], y[..., D // 2 :], cos[:num, None, : D // 2], sin[:num, None, : D // 2]
    ref = torch.cat((lo * c + -hi * s, hi * c + lo * s), -1).to(torch.bfloat16)
    g = qkv.to(gpu)
    ops.qk_norm_rope_(g, Hq, Hkv, D, w.to(gpu), w.to(gpu), 1e-6, cos.to(gpu), sin.to(gpu), 0)
    assert torch.equal(g.cpu().view(num, Hq + 2 * Hkv, D)[:, : Hq + Hkv], ref)
