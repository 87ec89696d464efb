"""The 16-byte kernels of nkv_rope_apply, nkv_camera_apply and
nkv_lift_lse_combine against the element-wise ones, which misaligned operands
still take: RoPE and the camera bit for bit, the lift (fp32 sums in another
order) to one bf16 rounding."""
import numpy as np
import pytest
import torch

from nanokv_amd import ops, synth
from oracle import oracle as orc
from tests._helpers import u16

pytestmark = pytest.mark.gpu


def _shift(t):
    """t at strides of its own, two elements off a 16-byte boundary."""
    buf = torch.zeros(t.numel() + 8, device=t.device, dtype=t.dtype)
    v = buf[2:2 + t.numel()].view(t.shape)
    v.copy_(t)
    return v


def _x(dev, B, S, H, D, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(B, S, H, D, generator=g)
    x[0, 0, 0, 0], x[0, S // 2, H - 1, D - 1] = float("inf"), float("nan")
    return x.to(torch.bfloat16).to(dev)


def _same(a, b):
    assert torch.equal(a.isnan(), b.isnan())
    assert (u16(a.nan_to_num()) == u16(b.nan_to_num())).all()


# one head, a full group of two and eight heads, ragged ones; pieces that end
# inside a block; past the few pieces that two heads a thread serve
@pytest.mark.parametrize("B,S,H,D", [(1, 1, 1, 8), (2, 17, 8, 128), (1, 33, 9, 96), (1, 130, 24, 64),
                                     (2, 2501, 9, 128), (1, 1366, 24, 128), (1, 1365, 24, 128)])
def test_rope_pieces(dev, B, S, H, D):
    x = _x(dev, B, S, H, D, S + H)
    g = torch.Generator().manual_seed(S)
    freqs = torch.polar(torch.ones(50, D // 2), 6.3 * torch.rand(50, D // 2, generator=g)).to(torch.complex128)
    rope = ops.RopeTable.from_freqs(freqs, dev)
    rows = torch.randint(-2, 60, (S,), generator=g).to(torch.int32).to(dev)
    _same(ops.rope_apply(x, rope, rows=rows), ops.rope_apply(_shift(x), rope, rows=rows, out=_shift(x)))


@pytest.mark.parametrize("layout,D", [("full", 128), ("full", 64), ("sf13", 128), ("sf13", 40)])
@pytest.mark.parametrize("B,S,H", [(1, 1, 1), (2, 37, 8), (1, 70, 17), (2, 4903, 17)])
def test_camera_pieces(dev, layout, D, B, S, H):
    x = _x(dev, B, S, H, D, S + D)
    P = synth.camera_matrices(3, seed=S)[2].to(dev)
    cam = ops.Camera(P, torch.tensor([2, 0, 1], dtype=torch.int32, device=dev), 16, layout)
    _same(ops.camera_apply(x, cam), ops.camera_apply(_shift(x), cam, out=_shift(x)))
    y = x.clone()
    _same(ops.camera_apply(y, cam, out=y), ops.camera_apply(x, cam))


@pytest.mark.parametrize("layout,D", [("full", 128), ("full", 64), ("sf13", 128)])
def test_camera_pieces_at_the_limits(dev, layout, D):
    """Products past fp32's range and below it, sums that cancel, zeros of both
    signs against negative entries: the element-wise kernel's bits, and the
    oracle's sum in 64 bits."""
    g = torch.Generator().manual_seed(D)
    x = torch.randn(1, 12, 9, D, generator=g)
    x[0, 0] = 0.0
    x[0, 1] = -0.0
    x[0, 2] = 3e38 * x[0, 2].sign()
    x[0, 3] = 3e38
    x[0, 4] *= 1e-30
    x[0, 5, :, ::3] = 3e38
    P = torch.randn(1, 3, 4, 4, 4, generator=g) * 2
    P[0, 0] = -P[0, 0].abs()
    P[0, 1, :, :, ::2] = 4.0                 # 4 x - 4 x of equal values past fp32
    P[0, 1, :, :, 1::2] = -4.0
    P[0, 2] *= 1e-12
    cam = ops.Camera(P.to(dev), torch.tensor([0, 1, 2], dtype=torch.int32, device=dev), 1, layout)
    x = x.to(torch.bfloat16).to(dev)
    rows = torch.arange(12, dtype=torch.int32, device=dev)
    for shift in range(3):                   # every row meets every matrix
        r = (rows + shift) % 3
        got = ops.camera_apply(x, cam, rows=r)
        _same(got, ops.camera_apply(_shift(x), cam, rows=r, out=_shift(x)))
        with np.errstate(over="ignore"):      # past the largest fp32: an infinity, as on the GPU
            ref = orc.camera_apply(u16(x[0]), P[0, r.cpu().long()].numpy(), layout)
        assert np.array_equal(orc.bf16_to_f32(ref), got[0].float().cpu().numpy(), equal_nan=True)


@pytest.mark.parametrize("low", [32, 64, 96])
@pytest.mark.parametrize("B,H,Q", [(1, 1, 1), (1, 2, 4), (1, 2, 5), (1, 2, 127), (2, 3, 161)])
def test_lift_pieces(dev, low, B, H, Q):
    g = torch.Generator().manual_seed(low + Q)
    native = torch.randn(2 * B, H, Q, 128, generator=g).to(torch.bfloat16).to(dev)
    lo = torch.randn(2 * B, H, Q, low, generator=g).to(torch.bfloat16)
    lo[-1, -1, -1, 5] = float("inf")     # one coordinate of one row: the others stay finite
    main = (torch.randn(H, low, 128, generator=g) / low ** 0.5).to(torch.bfloat16).to(dev)
    mix = (torch.randn(H, low // 4, 32, generator=g) / 4).to(torch.bfloat16).to(dev)
    nl, hl = (torch.randn(2 * B, H, Q, generator=g).to(dev) for _ in range(2))
    lo = lo.to(dev)
    got = ops.lift_lse_combine(native, nl, lo, main, mix, hl).float()
    ref = ops.lift_lse_combine(_shift(native), nl, _shift(lo), main, mix, hl).float()
    ok = ref.isfinite()
    assert torch.equal(ok, got.isfinite())
    # two roundings of sums that differ by fp32 rounding: one bf16 step
    assert ((got - ref).abs()[ok] <= ref.abs()[ok] * 2 ** -7 + 1e-6).all()
