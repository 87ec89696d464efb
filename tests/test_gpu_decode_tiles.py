"""The staged decode kernels (nkv_decode, nkv_decode_batch) against
decode_gemm_kernel, which a misaligned decoder and few rows of a low rank
still take: the same accumulation order, so the same bits."""
import pytest
import torch

from nanokv_amd import ops
from tests._helpers import u16

pytestmark = pytest.mark.gpu


def _codec(dev, N, HD, r, G, C, mean, seed, sdt=torch.float16):
    g = torch.Generator().manual_seed(seed)
    packed = torch.randint(0, 15, (1, N, r // 2), generator=g) * 16 + \
        torch.randint(0, 15, (1, N, r // 2), generator=g)
    scales = torch.rand(1, N, r // G, generator=g).to(sdt)
    w = (torch.randn(HD, r, generator=g) / r ** 0.5).to(torch.bfloat16)
    kw = {}
    if C:
        kw = dict(ids=torch.randint(0, C, (1, N), generator=g).to(torch.uint8).to(dev),
                  centers=torch.randn(1, C, HD, generator=g).to(torch.bfloat16).to(dev))
    m = torch.randn(HD, generator=g).to(dev) if mean else None
    return ops.Codec(packed=packed.to(torch.uint8).to(dev), scales=scales.to(dev),
                     w_dec=w.to(dev), group=G, mean=m, **kw)


def _misaligned(c):
    """The codec with its decoder 8 bytes off a 16-byte boundary."""
    buf = torch.empty(c.w_dec.numel() + 4, device=c.w_dec.device, dtype=torch.bfloat16)
    w = buf[4:].view(c.w_dec.shape)
    w.copy_(c.w_dec)
    assert w.data_ptr() % 16
    return ops.Codec(packed=c.packed, scales=c.scales, w_dec=w, group=c.group, ids=c.ids,
                     centers=c.centers, mean=c.mean)


# rows around the 64- and 128-row tiles, columns around the 128- and 256-wide
# ones, whole and half rank slices, groups of one chunk, a slice, the row
@pytest.mark.parametrize("N,HD,r,G,C,mean", [
    (1, 32, 32, 8, 3, True), (63, 160, 96, 24, 0, True), (65, 288, 64, 64, 5, False),
    (3, 32, 32, 8, 3, True), (17, 32, 160, 40, 0, True), (67, 16384, 96, 24, 0, True),
    (129, 544, 224, 224, 0, False), (8321, 1056, 160, 32, 7, True), (2000, 4128, 384, 48, 9, True)])
def test_decode_tiles_match_the_plain_kernel(dev, N, HD, r, G, C, mean):
    c = _codec(dev, N, HD, r, G, C, mean, seed=N + HD)
    if N > 1:
        c.scales[0, N // 2, 0] = float("inf")      # an overflowed fp16 scale
    rows = torch.tensor(sorted({0, N // 2, N - 1}), dtype=torch.int32, device=dev)
    for idx in (None, rows):
        got, ref = (ops.decode(x, HD, row_index=idx) for x in (c, _misaligned(c)))
        assert torch.equal(got.isnan(), ref.isnan())
        assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(ref))


@pytest.mark.parametrize("lens", [[1], [130, 1, 64], [37] * 18])
def test_decode_batch_is_each_decode(dev, lens):
    HD, r = 160, 96
    first = _codec(dev, 1, HD, r, 32, 4, True, seed=1)
    parts = []
    for i, n in enumerate(lens):
        c = _codec(dev, n, HD, r, 32, 4 + i, False, seed=10 + i)
        parts.append(ops.Codec(packed=c.packed, scales=c.scales, w_dec=first.w_dec, group=32,
                               ids=c.ids, centers=c.centers, mean=first.mean))
    got = ops.decode_batch(parts, HD)
    ref = torch.cat([ops.decode(p, HD) for p in parts], 1)
    assert (u16(got) == u16(ref)).all()
