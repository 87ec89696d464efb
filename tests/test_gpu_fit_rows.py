"""nkv_c64_fit_rows against the oracle's fit at the edges of its kernels: row
blocks of 16, center blocks of 32 (one, two and more), label scans of 2,048
rows, empty clusters, and bf16 rows equal to the same rows in fp32.  And the
quantiser's lane groups against the oracle."""
import numpy as np
import pytest
import torch

import oracle.oracle as orc
from nanokv_amd import _lib, ops
from tests._helpers import u16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,HD,C,iters", [
    (1, 1, 32, 1, 1), (2, 17, 96, 5, 2), (1, 47, 64, 32, 2), (1, 130, 288, 33, 3),
    (3, 65, 256, 64, 2), (1, 90, 32, 65, 2), (1, 2049, 64, 64, 2), (1, 4100, 32, 3, 1)])
def test_fit_rows_match_oracle(dev, B, S, HD, C, iters):
    g = torch.Generator().manual_seed(S + C)
    base = 2 * torch.randn(max(1, S // 9), HD, generator=g)
    x = (torch.randn(B, S, HD, generator=g) + base[torch.arange(S) % len(base)]).to(torch.bfloat16)
    x[:, S // 2] = x[:, 0]                           # equal rows: ties, empty clusters
    init = torch.randperm(S, generator=g)[:C].to(torch.int32)
    rc, rl = orc.c64_fit(x.float().numpy(), init.numpy(), iters)
    for rows in (x.to(dev), x.float().to(dev)):
        for start in (init, init.to(dev)):
            centers, labels, ids = ops.c64_fit_payload(rows, start, iters)
            assert np.array_equal(labels.cpu().numpy().astype(np.int64), rl)
            assert np.array_equal(ids.cpu().numpy().astype(np.int64), rl)
            assert np.array_equal(u16(centers), orc.f32_to_bf16(rc))


@pytest.mark.parametrize("B,S,HD,C", [(1, 40, 64, 33), (2, 130, 96, 64), (1, 300, 3072, 256)])
def test_fit_in_a_label_sized_workspace(dev, B, S, HD, C):
    """A workspace for the rows' labels alone serves fp32 rows; one byte less
    is refused."""
    g = torch.Generator().manual_seed(S)
    x = torch.randn(B, S, HD, generator=g)
    init = torch.randperm(S, generator=g)[:C].to(torch.int32)
    rc, rl = orc.c64_fit(x.numpy(), init.numpy(), 2)
    xd, rows = x.to(dev), init.to(dev)
    centers = torch.empty(B, C, HD, device=dev)
    labels = torch.empty(B, S, device=dev, dtype=torch.int32)
    need = -(-4 * B * S // 256) * 256
    assert need < _lib.lib().nkv_c64_fit_workspace_size(B, S, C)
    buf = torch.full((need + 4096,), 0x5a, device=dev, dtype=torch.uint8)
    for nbytes, want in ((need, _lib.NKV_OK), (need - 1, _lib.NKV_ERR_WORKSPACE)):
        assert _lib.lib().nkv_c64_fit(torch.cuda.current_stream().cuda_stream, xd.data_ptr(), B, S, HD,
                                      C, 2, rows.data_ptr(), centers.data_ptr(), labels.data_ptr(),
                                      buf.data_ptr(), nbytes) == want
    assert (buf[need:] == 0x5a).all()
    assert np.array_equal(labels.cpu().numpy().astype(np.int64), rl)
    assert np.array_equal(centers.cpu().numpy(), rc)


@pytest.mark.parametrize("rows,r,G", [(1, 8, 8), (5, 24, 24), (33, 64, 16), (7, 120, 40),
                                      (130, 384, 384), (9, 1032, 1032), (65, 192, 96)])
@pytest.mark.parametrize("mode", ["fp32", "bf16"])
def test_quantiser_lane_groups(dev, rows, r, G, mode):
    g = torch.Generator().manual_seed(rows + r)
    x = torch.randn(rows, r, generator=g)
    x[0, -1] = 50.0                                  # the last lane holds the maximum
    p, s = ops.quant_pack(x.to(dev), G, torch.bfloat16, mode)
    rp, rs, _ = orc.quant_pack(x.numpy(), G, "bf16", mode)
    assert np.array_equal(p.cpu().numpy(), rp)
    assert np.array_equal(u16(s), rs)
