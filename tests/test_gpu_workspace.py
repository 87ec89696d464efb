"""nkv_attend and nkv_fast_attend in a workspace smaller than their size query:
fewer key splits, the same attention within the rounding of the splits'
partials; nothing is written past the workspace; a workspace that no plan fits
is refused."""
import ctypes

import numpy as np
import pytest
import torch

from nanokv_amd import _lib, codec_native, ops
from tests._helpers import Scenario, max_abs_cos
from tests.test_gpu_fast import MAX_ABS, MIN_COS, _payload
from tests.test_plan import _check

pytestmark = pytest.mark.gpu

GUARD = 4096


def _in(call, args, out, nbytes):
    """call(stream, args, workspace, nbytes) in the front of a marked buffer."""
    buf = torch.full((nbytes + GUARD,), 0x5a, device=out.device, dtype=torch.uint8)
    out.fill_(float("nan"))
    rc = call(torch.cuda.current_stream().cuda_stream, ctypes.byref(args), buf.data_ptr(), nbytes)
    torch.cuda.synchronize()
    assert (buf[nbytes:] == 0x5a).all()
    return rc


@pytest.mark.parametrize("D", [128, 64])
def test_attend_in_a_smaller_workspace(dev, D):
    sc = Scenario(H=4, D=D, N=2000, Q=200, Nc=100, rK=64, rV=64, G=32, C=8, seed=D)
    key, value = sc.codecs(dev)
    lib = _lib.lib()
    q, kc, vc = sc.q.to(dev), sc.k_cur.to(dev), sc.v_cur.to(dev)   # the struct holds raw pointers
    args, out, lse, _ = ops._attend_args(q, kc, vc, key, value, sc.scale, None, True)
    full = lib.nkv_attend_workspace_size(ctypes.byref(args))
    shape = [(1, 4, 128, 200, 2000, 100, 64, 64, 0)]
    least = full - _check(shape)[2] + _check(shape, limit=1)[2]
    assert least < full
    ref, ref_lse = sc.reference(0)
    for nbytes in (full, full - 1, (least + full) // 2, least):
        assert _in(lib.nkv_attend, args, out, nbytes) == _lib.NKV_OK, nbytes
        diff, cos = max_abs_cos(out[0].float().cpu().numpy(), ref)
        assert diff <= 2e-2 and cos >= 0.9995, (nbytes, diff, cos)
        assert np.abs(lse[0].cpu().numpy() - ref_lse).max() < 2e-3
    assert _in(lib.nkv_attend, args, out, least - 1) == _lib.NKV_ERR_WORKSPACE
    assert out.isnan().all()


@pytest.mark.parametrize("Q,d", [(300, 64), (40, 32)])
def test_fast_attend_in_a_smaller_workspace(dev, Q, d):
    sc = Scenario(H=4, N=2600, Q=Q, Nc=60, rK=384, rV=384, G=32, C=16, with_mean=True, seed=Q)
    key, value = sc.codecs(dev)
    payload = _payload(sc, (0, 3), d, seed=d)
    groups = [g.tensors() for g in codec_native.ReaderLayer(payload, dev).groups]
    protect = np.arange(2400, 2600)
    low = np.arange(2400)
    rows = [torch.from_numpy(r.astype(np.int32)).to(dev) for r in (protect, low)]
    q, kc, vc = sc.q.to(dev), sc.k_cur.to(dev), sc.v_cur.to(dev)   # the struct holds raw pointers
    f, keep, full, out, lse, _ = ops._fast_args(q, kc, vc, key, value, *rows, groups, sc.scale, None,
                                                True)
    shapes = [(1, 4, 128, Q, 200, 60, 384, 384, 0)] + [
        (1, g.heads.numel(), g.d, Q, 2400, 0, 384, 384, 0) for g in groups]
    least = full - _check(shapes)[2] + _check(shapes, limit=1)[2]
    assert least < full
    lib = _lib.lib()
    ref = ops.fast_attend(q, kc, vc, key, value, *rows, groups, softmax_scale=sc.scale)
    for nbytes in (full, full - 1, (least + full) // 2, least):
        assert _in(lib.nkv_fast_attend, f, out, nbytes) == _lib.NKV_OK, nbytes
        diff, cos = max_abs_cos(out.float().cpu().numpy(), ref[0].float().cpu().numpy())
        assert diff <= MAX_ABS and cos >= MIN_COS, (nbytes, diff, cos)
        assert (lse - ref[1]).abs().max() < 2e-3
    assert _in(lib.nkv_fast_attend, f, out, least - 1) == _lib.NKV_ERR_WORKSPACE
    assert out.isnan().all()
