"""An encode with a workspace (search GEMM, decision and residual, projection
GEMM) against the same encode without one: ids, coefficients, codes and scales
bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

from nanokv_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _call(problems, scratch, **kw):
    """encode_batch of problems without a workspace, or (scratch) in one that
    the call has to use."""
    built = [ops._encode_args(p["x"], p["w_enc"], p.get("centers"), p.get("mean"), kw["group"],
                              kw["scale_dtype"], kw["quant_mode"], p.get("id_dtype"), None,
                              p.get("ids")) for p in problems]
    arr = (_lib.NkvEncodeArgs * len(built))(*(b[0] for b in built))
    buf = None
    if scratch:
        need = _lib.lib().nkv_encode_workspace_size(arr, len(built))
        assert need > 0
        buf = torch.full((need + 4096,), 0x5a, device=problems[0]["x"].device, dtype=torch.uint8)
        arr[0].workspace, arr[0].workspace_bytes = buf.data_ptr(), need
    _lib.check("nkv_encode_batch", _lib.lib().nkv_encode_batch(
        torch.cuda.current_stream().cuda_stream, arr, len(built)))
    if scratch:
        # the residual of the first row, at the front of it, was written, and nothing past it
        assert (buf[:problems[0]["x"].shape[1]] != 0x5a).any() and (buf[need:] == 0x5a).all()
    return [b[1] for b in built]


def _plain(problems, **kw):
    return _call(problems, False, **kw)


# rows around the 64- and 128-row tiles and past one pass of 4,096; widths of one
# stage and more; centers around the 128-wide tiles; column tiles 64, 96 and 128
@pytest.mark.parametrize("n,rows,HD,r,G,C,dtype,ids,mean", [
    (1, 1, 256, 32, 32, 1, torch.bfloat16, torch.uint8, True),
    (1, 63, 128, 96, 48, 5, torch.float32, torch.uint8, False),
    (2, 65, 256, 192, 64, 129, torch.bfloat16, torch.int16, True),
    (3, 129, 384, 64, 64, 0, torch.float32, torch.uint8, True),
    (1, 300, 3072, 384, 384, 257, torch.float32, torch.int16, False),
    (1, 130, 640, 160, 32, 1024, torch.float32, torch.int32, False),
    (2, 1100, 512, 384, 32, 256, torch.bfloat16, torch.uint8, True),
    (2, 3200, 256, 384, 128, 64, torch.bfloat16, torch.uint8, False),
    (1, 4300, 128, 32, 8, 7, torch.float32, torch.uint8, False),
    (2, 65, 1024, 192, 64, 129, torch.bfloat16, torch.int16, True),
    (2, 1100, 1024, 384, 32, 256, torch.bfloat16, torch.uint8, True),
    (2, 3200, 2048, 384, 128, 64, torch.bfloat16, torch.uint8, False),
    (1, 4300, 2048, 224, 32, 0, torch.float32, torch.uint8, False),
    (1, 63, 128, 96, 48, 300, torch.float32, torch.int16, False),
    (1, 4300, 640, 32, 8, 64, torch.float32, torch.uint8, False)])
def test_staged_encode_is_the_plain_one(dev, n, rows, HD, r, G, C, dtype, ids, mean):
    g = torch.Generator().manual_seed(rows + HD + C)
    problems = []
    for i in range(n):
        p = {"w_enc": torch.randn(r, HD, generator=g).to(torch.bfloat16).to(dev)}
        x = torch.randn(rows + 1, HD, generator=g)
        if C:
            c = torch.randn(C, HD, generator=g)
            if C > 4:
                c[3] = c[1]                          # equal centers: ties
                c[2] = c[1] * (1 + 2 ** -7)          # near ones: exact comparisons
            c = c.to(torch.bfloat16)
            x = x + c.float()[torch.randint(0, C, (rows + 1,), generator=g)]
            p["centers"], p["id_dtype"] = c.to(dev), ids
        if mean:
            p["mean"] = torch.randn(HD, generator=g).to(dev)
        # each problem has its own row count; one row is not finite
        m = rows - 7 * i if rows > 40 else rows
        x[m // 2, 5] = float("nan")
        wide = torch.zeros(m, 2 * HD, dtype=dtype)
        wide[:, :HD] = x[:m].to(dtype)
        strided = HD % 256 == 0 and C <= 256         # a view of a wider projection
        p["x"] = wide.to(dev)[:, :HD] if strided else wide[:, :HD].contiguous().to(dev)
        problems.append(p)
    for mode in ("fp32", "bf16"):
        kw = dict(group=G, scale_dtype=torch.float16, quant_mode=mode)
        ref = _plain(problems, **kw)
        got = ops.encode_batch(problems, **kw)
        # (narrow rows gain nothing from a workspace)
        if (n, HD) not in ((2, 256), (2, 512)) and (HD > 128 or C > 64):
            got += _call(problems, True, **kw)
        for a, b in zip(got, ref + ref):
            for name in ("ids", "coeff", "packed", "scales"):
                if b[name] is None:
                    continue
                assert torch.equal(a[name].nan_to_num() if a[name].is_floating_point() else a[name],
                                   b[name].nan_to_num() if b[name].is_floating_point() else b[name]), name


def test_workspace_size_and_short_workspace(dev):
    """The size is bounded in the rows, and a workspace below it is not used."""
    lib = _lib.lib()
    x = torch.randn(100, 256, device=dev)
    w = torch.randn(32, 256, device=dev).to(torch.bfloat16)
    c = torch.randn(9, 256, device=dev).to(torch.bfloat16)
    args, out, _ = ops._encode_args(x, w, c, None, 32, torch.float16, "fp32", None, None, None)
    need = lib.nkv_encode_workspace_size(ctypes.byref(args), 1)
    assert need > 0
    args.rows = 10 ** 7
    assert lib.nkv_encode_workspace_size(ctypes.byref(args), 1) < 200 << 20
    args.rows = 100
    scratch = torch.zeros(need, device=dev, dtype=torch.uint8)
    args.workspace, args.workspace_bytes = scratch.data_ptr(), need - 1
    _lib.check("nkv_encode", lib.nkv_encode(torch.cuda.current_stream().cuda_stream,
                                            ctypes.byref(args)))
    assert not scratch.any()
    assert torch.equal(out["ids"], ops.encode(x, w, centers=c)["ids"])


@pytest.mark.parametrize("C", [9, 300, 1024])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_search_of_infinities_and_overflowing_sums(dev, C, dtype):
    """Rows and centers whose fp32 sums overflow take the center that 64 bits
    give; a row with a NaN takes center 0: with a workspace, without one and
    in nkv_assign."""
    if dtype == torch.bfloat16 and C > 256:
        pytest.skip("bf16 rows are searched against at most 256 centers")
    g = torch.Generator().manual_seed(C)
    x = torch.randn(70, 256, generator=g)
    c = torch.randn(C, 256, generator=g).to(torch.bfloat16)
    c[c == 0] = 1.0                       # no infinity times zero
    c[2] *= 1e20                          # ||c||^2 overflows fp32
    x[3, 7] = float("inf")
    x[4, 9] = float("-inf")
    x[5, 11] = 3.3e38
    x[6] *= 1e30
    x[7, 13] = float("nan")
    if dtype == torch.float32:
        x[8, 1] = 3.4e38                  # finite, past the largest bf16
    x = x.to(dtype)
    with np.errstate(invalid="ignore"):
        xd, cd = x.double().numpy(), c.double().numpy()
        dist = (cd * cd).sum(1)[None] - 2.0 * (xd[:, None, :] * cd[None]).sum(2)
    want = np.argmin(dist, axis=1)        # the first of equal ones; NaN: 0
    w = torch.randn(64, 256, generator=g).to(torch.bfloat16).to(dev)
    problem = {"x": x.to(dev), "w_enc": w, "centers": c.to(dev), "id_dtype": torch.int32}
    got = ops.encode_batch([problem], group=32)[0]["ids"]
    assert np.array_equal(got.cpu().numpy(), want)
    plain = _plain([problem], group=32, scale_dtype=torch.float16, quant_mode="fp32")[0]["ids"]
    assert np.array_equal(plain.cpu().numpy(), want)
    if dtype == torch.float32:
        assert np.array_equal(ops.assign(problem["x"], problem["centers"], torch.int32).cpu().numpy(), want)
