"""The staged schedule's workspace plan against the extents its kernels write
(host arithmetic of the library, no GPU).

Every staged call plans one workspace: per partition its tile images (K and
V^T per 128-key tile, at the partition's K/Q width), then its split partials.
nkv_plan_check runs the library's planner and checks, from the same tile
format the decode and flash kernels address the tiles with, that each
partition's last V^T image and its partials end inside its slice.  The same
check runs inside every staged call before any launch.  A decode that wrote
the V^T images of a 32- or 64-wide partition at the 128-wide tile stride
(a layout mistake that once faulted a GPU run) is caught here, on the CPU.
The same check holds the decode launch's block plan to what the kernel
assumes: per codec a multiple of 8 blocks with ranges of at most 24 tiles,
and current-key blocks whenever a partition has current tiles.
"""
import ctypes

import pytest

from nanokv_amd import _lib


def _check(parts, v_dk=0, limit=0):
    lib = _lib.lib()
    fn = lib.nkv_plan_check
    fn.argtypes = [ctypes.POINTER(ctypes.c_int64), ctypes.c_int, ctypes.c_int,
                   ctypes.POINTER(ctypes.c_size_t)]
    fn.restype = ctypes.c_int
    flat = [v for p in parts for v in p]
    arr = (ctypes.c_int64 * len(flat))(*flat)
    total = ctypes.c_size_t(limit)
    rc = fn(arr, len(parts), v_dk, ctypes.byref(total))
    return rc, lib.nkv_last_error().decode(), total.value


# (B, H, dk, Q, n_rows, Nc, rK, rV, camera)
CFG1 = (1, 24, 128, 1560, 12480, 1560, 384, 384, 0)
CFG2 = (1, 24, 128, 780, 49920, 780, 384, 256, 0)
CFG3_NATIVE = (1, 24, 128, 1560, 3120, 1560, 384, 384, 0)


def _tiles(H, dk, n_rows, Nc, B=1):
    chunks = -(-n_rows // 256) + -(-Nc // 256)
    return B * H * 2 * chunks * 128 * (dk + 128) * 2


@pytest.mark.parametrize("parts", [
    [CFG1],
    [CFG2],
    [(2, 3, 128, 100, 300, 0, 128, 64, 0)],          # last history tile empty (300 % 256 <= 128)
    [(1, 2, 128, 33, 1, 1, 64, 64, 1)],               # one key each, camera (stage8 decode)
    [CFG3_NATIVE, (1, 18, 32, 1560, 9360, 0, 384, 384, 0)],
    [CFG3_NATIVE, (1, 6, 128, 1560, 9360, 0, 384, 384, 0),
     (1, 6, 32, 1560, 9360, 0, 384, 384, 0), (1, 12, 64, 1560, 9360, 0, 384, 384, 0)],
    [(2, 4, 128, 1024, 700, 200, 256, 128, 0), (2, 4, 64, 1024, 1000, 0, 256, 128, 0)],
])
def test_plan_extents_fit(parts):
    rc, err, total = _check(parts)
    assert rc == _lib.NKV_OK, err
    # the plan holds at least every partition's tile images
    assert total >= sum(_tiles(p[1], p[2], p[4], p[5], p[0]) for p in parts)


def test_cfg1_workspace_is_the_documented_size():
    rc, err, total = _check([CFG1])
    assert rc == _lib.NKV_OK, err
    tiles = _tiles(24, 128, 12480, 1560)
    assert tiles == 24 * 112 * 64 * 1024          # 176.2 MB of tile images
    assert total - tiles == pytest.approx(29.8e6, rel=0.01)   # split partials


@pytest.mark.parametrize("dk", [32, 64])
def test_v_images_at_the_128_wide_stride_are_caught(dk):
    """The V^T images of a narrow partition addressed with the 128-wide tile
    format run past its tiles: the check names the last V^T image."""
    parts = [CFG3_NATIVE, (1, 18, dk, 1560, 9360, 0, 384, 384, 0)]
    rc, err, _ = _check(parts, v_dk=128)
    assert rc == _lib.NKV_ERR_INVALID
    assert "partition 1" in err and "last V^T image" in err
    # the partition's own width fits
    assert _check(parts, v_dk=dk)[0] == _lib.NKV_OK


def test_unstaged_partitions_are_refused():
    # a 32-wide reader with ranks above the resident decoder's 384 runs the
    # key-chunk kernel, not the staged plan; with the camera and ranks up to
    # 384 it is staged
    rc, err, _ = _check([(1, 4, 32, 64, 512, 0, 448, 128, 1)])
    assert rc == _lib.NKV_ERR_INVALID and "not staged" in err
    assert _check([(1, 4, 32, 64, 512, 0, 384, 128, 1)])[0] == _lib.NKV_OK


@pytest.mark.parametrize("B,H,n_rows,Nc,rK,rV", [
    (1, 24, 12480, 1560, 384, 384),    # cfg1
    (1, 24, 49920, 780, 384, 256),     # cfg2: K and V in two launches
    (1, 1, 1, 1, 64, 64),              # one tile of each
    (3, 5, 128 * 37 - 5, 700, 384, 384),
    (2, 64, 300, 5000, 128, 128),      # more current than history tiles
    (1, 8, 2_000_000, 0, 384, 384),    # ranges pinned at 24 tiles
    (1, 24, 0, 1560, 384, 384),        # current keys only
    (4, 40, 12480, 1560, 192, 320),
])
def test_decode_block_plan(B, H, n_rows, Nc, rK, rV):
    rc, err, _ = _check([(B, H, 128, 1024, n_rows, Nc, rK, rV, 0)])
    assert rc == _lib.NKV_OK, err


@pytest.mark.parametrize("parts", [
    [(1, 8, 128, 256, 2048, 256, 64, 64, 0)],         # many splits of few tiles
    [CFG1],
    # one short partition before a long one: the first candidate splits are
    # neither the fewest nor always the ones that fit
    [(1, 4, 128, 300, 200, 60, 384, 384, 0), (1, 4, 64, 300, 4000, 0, 384, 384, 0)],
    [CFG3_NATIVE, (1, 6, 128, 1560, 9360, 0, 384, 384, 0),
     (1, 6, 32, 1560, 9360, 0, 384, 384, 0), (1, 12, 64, 1560, 9360, 0, 384, 384, 0)],
])
def test_plan_fits_a_smaller_workspace(parts):
    """Fewer splits down to one each; below that the least plan, which the
    caller refuses."""
    full = _check(parts)[2]
    least = _check(parts, limit=1)[2]
    areas = [p[0] * p[1] * -(-p[3] // 32) * 32 * (128 * 2 + 8) for p in parts]
    assert least == sum(_tiles(p[1], p[2], p[4], p[5], p[0]) for p in parts) + \
        sum(-(-a // 256) * 256 for a in areas)
    assert full > least
    for limit in (least, least + 1, (least + full) // 2, full - 1):
        rc, err, total = _check(parts, limit=limit)
        assert rc == _lib.NKV_OK, err
        assert least <= total <= limit
    for limit in (full, full + 1, 1 << 40, 0):
        assert _check(parts, limit=limit)[2] == full
    assert _check(parts, limit=least - 1)[2] == least


@pytest.mark.parametrize("n,rows,HD,r,C,bf16,used", [
    # against the general kernels (other widths, more centers): by centers x width
    (1, 5000, 256, 64, 257, False, True), (2, 50, 384, 64, 1, False, True), (2, 50, 128, 64, 191, False, False),
    (2, 50, 128, 64, 192, False, True), (2, 5000, 384, 64, 64, False, False), (1, 5000, 640, 64, 64, False, True),
    (2, 50, 384, 64, 0, False, True), (2, 50, 128, 64, 0, False, False), (1, 5000, 1152, 384, 0, False, False),
    (1, 8192, 3200, 64, 0, False, True), (1, 8193, 3200, 64, 0, False, False), (1, 8193, 3200, 224, 0, False, True),
    # against the batched ones: one pass (4,096 rows of all problems)
    (1, 4096, 1024, 64, 0, True, True), (1, 4096, 768, 384, 0, True, False), (2, 2048, 1024, 64, 64, True, True),
    (2, 64, 768, 64, 64, True, False), (1, 4096, 256, 64, 64, True, True), (1, 4096, 512, 64, 64, False, True),
    (1, 512, 256, 64, 64, False, True), (1, 513, 256, 64, 64, False, False),
    # more than a pass: wide rows and more than one column block of the projection
    (1, 4097, 2048, 224, 0, True, True), (1, 4097, 2048, 192, 0, True, False), (1, 4097, 1792, 384, 0, True, False),
    (1, 4097, 3072, 384, 256, True, True), (1, 4097, 3072, 384, 256, False, False),
    (2, 2049, 3072, 384, 0, False, True), (2, 2049, 3072, 96, 64, True, False)])
def test_encode_workspace_is_asked_for_where_it_pays(n, rows, HD, r, C, bf16, used):
    args = (_lib.NkvEncodeArgs * n)()
    for a in args:
        a.rows, a.HD, a.r, a.group, a.scale_dtype = rows, HD, r, 32, _lib.NKV_DTYPE_FP16
        a.num_centers, a.id_bytes = C, 2
        setattr(a, "x_bf16" if bf16 else "x", 256)     # only looked at
        a.w_enc = a.coeff = a.packed = a.scales = 256
        if C:
            a.centers = a.ids = 256
    lib = _lib.lib()
    need = lib.nkv_encode_workspace_size(args, n)
    assert lib.nkv_last_error() == b"" and (need > 0) == used
