"""Kernels that take more than 64 KB of dynamic LDS have that attribute set on
the device they are launched on, also when a process uses a second one: the
library runs in a process of its own over stand-ins for the HIP calls (nothing
is launched, no GPU is needed), which note the attribute per device."""
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

from nanokv_amd import _lib

SHIM = r"""
#include <stddef.h>
typedef struct { unsigned x, y, z; } dim3;
enum { MAXN = 256 };
static int cur, n, launches, large, missing;
static struct { int dev; const void* f; int bytes; } set[MAXN];
static struct { dim3 g, b; size_t s; void* st; } call;
void shim_device(int d) { cur = d; launches = large = missing = 0; }
int shim_launches(void) { return launches; }
int shim_large(void) { return large; }
int shim_missing(void) { return missing; }
int hipGetDevice(int* d) { *d = cur; return 0; }
int hipGetLastError(void) { return 0; }
int hipFuncSetAttribute(const void* f, int attr, int v) {
    if (n < MAXN) { set[n].dev = cur; set[n].f = f; set[n++].bytes = v; }
    return 0;
}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, void* st) {
    call.g = g; call.b = b; call.s = s; call.st = st;
    return 0;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, void** st) {
    *g = call.g; *b = call.b; *s = call.s; *st = call.st;
    return 0;
}
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t s, void* st) {
    ++launches;
    if (s > 65536) {
        int i, ok = 0;
        ++large;
        for (i = 0; i < n; ++i) ok |= set[i].dev == cur && set[i].f == f && (size_t)set[i].bytes >= s;
        missing += !ok;
    }
    return 0;
}
"""

CALLS = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # before the library: its symbols come first
from nanokv_amd import _lib
lib = _lib.lib()
P = 1 << 20                                               # never read: nothing is launched

def codec(r, centers):
    c = _lib.NkvCodec(P, P, P if centers else None, P if centers else None, P, None, r, 32,
                      _lib.NKV_DTYPE_FP16)
    if centers:
        c.id_bytes, c.num_centers = 1, centers
    return c

def decode(rows, HD):
    a = _lib.NkvDecodeArgs(1, HD, rows, rows, None, codec(384, 16))
    a.out = P
    return lib.nkv_decode(None, ctypes.byref(a))

def encode(rows, r, bf16, scratch):
    a = _lib.NkvEncodeArgs()
    a.rows, a.HD, a.r, a.group, a.scale_dtype = rows, 512, r, 32, _lib.NKV_DTYPE_FP16
    a.num_centers, a.id_bytes = 16, 1
    if bf16: a.x_bf16 = P
    else: a.x = P
    a.centers = a.w_enc = a.ids = a.coeff = a.packed = a.scales = P
    if scratch:
        a.workspace, a.workspace_bytes = P, lib.nkv_encode_workspace_size(ctypes.byref(a), 1)
        assert a.workspace_bytes
    return lib.nkv_encode(None, ctypes.byref(a))

def attend():
    B, H, D, Q, N = 1, 4, 128, 200, 2000
    a = _lib.NkvAttendArgs()
    a.B, a.H, a.D, a.Q, a.N, a.softmax_scale = B, H, D, Q, N, 1.0
    a.q = a.out = P
    a.q_sb, a.q_st, a.q_sh = Q * H * D, H * D, D
    a.o_sb, a.o_st, a.o_sh = Q * H * D, H * D, D
    a.key, a.value = codec(384, 16), codec(384, 16)
    need = lib.nkv_attend_workspace_size(ctypes.byref(a))
    return lib.nkv_attend(None, ctypes.byref(a), P, need)

# (call, whether some of its launches take more than 64 KB)
calls = [(lambda: decode(8192, 3072), True), (lambda: decode(40, 256), False), (attend, True)]
calls += [(lambda r=r, b=b, s=s: encode(rows, r, b, s), True) for rows, r in ((64, 64), (3000, 384), (4096, 480))
          for b in (False, True) for s in (False, True)]
for i, (call, large) in enumerate(calls):
    for dev in (0, 1, 0):
        shim.shim_device(dev)
        rc = call()
        assert rc == 0, (i, dev, rc, lib.nkv_last_error())
        assert shim.shim_launches() > 0 and (shim.shim_large() > 0) == large, (i, dev)
        assert shim.shim_missing() == 0, (i, dev, shim.shim_missing())
print("ok")
"""


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs a C compiler")
def test_dynamic_lds_is_set_on_every_device(tmp_path):
    src, so = tmp_path / "shim.c", tmp_path / "libshim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(src), "-o", str(so)], check=True)
    assert _lib.LIB_PATH.exists()
    run = subprocess.run([sys.executable, "-c", CALLS, str(so)], capture_output=True, text=True,
                         cwd=Path(__file__).resolve().parent.parent, timeout=120)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stdout + run.stderr
