"""Launches on a second device of the same process, with the runtime's calls answered by a stand-in: the limit of dynamic LDS
above 64 KB belongs to a kernel on a device and has to be raised on each."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "apnn-tc_amd", "lib", "libapnn_tc.so")

STAND_IN = r"""
#include <stddef.h>
int stand_in_device, stand_in_raised[2], stand_in_launches[2];
int hipGetDevice(int *d) { *d = stand_in_device; return 0; }
int hipFuncSetAttribute(const void *f, int attr, int value) { (void)f; (void)attr; (void)value; stand_in_raised[stand_in_device]++; return 0; }
typedef struct { unsigned x, y, z; } d3;
int hipLaunchKernel(const void *f, d3 g, d3 b, void **a, size_t lds, void *s) {
  (void)f; (void)g; (void)b; (void)a; (void)lds; (void)s;
  stand_in_launches[stand_in_device]++;
  return 0;
}
int __hipPushCallConfiguration(d3 g, d3 b, size_t lds, void *s) { (void)g; (void)b; (void)lds; (void)s; return 0; }
int __hipPopCallConfiguration(d3 *g, d3 *b, size_t *lds, void **s) { (void)g; (void)b; *lds = 0; *s = 0; return 0; }
int hipGetLastError(void) { return 0; }
int hipDeviceGetAttribute(int *v, int attr, int dev) { (void)attr; (void)dev; *v = 256; return 0; }
int hipGetSymbolAddress(void **p, const void *s) { static int word[4]; (void)s; *p = word; return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t lds) { (void)f; (void)b; (void)lds; *n = 1; return 0; }
"""

CALLS = r"""
import ctypes, sys
sys.path.insert(0, %r)
import pkg
A = pkg.load()
L = A.lib()
S = ctypes.CDLL(%r)
device, raised = ctypes.c_int.in_dll(S, "stand_in_device"), (ctypes.c_int * 2).in_dll(S, "stand_in_raised")
launches = (ctypes.c_int * 2).in_dll(S, "stand_in_launches")
def conv(path, tile, C, R, xb, epi):
    d = A.ConvDesc(W=0x1000, X=0x1000, O=0x1000, batch=8, H=56, Wd=56, cin_pad=C, COUT=256, R=R, S=R, stride=1, pad=R // 2, halo=0,
                   wb=1, xb=xb, weight_mode=1, epi=epi, path=path | ((tile + 1) << 8))
    return L.apnn_conv(ctypes.byref(d), None)
codes = A.Epilogue(mode=A.EPI_BN, out_bits=4, thresholds=0x1000)
calls = {
    "patch": lambda: conv(A.PATH_MFMA_PATCH, 3, 64, 5, 2, A.Epilogue()),
    "async": lambda: conv(A.PATH_MFMA, 7, 256, 3, 4, codes),
    "mfma": lambda: conv(A.PATH_MFMA, 1, 256, 3, 8, codes),
    "xs": lambda: conv(A.PATH_MFMA_XS, 7, 256, 3, 4, A.Epilogue()),
    "rows": lambda: L.apnn_conv_i8_bn_pack(0x1000, 0x1000, 0x1000, 0x1000, 8, 224, 224, 3, 64, 11, 11, 4, 5, 2, 128, None),
    "c4": lambda: L.apnn_conv_i8_bn(0x1000, 0x1000, 0x1000, 0x1000, None, 8, 64, 64, 4, 64, 15, 15, 1, 7, 2, 128, None),
}
for name, call in calls.items():
    seen = []
    for dev in (0, 0, 1, 1):
        device.value = dev
        before = raised[dev], launches[dev]
        rc = call()
        assert rc == 0 and launches[dev] == before[1] + 1, (name, rc, launches[dev])
        seen.append(raised[dev] - before[0])
    print(name, *seen)
"""


@pytest.mark.skipif(not os.path.exists(LIB), reason="needs the built library")
def test_lds_limit_is_raised_on_every_device(tmp_path):
    src, so = tmp_path / "stand_in.c", tmp_path / "stand_in.so"
    src.write_text(STAND_IN)
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    out = subprocess.run([sys.executable, "-c", CALLS % (os.path.join(ROOT, "tests"), str(so))], text=True, capture_output=True,
                         env=dict(os.environ, LD_PRELOAD=str(so)), timeout=120)
    assert out.returncode == 0, out.stderr[-2000:]
    seen = {line.split()[0]: line.split()[1:] for line in out.stdout.splitlines() if len(line.split()) == 5}
    assert set(seen) == {"patch", "async", "mfma", "xs", "rows", "c4"}, out.stdout
    raised = {name: s for name, s in seen.items() if s != ["0"] * 4}
    assert {"patch", "rows"} <= set(raised), seen  # more than 64 KB of LDS
    assert all(s == ["1", "0", "1", "0"] for s in raised.values()), seen
