"""A launch that fails ends a call of several launches: the ones behind it, which would work on what it left out, are not sent.  On the host, with the
runtime's launch functions by stand-ins of which the one asked for fails."""
import shutil
import subprocess
import sys

import pytest

STAND_INS = r"""
extern "C" {
static int launches, fails, last;
void fail_at(int n) { launches = last = 0, fails = n; }
int launched() { return launches; }
int hipLaunchKernel(const void *, unsigned long long, unsigned, unsigned long long, unsigned, void **, unsigned long, void *) {
  if (++launches != fails) return 0;
  return last = 719;   // (kept until it is asked for)
}
int __hipPushCallConfiguration(unsigned long long, unsigned, unsigned long long, unsigned, unsigned long, void *) { return 0; }
int __hipPopCallConfiguration(void *, void *, unsigned long *, void **) { return 0; }
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipGetLastError() { const int e = last; last = 0; return e; }
}
"""

CALLS = r"""
import ctypes, sys
stand_ins = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
class Act(ctypes.Structure):
    _fields_ = [("fields", ctypes.c_int64 * 8)]
class Args(ctypes.Structure):
    _fields_ = ([(n, ctypes.c_void_p) for n in "x router correction gate_up down act weights place out workspace".split()]
                + [(n, ctypes.c_int64) for n in "x_stride ws_bytes".split()]
                + [(n, ctypes.c_int) for n in "rows k router_k outputs top groups keep route_flags experts tile_m ff width weigh_inputs".split()] + [("scale", ctypes.c_float)])
act, p = Act(), 4096      # (an address that the host does not look at)
for rows, dtype in ((16, int(sys.argv[3])), (17, int(sys.argv[3]))):
    a = Args(x=p, router=p, gate_up=p, down=p, act=ctypes.addressof(act), weights=p, place=p, out=p, workspace=p, x_stride=64, ws_bytes=1 << 20, rows=rows, k=64, router_k=64,
             outputs=8, top=2, groups=1, keep=1, experts=8, tile_m=16, ff=64, width=64, scale=1.0)
    stand_ins.fail_at(0)
    print(lib.mv_moe_mlp(ctypes.byref(a), dtype, None), stand_ins.launched(), end=" ")
    for n in range(1, stand_ins.launched() + 1):
        stand_ins.fail_at(n)
        print(lib.mv_moe_mlp(ctypes.byref(a), dtype, None), stand_ins.launched(), end=" ")
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="no C++ compiler")
def test_experts_in_one_call(tmp_path):
    from minivllm_amd import hip_ops

    (tmp_path / "stand_ins.cpp").write_text(STAND_INS)
    lib = str(tmp_path / "stand_ins.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", lib, str(tmp_path / "stand_ins.cpp")], check=True)
    out = subprocess.run([sys.executable, "-c", CALLS, lib, hip_ops.LIB_PATH, str(hip_ops.MV_BF16)], check=True, capture_output=True, text=True, timeout=60).stdout
    # router with grouping and two products; router, grouping and two products
    assert out.split() == "0 3 719 1 719 2 719 3".split() + "0 4 719 1 719 2 719 3 719 4".split()
