"""What entry points send to the GPU, on the host: the runtime's launch functions by stand-ins that count the launches, keep the last one's size and let one fail."""
import ctypes
import json
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.skipif(not shutil.which("g++"), reason="no C++ compiler")

STAND_INS = r"""
extern "C" {
static int launches, fails, last;
static unsigned long long threads, blocks;
void fail_at(int n) { launches = last = 0, fails = n; }
int launched() { return launches; }
int threads_x() { return (int)(threads & 0xffffffff); }
int blocks_y() { return (int)(blocks >> 32); }
int hipLaunchKernel(const void *, unsigned long long grid, unsigned, unsigned long long block, unsigned, void **, unsigned long, void *) {
  threads = block, blocks = grid;
  if (++launches != fails) return 0;
  return last = 719;   // (kept until it is asked for)
}
static struct { unsigned long long grid, block; unsigned grid_z, block_z; } pushed;
int __hipPushCallConfiguration(unsigned long long grid, unsigned grid_z, unsigned long long block, unsigned block_z, unsigned long, void *) {
  pushed = {grid, block, grid_z, block_z};
  return 0;
}
int __hipPopCallConfiguration(unsigned *grid, unsigned *block, unsigned long *shared, void **stream) {
  grid[0] = (unsigned)pushed.grid, grid[1] = (unsigned)(pushed.grid >> 32), grid[2] = pushed.grid_z;
  block[0] = (unsigned)pushed.block, block[1] = (unsigned)(pushed.block >> 32), block[2] = pushed.block_z;
  *shared = 0, *stream = 0;
  return 0;
}
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipGetLastError() { const int e = last; last = 0; return e; }
}
"""

START = r"""
import ctypes, sys
stand_ins = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
dtype, p = int(sys.argv[3]), 4096      # (an address that the host does not look at)
"""

EXPERTS = START + r"""
class Act(ctypes.Structure):
    _fields_ = [("fields", ctypes.c_int64 * 8)]
class Args(ctypes.Structure):
    _fields_ = ([(n, ctypes.c_void_p) for n in "x router correction gate_up down act weights place out workspace".split()]
                + [(n, ctypes.c_int64) for n in "x_stride ws_bytes".split()]
                + [(n, ctypes.c_int) for n in "rows k router_k outputs top groups keep route_flags experts tile_m ff width weigh_inputs".split()] + [("scale", ctypes.c_float)])
act = Act()
for rows in (16, 17):
    a = Args(x=p, router=p, gate_up=p, down=p, act=ctypes.addressof(act), weights=p, place=p, out=p, workspace=p, x_stride=64, ws_bytes=1 << 20, rows=rows, k=64, router_k=64,
             outputs=8, top=2, groups=1, keep=1, experts=8, tile_m=16, ff=64, width=64, scale=1.0)
    stand_ins.fail_at(0)
    print(lib.mv_moe_mlp(ctypes.byref(a), dtype, None), stand_ins.launched(), end=" ")
    for n in range(1, stand_ins.launched() + 1):
        stand_ins.fail_at(n)
        print(lib.mv_moe_mlp(ctypes.byref(a), dtype, None), stand_ins.launched(), end=" ")
"""

# one call per dict of sys.argv[6]: the fields of the arguments' struct (names and type codes in sys.argv[5]) that are not a pointer or 0 -> launches, y of the last one
STRUCT = START + r"""
import json
fields = [(n, {"P": ctypes.c_void_p, "l": ctypes.c_int64, "q": ctypes.c_int64, "i": ctypes.c_int, "f": ctypes.c_float}[t]) for n, t in json.loads(sys.argv[5])]
Args = type("Args", (ctypes.Structure,), {"_fields_": fields})
for case in json.loads(sys.argv[6]):
    a = Args(**{n: p for n, t in fields if t is ctypes.c_void_p}, **case)
    stand_ins.fail_at(0)
    rc = getattr(lib, sys.argv[4])(ctypes.byref(a), *eval(sys.argv[7]))
    print(*((stand_ins.launched(), stand_ins.blocks_y()) if rc == 0 else (rc, rc)), end=" ")
"""

ROTATION = START + r"""
i, v, f = ctypes.c_int, ctypes.c_void_p, ctypes.c_float
q = ctypes.c_int64
for heads, kv, dim, norm, cache, tokens in eval(sys.argv[4]):
    w, c = p if norm else None, p if cache else None
    rc = lib.mv_rope_qk_store_ex(v(p), v(p), v(p), q(16384), q(16384), q(16384), v(p), v(p), v(p), q(64), v(w), v(w), f(1e-6), v(p), None if cache else v(p), v(c), v(c), v(c),
                                 q(64), i(tokens), i(heads), i(kv), i(dim), i(dtype), None, None)
    print(stand_ins.threads_x() if rc == 0 else rc, end=" ")
"""


@pytest.fixture(scope="module")
def call(tmp_path_factory):
    from minivllm_amd import hip_ops

    folder = tmp_path_factory.mktemp("stand_ins")
    (folder / "stand_ins.cpp").write_text(STAND_INS)
    lib = str(folder / "stand_ins.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", lib, str(folder / "stand_ins.cpp")], check=True)

    def run(program, dtype, *more):
        return subprocess.run([sys.executable, "-c", program, lib, hip_ops.LIB_PATH, str(dtype), *more], check=True, capture_output=True, text=True, timeout=60).stdout.split()
    return run


def _launches(call, entry, struct, dtype, cases, more="dtype, None"):
    """-> (launches, y of the last one) of each case."""
    fields = json.dumps([(n, t._type_) for n, t in struct._fields_])
    out = list(map(int, call(STRUCT, dtype, entry, fields, json.dumps(cases), more)))
    return list(zip(out[::2], out[1::2]))


def test_a_launch_that_fails_ends_the_experts(call):
    """The launches behind it would work on what it left out: they are not sent."""
    from minivllm_amd import hip_ops

    # router with grouping and two products; router, grouping and two products
    assert call(EXPERTS, hip_ops.MV_BF16) == "0 3 719 1 719 2 719 3".split() + "0 4 719 1 719 2 719 3 719 4".split()


# heads, heads of keys and values, columns, norms, cache: tokens -> threads of a token: the lines by the rows that a wave would have one behind the other
ROTATIONS = {(16, 8, 128, True, True): {512: 256, 513: 128, 1408: 128, 1409: 64}, (28, 4, 128, False, True): {512: 256, 513: 128, 900: 128, 901: 64},
             (24, 8, 128, True, True): {768: 256, 769: 128, 1760: 128, 1761: 64}, (64, 8, 128, True, True): {1025: 256, 2048: 256, 2049: 128, 3520: 128, 3521: 64},
             (64, 8, 64, False, True): {768: 256, 769: 128, 1400: 128, 1401: 64}, (4, 1, 128, True, True): {512: 256, 513: 64}, (1, 1, 64, False, False): {513: 64},
             (40, 40, 128, False, True): {513: 256, 9000: 256}, (40, 40, 128, False, False): {768: 256, 769: 128, 1401: 64},
             (32, 8, 256, True, True): {768: 256, 769: 128, 3168: 128, 3169: 64}, (32, 16, 256, True, True): {769: 128, 9000: 128}}


def test_waves_of_a_token(call):
    from minivllm_amd import hip_ops

    cases = [(*k, t) for k, v in ROTATIONS.items() for t in v]
    want = [n for v in ROTATIONS.values() for n in v.values()]
    for dtype in (hip_ops.MV_BF16, hip_ops.MV_F16):
        assert list(map(int, call(ROTATION, dtype, repr(cases)))) == want
    assert set(call(ROTATION, hip_ops.MV_F32, repr(cases))) == {"256"}


def test_grouping_by_the_router(call):
    """Up to 16 tokens of 16 bits, and 256 pairs and experts together."""
    from minivllm_amd import hip_ops as H

    cases = {(1, 8): 3, (16, 4): 3, (16, 8): 3, (15, 16): 3, (16, 16): 4, (17, 1): 4}
    fields = [dict(x_stride=64, ws_bytes=1 << 20, rows=r, k=64, router_k=64, outputs=16, top=t, groups=1, keep=1, experts=16, tile_m=16, ff=64, width=64, scale=1.0)
              for r, t in cases]
    assert ctypes.sizeof(H.GateAct) <= 32
    program = STRUCT.replace("for case in", "act = (ctypes.c_int64 * 4)()\nfor case in").replace("**case)", "**case)\n    a.act = ctypes.addressof(act)")
    names = json.dumps([(n, t._type_) for n, t in H.MvMoeMlpArgs._fields_])
    for dtype, want in ((H.MV_BF16, list(cases.values())), (H.MV_F16, list(cases.values())), (H.MV_F32, [4] * len(cases))):
        assert list(map(int, call(program, dtype, "mv_moe_mlp", names, json.dumps(fields), "dtype, None")))[::2] == want


# (heads of a group, groups, p, n, sequences, tokens of all, of the longest) -> along with the preparation, bf16 and one decay per head.  Turns of a workgroup's threads: one; two;
# three and four; a head a group of 1.5, three and four
ALONG = {(2, 8, 64, 64, 1, 700, 700): True, (2, 8, 64, 32, 4, 15000, 4000): True, (2, 8, 64, 32, 16, 18000, 1490): False, (2, 8, 128, 128, 1, 256, 256): True,
         (2, 8, 128, 128, 1, 257, 257): False, (2, 8, 128, 128, 3, 704, 280): False, (2, 8, 128, 128, 4, 704, 280): True, (2, 8, 128, 128, 16, 18000, 1490): True,
         (2, 8, 256, 128, 1, 60, 60): False, (2, 8, 256, 128, 16, 18000, 1490): False, (1, 8, 64, 64, 1, 341, 341): True, (1, 8, 64, 64, 1, 383, 383): False,
         (1, 8, 64, 64, 1, 448, 448): True, (1, 8, 128, 128, 16, 704, 60): False, (1, 8, 128, 128, 16, 1024, 171): True,
         (1, 8, 256, 128, 16, 18000, 1490): False, (4, 2, 64, 64, 16, 18000, 1490): False}


def test_convolution_along_with_the_preparation(call):
    from minivllm_amd import hip_ops as H

    def fields(per, groups, p, n, seqs, total, longest, taps=4, channel=0):
        heads, channels = per * groups, groups * (per * p + 2 * n)
        return dict(x_stride=channels, beta_stride=heads, a_stride=heads * (n if channel else 1), out_stride=heads * p, slots=seqs, ws_bytes=1 << 34, n_seqs=seqs, max_q=longest,
                    total_q=total, channels=channels, taps=taps, heads=heads, groups=groups, p=p, p_true=p, n=n, k_off=heads * p, q_off=heads * p + groups * n,
                    channel_decay=channel)
    run = lambda cases, dtype: [n for n, _ in _launches(call, "mv_delta_prefill_conv", H.MvDeltaArgs, dtype, cases, "ctypes.c_void_p(p), dtype, 0, None")]
    assert run([fields(*k) for k in ALONG], H.MV_BF16) == [2 if v else 3 for v in ALONG.values()]
    # other taps, and more heads than two of a group, never; heads of 16 bits otherwise, and decays per channel: by their sizes alone, with or without it the same launches
    assert run([fields(2, 8, 64, 64, 1, 100, 100, taps=t) for t in (1, 2, 3, 5)], H.MV_BF16) == [3] * 4
    some = [(1, 4, 64, 64), (1, 4, 128, 64), (1, 4, 144, 96), (1, 4, 80, 32), (2, 4, 64, 64)]
    for dtype in (H.MV_BF16, H.MV_F16):
        got = run([fields(*k, 1, 100, 100, channel=1) for k in some], dtype)
        assert [b - got[0] for b in got] == [0, 0, 1, 1, 1]


def test_tokens_of_a_convolution(call):
    """Eight a workgroup up to 1700 workgroups of 32."""
    from minivllm_amd import hip_ops as H

    def fields(taps, seqs, longest, channels):
        return dict(x_stride=channels, out_stride=channels, slots=seqs, n_seqs=seqs, max_q=longest, channels=channels, taps=taps, heads=2, groups=1, p=16, n=32, b_off=32, c_off=64)
    cases = {(4, 10, 170 * 32, 512): 680, (4, 10, 170 * 32 + 1, 512): 171, (2, 10, 170 * 32, 512): 680, (8, 10, 170 * 32, 512): 680, (8, 10, 170 * 32 + 1, 512): 171,
             (4, 10, 170 * 32, 544): 170, (1, 1, 1, 96): 1}
    for dtype in (H.MV_BF16, H.MV_F16):
        assert _launches(call, "mv_causal_conv", H.MvSsmArgs, dtype, [fields(*k) for k in cases]) == [(1, y) for y in cases.values()]
    assert _launches(call, "mv_causal_conv", H.MvSsmArgs, H.MV_F32, [fields(4, 10, 170 * 32, c) for c in (256, 288)]) == [(1, 680), (1, 170)]
