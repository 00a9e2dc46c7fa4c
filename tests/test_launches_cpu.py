"""What the library launches, on the CPU: launch_stub.cpp takes the place of
the HIP runtime's launch calls in a child process and records them (operands
are fake addresses that nothing reads)."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
PRELUDE = """
import ctypes, importlib, sys, threading
stub = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
q = importlib.import_module("355_1_trans_amd")
L, P = q.lib(), ctypes.c_void_p

def launches():
    out = []
    for i in range(stub.stub_count()):
        v = (ctypes.c_longlong * 6)()
        stub.stub_launch(i, v)
        out.append(tuple(v))
    return out

def far(i):
    return (1 << 44) + (i << 38)

def mx_kargs(at, m, n, k, fp4=False):
    kb, kg = k // 2 if fp4 else k, k // 32
    p = [far(5 * at + j) for j in range(5)]
    return q.Kargs(p[0], p[1], p[2], m, n, k, 1, kb, kb, n, m * kb, n * kb, m * n, p[3], p[4], kg, kg, m * kg, n * kg)

def bs_kargs(at, m, n, k):
    kg, p = k // 128, [far(5 * at + j) for j in range(5)]
    return q.Kargs(p[0], p[1], p[2], m, n, k, 1, k, 128, n, m * k, n * k, m * n, p[3], p[4], 1 if m > 1 else m, kg,
                   m * kg, (n + 127) // 128 * kg)

def mx4s_kargs(at, m, n, k):
    p = [far(5 * at + j) for j in range(5)]
    return q.Mxfp4Kargs(p[0], p[1], p[2], m, n, k, 1, k // 2, k // 2, n, m * k // 2, n * k // 2, m * n, p[3], p[4],
                        k, k, (m + 31) // 32 * k, (n + 31) // 32 * k, 0)
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = tmp_path_factory.mktemp("stub") / "launch_stub.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__=1",
                    "-I", os.environ.get("ROCM_PATH", "/opt/rocm") + "/include", str(HERE / "launch_stub.cpp"),
                    "-o", str(so)], check=True)
    return so


def _child(stub, body):
    """Runs `body` behind the stub; what it prints."""
    res = subprocess.run([sys.executable, "-c", PRELUDE + body, str(stub), str(HERE.parent)], capture_output=True,
                         text=True, timeout=300)
    assert res.returncode == 0, res.stdout + res.stderr
    return res.stdout.split()


# plans of more than one launch over their workspace: partial planes and their
# sum (ring kernel in its three families, 128 x 128 kernel, one-by-four and
# four-wave kernels split over K), a scale copy before its kernel
SHARED = {    # plan: (a kernel of it, call)
    "ring_mxfp8": ("ring_gemm<", "mx8(mx_kargs(%d, 32, 1536, 7168))"),
    "ring_bs": ("ring_gemm<", "bs(bs_kargs(%d, 64, 2112, 7168))"),
    "ring_aiter": ("ring_gemm<", "mx4s(mx4s_kargs(%d, 57, 2048, 8192))"),
    "mid": ("mid_gemm<", "mx8(mx_kargs(%d, 128, 7168, 16384))"),
    "quad_split": ("splitk_reduce<", "mx4s(mx4s_kargs(%d, 256, 2112, 7168))"),
    "wide_split": ("splitk_reduce<", "mx8(mx_kargs(%d, 512, 12288, 7168))"),
    "wide_panels": ("wide_gemm<", "mx8(mx_kargs(%d, 4096, 8192, 8192))"),
    "noalloc": ("mid_gemm<", "noalloc(mx_kargs(%d, 128, 7168, 16384, True))"),
}
SHARED_BODY = """
ws = far(100)

def shared(fn, query, a):
    need = query(ctypes.byref(a))
    assert need > 0
    return lambda: fn(ctypes.byref(a), 1, P(ws), need, None)

def mx8(a):
    return shared(L.gemm_a8w8_mxfp8, L.gemm_a8w8_mxfp8_workspace_bytes, a)

def bs(a):
    return shared(L.gemm_a8w8_blockscale_bpreshuffle, L.gemm_a8w8_blockscale_bpreshuffle_workspace_bytes, a)

def mx4s(a):
    return shared(lambda p, out, w, b, s: L.gemm_a4w4_mxfp4_bpreshuffle_kid(p, out, 0, w, b, s),
                  lambda p: L.gemm_a4w4_mxfp4_bpreshuffle_kid_workspace_bytes(p, 0), a)

def noalloc(a):
    return lambda: L.gemm_a4w4_mxfp4_noalloc(ctypes.byref(a), 1, None)

# the same plan from two threads, and a plan of one launch over the workspace from a third
calls = [%s, %s, %s]
assert calls[0]() == 0 and "%s" in q.last_launch(), q.last_launch()
stub.stub_reset(0)
assert calls[0]() == 0
per_call = stub.stub_count()
assert per_call > 1, per_call
stub.stub_reset(2000)
start = threading.Barrier(3)

def worker(call):
    start.wait()
    for _ in range(4):
        assert call() == 0

threads = [threading.Thread(target=worker, args=(c,)) for c in calls]
[t.start() for t in threads]
[t.join() for t in threads]
got = launches()
assert len(got) == 8 * per_call + 4, len(got)
apart, i = 0, 0
single = next(t for t in {g[0] for g in got} if sum(g[0] == t for g in got) == 4)
while i < len(got):
    n = 1 if got[i][0] == single else per_call
    apart += any(g[0] != got[i][0] for g in got[i:i + n])
    i += n
print(apart)
"""


@pytest.mark.parametrize("plan", list(SHARED))
def test_launches_of_a_shared_workspace_stay_together(stub, plan):
    """Threads that share a stream share its workspace: between the launches
    of one call that write and read it, no other call's launch may be queued."""
    one = "noalloc(mx_kargs(2, 4, 7168, 32768, True))" if plan == "noalloc" else "bs(bs_kargs(2, 32, 1536, 7168))"
    name, call = SHARED[plan]
    assert _child(stub, SHARED_BODY % (call % 0, call % 1, one, name)) == ["0"]


# shapes whose split ring plan (grouped: split plan) takes the place of one that needs no workspace
KEPT = {
    "mxfp8": "L.gemm_a8w8_mxfp8, L.gemm_a8w8_mxfp8_workspace_bytes, mx_kargs(0, 32, 2112, 8192)",
    "mxfp4": "L.gemm_a4w4_mxfp4, L.gemm_a4w4_mxfp4_workspace_bytes, mx_kargs(0, 40, 4096, 16384, True)",
    "bs": "L.gemm_a8w8_blockscale_bpreshuffle, L.gemm_a8w8_blockscale_bpreshuffle_workspace_bytes, "
          "bs_kargs(0, 4, 2112, 16384)",
    "bypass": "L.gemm_a8w8_blockscale_ldsbypass, L.gemm_a8w8_blockscale_ldsbypass_workspace_bytes, "
              "bypass_kargs(0, 4, 2112, 16384)",
}
KEPT_BODY = """
def bypass_kargs(at, m, n, k):
    kg, p = k // 128, [far(5 * at + j) for j in range(5)]
    return q.LdsBypassKargs(p[0], None, p[1], p[2], m, n, k, 1, k, 128, n, m * k, n * k, m * n, p[3], p[4],
                            1 if m > 1 else m, kg, m * kg, (n + 127) // 128 * kg, (n + 15) // 16 * 16 * k)

fn, query, a = %s
need, ws = query(ctypes.byref(a)), far(100)
b = a.ptr_b_pp if hasattr(a, "ptr_b_pp") else a.ptr_b
assert need > 0

def call(p, size):
    st = fn(ctypes.byref(a), 1, P(p), size, None)
    return st, q.last_launch().split("<")[0]

st, plain = call(None, 0)
assert st == 0 and plain != "ring_gemm", (st, plain)
print(call(ws, need) == (0, "ring_gemm"))
print(all(call(p, size) == (0, plain) for p, size in ((ws + 16, need), (a.ptr_c, need), (b, need), (ws, need - 1))))
"""


@pytest.mark.parametrize("entry", list(KEPT))
def test_a_workspace_no_plan_can_use_is_no_error(stub, entry):
    """Where the plan without the ring kernel needs no workspace, one that is
    unaligned, on an operand or too small leaves the call to that plan."""
    assert _child(stub, KEPT_BODY % KEPT[entry]) == ["True", "True"]


GROUPED_BODY = """
ks = (q.Kargs * 3)(*[bs_kargs(i, 32, n, k) for i, (n, k) in enumerate([(2112, 7168), (4096, 7168), (7168, 2048)])])
fn, ws = L.gemm_a8w8_blockscale_bpreshuffle_grouped, far(100)
need = L.gemm_a8w8_blockscale_bpreshuffle_grouped_workspace_bytes(ks, 3)
assert need > 0
for p, size in ((None, 0), (ws, need), (ws + 16, need), (ks[1].ptr_c, need), (ks[2].ptr_b, need), (ws, need - 1)):
    print(fn(ks, 3, 1, 0, P(p), size, None))
"""


def test_grouped_workspace_no_plan_can_use_is_no_error(stub):
    """The grouped entries alike: three problems that also run unsplit."""
    assert _child(stub, GROUPED_BODY) == ["0"] * 6


QUANT_BODY = """
x, c, s = far(0), far(10), far(20)
k, kg = (1 << 31) - 128, ((1 << 31) - 128) // 128
for fn, args, tile in (
        (L.qgemm_quant_fp8_blockscale_act, (c, k, s, kg, 1), 1024),
        (L.qgemm_quant_fp8_blockscale_act, (c, k, s, 1, 8), 256),
        (L.qgemm_quant_fp8_e8m0_act, (c, k, s, 1, 8), 256), (L.qgemm_quant_mxfp8, (c, k, s, 4 * kg, 0), 1024),
        (L.qgemm_quant_mxfp4, (c, k // 2, s, 4 * kg, 0), 1024), (L.qgemm_quant_mxfp4, (c, k // 2, s, 4 * kg, 1), 256)):
    stub.stub_reset(0)
    st = fn(P(x), 1, 1, k, k, P(args[0]), args[1], P(args[2]), *args[3:], None)
    # every tile of the row; the shuffled scales' tiles take 32 rows in one pass of four
    print(st == 0 and stub.stub_count() == 1 and launches()[0][1] == (k + tile - 1) // tile)
"""


def test_quantizers_take_the_longest_row(stub):
    """One row of 2^31 - 128 elements: the tile count is one past what int
    arithmetic on the rounded-up K holds."""
    assert _child(stub, QUANT_BODY) == ["True"] * 6


MANY_ROWS_BODY = """
x, c, s, rows = far(0), far(10), far(20), (1 << 29) + 64    # K = 32, shuffled: 32 rows a workgroup
for fn, row in ((L.qgemm_quant_mxfp8, 32), (L.qgemm_quant_mxfp4, 16)):
    stub.stub_reset(0)
    st = fn(P(x), 1, rows, 32, 32, P(c), row, P(s), 1, 1, None)
    got = launches()
    fits = all(g[1] * 256 < 1 << 32 and g[2:5] == (1, 1, 256) for g in got)
    # (the 96 rows left take 8 rows a workgroup)
    print(st == 0 and fits and [g[1] for g in got] == [(1 << 24) - 1, 12])
"""


def test_quantizers_take_more_tiles_than_one_grid_dimension(stub):
    """More than 2^24 workgroups of 256 threads: past what one dimension of a
    grid may count."""
    assert _child(stub, MANY_ROWS_BODY) == ["True"] * 2
