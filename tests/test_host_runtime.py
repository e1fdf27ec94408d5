"""libaxhip.so's host side against a stand-in for the HIP runtime (hip_runtime_stub.c): what it allocates and launches, and how it takes refusals.  Each test in a
process of its own, without a GPU; no kernel runs."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, sys
sys.path.insert(0, %r)
class Launch(C.Structure):
    _fields_ = [("kernel", C.c_char * 256), ("grid", C.c_uint32 * 3), ("block", C.c_uint32 * 3), ("shared", C.c_uint64), ("args", C.c_uint64 * 7), ("order", C.c_int32)]
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
stub.stub_launch.restype, stub.stub_set_free.argtypes = C.POINTER(Launch), [C.c_size_t]
from axiom_amd import AxHip
hip = AxHip()
L = hip.L
MIB = 1 << 20
A, B, D = 1 << 45, 1 << 46, 1 << 47                # operands that nothing reads
def launched():
    assert stub.stub_launches() <= 4096
    return [stub.stub_launch(i).contents for i in range(stub.stub_launches())]
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["gcc", "-std=gnu11", "-O1", "-Wall", "-Werror", "-fPIC", "-shared", "-I/opt/rocm/include", os.path.join(HERE, "hip_runtime_stub.c"), "-o", out], check=True)
    return out


def run(stub, body):
    r = subprocess.run([sys.executable, "-c", PRELUDE % ROOT + body, stub], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return r.stdout


def test_start_on_a_device_that_is_nearly_full(stub):
    """100 MiB free: the workspace starts with 64 MiB, and the refused larger block is no error of the calls that follow."""
    run(stub, """
stub.stub_set_free(100 * MIB)
hip.check(L.axhip_init())
have = C.c_size_t()
hip.check(L.axhip_workspace_reserve(0, C.byref(have)))
assert have.value == 64 * MIB, have.value
assert hip.last_error() == "", hip.last_error()
hip.check(L.axhip_sgemm(0, 0, 64, 64, 64, 1.0, A, 64, B, 64, 0.0, D, 64, None, 0))
assert len(launched()) == 1
""")


def test_start_on_a_full_device_is_refused(stub):
    """... and goes well once there is room, the first launch too."""
    run(stub, """
stub.stub_set_free(50 * MIB)
assert L.axhip_init() == 2 and "out of device memory" in hip.last_error()
stub.stub_set_free(1000 * MIB)
hip.check(L.axhip_sgemm(0, 0, 64, 64, 64, 1.0, A, 64, B, 64, 0.0, D, 64, None, 0))
have = C.c_size_t()
hip.check(L.axhip_workspace_reserve(0, C.byref(have)))
assert have.value == 160 * MIB
""")


def test_a_refused_allocation_is_the_error_of_its_own_call_only(stub):
    """The workspace, and the vector of ones that column sums of many rows multiply by."""
    run(stub, """
hip.check(L.axhip_init())
stub.stub_set_free(10 * MIB)
assert L.axhip_workspace_reserve(2000 * MIB, None) == 2 and "workspace" in hip.last_error()
hip.check(L.axhip_fill_f32(A, 1.0, 1000))
assert L.axhip_sum_axis(A, 1, 100 * MIB, 2048, D) == 2 and "ones" in hip.last_error()
hip.check(L.axhip_fill_f32(A, 1.0, 1000))
""")


@pytest.mark.parametrize("S,dk,H,B", [(129, 4, 1, 8500001), (129, 36, 1, 9000000), (129, 68, 1, 9000000), (129, 100, 1, 9000000), (200, 32, 7, 1300000), (4096, 4, 1 << 20, 1),
                                      (2049, 4, 999999, 3), (128, 8, 1, 20000000)])
@pytest.mark.parametrize("causal", [0, 1])
def test_attention_over_more_tiles_than_a_grid_holds(stub, S, dk, H, B, causal):
    """2^24 workgroups of 256 threads are 2^32 threads, one more than a launch may have: the heads go in pieces, of whole batches or within one."""
    run(stub, """
S, dk, H, B, causal = %r
hip.check(L.axhip_init())
O, lse = 1 << 48, 1 << 49
if H == 1:
    hip.check(L.axhip_sdpa_fwd(A, B_ptr, D, O, lse, B, S, dk, 0.5, causal))
else:
    hip.check(L.axhip_sdpa_fwd_rows(A, B_ptr, D, H * dk, O, H * dk, lse, B, H, S, dk, 0.5, causal))
at = 0                                              # heads so far
for x in launched():
    b, h = divmod(at, H)
    assert list(x.args[:4]) == [p + 4 * (b * S * H + h) * dk for p in (A, 1 << 46, D, O)] and x.args[4] == lse + 4 * at * S and x.args[6] == S
    n = x.args[5]
    assert n %% H == 0 or h + n <= H
    a_head = -(-S // (x.block[0] // 2))
    assert x.grid[0] in (a_head * n, (a_head + 1) // 2 * n)
    at += n
assert at == B * H
""".replace("B_ptr", "1 << 46") % ((S, dk, H, B, causal),))
