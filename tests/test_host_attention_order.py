"""Which workgroup of causal attention takes which query tile, on the host: the order of single tiles, and what is chosen for a shape (256 CUs).  Without a GPU."""
import os
import subprocess

import pytest

from test_host_runtime import HERE, ROOT, run, stub  # noqa: F401  (stub is a fixture)

PAIRS, GROUPS = -2, -1


def test_order_of_single_tiles(tmp_path):
    """Every tile once; the last heads longest first; those before in groups whose heads stay on an XCD and whose lengths are the same over its shader engines."""
    exe = str(tmp_path / "order")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I" + os.path.join(ROOT, "axiom_amd", "csrc", "hip"), os.path.join(HERE, "causal_order_driver.cpp"),
                    "-o", exe], check=True)
    cases = [(heads, nq, resident) for heads in (1, 7, 8, 31, 32, 33, 63, 64, 65, 127, 200, 257, 512, 1021, 3000) for nq in (1, 2, 3, 4, 5, 8, 9, 19, 64) for resident in (256, 512)]
    out = subprocess.run([exe], input="".join("%d %d %d\n" % c for c in cases), capture_output=True, text=True, check=True).stdout.split("\n")
    for (heads, nq, resident), line in zip(cases, out):
        word, first, last = line.rsplit(" ", 2)
        assert word == "ok" and int(first) + int(last) == heads, (heads, nq, resident, line)
        # of those that go longest first over all there are enough to even out the ends, and not a group too many
        assert int(first) == 0 or 2 * resident <= nq * int(last) < 2 * resident + nq * 33


# (heads, S, head size, what goes out: pairs, groups of eight heads, or single tiles with so many heads longest first over all)
CHOICES = [(512, 1024, 128, 160), (256, 2048, 96, 96), (1049, 1042, 64, 121), (728, 991, 96, 152), (96, 1000, 80, 96), (8, 16384, 64, PAIRS), (8, 8192, 64, PAIRS), (16, 8192, 32, 16),
           (12, 7662, 80, PAIRS), (12, 6000, 80, 12), (8, 16384, 128, PAIRS), (5, 12000, 128, GROUPS), (25, 1262, 96, GROUPS), (64, 1024, 128, PAIRS), (32, 2048, 64, PAIRS)]


@pytest.mark.parametrize("heads,S,dk,order", CHOICES)
def test_choice_of_order(stub, heads, S, dk, order):  # noqa: F811
    run(stub, """
heads, S, dk, order = %r
hip.check(L.axhip_init())
hip.check(L.axhip_sdpa_fwd(A, 1 << 46, D, 1 << 48, None, heads, S, dk, 0.5, 1))
x, = launched()
assert "few" not in x.kernel.decode()
assert x.order == order, x.order
tiles = -(-S // (x.block[0] // 2))
assert x.grid[0] == heads * ((tiles + 1) // 2 if order == -2 else tiles)
""" % ((heads, S, dk, order),))


# (heads, S, head size, waves a workgroup): geometry 96 under the mask, both sides of each line
WAVES = [(32, 1024, 96, 4), (24, 2000, 96, 4), (25, 1793, 96, 8), (17, 2358, 80, 4), (90, 400, 96, 8), (44, 600, 80, 8), (42, 600, 80, 4), (8, 7662, 80, 4), (9, 7662, 80, 8), (28, 1786, 96, 8)]


@pytest.mark.parametrize("heads,S,dk,waves", WAVES)
def test_waves_of_geometry_96(stub, heads, S, dk, waves):  # noqa: F811
    run(stub, """
heads, S, dk, waves = %r
hip.check(L.axhip_init())
hip.check(L.axhip_sdpa_fwd(A, 1 << 46, D, 1 << 48, None, heads, S, dk, 0.5, 1))
x, = launched()
assert "few" not in x.kernel.decode() and x.block[0] == 64 * waves, (x.kernel, x.block[0])
""" % ((heads, S, dk, waves),))
