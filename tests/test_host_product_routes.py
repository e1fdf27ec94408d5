"""Which single fp32 products go over planes of terms (gemm_planes.hip) and which in ranges of K in one launch (gemm_strips.hip), on the host (256 CUs): sizes on both sides of
the rules' lines.  Without a GPU."""
import pytest

from test_host_runtime import run, stub  # noqa: F401  (stub is a fixture)

ROUTES = [("nn", 2000, 4096, 1024, True), ("nn", 2000, 3072, 1024, True), ("nt", 2112, 2432, 2403, True), ("tn", 1288, 3985, 767, True), ("nn", 2000, 1024, 4096, False),
          ("nn", 1024, 1024, 1024, False), ("nn", 2048, 4096, 479, False), ("nt", 3392, 29824, 480, True),
          # a K above 4096 near the line
          ("nt", 1498, 2020, 7312, False), ("nt", 2208, 1248, 6112, False), ("nt", 1725, 1913, 6752, False), ("nn", 2368, 1248, 6304, False), ("nn", 1152, 2496, 5472, False),
          ("nn", 1120, 2528, 7040, False), ("nt", 1817, 1656, 4603, False), ("tn", 1495, 1819, 5230, True), ("nn", 1706, 3467, 5049, True), ("nn", 2048, 3328, 4672, True),
          # more than the workspace starts with (160 MiB): never, whatever it holds
          ("nn", 4096, 4096, 4096, False)]


@pytest.mark.parametrize("order,M,N,K,planes", ROUTES)
def test_planes_are_taken(stub, order, M, N, K, planes):  # noqa: F811
    run(stub, """
order, M, N, K, planes = %r
hip.check(L.axhip_init())
hip.check(L.axhip_workspace_reserve(400 * MIB, None))
ta, tb = order[0] == "t", order[1] == "t"
hip.check(L.axhip_sgemm(ta, tb, M, N, K, 1.0, A, M if ta else K, B, K if tb else N, 0.0, D, N, None, 0))
assert ("planes" in hip.last_kernel()) == planes, hip.last_kernel()
assert not planes or [x.kernel.decode().count("k_cut_planes") for x in launched()] == [1, 0]
""" % ((order, M, N, K, planes),))


# (order, M, N, K, whether in ranges): 65 to 100 tiles, on and off the 16-byte grid
RANGES = [("nn", 96, 1024, 1600, True), ("nn", 96, 1024, 1604, False), ("nn", 123, 601, 1600, True), ("nn", 123, 601, 1601, False), ("nt", 1360, 64, 1280, True), ("nt", 1360, 64, 1284, False),
          ("nt", 335, 205, 1279, True), ("nt", 335, 205, 2200, False), ("nt", 1368, 34, 2322, False), ("tn", 96, 1056, 2600, True), ("tn", 96, 1056, 2601, False), ("tn", 123, 601, 1950, True),
          ("tn", 123, 601, 1951, False), ("nt", 64, 1024, 2600, True), ("nt", 64, 1024, 2604, False), ("nt", 100, 10, 4608, True), ("nt", 100, 10, 4612, False)]


@pytest.mark.parametrize("order,M,N,K,ranges", RANGES)
def test_ranges_are_taken(stub, order, M, N, K, ranges):  # noqa: F811
    run(stub, """
order, M, N, K, ranges = %r
hip.check(L.axhip_init())
ta, tb = order[0] == "t", order[1] == "t"
hip.check(L.axhip_sgemm(ta, tb, M, N, K, 1.0, A, M if ta else K, B, K if tb else N, 0.0, D, N, None, 0))
assert (hip.last_kernel() == "sgemm_%%s_ranges32x3" %% order) == ranges, hip.last_kernel()
assert len(launched()) == 1 or not ranges
""" % ((order, M, N, K, ranges),))
