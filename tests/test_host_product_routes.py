"""Which single fp32 products go over planes of terms (gemm_planes.hip), on the host (256 CUs): sizes on both sides of the rule's lines.  Without a GPU."""
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
