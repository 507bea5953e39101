"""The library's host code on a HIP runtime without a GPU (tests/hip_stub.py):
launch sizes, and what happens where an allocation is refused."""
import pytest

import hip_stub


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    return hip_stub.build(tmp_path_factory.mktemp("hip_stub"))


@pytest.mark.parametrize("rule,bc", [("RDF_REF_GPU", "BC_PERIODIC"), ("RDF_RBINS", "BC_PERIODIC"),
                                     ("RDF_REF_CPU", "BC_NONE"), ("RDF_RBINS", "BC_WALL")])
def test_rdf_counts_of_a_workgroup_fit_32_bits(so, rule, bc):
    """The all-pairs RDF pass counts a workgroup's pairs in 32-bit words: at every
    N that lj_create takes, no workgroup may meet 2^32 pairs.  Group g of 256
    particles meets the units of 32 particles from its own first one on; the units
    of all groups are cut into one run per workgroup, as even as possible."""
    hip_stub.run(so, f"""
for N in [1, 255, 257, 400, 16384, 70000, 131072, 1000003, 10400000, 15000001, (1 << 24) + 1,
          (1 << 26) - 31, 1 << 26]:
    s = ljamd.LJSystem(N, 0.85, 1.0, boundary=ljamd.{bc}, jslices=1)
    kernels()
    s.rdf(ljamd.{rule}, 256)
    grid = [g for n, g in kernels() if "k_rdf_fx" in n or "k_rdf_wall" in n]
    assert len(grid) == 1, grid
    nu, ng = -(-N // 32), -(-N // 256)
    units = ng * nu - 4 * ng * (ng - 1)
    run = -(-units // grid[0])
    assert run * 32 * 256 < 1 << 32, (N, grid, run)
    if N <= 1000003:  # sizes in use: as many runs as ever
        assert grid[0] <= 8 * 256 * 6, (N, grid)
    s.close()
""", env={"LJ_RDF_CELLS": "0"})
