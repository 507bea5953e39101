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


@pytest.mark.parametrize("refused", range(9))
def test_rdf_cell_lists_without_room(so, refused):
    """Steps that sample the RDF through the cell lists are captured with the lists'
    addresses.  A later lj_rdf that grows the lists frees them first: the captured
    steps are dropped also where one of the new arrays finds no room, nothing
    half-allocated stays, and both passes go on over all pairs."""
    hip_stub.run(so, f"""
s = ljamd.LJSystem(16384, 0.85, 1.0)
s.set_step_sampling(ljamd.SAMPLE_RDF_SUM, rdf_rule=ljamd.RDF_REF_GPU, rdf_nbins=256)
s.rdf(ljamd.RDF_RBINS, 1000)  # all pairs: the histogram and table of 1000 bins
s.Integrate(0.005, 3)
dr2 = L.lib().lj_rdf_dr2_default(16384) * 256 / 1000
assert any("k_rdf_cells" in n for n, _ in kernels())
held, captured = stub.stub_live(), stub.stub_instantiated()
stub.stub_fail_in({refused}, 0)
try:
    s.rdf(ljamd.RDF_REF_GPU, 1000, dr2)
finally:
    stub.stub_fail_in(-1, 0)
    # the captured steps are gone before anything else can run them
    assert stub.stub_graphs() == 0, "captured steps hold freed lists"
assert stub.stub_refused() > 0
names = [n for n, _ in kernels()]
assert any("k_rdf_fx" in n for n in names) and not any("k_rdf_cells" in n for n in names)
assert stub.stub_live() < held
s.Integrate(0.005, 3)
assert stub.stub_instantiated() > captured
names = [n for n, _ in kernels()]
assert any("k_rdf_fx" in n for n in names) and not any("k_rdf_cells" in n for n in names)
s.step_rdf_counts()
# room again: the next pass takes the lists
s.rdf(ljamd.RDF_REF_GPU, 1000, dr2)
assert any("k_rdf_cells" in n for n, _ in kernels())
s.close()
assert stub.stub_live() == 0
""")


@pytest.mark.parametrize("boxes,N,small", [(16, 400, 1), (1310, 200, 1), (2621, 200, 0), (5242, 200, 0),
                                           (768, 512, 1), (769, 512, 0), (262, 1000, 1),
                                           (524, 1000, 0), (262, 2000, 1), (131, 4000, 1),
                                           (8, 10000, 1), (1, 100000, 1)])
def test_untuned_batch_route(so, boxes, N, small):
    """Untuned batches of many small boxes keep the default tiling's launches, which
    the one-launch step is slower than there; a tuning always selects its own."""
    hip_stub.run(so, f"""
b = ljamd.LJBatch(np.full({boxes}, {N}, np.int32), np.full({boxes}, .5), np.full({boxes}, 1.))
def step_kernels():
    kernels()
    b.integrate(0.005, 1)
    return [n for n, _ in kernels()]
one, tiled = "k_batch_small", "k_batch_force"
assert any((one if {small} else tiled) in n for n in step_kernels())
assert not any((tiled if {small} else one) in n for n in step_kernels())
b.set_tuning(2, 256, 0)
names = step_kernels()
assert any(tiled in n for n in names) and not any(one in n for n in names)
""")


def test_batch_returns_to_its_default_step(so):
    """What lj_batch_get_tuning gives for a new batch sets the new batch's step again,
    and the autotuner keeps the one-launch step where that is faster (here, where
    time is launches, always within its sizes), leaving the batch's arrays alone."""
    hip_stub.run(so, """
b = ljamd.LJBatch(np.full(16, 400, np.int32), np.full(16, .5), np.full(16, 1.))
def one_launch():
    kernels()
    b.integrate(0.005, 1)
    return any("k_batch_small" in n for n, _ in kernels())
fresh = b.tuning()
assert one_launch()
b.set_tuning(*fresh)
assert one_launch() and b.tuning() == fresh
b.set_tuning(1, 512, 0, 1)
assert not one_launch()
b.set_tuning(*fresh)
assert one_launch()
live = stub.stub_live()
best, us = b.autotune(reps=2)
assert best == b.tuning() == fresh and us < 1.5 and one_launch()
# no room for the copies it times steps on: the best tiling
stub.stub_fail_in(0, 0)
best, _ = b.autotune(reps=2)
stub.stub_fail_in(-1, 0)
assert best == b.tuning() != fresh and not one_launch()
big = ljamd.LJBatch(np.full(2000, 400, np.int32), np.full(2000, .5), np.full(2000, 1.))
best, _ = big.autotune(reps=2)
assert best == big.tuning() != fresh
""")


@pytest.mark.parametrize("once", [1, 0])
@pytest.mark.parametrize("refused", range(3))  # two arrays of slots, one of totals
def test_batch_tuning_without_room(so, refused, once):
    """A tuning whose tables find no room leaves the batch as it was tuned before, or,
    where the old tables find none either, with calls that refuse to run; never
    with captured steps, or a tuning, that do not fit the tables."""
    hip_stub.run(so, f"""
b = ljamd.LJBatch(np.full(32, 1000, np.int32), np.full(32, .5), np.full(32, 1.))
b.set_tuning(2, 2048, 0)
b.integrate(0.005, 1)
captured = stub.stub_instantiated()
stub.stub_fail_in({refused}, {once})
try:
    b.set_tuning(1, 256, 0, 1)
    assert False
except ljamd.LJError:
    pass
assert stub.stub_graphs() == 0, "captured steps hold freed tables"
assert b.tuning() == (2, 2048, 0, 0)
kernels()
if {once} or {refused} == 2:  # the old tables need no totals
    b.integrate(0.005, 1)
    assert stub.stub_instantiated() > captured
    assert any("k_batch_force" in n for n, _ in kernels())
else:
    for call in (lambda: b.integrate(0.005, 1), b.compute_forces, b.time_force):
        try:
            call()
            assert False
        except ljamd.LJError as e:
            assert "no tables" in str(e)
    assert not kernels()
    stub.stub_fail_in(-1, 0)
    b.set_tuning(1, 256, 0, 1)
    b.integrate(0.005, 1)
    assert any("k_batch_force_n3" in n for n, _ in kernels())
""")


def test_refused_allocation_is_told_once(so):
    """A call that found no room says so; the next call, which needs none, runs."""
    hip_stub.run(so, """
s = ljamd.LJSystem(400, 0.5, 1.0)
s.Integrate(0.005, 1)
stub.stub_fail_in(0, 1)
try:
    s.trajectory_loss(0.005, 2)
    assert False
except ljamd.LJError as e:
    assert "hipMalloc" in str(e)
s.CalculateForces()
s.Integrate(0.005, 1)
""")


@pytest.mark.parametrize("N", [400, 5000])
def test_adjoint_arrays_without_room(so, N):
    """The differentiable path's arrays are allocated all or not at all: a call after
    one that found no room starts again instead of using what is missing."""
    hip_stub.run(so, f"""
def first(s):
    n = stub.stub_mallocs()
    s.trajectory_grad(0.005, 6, 3)
    return stub.stub_mallocs() - n
with ljamd.LJSystem({N}, 0.5, 1.0) as s:
    whole = first(s)
assert whole > 15
for refused in range(whole):
    with ljamd.LJSystem({N}, 0.5, 1.0) as s:
        live = stub.stub_live()
        stub.stub_fail_in(refused, 1)
        try:
            first(s)
            assert False
        except ljamd.LJError:
            pass
        if refused < whole - 2:  # before the checkpoints and the segment's states
            assert stub.stub_live() == live
            assert first(s) == whole
        else:
            assert first(s) == whole - refused
    assert stub.stub_live() == 0
""")


@pytest.mark.parametrize("refused", range(2))
def test_step_sampling_without_room(so, refused):
    """Sampling more bins than before where the histogram or its table finds no room:
    the captured steps, which hold the old ones, are dropped and nothing is sampled."""
    hip_stub.run(so, f"""
s = ljamd.LJSystem(400, 0.5, 1.0)
s.set_step_sampling(ljamd.SAMPLE_RDF_SUM, rdf_rule=ljamd.RDF_REF_CPU, rdf_nbins=100)
s.Integrate(0.005, 2)
stub.stub_fail_in({refused}, 1)
try:
    s.set_step_sampling(ljamd.SAMPLE_RDF_SUM, rdf_rule=ljamd.RDF_REF_CPU, rdf_nbins=500)
    assert False
except ljamd.LJError:
    pass
assert stub.stub_graphs() == 0, "captured steps hold a freed histogram"
kernels()
s.Integrate(0.005, 2)
assert not any("rdf" in n for n, _ in kernels())
s.set_step_sampling(ljamd.SAMPLE_RDF_SUM, rdf_rule=ljamd.RDF_REF_CPU, rdf_nbins=500)
s.Integrate(0.005, 2)
assert any("rdf" in n for n, _ in kernels())
""")


@pytest.mark.parametrize("split", ["", "0", "1"])
def test_noalloc_forces_at_every_size(so, split):
    """calculateNForcesNoAlloc serves every N up to 65536 whatever groups
    LJ_PAIR_ONCE_SPLIT asks for, with the launches of calculateNForces."""
    hip_stub.run(so, """
p, f = C.c_void_p(), C.c_void_p()
L.lib().allocateArray(C.byref(p), 65536)
L.lib().allocateArray(C.byref(f), 65536)
def force_pass(call, N):
    kernels()
    rc = call(p, f, None, N, 30., 1, None, 0.1, 256, 1)
    got = [k for k in kernels() if "force" in k[0]]
    assert got, N
    return rc, got
for N in [1, 400, 3071, 3072, 5003, 16384, 23039, 23040, 24001, 32767, 32768, 32769, 65536]:
    rc, got = force_pass(L.lib().calculateNForcesNoAlloc, N)
    assert rc == 0 and got == force_pass(L.lib().calculateNForces, N)[1], (N, rc, got)
""", env={"LJ_PAIR_ONCE_SPLIT": split} if split else {})


def test_force_call_scratch_settles(so):
    """calculateNForces on boxes of two sizes in turn allocates for each once; where the
    pair-once sums find no room it takes the sliced pass, and later them again."""
    hip_stub.run(so, """
p, f = C.c_void_p(), C.c_void_p()
L.lib().allocateArray(C.byref(p), 65536)
L.lib().allocateArray(C.byref(f), 65536)
rdf = np.zeros(256, np.int32)
def call(N):
    kernels()
    n, r = stub.stub_mallocs(), stub.stub_refused()
    L.lib().calculateNForces(p, f, None, N, 40., 1, rdf.ctypes.data, 0.02, 256, 1)
    names = [k for k, _ in kernels()]
    assert any("force" in k for k in names) and any("rdf" in k for k in names), N
    return stub.stub_mallocs() - n, stub.stub_refused() - r, any("k_force_n3" in k for k in names)
first = [call(N) for N in (30000, 40000, 400)]
assert first[0][2] and not first[1][2]
for N in (30000, 40000, 400) * 2:
    assert call(N)[0] == 0, N
L.lib().threadExit()
stub.stub_refuse_above(50 << 20)  # 30000: 57 MB of entries
assert call(30000)[1:] == (1, False)
stub.stub_refuse_above(1 << 40)
assert call(30000)[1:] == (0, True)
""")


def test_fp64_context_without_room_for_pair_once(so):
    """The FP64 mode's slots of every pair once take 2 GiB at N = 131072; a device with
    less room serves the size with the sliced pass."""
    hip_stub.run(so, """
def passes(**kw):
    with ljamd.LJSystem(131072, 0.3, 1.0, precision=ljamd.PREC_FP64, **kw) as s:
        kernels()
        s.Integrate(0.002, 2)
        s.CalculateForces()
        return [k for k in kernels() if "k_force64" in k[0]]
once = passes()
assert once and all("k_force64_n3" in n for n, _ in once)
assert stub.stub_live() == 0
stub.stub_refuse_above(1 << 30)
sliced = passes()
assert stub.stub_refused() == 1
stub.stub_refuse_above(1 << 40)
assert sliced and not any("n3" in n for n, _ in sliced) and len(sliced) == len(once)
stub.stub_refuse_above(1 << 20)
try:
    passes()
    assert False
except ljamd.LJError:
    pass
assert stub.stub_live() == 0
""")


def test_gradient_timing_events(so):
    """The gradient's timing takes a bounded number of events however many segments the
    sweep has, none where no times are asked for, and still covers every segment (one
    launch of the stub is a microsecond: a one-step segment's recomputation takes two,
    the last segment's none)."""
    hip_stub.run(so, """
s = ljamd.LJSystem(400, 0.5, 1.0)
out, g = np.zeros(3), np.zeros(2)
before = stub.stub_events()
assert L.lib().lj_trajectory_grad(s.h, 0.005, 600, 1, 1.0, 1.0, out.ctypes.data, g.ctypes.data,
                                  None, None, None) == 0
assert stub.stub_events() == before
for M in (1, 31, 32, 33, 600):
    times = s.trajectory_grad(0.005, M, 1)[3]
    assert stub.stub_events() - before <= 67
    assert abs(times[1] - 2e-3 * (M - 1)) < 1e-6 * M, (M, times)
    assert times[0] >= 1e-3 * M and times[2] >= 1e-3 * M, (M, times)
s.close()
assert stub.stub_events() == 0
""")
