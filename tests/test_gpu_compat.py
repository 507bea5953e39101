"""The compatibility set (reference MDSystem.cu:155-299) on the device: the
forces, pressure and RDF that the reference class's GPU branch
(MDSystem.cpp:240-251) reads from calculateNForces, against the FP64 oracle and
the oracle's GPU-rule RDF.  The reference class itself, compiled with
USE_CUDA_TOOLKIT and linked against libljhip.so, is checked on the CPU
(tests/test_ref_class_link.py): the compiled reference stays on the machine
that has its sources."""
import numpy as np
import pytest

import ljamd
from helpers import force_errors, perturbed_state, rel, xyz
from oracle_lib import ORC, RDF_REF_GPU, forces_fp64, rdf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,rho,periodic", [(400, 0.05, 1), (2048, 0.85, 1), (2048, 0.85, 0),
                                            (16384, 0.85, 1), (257, 0.3, 1)])
def test_calculateNForces_semantics(N, rho, periodic):
    """Force = (4 sum r s, sum (r^-12 - r^-6)), pressure = sum (4/6) r.f, RDF GPU rule."""
    L, pos, _ = perturbed_state(N, rho, 1.0, seed=41)
    print(f"\n[case] compat N={N} periodic={periodic}", flush=True)
    dr2 = ORC.orc_rdf_dr2(N)
    arr = ljamd.CompatArrays(N)
    try:
        frc, pressure, rdf_got = arr.calculate(pos, np.float32(L), periodic, dr2)
    finally:
        arr.close()
    F64, ew, E, W = forces_fp64(pos, float(np.float32(L)), periodic, skip_r2=1e-6)
    err = force_errors(xyz(frc), F64)
    assert err["global_rel"] <= 2e-6 and err["max_rel_floor"] <= 1e-5, err
    w = frc.reshape(N, 4)[:, 3]
    assert np.max(np.abs(w - ew[:, 0]) / np.maximum(np.abs(ew[:, 0]), 1.0)) <= 1e-5
    assert rel(pressure, W / 3.0) <= 1e-6
    exp = rdf(pos, float(np.float32(L)), periodic, RDF_REF_GPU, 256, dr2=dr2)
    assert np.array_equal(rdf_got.astype(np.int64), exp)


def test_coincident_particles_skipped():
    """r^2 <= 1e-6 pairs are skipped (MDSystem.cu:37): a duplicated particle
    contributes nothing."""
    N, rho = 300, 0.3
    L, pos, _ = perturbed_state(N, rho, 1.0, seed=7)
    p = pos.reshape(N, 4).copy()
    p[5, :3] = p[4, :3]
    arr = ljamd.CompatArrays(N)
    try:
        frc, pressure, rdf_got = arr.calculate(p.reshape(-1), np.float32(L), 1, 0.1)
    finally:
        arr.close()
    assert np.all(np.isfinite(frc))
    F64, _, _, W = forces_fp64(p.reshape(-1), float(np.float32(L)), 1, skip_r2=1e-6)
    assert force_errors(xyz(frc), F64)["global_rel"] <= 2e-6


def test_compat_errors_do_not_crash():
    # null device arrays: reported, not a crash
    ljamd.lib().calculateNForces(None, None, None, 10, 1.0, 1, None, 0.1, 256, 1)
    assert b"null" in ljamd.lib().lj_last_error()


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("N", [2, 33, 1000, 5000])
def test_excluded_pairs(N, periodic):
    """Pairs at r^2 <= 1e-6 are left out of the force (MDSystem.cu:37), wherever
    in a block of 32 j they fall and whatever else the block holds: copies of
    particles at the same place and 5e-4 away, against FP64 with the same rule."""
    rho = 0.3 if N > 2 else 0.01
    L, pos, _ = perturbed_state(N, rho, 1.0, seed=79)
    p = pos.reshape(N, 4).copy()
    for a, b, d in ((0, 1, 0.0),) if N == 2 else ((0, 1, 0.0), (2, N - 1, 0.0), (5, 32, 5e-4), (31, 6, 0.0)):
        p[b] = p[a]
        p[b, 0] += np.float32(d)
    print(f"\n[case] excluded pairs N={N} periodic={periodic}", flush=True)
    arr = ljamd.CompatArrays(N)
    f, pr, _ = arr.calculate(p.reshape(-1), L, periodic, 0.1)
    arr.close()
    F64, _, E, W = forces_fp64(p.reshape(-1), float(np.float32(L)), periodic, skip_r2=1e-6)
    assert np.all(np.isfinite(f))
    if N == 2:  # the only pair is left out
        assert not np.any(F64) and not np.any(f)
    else:
        err = force_errors(xyz(f), F64)
        assert err["global_rel"] <= 2e-6 and err["max_rel_floor"] <= 1e-5, err
    assert abs(pr - W / 3.0) <= 1e-5 * max(abs(W / 3.0), 1e-3)


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("N", [3072, 4097, 8192, 16385])
def test_excluded_pairs_every_pair_once(N, periodic):
    """The same where every pair is taken once (groups of 128: 3072 and 4097,
    whose last group holds one particle; of 256: 8192 and 16385): pairs to leave
    out inside a group, between two, and with the last particle; the RDF beside
    it as the oracle's."""
    rho = 0.3
    L, pos, _ = perturbed_state(N, rho, 1.0, seed=80)
    p = pos.reshape(N, 4).copy()
    for a, b, d in ((0, 1, 0.0), (2, N - 1, 0.0), (70, 200, 5e-4), (300, 900, 0.0), (1000, 3000, 0.0)):
        p[b] = p[a]
        p[b, 0] += np.float32(d)
    dr2 = ORC.orc_rdf_dr2(N)
    arr = ljamd.CompatArrays(N)
    f, pr, got = arr.calculate(p.reshape(-1), L, periodic, dr2)
    arr.close()
    F64, _, E, W = forces_fp64(p.reshape(-1), float(np.float32(L)), periodic, skip_r2=1e-6)
    assert np.all(np.isfinite(f))
    err = force_errors(xyz(f), F64)
    assert err["global_rel"] <= 2e-6 and err["max_rel_floor"] <= 1e-5, err
    assert abs(pr - W / 3.0) <= 1e-5 * max(abs(W / 3.0), 1e-3)
    exp = rdf(p.reshape(-1), float(np.float32(L)), periodic, RDF_REF_GPU, 256, dr2=dr2)
    assert np.array_equal(got.astype(np.int64), exp)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("N", [600, 3500, 8192])
def test_exact_ties(N, axis):
    """Particles on the two planes x = 0 and x = L/2 (or of y, of z): the x
    separation of a pair is 0 or exactly half the box, so F_x comes from the ties
    alone, each particle drawn towards the image that rounding half away from zero
    picks (+L/2 for the lower x, MDSystem.cu:31-33).  All terms of a particle's sum have the same
    sign, N/2 of them in float sums of at most 128: 1e-5 relative."""
    L = 16.0
    rng = np.random.default_rng(5)
    p = np.zeros((N, 4), np.float32)
    up = rng.permutation(N) % 2 == 1
    others = [a for a in range(3) if a != axis]
    p[:, axis] = np.where(up, L / 2, 0.0)
    k = int(np.ceil(np.sqrt(N)))
    g = rng.permutation(k * k)[:N]
    p[:, others[0]] = (g // k + 0.5 + 0.3 * rng.uniform(-1, 1, N)) * (L / k)
    p[:, others[1]] = (g % k + 0.5 + 0.3 * rng.uniform(-1, 1, N)) * (L / k)
    arr = ljamd.CompatArrays(N)
    f, _, _ = arr.calculate(p.reshape(-1), L, True, 0.1)
    arr.close()
    q = p.astype(np.float64)
    F = np.zeros(N)
    for i in range(N):
        o = up != up[i]
        d = q[i, others] - q[o][:, others]
        d -= L * np.round(d / L)
        r2 = (L / 2) ** 2 + np.sum(d * d, axis=1)
        F[i] = (1.0 if not up[i] else -1.0) * np.sum(24.0 * (2.0 / r2 ** 7 - 1.0 / r2 ** 4)) * (L / 2)
    assert np.max(np.abs(f.reshape(N, 4)[:, axis] - F) / np.abs(F)) <= 1e-5


@pytest.mark.parametrize("N", [1000, 3072, 5003])
def test_coordinate_that_is_no_number(N):
    """A hard-wall box with one NaN coordinate: r^2 of its particle's pairs is not
    comparable, so they are left out like those at r^2 <= 1e-6, whichever pass finds
    them (its least r^2 does not show them, its sums do).  Only the axis of the NaN
    has no force, since NaN times a factor of 0 is NaN; the others, the energies and
    the pressure are those of the box without the particle (the bounds are the
    other tests')."""
    L, pos, _ = perturbed_state(N, 0.3, 1.0, seed=81)
    k = N - 70
    p = pos.reshape(N, 4).copy()
    p[k, 0] = np.nan
    arr = ljamd.CompatArrays(N)
    f, pr, _ = arr.calculate(p.reshape(-1), L, False, 0.1)
    arr.close()
    rest = np.arange(N) != k
    F64, ew, E, W = forces_fp64(p[rest].reshape(-1), float(np.float32(L)), False, skip_r2=1e-6)
    f = f.reshape(N, 4)
    assert np.all(np.isnan(f[:, 0])) and not np.any(f[k, 1:])
    got, exp = xyz(f[rest]), np.asarray(F64)[:, :3].copy()
    got[:, 0] = exp[:, 0] = 0.0
    err = force_errors(got, exp)
    assert err["global_rel"] <= 2e-6 and err["max_rel_floor"] <= 1e-5, err
    assert np.max(np.abs(f[rest, 3] - ew[:, 0]) / np.maximum(np.abs(ew[:, 0]), 1.0)) <= 1e-5
    assert abs(pr - W / 3.0) <= 1e-5 * max(abs(W / 3.0), 1e-3)
