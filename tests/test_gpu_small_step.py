"""The one-launch time step and trajectory gradient of small boxes (N <= 4096 without an explicit choice
of force pass) at the edges of its tiles: box sizes around the particle counts
at which its tile (4, 8, 16 particles per workgroup) and its LDS chunk (2048
particles) change, against the reference CPU path restated in the oracle."""
import numpy as np
import pytest

import ljamd
from helpers import perturbed_state, xyz
from oracle_lib import OracleSystem, traj_grad_fp64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", [ljamd.BC_PERIODIC, ljamd.BC_WALL, ljamd.BC_NONE])
@pytest.mark.parametrize("N,canon", [
    (1, ljamd.EVN), (2, ljamd.EVN), (3, ljamd.TVN), (5, ljamd.EVN), (255, ljamd.TVN), (1023, ljamd.EVN),
    (1024, ljamd.TVN), (1025, ljamd.EVN), (2047, ljamd.TVN), (2048, ljamd.EVN), (2049, ljamd.TVN),
    (4095, ljamd.EVN), (4096, ljamd.TVN), (4097, ljamd.EVN)])
def test_small_step_edges(N, canon, bc):
    # 10 steps (an 8-step graph and two single steps); tolerances as for the
    # trajectories of test_gpu_step.py over as many steps, relative to the
    # energy per particle where that exceeds 1
    rho, dt, steps = (0.1 if N < 64 else 0.7), 0.004, 10
    L, pos, vel = perturbed_state(N, rho, 1.2, seed=61)
    if N == 1:
        vel = np.array([0.5, -0.25, 0.125, 0.0], np.float32)
    print(f"\n[case] small step N={N} canon={canon} bc={bc}", flush=True)
    o = OracleSystem(N, 1.2, rho, canon, bc, nthreads=8)
    o.set_state(pos, vel)
    o.forces()
    o.params()
    ho = o.integrate(dt, steps)
    for prec in (ljamd.PREC_FP32, ljamd.PREC_COMPENSATED):
        with ljamd.LJSystem(N, rho, 1.2, canonical=canon, boundary=bc, precision=prec) as g:
            g.set_state(pos, vel)
            g.CalculateForces()
            g.CalculateParameters()
            hg = g.Integrate(dt, steps)
            obs = g.observables()
            pg, vg = xyz(g.pos), xyz(g.vel)
            full = g.CalculateForces()
        scale = max(1.0, np.max(np.abs(ho[:, 3])) / N)
        assert np.max(np.abs(hg[:, 0] - ho[:, 0])) / N <= 2e-6 * scale
        assert np.max(np.abs(hg[:, 1] - ho[:, 1])) <= 2e-5 * scale
        assert np.max(np.abs(pg - xyz(o.pos))) <= 1e-5 * max(1.0, L)
        assert np.max(np.abs(vg - xyz(o.vel))) <= 1e-4 * np.max(np.abs(xyz(o.vel)))
        assert obs["step"] == steps and obs["av_iters"] >= steps
        # the step's V and W are those of a separate evaluation at its positions
        assert abs(obs["V"] - full["V"]) <= 2e-6 * N * scale
        assert abs(obs["W"] - full["W"]) <= 1e-5 * max(abs(full["W"]), N * scale)


@pytest.mark.parametrize("bc", [ljamd.BC_PERIODIC, ljamd.BC_NONE])
@pytest.mark.parametrize("N,M,k", [(2, 6, 4), (17, 5, 5), (1025, 6, 4), (2049, 4, 1), (4096, 4, 3)])
def test_small_gradient_edges(N, M, k, bc):
    """Forward, recompute and reverse sweep in one-launch steps (the last
    checkpoint interval whole, partial, one step long and the only one) against
    the FP64 adjoint, with the tolerances of test_gpu_adjoint.py."""
    rho, dt = (0.1 if N < 64 else 0.6), 0.004
    L, pos, vel = perturbed_state(N, rho, 1.0, seed=67)
    print(f"\n[case] small gradient N={N} M={M} k={k} bc={bc}", flush=True)
    with ljamd.LJSystem(N, rho, 1.0, boundary=bc) as s:
        s.set_state(pos, vel)
        loss = s.trajectory_loss(dt, M)
        out, g2, dx0, _ = s.trajectory_grad(dt, M, k)
        again = s.trajectory_grad(dt, M, M)
    assert np.array_equal(out, loss)
    assert np.array_equal(g2, again[1]) and np.array_equal(dx0, again[2])
    ref, ref_g2, ref_dx = traj_grad_fp64(xyz(pos), xyz(vel), L, int(bc == ljamd.BC_PERIODIC), 1.0, 1.0,
                                         dt, M)
    assert abs(out[0] - ref[0]) <= 1e-5 * abs(ref[0])
    assert np.all(np.abs(g2 - ref_g2) <= 1e-4 * np.abs(ref_g2) + 1e-6)
    assert np.linalg.norm(dx0[:, :3] - ref_dx) <= 1e-4 * np.linalg.norm(ref_dx) + 1e-6
