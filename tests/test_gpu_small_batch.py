"""The one-launch time steps of a batch whose tuning was not set, at the edges
of their tiles (16 particles) and LDS chunks (2048): box sizes 1 to 4097 in one
batch, against the separate kernels of a sliced tuning (the default tuning, set
again, gives the one-launch step's bits), and in any split of the run."""
import numpy as np
import pytest

import ljamd
from helpers import rel, xyz

pytestmark = pytest.mark.gpu

N = np.array([2, 15, 16, 17, 64, 400, 2047, 2048, 2049, 4097], np.int32)
RHO = np.array([0.02, 0.1, 0.2, 0.3, 0.4, 0.05, 0.5, 0.85, 0.6, 0.7])
T0 = np.linspace(0.8, 2.0, N.size)


@pytest.mark.parametrize("bc", [ljamd.BC_PERIODIC, ljamd.BC_WALL, ljamd.BC_NONE])
@pytest.mark.parametrize("canon", [ljamd.EVN, ljamd.TVN])
def test_small_batch_edges(canon, bc):
    # tolerances: those of the single-box comparison of test_gpu_batch.py
    steps = 20
    print(f"\n[case] small batch canon={canon} bc={bc}", flush=True)
    out = []
    for chunks, tuning in (([steps], None), ([7, 13], None), ([steps], (1, 512, 8, 0)),
                           ([steps], (1, 512, 4, 0))):
        with ljamd.LJBatch(N, RHO, T0, canonical=canon, boundary=bc, seed=31) as b:
            if tuning:
                b.set_tuning(*tuning)
            h = np.concatenate([b.integrate_hist(0.004, c) for c in chunks])
            obs = b.observables()
            f = [b.get_array(ljamd.ARRAY_FORCE, box=k) for k in range(N.size)]
            p = [b.get_array(ljamd.ARRAY_POS, box=k) for k in range(N.size)]
            v = [b.get_array(ljamd.ARRAY_VEL, box=k) for k in range(N.size)]
            st = b.stats()
            b.compute_forces()
            full = b.observables()
        out.append((h, obs, p, v, f, st, full))
    a, split, again, sliced = out
    for o in (split, again):
        for x, y in zip((a[0], a[5], *a[2], *a[3], *a[4]), (o[0], o[5], *o[2], *o[3], *o[4])):
            assert np.array_equal(x, y)
    assert any(not np.array_equal(x, y) for x, y in zip(a[3], sliced[3]))  # another route
    assert np.all(a[5][:, 0] == steps) and np.array_equal(a[5][:, 9], sliced[5][:, 9])
    for k in range(N.size):
        assert np.max(np.abs(a[0][:, k, 0] - sliced[0][:, k, 0])) / N[k] <= 2e-5, k
        assert np.max(np.abs(xyz(a[2][k]) - xyz(sliced[2][k]))) <= 4e-5, k
        assert np.max(np.abs(xyz(a[3][k]) - xyz(sliced[3][k]))) <= 1e-3, k
        assert abs(a[1][k]["V"] - a[6][k]["V"]) <= 1e-6 * max(abs(a[6][k]["V"]), N[k]), k
        assert abs(a[1][k]["W"] - a[6][k]["W"]) <= 1e-5 * max(abs(a[6][k]["W"]), N[k]), k
        e = np.sum(a[4][k].reshape(-1, 4)[:, 3].astype(np.float64)) * 2.0
        assert rel(e, a[1][k]["V"]) <= 1e-5 or abs(e) < 1e-5, k


def test_autotune_keeps_the_one_launch_step():
    """16 boxes of 400, where the one-launch step takes a third of the best tiling's
    time: the autotuner leaves it on, and the batch's state alone."""
    n, r, t = np.full(16, 400, np.int32), np.linspace(0.05, 0.8, 16), np.full(16, 1.4)
    print("\n[case] autotune 16 of 400", flush=True)
    out = []
    for tune in (False, True):
        with ljamd.LJBatch(n, r, t, seed=5) as b:
            b.integrate(0.004, 5)
            fresh = b.tuning()
            if tune:
                best, us = b.autotune(reps=3)
                print(f"  {best} {us:.1f} us", flush=True)
                assert best == b.tuning() == fresh
            a = [b.get_array(k) for k in (ljamd.ARRAY_POS, ljamd.ARRAY_VEL, ljamd.ARRAY_FORCE)]
            h = b.integrate_hist(0.004, 20)
            out.append((*a, h, b.stats(), b.get_array(ljamd.ARRAY_POS), b.get_array(ljamd.ARRAY_VEL)))
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("n,steps", [([10007, 300, 5003, 1], 8), ([40001], 2)])
@pytest.mark.parametrize("canon", [ljamd.EVN, ljamd.TVN])
def test_large_boxes_untuned(canon, n, steps):
    """Boxes well above the sizes a single box takes in one launch, against the
    sliced tuning, with the bounds of the small boxes.  (A single particle's seeded
    velocity, without its mean and scaled to T, is no number: alike on both sides.)"""
    def gap(x, y):
        no = np.isnan(x)
        assert np.array_equal(no, np.isnan(y))
        return np.max(np.abs(np.where(no, 0.0, x - y)))

    n = np.array(n, np.int32)
    print(f"\n[case] large untuned batch {n} canon={canon}", flush=True)
    out = []
    for tuning in (None, (1, 512, 4, 0)):
        with ljamd.LJBatch(n, np.full(n.size, 0.6), np.full(n.size, 1.2), canonical=canon, seed=33) as b:
            if tuning:
                b.set_tuning(*tuning)
            h = b.integrate_hist(0.004, steps)
            out.append((h, *[[b.get_array(a, box=k) for k in range(n.size)]
                             for a in (ljamd.ARRAY_POS, ljamd.ARRAY_VEL)]))
    (h, p, v), (hs, ps, vs) = out
    for k in range(n.size):
        assert np.any(np.isnan(h[:, k])) == (n[k] == 1)
        assert gap(h[:, k, 0], hs[:, k, 0]) / n[k] <= 2e-5, k
        assert gap(xyz(p[k]), xyz(ps[k])) <= 4e-5, k
        assert gap(xyz(v[k]), xyz(vs[k])) <= 1e-3, k


def test_many_small_boxes_untuned():
    """2000 boxes of 200, beyond the one-launch step's sizes: the default tiling's
    step, whose bits do not depend on how its items are handed out."""
    n = np.full(2000, 200, np.int32)
    out = []
    for tuning in (None, (1, 512, 4, 0)):
        with ljamd.LJBatch(n, np.full(2000, 0.5), np.full(2000, 1.0), seed=34) as b:
            if tuning:
                b.set_tuning(*tuning)
            h = b.integrate_hist(0.004, 9)
            out.append((h, b.get_array(ljamd.ARRAY_POS), b.get_array(ljamd.ARRAY_VEL),
                        b.get_array(ljamd.ARRAY_FORCE)))
    for x, y in zip(*out):
        assert np.array_equal(x, y)
