"""Barnes-Hut gravity on the GPU against FP64 direct summation."""
import numpy as np
import pytest

import oracle
from sph_2_amd import ic

pytestmark = pytest.mark.gpu


def rel_rms(a, b):
    return float(np.sqrt(((a - b) ** 2).sum() / (b ** 2).sum()))


@pytest.fixture(scope="module")
def plummer():
    p = ic.plummer(40000, seed=4, eps=0.01)
    rows = np.arange(0, 40000, 17)
    ref = oracle.gravity(p.pos, p.m, p.eps, 1.0, rows=rows)
    return p, rows, ref


def test_bh_error_decreases_with_theta(gpu, plummer):
    from sph_2_amd import libsx

    p, rows, ref = plummer
    errs = []
    for theta in (0.7, 0.5, 0.3, 0.1):
        acc, st = libsx.getAcc_g_bh(p.pos, p.m, 1.0, p.eps, theta, return_stats=True)
        assert st["overflow"] == 0
        errs.append(rel_rms(acc[rows], ref))
    assert errs[0] > errs[1] > errs[2] > errs[3]
    assert errs[0] < 2e-2 and errs[1] < 1e-2 and errs[2] < 3e-3 and errs[3] < 2e-4


def test_bh_tree_covers_every_particle(gpu, plummer):
    """theta -> 0 opens every cell: the walk reduces to the direct sum."""
    from sph_2_amd import libsx

    p, rows, ref = plummer
    small = ic.plummer(3000, seed=9, eps=0.05)
    acc, st = libsx.getAcc_g_bh(small.pos, small.m, 1.0, small.eps, 1e-6, return_stats=True)
    ref2 = oracle.gravity(small.pos, small.m, small.eps, 1.0)
    assert st["interactions"] == 3000 * 3000
    assert rel_rms(acc, ref2) < 1e-5


def test_bh_rows_and_duplicates(gpu):
    """Coincident particles end in unsplittable leaves; rows select targets."""
    from sph_2_amd import libsx

    p = ic.plummer(5000, seed=2, eps=0.02)
    pos = p.pos.copy()
    pos[100:140] = pos[7]          # 41 particles at one point
    acc = libsx.getAcc_g_bh(pos, p.m, 1.0, p.eps, 0.4, nbeg=50, nend=300)
    ref = oracle.gravity(pos, p.m, p.eps, 1.0, rows=np.arange(50, 300))
    assert acc.shape == (250, 3)
    assert rel_rms(acc, ref) < 5e-3


def test_plan_step_with_tree_gravity(gpu):
    """The step with Barnes-Hut gravity: theta -> 0 reproduces the direct-sum
    step; theta = 0.5 stays within the tree's force error; the SPH part of
    the bootstrap is identical (same positions, same neighbour decisions)."""
    from sph_2_amd.plan import SphPlan

    e = ic.evrard(8192, seed=21)
    p = oracle.Params()
    s0 = oracle.bootstrap(oracle.State(e.pos, e.vel, e.u, e.m, e.h), p)
    out = {}
    for theta in (0.0, 1e-6, 0.5):
        pl = SphPlan(8192)
        pl.set_gravity_bh(theta)
        pl.load(e.pos, e.vel, e.u, e.m, e.h)
        pl.init()
        st0 = pl.state()
        pl.step(2, 1e-4)
        out[theta] = (st0, pl.state(), pl.counters())
        pl.close()
    d0, d1, _ = out[0.0]
    for theta in (1e-6, 0.5):
        b0, b1, cnt = out[theta]
        assert cnt["bh_overflow"] == 0
        assert np.array_equal(b0["h"], d0["h"]) and np.array_equal(b0["rho"], d0["rho"])
        tol = 1e-5 if theta < 1e-3 else 3e-3
        assert rel_rms(b0["acc_g"], s0.acc_g) < tol
        assert rel_rms(b1["acc_g"], d1["acc_g"]) < tol
        assert rel_rms(b1["pos"], d1["pos"]) < 1e-9
    assert rel_rms(out[1e-6][0]["acc_g"], d0["acc_g"]) < 1e-5
    assert rel_rms(d0["acc_g"], s0.acc_g) < 1e-5


def test_plan_tree_gravity_rejected_in_fp64_mode(gpu):
    from sph_2_amd.plan import SphPlan

    pl = SphPlan(1024, mode="fp64")
    with pytest.raises(Exception):
        pl.set_gravity_bh(0.5)
    pl.close()


@pytest.mark.parametrize("theta,tol_pot,tol_acc", [(0.5, 3e-4, 3e-3), (0.3, 1e-4, 1e-3),
                                                   (0.1, 5e-6, 2e-5), (1e-6, 1e-6, 1e-5)])
def test_bh_potential(gpu, theta, tol_pot, tol_acc):
    """The walk's potential and accelerations (the deep walk below theta
    0.35, the shallow one above) against the FP64 direct sum, which theta ->
    0 reproduces to FP32 round-off (measured on this input: potential 1e-4,
    3e-5, 7e-7, 3e-8 and accelerations 8e-4, 2e-4, 3e-6, 1.4e-7 relative RMS
    at theta 0.5, 0.3, 0.1, 1e-6)."""
    from sph_2_amd import libsx

    p = ic.plummer(6000, seed=5, eps=0.02)
    acc, pot = libsx.getAcc_g_bh(p.pos, p.m, 1.0, p.eps, theta, return_potential=True)
    acc_o, pot_o = oracle.gravity(p.pos, p.m, p.eps, 1.0, potential=True)
    assert rel_rms(pot, pot_o) < tol_pot
    assert rel_rms(acc, acc_o) < tol_acc


@pytest.mark.parametrize("n", [1, 63, 2049, 8192, 8193, 32768, 32769, 98305])
def test_bh_waves_of_a_group_cover_every_pair(gpu, n):
    """Groups walked by several waves (eight, four, two or one for a whole run by
    its size, and parts for outliers beside full cells): every particle is summed
    once at an opening angle that opens every cell, and its force is the direct
    sum's to FP32 rounding (1e-5 relative RMS, the bar of the tree that covers
    every particle)."""
    from sph_2_amd import libsx

    p = ic.plummer(n, seed=31, eps=0.02)
    acc, pot, st = libsx.getAcc_g_bh(p.pos, p.m, 1.0, p.eps, 1e-6, return_potential=True,
                                     return_stats=True)
    assert st["interactions"] == n * n and st["overflow"] == 0
    rows = np.unique(np.r_[np.argsort((p.pos ** 2).sum(1))[-40:], np.linspace(0, n - 1, 40).astype(int)])
    rows = rows[(rows >= 0) & (rows < n)]
    if n > 1:
        ref = oracle.gravity(p.pos, p.m, p.eps, 1.0, rows=rows)
        assert rel_rms(acc[rows], ref) < 1e-5
    plain = libsx.getAcc_g_bh(p.pos, p.m, 1.0, p.eps, 1e-6)
    assert rel_rms(plain, acc) < 1e-6 if n > 1 else np.array_equal(plain, acc)
    again = libsx.getAcc_g_bh(p.pos, p.m, 1.0, p.eps, 1e-6)
    assert np.array_equal(plain, again)


@pytest.mark.parametrize("n,each", [(9, 9), (900, 9), (9000, 9), (9000, 100), (40000, 2)])
def test_bh_deep_trees(gpu, n, each):
    """Clusters of coincident particles: chains of cells down to the deepest
    level, more levels and more cells than the build starts with, and leaves
    that hold more than eight.  Every particle is summed once (an angle of 1e-7
    opens the deepest cells too, whose side is 2^-21 of the box's: s / theta is
    4.8 box sides)."""
    from sph_2_amd import libsx

    c = ic.plummer(max(2, n // each), seed=32, eps=0.05)
    pos = np.repeat(c.pos, each, axis=0)[:n]
    m = np.full(n, 1.0 / n)
    eps = np.full(n, 0.05)
    acc, st = libsx.getAcc_g_bh(pos, m, 1.0, eps, 1e-7, return_stats=True)
    assert st["interactions"] == n * n and st["overflow"] == 0
    assert each <= 8 or st["depth"] == 21 or n == 9
    rows = np.linspace(0, n - 1, 50).astype(int)
    ref = oracle.gravity(pos, m, eps, 1.0, rows=rows)
    assert np.sqrt(((acc[rows] - ref) ** 2).sum()) < 1e-5 * max(1.0, np.sqrt((ref ** 2).sum()))
