"""Gravity of a plan whose softening is h: the softened pairs summed with the
density (over the lists, or by the walk where a list overflows or the lists are
off), the others as clamped point masses, by every kernel that takes them: the
tiled sum with and without a j split, the symmetric sum with full, partial and
single blocks.  Against the FP64 sum of the same state; the bar is 1e-6 relative
RMS (a pair's FP32 factor is good to a few 2^-24, and both sides of a softened
pair's difference carry it)."""
import numpy as np
import pytest

import oracle
from sph_2_amd import ic

pytestmark = pytest.mark.gpu


def _check(n, cfg, masses="equal", lists=True, wide=False):
    from sph_2_amd.plan import SphPlan

    e = ic.evrard(n, seed=21)
    kw = {}
    if masses == "varied":
        w = np.random.default_rng(3).uniform(0.5, 1.5, n)
        e.m = w / w.sum()
    if wide:  # lengths that no iteration narrows: more than 128 neighbours for some
        e.h = np.where(e.pos[:, 0] > 0.3, 2.0 * e.h, e.h)
        kw = dict(max_iter=1)
    pl = SphPlan(n, **kw)
    pl.set_gravity_config(*cfg)
    pl.set_neighbor_lists(lists)
    pl.load(e.pos, e.vel, e.u, e.m, e.h)
    pl.init()
    s, c = pl.state(), pl.counters()
    pl.close()
    if wide:
        assert (c["nbr_overflow"] > 0) == lists
    want = oracle.gravity(s["pos"], e.m, s["h"])
    err = np.sqrt(((s["acc_g"] - want) ** 2).sum() / (want ** 2).sum())
    assert err < 1e-6, err


@pytest.mark.parametrize("masses", ["equal", "varied"])
@pytest.mark.parametrize("cfg", [(1, 256, 1), (1, 256, 16), (2, 512, 3), (4, 512, 1), (8, 512, 1),
                                 (8, 512, 3)])
@pytest.mark.parametrize("n", [65, 513, 2500])
def test_soft_gravity(gpu, n, cfg, masses):
    _check(n, cfg, masses)


@pytest.mark.parametrize("n", [512, 640, 641, 1151, 9000])
def test_symmetric_blocks(gpu, n):
    _check(n, (8, 512, 2))


@pytest.mark.parametrize("lists", [True, False])
@pytest.mark.parametrize("cfg", [(1, 256, 16), (8, 512, 1)])
def test_soft_gravity_by_the_walk(gpu, cfg, lists):
    _check(6000, cfg, lists=lists, wide=True)


def test_tuner_times_the_steps_of_a_plan(gpu, monkeypatch):
    """The shape table is for the kernels of a resident run, not for those of the
    stateless call."""
    from sph_2_amd import autotune, libsx

    def never(*a, **kw):
        raise AssertionError("stateless gravity call")

    monkeypatch.setattr(libsx, "getAcc_g_smth", never)
    best, res = autotune.tune_gravity(1500, reps=1, write=False)
    assert ",".join(map(str, best)) in res and all(v > 0.0 for v in res.values())
    assert {"1,256,1", "2,1024,4", "8,512,1", "8,512,64"} <= set(res)
