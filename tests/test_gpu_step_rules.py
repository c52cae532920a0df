"""The step rules of the smoothing length (h_mode 2-5) where the window of
distances that replaces their walks is hardest to find: starts far from the
band, more particles at one distance than the window holds, a run smaller than
the band, passes that end outside the window.  Every h, count and pass count
bit for bit the oracle's."""
import numpy as np
import pytest

import oracle
from sph_2_amd import ic

pytestmark = pytest.mark.gpu


def _case(name):
    e = ic.evrard(1500, seed=4)
    if name == "guess":
        return e.pos, e.h
    if name == "starts":  # from a fifth to five times the length
        return e.pos, e.h * np.geomspace(0.2, 5.0, e.n)
    if name == "lattice":  # shells of up to 48 particles at one distance
        g = np.arange(11.0)
        pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
        return pos, np.full(len(pos), 1.3)
    if name == "coincident":  # 80 particles on one point among others
        pos = e.pos[:700].copy()
        pos[100:180] = pos[100]
        return pos, e.h[:700]
    if name == "few":  # fewer particles than the band asks for
        return e.pos[:50], np.full(50, 0.3)
    if name == "just_enough":  # 65: the band can be met, never passed
        return e.pos[:65], np.full(65, 0.9)
    raise AssertionError(name)


@pytest.mark.parametrize("h_mode", [2, 3, 4, 5])
@pytest.mark.parametrize("name", ["guess", "starts", "lattice", "coincident", "few", "just_enough"])
def test_step_rules_match_the_oracle(gpu, name, h_mode):
    import warnings

    from sph_2_amd import libsx

    pos, h0 = _case(name)
    ho, ko, ito, _ = oracle.smoothing(pos, h0, p=oracle.Params(h_mode=h_mode))
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", RuntimeWarning)  # the pass limit, as in the oracle
        h, k, it = libsx.smoothing_h(pos, h0, h_mode=h_mode)
    assert np.array_equal(h, ho)
    assert np.array_equal(k, ko)
    assert np.array_equal(it, ito)


@pytest.mark.parametrize("h_mode", [2, 4, 5])
@pytest.mark.parametrize("nngb,ndown,nup", [(64, 44, 84), (64, 35, 93), (64, 35, 94), (64, 20, 110),
                                            (200, 170, 230), (32, 1, 33), (32, 0, 40), (500, 480, 520)])
def test_bands(gpu, nngb, ndown, nup, h_mode):
    """Bands that nearly fill the window's 64 distances, the widest that takes one
    (35 to 93), those that take none, and other neighbour numbers."""
    import warnings

    from sph_2_amd import libsx

    e = ic.evrard(900, seed=6)
    h0 = e.h * np.geomspace(0.5, 2.0, e.n) * (nngb / 64.0) ** (1.0 / 3.0)
    kw = dict(h_mode=h_mode, nngb=nngb, ndown=ndown, nup=nup)
    ho, ko, ito, _ = oracle.smoothing(e.pos, h0, p=oracle.Params(**kw))
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", RuntimeWarning)
        h, k, it = libsx.smoothing_h(e.pos, h0, **kw)
    assert np.array_equal(h, ho) and np.array_equal(k, ko) and np.array_equal(it, ito)


def test_wide_band_costs_no_more(gpu):
    """From 1.3 times the length the passes are many for any band.  A band of 41
    counts, which the window still holds, takes about what the narrow one takes;
    searching for its window in vain took a walk for each of 100 passes."""
    import time

    from sph_2_amd import libsx

    e = ic.evrard(16384, seed=6)
    h0 = 1.3 * libsx.smoothing_h(e.pos, e.h)[0]

    def best(**kw):
        t = []
        for _ in range(6):
            t0 = time.perf_counter()
            libsx.smoothing_h(e.pos, h0, h_mode=2, max_iter=200, **kw)
            t.append(time.perf_counter() - t0)
        return min(t)

    narrow = best(nngb=64, ndown=59, nup=69)
    wide = best(nngb=64, ndown=44, nup=84)
    assert wide < 2.5 * narrow, (wide, narrow)


def test_far_starts_cost_no_more(gpu):
    """Starts from a third of the length to three times it find their windows too:
    some 1.5 times what starts from the guess take, where one target walked pass by
    pass (400 of them) takes five."""
    import time

    from sph_2_amd import libsx

    e = ic.evrard(98304, seed=17)
    h0 = e.h.copy()
    h0[::7] *= np.geomspace(1.0 / 3.0, 3.0, len(h0[::7]))

    def best(h):
        t = []
        for _ in range(6):
            t0 = time.perf_counter()
            libsx.smoothing_h(e.pos, h, h_mode=5)
            t.append(time.perf_counter() - t0)
        return min(t)

    near, far = best(e.h), best(h0)
    assert far < 3.0 * near, (far, near)


@pytest.mark.parametrize("h_mode", [2, 4, 5])
@pytest.mark.parametrize("n", [24576, 24577, 98304, 98305])
def test_step_rules_at_every_group_size(gpu, n, h_mode):
    """A quarter, a half and a whole bucket per group (384 / 385 and 1,536 / 1,537
    buckets, the last one partial), from the guess, from starts up to three times
    off among them with 80 particles on one point, and (rules with one) from the eq.
    31 start of a step later: sampled rows, the clustered ones among them."""
    import warnings

    from sph_2_amd import libsx

    e = ic.evrard(n, seed=17)
    # (10,001 passes for h_mode 5's clustered rows: one of them)
    rows = np.unique(np.r_[0:32 if h_mode == 5 else 64, 40, np.linspace(0, n - 1, 160).astype(int)])
    p = oracle.Params(h_mode=h_mode)

    def check(pos, h0, **kw):
        ho, ko, ito, _ = oracle.smoothing(pos, h0, p=p, rows=rows, **kw)
        with warnings.catch_warnings():
            warnings.simplefilter("ignore", RuntimeWarning)
            if kw:
                out = libsx._smoothing(pos, h0, kw["k_prev"], kw["divV"], kw["dt"], None, None,
                                       "mixed", 0, h_mode=h_mode)
            else:
                out = libsx.smoothing_h(pos, h0, h_mode=h_mode)
        for got, want in zip(out, (ho, ko, ito)):
            assert np.array_equal(got[rows], want)
        return out

    check(e.pos, e.h)
    pos, h0 = e.pos.copy(), e.h.copy()
    h0[::7] *= np.geomspace(1.0 / 3.0, 3.0, len(h0[::7]))
    pos[32:112] = pos[32]
    check(pos, h0)
    if h_mode != 5:
        h, k, _ = libsx.smoothing_h(e.pos, e.h)
        r = np.sqrt((e.pos ** 2).sum(axis=1))
        vel = -0.8 / (0.3 + r)[:, None] * e.pos
        check(e.pos + 1e-3 * vel, h, k_prev=k, divV=-0.8 * (0.9 + 2.0 * r) / (0.3 + r) ** 2, dt=1e-3)
