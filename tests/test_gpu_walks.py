"""The candidate walks at the sizes where their shape changes (an eighth, a
quarter, a half or a whole bucket per group: 256 / 257, 384 / 385, 1,536 / 1,537
and 3,072 / 3,073 buckets), with a partial last bucket, and where the FP32 screen of the FP64 distance test
is hardest: coordinates far from the origin, units far from one, distances that
equal the radius.  Counts and smoothing lengths bit for bit the oracle's."""
import numpy as np
import pytest

import oracle
from sph_2_amd import ic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 65, 1000, 16384, 16385, 24576, 24577, 98304, 98305, 196608, 196650])
def test_walk_shapes(gpu, n):
    from sph_2_amd import libsx

    e = ic.evrard(n, seed=11)
    rows = np.unique(np.r_[0:min(n, 200), np.linspace(0, n - 1, min(n, 300)).astype(int)])
    h, k, it = libsx.smoothing_h(e.pos, e.h)
    ho, ko, ito, _ = oracle.smoothing(e.pos, e.h, rows=rows)
    assert np.array_equal(h[rows], ho) and np.array_equal(k[rows], ko)
    assert np.array_equal(it[rows], ito)
    rho, cnt = libsx.getDensity(e.pos, e.m, h, return_count=True)
    rho_o, cnt_o = oracle.density(e.pos, e.m, h, rows=rows)
    assert np.array_equal(cnt[rows], cnt_o)
    assert np.max(np.abs(rho[rows] / rho_o - 1.0)) < 1e-6


@pytest.mark.parametrize("shift,scale", [(1e6, 1.0), (0.0, 3.0e21), (0.0, 1e-150), (0.0, 1e150)])
def test_walk_frames(gpu, shift, scale):
    """Offsets and units: the counts only compare distances, so any scale does."""
    from sph_2_amd import libsx

    e = ic.evrard(3000, seed=12)
    pos, h0 = e.pos * scale + shift, e.h * scale
    h, k, _ = libsx.smoothing_h(pos, h0)
    ho, ko, _, _ = oracle.smoothing(pos, h0)
    assert np.array_equal(h, ho) and np.array_equal(k, ko)


def test_walk_distances_at_the_radius(gpu):
    """A cubic lattice with h = 1 and 1.5: thousands of pairs lie exactly at r =
    h_i + h_j, which counts them, and every batch holds one."""
    from sph_2_amd import libsx

    g = np.arange(14.0)
    pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    m = np.full(len(pos), 1.0 / len(pos))
    for h in (1.0, 1.5):
        hh = np.full(len(pos), h)
        rho, cnt = libsx.getDensity(pos, m, hh, return_count=True)
        rho_o, cnt_o = oracle.density(pos, m, hh)
        assert np.array_equal(cnt, cnt_o)
        assert np.max(np.abs(rho / rho_o - 1.0)) < 1e-6


def test_lists_of_the_stateless_calls_overflow(gpu):
    """Particles with more neighbours than a list holds beside others without:
    the stateless density, div/curl and hydro take the walk for those buckets."""
    from sph_2_amd import libsx

    e = ic.evrard(6000, seed=13)
    rng = np.random.default_rng(5)
    v = rng.standard_normal((e.n, 3))
    h = np.where(e.pos[:, 0] > 0.4, 2.0 * e.h, e.h)
    rho, cnt = libsx.getDensity(e.pos, e.m, h, return_count=True)
    rho_o, cnt_o = oracle.density(e.pos, e.m, h)
    assert cnt_o.max() > 128 and cnt_o.min() < 128
    assert np.array_equal(cnt, cnt_o)
    assert np.max(np.abs(rho / rho_o - 1.0)) < 1e-6
    dv, cv = libsx.div_curlVel(e.pos, v, rho_o, e.m, h)
    dvo, cvo = oracle.divcurl(e.pos, v, rho_o, e.m, h)
    P, c = (2.0 / 3.0) * rho_o * e.u, np.sqrt(10.0 / 9.0 * e.u)
    acc, du = libsx.getAcc_sph_dU(e.pos, v, rho_o, P, c, h, e.m, balsara=1, divV=dvo, curlV=cvo)
    acco, duo = oracle.hydro(e.pos, v, rho_o, P, c, h, e.m, dvo, cvo, oracle.Params(balsara=1))
    for a, b in ((dv, dvo), (cv, cvo), (acc, acco), (du, duo)):
        assert np.sqrt(((a - b) ** 2).sum() / (b ** 2).sum()) < 1e-5


@pytest.mark.parametrize("n", [1, 17, 63, 32768, 32769, 33001])
def test_list_passes_equal_the_walks(gpu, n):
    """The list passes on both sides of 512 buckets (four lanes a particle and
    the overflowed buckets walked in the same launch; above it the walks in a
    launch of their own), with partial buckets: the lists give the walks' bits,
    with lists that overflow and without."""
    from sph_2_amd.plan import SphPlan

    for wide in (False, True):
        e = ic.evrard(n, seed=23)
        kw = {}
        if wide:
            e.h = np.where(e.pos[:, 0] > 0.3, 3.0 * e.h, e.h)
            kw = dict(max_iter=1)
        outs = []
        for lists in (True, False):
            pl = SphPlan(n, **kw)
            pl.set_cell_level(0)
            pl.set_neighbor_lists(lists)
            pl.load(e.pos, e.vel, e.u, e.m, e.h)
            pl.init()
            pl.step(1, 1e-4)
            outs.append(pl.state())
            c = pl.counters()
            pl.close()
            if lists and n > 1000:
                assert (c["buckets"] <= 512) == (n <= 32768), c
                assert (c["nbr_overflow"] > 0) == wide, c
        for f in outs[0]:
            assert np.array_equal(outs[0][f], outs[1][f]), (f, wide)


def _capped_ok(call, *a, **kw):
    import warnings

    with warnings.catch_warnings():
        warnings.simplefilter("ignore", RuntimeWarning)  # the odd particle finds no length
        return call(*a, **kw)


@pytest.mark.parametrize("h_mode", [0, 2, 5])
@pytest.mark.parametrize("where", [(np.inf, 0.1, 0.1), (0.1, -np.inf, 0.1), (np.inf, -np.inf, np.inf)])
def test_infinite_position_beside_valid_rows(gpu, where, h_mode):
    """A particle at infinity has no neighbours and is nobody's: the other rows,
    those of its own group among them, are what they are without it."""
    from sph_2_amd import libsx

    e = ic.evrard(700, seed=31)
    pos = e.pos.copy()
    pos[333] = where
    rows = np.delete(np.arange(e.n), 333)
    h, k, it = _capped_ok(libsx.smoothing_h, pos, e.h, h_mode=h_mode)
    ho, ko, ito, _ = oracle.smoothing(pos, e.h, p=oracle.Params(h_mode=h_mode), rows=rows)
    assert np.array_equal(h[rows], ho) and np.array_equal(k[rows], ko) and np.array_equal(it[rows], ito)
    rho, cnt = libsx.getDensity(pos, e.m, e.h, return_count=True)
    rho_o, cnt_o = oracle.density(pos, e.m, e.h, rows=rows)
    assert np.array_equal(cnt[rows], cnt_o)
    assert np.max(np.abs(rho[rows] / rho_o - 1.0)) < 1e-6


@pytest.mark.parametrize("huge", [1e10, 1e18, 1e19, 1e25, 1e100, 1e200, np.inf])
def test_huge_h_beside_valid_rows(gpu, huge):
    """One particle with a huge or infinite h: everybody's neighbour, with no
    weight, and no more to the rows beside it."""
    from sph_2_amd import libsx

    e = ic.evrard(700, seed=32)
    h = e.h.copy()
    h[100] = huge
    rho, cnt = libsx.getDensity(e.pos, e.m, h, return_count=True)
    rho_o, cnt_o = oracle.density(e.pos, e.m, h)
    assert np.array_equal(cnt, cnt_o)
    ok = np.arange(e.n) != 100
    assert np.max(np.abs(rho[ok] / rho_o[ok] - 1.0)) < 1e-6
    assert rho[100] == pytest.approx(rho_o[100], rel=1e-5, abs=1e-30)
    if huge < np.inf:
        # far particles, one of which only that h reaches
        pos = e.pos.copy()
        pos[200] = (0.0, 1.5 * huge, 0.0)
        pos[201] = (0.5 * huge, 0.0, 0.0)
        cnt = libsx.getDensity(pos, e.m, h, return_count=True)[1]
        assert np.array_equal(cnt, oracle.density(pos, e.m, h)[1])


@pytest.mark.parametrize("h_mode", [0, 2, 5])
def test_infinite_start_beside_valid_rows(gpu, h_mode):
    """A particle whose iteration starts from an infinite length, and the rows
    of its group."""
    from sph_2_amd import libsx

    e = ic.evrard(700, seed=33)
    h0 = e.h.copy()
    h0[400] = np.inf
    rows = np.delete(np.arange(e.n), 400)
    h, k, it = _capped_ok(libsx.smoothing_h, e.pos, h0, h_mode=h_mode)
    ho, ko, ito, _ = oracle.smoothing(e.pos, h0, p=oracle.Params(h_mode=h_mode), rows=rows)
    assert np.array_equal(h[rows], ho) and np.array_equal(k[rows], ko) and np.array_equal(it[rows], ito)


@pytest.mark.parametrize("shift", [0.0, 2.0 ** 46, 2.0 ** 51, 2.0 ** 52])
def test_far_offsets(gpu, shift):
    """Particles so far from the origin that the middle of a group's box is
    rounded by a good part of the search radius: a lattice whose pairs lie on the
    radius, and a sphere."""
    from sph_2_amd import libsx

    g = np.arange(14.0)
    pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3) + shift
    m = np.full(len(pos), 1.0 / len(pos))
    for r in (2.0, 3.0):
        hh = np.full(len(pos), 0.5 * r)
        cnt = libsx.getDensity(pos, m, hh, return_count=True)[1]
        assert np.array_equal(cnt, oracle.density(pos, m, hh)[1])
        for h_mode in (0, 2):
            h, k, it = _capped_ok(libsx.smoothing_h, pos, hh, h_mode=h_mode)
            ho, ko, ito, _ = oracle.smoothing(pos, hh, p=oracle.Params(h_mode=h_mode))
            assert np.array_equal(h, ho) and np.array_equal(k, ko) and np.array_equal(it, ito)
    e = ic.evrard(3000, seed=34)
    pos, h0 = 64.0 * e.pos + shift * np.array([1.0, -0.75, 0.875]), 64.0 * e.h
    cnt = libsx.getDensity(pos, e.m, h0, return_count=True)[1]
    assert np.array_equal(cnt, oracle.density(pos, e.m, h0)[1])


def test_large_lists_are_given_back(gpu):
    """The stateless calls hold the neighbour lists of small runs only: after
    div/curl of 5,000,000 particles (3 GB of lists, 1.3 GB of particle arrays) the
    device has that memory again, and smaller calls in the same context, whose
    lists are made anew, give what a context of their own gives."""
    import ctypes as C

    from sph_2_amd import _lib

    L = _lib.load()
    st = _lib.stream_handle()
    rng = np.random.default_rng(2)

    def divcurl(ctx, n):
        pos, m = _lib.dev(rng.random((n, 3))), _lib.dev(np.full(n, 1.0 / n))
        v = _lib.dev(rng.standard_normal((n, 3)))
        h = _lib.dev(np.full(n, 0.62 * (64.0 / (4.19 * n)) ** (1.0 / 3.0)))
        div, curl = (gpu.empty(n, dtype=gpu.float64, device="cuda") for _ in range(2))
        args = [a.data_ptr() for a in (pos, v, m, m, h)]  # (rho: any)

        def call(c, a, b):
            assert L.sphx_div_curlVel(c, _lib.MIXED, n, *args, 0, n, a.data_ptr(), b.data_ptr(), st) == 0

        call(ctx, div, curl)
        gpu.cuda.synchronize()
        own = C.c_void_p()
        assert L.sphx_ctx_create(0, C.byref(own)) == 0
        want = gpu.empty_like(div), gpu.empty_like(curl)
        call(own, *want)
        gpu.cuda.synchronize()
        assert L.sphx_ctx_destroy(own) == 0
        assert gpu.equal(div, want[0]) and gpu.equal(curl, want[1])

    ctx = C.c_void_p()
    assert L.sphx_ctx_create(0, C.byref(ctx)) == 0
    divcurl(ctx, 2000)
    gpu.cuda.empty_cache()
    free = gpu.cuda.mem_get_info()[0]
    divcurl(ctx, 5_000_000)
    gpu.cuda.empty_cache()
    taken = free - gpu.cuda.mem_get_info()[0]
    assert taken < 2.0e9, taken
    for n in (1080, 2000, 100_000, 1_000_001):
        divcurl(ctx, n)
    gpu.cuda.synchronize()
    gpu.cuda.empty_cache()
    taken = free - gpu.cuda.mem_get_info()[0]
    assert taken < 4.5e9, taken
    assert L.sphx_ctx_destroy(ctx) == 0


def test_overflowing_lists_are_walked_by_the_whole_device(gpu):
    """Eight times the neighbours, so that every list overflows: the walks that
    take their place cost a few times the list passes (2 to 4 here), not the
    fiftyfold that 17 waves took for 1,028 buckets."""
    import time

    from sph_2_amd import libsx

    e = ic.evrard(65752, seed=3)
    v = np.random.default_rng(1).standard_normal((e.n, 3))

    def best(f):
        t = []
        for _ in range(4):
            t0 = time.perf_counter()
            f()
            t.append(time.perf_counter() - t0)
        return min(t)

    rho = libsx.getDensity(e.pos, e.m, e.h)
    for f in (lambda h: libsx.getDensity(e.pos, e.m, h), lambda h: libsx.div_curlVel(e.pos, v, rho, e.m, h)):
        narrow, wide = best(lambda: f(e.h)), best(lambda: f(2.0 * e.h))
        assert wide < 8.0 * narrow, (wide, narrow)
