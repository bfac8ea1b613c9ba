"""Several steps per launch on small lattices (tiles in LDS) against one
launch per step.

STEP_NO_GRAPH launches every step by itself through the kernels that the
parity tests pin to the oracle; the tiles must give the same bits.  Sizes lie
at the edges of the tiles (8 to 24 stored nodes a side), step counts at every
remainder of a launch and past a captured graph."""
import numpy as np
import pytest

import lbm_amd as L
from test_gpu_march import POLICIES, make, random_class, state

pytestmark = pytest.mark.gpu

SIZES = [(3, 3), (3, 200), (200, 3), (7, 9), (8, 8), (9, 17), (16, 15), (40, 96), (128, 130), (129, 128), (225, 231),
         (401, 403), (240, 1201)]


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED, L.F16_SHIFTED])
@pytest.mark.parametrize("nr,nc", SIZES)
def test_same_bits_as_single_steps(nr, nc, storage):
    rng = np.random.default_rng(1000 * nr + nc)
    for case in range(3):
        cls = random_class(rng, nr, nc, (0.0, 0.15, 0.4)[case])
        policies = (POLICIES[case], POLICIES[(case + nr) % 3])
        collision = (L.BGK, L.TRT)[(case + nc) % 2]
        p0 = state(rng, nc, nr)
        vals = int(rng.integers(1 << 30))
        lats = [make(cls, np.random.default_rng(vals), storage, collision, policies) for _ in range(2)]
        for lat in lats:
            lat.upload_populations(p0)
        done = 0
        for n in ((1, 2, 7), (9, 3, 100), (8, 5, 33))[case]:
            # new prescribed values before every call
            ux = rng.uniform(-0.02, 0.02)
            for lat, flags in zip(lats, (0, L.STEP_NO_GRAPH)):
                k = len(lat.open_nodes(0))
                lat.set_open_values(0, ux=np.full(k, ux), rho=np.full(k, 1.0 + ux / 4))
                lat.step(n, flags | L.STEP_MACRO | L.STEP_CHECK)
            done += n
            a, b = lats
            assert a.time == b.time == done
            for x, y in zip(a.macro(), b.macro()):
                assert np.array_equal(x, y)
            assert np.array_equal(a.populations(), b.populations()), (nr, nc, case, n)
            assert np.array_equal(a.after_collision(), b.after_collision())
        for lat in lats:
            lat.close()


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED, L.F16_SHIFTED])
def test_planes(storage):
    rng = np.random.default_rng(2)
    cls = random_class(rng, 150, 170, 0.2)
    p0 = state(rng, 170, 150)
    out = []
    for options in (0, L.OPT_PLANAR_LAYOUT):
        lat = L.Lattice(cls, tau=0.8, storage=storage, options=options)
        lat.upload_populations(p0)
        lat.step(77)
        out.append(lat.populations())
        lat.close()
    assert np.array_equal(*out)


def test_flags_of_inner_steps():
    """A NaN, or an FP16 value beyond the format, that appears within a
    launch is reported by the check after it; nothing is reported for the
    tiles' spoilt rings."""
    cls = L.geometry_channel(80, 90)
    rng = np.random.default_rng(3)
    p = state(rng, 90, 80)
    for storage in (L.F64, L.F32_SHIFTED, L.F16_SHIFTED):
        lat = L.Lattice(cls, storage=storage, tau=0.8)
        lat.upload_populations(p)
        lat.step(40, L.STEP_CHECK)
        bad = p.copy()
        bad[3, 40, 41] = np.nan
        lat.upload_populations(bad)
        with pytest.raises(L.LbmError) as e:
            lat.step(5, L.STEP_CHECK)
        assert e.value.code == L.ERR_NAN
        lat.close()
    # |f - w| S beyond the format from the upload on: whatever single steps say
    codes = []
    for flags in (0, L.STEP_NO_GRAPH):
        lat = L.Lattice(cls, storage=L.F16_SHIFTED, tau=0.8, f16_scale=2.0 ** 23)
        lat.upload_populations(p)
        with pytest.raises(L.LbmError) as e:
            lat.step(6, flags | L.STEP_CHECK)
        codes.append(e.value.code)
        lat.close()
    assert codes[0] == codes[1]


def test_range_is_reported_from_tiles():
    """An inlet velocity whose equilibrium leaves the FP16 range: |f1 - w1| =
    1/9 (3 u + 3 u^2) = 0.08 at u = 0.2, times S = 2^20 = 83886 > 65504."""
    cls = L.geometry_channel(80, 90)
    lat = L.Lattice(cls, storage=L.F16_SHIFTED, tau=0.8, f16_scale=2.0 ** 20)
    lat.init_equilibrium()
    lat.step(3, L.STEP_CHECK)
    n = len(lat.open_nodes(0))
    lat.set_open_values(0, ux=np.full(n, 0.2))
    with pytest.raises(L.LbmError) as e:
        lat.step(1, L.STEP_CHECK)
    assert e.value.code == L.ERR_RANGE
    lat.close()


@pytest.mark.parametrize("nr,nc", [(24, 24), (57, 61), (129, 129), (230, 290), (400, 410)])
def test_partially_saturated_obstacles(nr, nc):
    """Obstacles of every weight through the tiles against single steps,
    across calls and captured graphs."""
    rng = np.random.default_rng(nr)
    cls = random_class(rng, nr, nc, 0.1)
    p0 = state(rng, nc, nr)
    lats = [make(cls, np.random.default_rng(1), L.F64, (L.BGK, L.TRT)[nr % 2], POLICIES[:2]) for _ in range(2)]
    nob = int(lats[0].node_counts()[6])
    b = rng.random(nob)
    for lat, flags in zip(lats, (0, L.STEP_NO_GRAPH)):
        lat.set_partial_bounce_back(0.9, b)
        lat.upload_populations(p0)
        for n in (1, 2, 13, 97):
            lat.step(n, flags | L.STEP_MACRO)
    x, y = lats
    assert np.array_equal(x.populations(), y.populations())
    for u, v in zip(x.macro(), y.macro()):
        assert np.array_equal(u, v)
    assert x.lift_drag() == y.lift_drag()
    for lat in lats:
        lat.close()


@pytest.mark.parametrize("storage", [L.F64, L.F16_SHIFTED])
@pytest.mark.parametrize("nr,nc", [(40, 96), (300, 700)])
def test_new_values_every_step(nr, nc, storage):
    """More new values in flight than the waiting slots hold, values that are
    replaced before any step reads them, and steps that take them together
    with older ones; against single steps that wait for every value."""
    rng = np.random.default_rng(nc)
    cls = random_class(rng, nr, nc, 0.1)
    p0 = state(rng, nc, nr)
    lats = [make(cls, np.random.default_rng(4), storage, L.BGK, (L.ZOUHE_VELOCITY, L.ZOUHE_PRESSURE))
            for _ in range(2)]
    n0, n1 = (len(lats[0].open_nodes(k)) for k in (0, 1))
    values = rng.uniform(-0.02, 0.02, (60, 3))
    for lat in lats:
        lat.upload_populations(p0)
    for k, (x, y, r) in enumerate(values):
        for lat, flags in zip(lats, (0, L.STEP_NO_GRAPH)):
            if k % 7 == 3:
                lat.set_open_values(0, ux=np.full(n0, 9.0 * x))    # replaced below
            lat.set_open_values(0, ux=np.full(n0, x), uy=np.full(n0, y))
            if k % 3 == 0:
                lat.set_open_values(1, rho=np.full(n1, 1.0 + r / 4))
            lat.step(1 + (k % 5) * (k % 2), flags)
            if flags:
                lat.synchronize()
    assert np.array_equal(lats[0].populations(), lats[1].populations())
    for lat in lats:
        lat.close()
