"""Several steps per launch (marching waves) against one launch per step.

STEP_NO_GRAPH launches every step by itself through the kernels that the
parity tests pin to the oracle; the marching launches must give the same
bits.  Sizes lie at the edges of the windows (64 - 2K rows for K = 2 .. 5
steps: 60, 58, 56, 54) and of the columns that the first and last columns
influence (2K + 3), step counts at every remainder of a launch and of a
captured graph."""
import numpy as np
import pytest

import lbm_amd as L

pytestmark = pytest.mark.gpu

POLICIES = (L.ZOUHE_VELOCITY, L.ZOUHE_PRESSURE, L.OPEN_NOOP)


def random_class(rng, nr, nc, solid):
    """Every kind of perimeter: walls, open nodes of both lists and plain
    fluid nodes, on all four sides and the corners; discs of one node up."""
    cls = np.where(rng.random((nc, nr)) < solid, L.OBSTACLE, L.FLUID).astype(np.uint8)
    kinds = np.array([L.BOUNDARY, L.INLET, L.OUTLET, L.FLUID], np.uint8)
    for side in (np.s_[0, :], np.s_[-1, :], np.s_[:, 0], np.s_[:, -1]):
        n = cls[side].shape[0]
        cls[side] = np.repeat(rng.choice(kinds, (n + 6) // 7), 7)[:n]
    return cls


def make(cls, rng, storage, collision, policies):
    lat = L.Lattice(cls, collision=collision, tau=0.8, tau_even=0.7, tau_odd=0.9, inlet_policy=policies[0],
                    outlet_policy=policies[1], storage=storage)
    for which in (0, 1):
        n = len(lat.open_nodes(which))
        lat.set_open_values(which, ux=rng.uniform(-0.02, 0.02, n), uy=rng.uniform(-0.02, 0.02, n),
                            rho=rng.uniform(0.99, 1.01, n))
    return lat


def state(rng, nc, nr):
    w = np.array([4 / 9] + [1 / 9] * 4 + [1 / 36] * 4)
    return w[:, None, None] * (1.0 + rng.uniform(-0.02, 0.02, (9, nc, nr)))


# windows end at these row counts (wide lattices), chunks at these column
# counts (tall ones); all of the sizes that take several steps a launch
SIZES = [(3, 100100), (53, 5700), (54, 5560), (55, 5460), (56, 5370), (57, 5301), (58, 5190), (60, 5003), (64, 4700),
         (65, 4630), (112, 2680), (113, 2670), (33400, 9), (30100, 10), (27300, 11), (25100, 12), (23100, 13),
         (21500, 14), (560, 541)]


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
@pytest.mark.parametrize("nr,nc", SIZES)
def test_same_bits_as_single_steps(nr, nc, storage):
    rng = np.random.default_rng(1000 * nr + nc)
    for case in range(3):
        cls = random_class(rng, nr, nc, (0.0, 0.15, 0.4)[case])
        policies = (POLICIES[case], POLICIES[(case + nr) % 3])
        collision = (L.BGK, L.TRT)[(case + nc) % 2]
        p0 = state(rng, nc, nr)
        vals = int(rng.integers(1 << 30))
        for n in ((3, 5, 10), (4, 6, 47), (7, 8, 9))[case]:
            lats = [make(cls, np.random.default_rng(vals), storage, collision, policies) for _ in range(2)]
            for lat, flags in zip(lats, (0, L.STEP_NO_GRAPH)):
                lat.upload_populations(p0)
                lat.step(n, flags | L.STEP_MACRO)
            a, b = lats
            assert a.time == b.time == n
            assert np.array_equal(a.populations(), b.populations()), (nr, nc, case, n)
            for x, y in zip(a.macro(), b.macro()):
                assert np.array_equal(x, y)
            for lat in lats:
                lat.close()


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
def test_long_chunks(storage):
    """A lattice whose waves walk the longest chunks (and, in FP64, take 5
    steps a launch), over more than one captured graph."""
    nr, nc = 1100, 4000
    rng = np.random.default_rng(5)
    cls = random_class(rng, nr, nc, 0.2)
    p0 = state(rng, nc, nr)
    lats = [make(cls, np.random.default_rng(9), storage, L.BGK, POLICIES[:2]) for _ in range(2)]
    for lat, flags in zip(lats, (0, L.STEP_NO_GRAPH)):
        lat.upload_populations(p0)
        lat.step(93, flags)
    a, b = lats
    assert np.array_equal(a.populations(), b.populations())
    # new prescribed values between calls, and a shape set by hand
    for lat, flags in zip(lats, (0, L.STEP_NO_GRAPH)):
        n = len(lat.open_nodes(0))
        lat.set_open_values(0, ux=np.full(n, 0.01))
        lat.step(9, flags)
    a.set_launch(1)
    for lat in lats:
        lat.step(5)
    a.set_launch(0)
    for lat in lats:
        lat.step(6)
    assert np.array_equal(a.populations(), b.populations())
    for lat in lats:
        lat.close()


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
def test_nan_is_reported(storage):
    """A NaN that appears inside a launch of several steps is reported by
    the check after it."""
    cls = L.geometry_channel(80, 90)
    lat = L.Lattice(cls, storage=storage, tau=0.8)
    p = state(np.random.default_rng(3), 90, 80)
    lat.upload_populations(p)
    lat.step(8, L.STEP_CHECK)
    p[3, 40, 41] = np.nan
    lat.upload_populations(p)
    with pytest.raises(L.LbmError) as e:
        lat.step(8, L.STEP_CHECK)
    assert e.value.code == L.ERR_NAN
    lat.close()


@pytest.mark.parametrize("big", [[], [(900, 1300)]])
@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
def test_ensemble_same_bits_as_single_steps(storage, big):
    """Samples of every small size beside larger ones, all kinds of
    perimeter: the ensemble's marching launches against its single steps."""
    shapes = [(3, 3), (5, 9), (57, 10), (56, 11), (64, 12), (113, 40), (300, 200), (129, 700)] + big
    rng = np.random.default_rng(17)
    classes = [random_class(rng, nr, nc, 0.15) for nr, nc in shapes]
    states = [state(rng, nc, nr) for nr, nc in shapes]
    out = []
    for flags in (0, L.STEP_NO_GRAPH):
        lats = [make(c, np.random.default_rng(k), storage, L.TRT, POLICIES[:2]) for k, c in enumerate(classes)]
        for lat, p in zip(lats, states):
            lat.upload_populations(p)
        with L.Batch(lats) as b:
            for n in (1, 4, 5, 43):
                b.step(n, flags)
            lats[6].set_open_values(0, ux=np.full(len(lats[6].open_nodes(0)), 0.005))
            b.step(13, flags)
        assert all(lat.time == 66 for lat in lats)
        out.append([lat.populations() for lat in lats])
        for lat in lats:
            lat.close()
    for shape, x, y in zip(shapes, *out):
        assert np.array_equal(x, y), shape


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
@pytest.mark.parametrize("nr,nc", [(56, 5370), (113, 2670), (30100, 10), (2051, 2047)])
def test_planes(nr, nc, storage):
    """The layout of lattices beyond 4 GiB a buffer, asked for: one stripe of
    windows, several, all windows on the perimeter, and the large lattices'
    launches, at every remainder of a launch."""
    rng = np.random.default_rng(nr + nc)
    cls = random_class(rng, nr, nc, 0.15)
    p0 = state(rng, nc, nr)
    for n in (3, 4, 5, 10, 46):
        out = []
        for options, flags in ((L.OPT_PLANAR_LAYOUT, 0), (L.OPT_PLANAR_LAYOUT, L.STEP_NO_GRAPH)):
            lat = L.Lattice(cls, tau=0.8, inlet_policy=L.ZOUHE_PRESSURE, outlet_policy=L.OPEN_NOOP, storage=storage,
                            options=options)
            lat.set_open_values(0, rho=np.full(len(lat.open_nodes(0)), 1.001))
            assert lat.layout() == L.LAYOUT_PLANES
            lat.upload_populations(p0)
            lat.step(n, flags)
            out.append(lat.populations())
            lat.close()
        assert np.array_equal(*out), n
