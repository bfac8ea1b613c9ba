"""Steps per launch: what is in use can be read, set by hand and brought back,
for a lattice and for an ensemble; the results keep their bits."""
import numpy as np
import pytest

import lbm_amd as L
from test_gpu_march import POLICIES, make, random_class, state

pytestmark = pytest.mark.gpu

# tiles, marching waves of 4 steps, and of 5 (FP64)
SIZES = [(129, 130), (560, 541), (2060, 2040)]


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
@pytest.mark.parametrize("nr,nc", SIZES)
def test_lattice(nr, nc, storage):
    rng = np.random.default_rng(nr)
    cls = random_class(rng, nr, nc, 0.1)
    p0 = state(rng, nc, nr)
    lat = make(cls, np.random.default_rng(1), storage, L.BGK, POLICIES[:2])
    default = lat.steps_per_launch()
    assert default > 1
    lat.set_launch(2)
    assert lat.steps_per_launch() == 1
    lat.set_launch(0)
    assert lat.steps_per_launch() == default
    with pytest.raises(L.LbmError):
        lat.set_steps_per_launch(-1)
    want = None
    for k in (1, 2, 3, 4, default, 100, 0):
        lat.set_steps_per_launch(k)
        assert lat.steps_per_launch() == min(k or default, default)
        lat.upload_populations(p0)
        lat.step(93)
        p = lat.populations()
        want = p if want is None else want
        assert np.array_equal(p, want), k
    # a tuned choice, on another lattice of the same geometry
    lat.autotune(2)
    tuned = lat.launch(), lat.occupancy(), lat.steps_per_launch()
    other = make(cls, np.random.default_rng(1), storage, L.BGK, POLICIES[:2])
    other.set_launch(tuned[0])
    other.set_occupancy(tuned[1])
    other.set_steps_per_launch(tuned[2])
    assert (other.launch(), other.occupancy(), other.steps_per_launch()) == tuned
    other.upload_populations(p0)
    other.step(93)
    assert np.array_equal(other.populations(), want)
    lat.close()
    other.close()


def test_ensemble():
    rng = np.random.default_rng(3)
    shapes = [(300, 200), (129, 700), (200, 250)]
    lats = [make(random_class(rng, nr, nc, 0.1), np.random.default_rng(k), L.F32_SHIFTED, L.TRT, POLICIES[:2])
            for k, (nr, nc) in enumerate(shapes)]
    states = [state(rng, nc, nr) for nr, nc in shapes]
    with L.Batch(lats) as b:
        default = b.steps_per_launch()
        segments, blocks = b.launch()
        b.set_launch(segments, blocks)
        assert b.steps_per_launch() == 1
        out = []
        for k, n in ((1, 1), (3, 1), (4, 4), (100, 4), (0, default)):
            b.set_steps_per_launch(k)
            assert b.steps_per_launch() == n
            for lat, p in zip(lats, states):
                lat.upload_populations(p)
            b.step(45)
            out.append([lat.populations() for lat in lats])
        for x in out[1:]:
            assert all(np.array_equal(p, q) for p, q in zip(out[0], x))
        b.set_launch(segments, blocks)
        b.set_steps_per_launch(0)
        assert b.steps_per_launch() == default
    for lat in lats:
        lat.close()


def test_without_geometry_it_is_an_error():
    import ctypes as C
    with L.Lattice(L.geometry_channel(40, 96), storage=L.F16_SHIFTED) as lat:
        assert lat.steps_per_launch() > 1
    assert L.lib().lbm_get_steps_per_launch(None, C.byref(C.c_int32())) == L.ERR_INVALID


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
def test_mostly_dry_lattices_take_single_steps(storage):
    """The rule's line, seen from outside, and the same bits either side of it."""
    nr = nc = 600
    p0 = state(np.random.default_rng(2), nc, nr)
    for wet, single in ((0.2, True), (0.8, False)):
        cls = np.full((nc, nr), L.OBSTACLE, np.uint8)
        cls[1:int(wet * nc), 1:nr - 1] = L.FLUID
        lat = L.Lattice(cls, storage=storage, tau=0.8)
        assert (lat.steps_per_launch() == 1) == single
        out = []
        for k in (0, 1, 4):
            lat.set_steps_per_launch(k)
            lat.upload_populations(p0)
            lat.step(45)
            out.append(lat.populations())
        assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
        lat.close()


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
def test_ensembles_of_any_shape_keep_their_bits(storage):
    """Several steps per launch asked for, whatever the rule says: samples of
    every small size, mostly dry ones, wet first and last rows."""
    rng = np.random.default_rng(23)
    classes = [random_class(rng, nr, nc, 0.15) for nr, nc in [(3, 3), (5, 9), (57, 10), (56, 11), (64, 12), (113, 40),
                                                              (200, 64), (129, 300)]]
    for nr, nc in ((300, 200), (128, 400)):
        dry = np.full((nc, nr), L.OBSTACLE, np.uint8)
        dry[1:20, 1:nr - 1] = L.FLUID
        classes.append(dry)
    lids = np.zeros((250, 64), np.uint8)
    lids[0] = lids[-1] = L.BOUNDARY
    lids[1:-1, 0], lids[1:-1, -1] = L.INLET, L.OUTLET
    classes += [lids] * 3
    states = [state(rng, *c.shape) for c in classes]
    out = []
    for k in (1, 4, 0):
        lats = [make(c, np.random.default_rng(s), storage, L.BGK, POLICIES[:2]) for s, c in enumerate(classes)]
        for lat, p in zip(lats, states):
            lat.upload_populations(p)
        with L.Batch(lats) as b:
            b.set_steps_per_launch(k)
            assert k == 0 or b.steps_per_launch() == k
            b.step(47)
        out.append([lat.populations() for lat in lats])
        for lat in lats:
            lat.close()
    for s in range(len(classes)):
        assert np.array_equal(out[0][s], out[1][s]) and np.array_equal(out[0][s], out[2][s]), classes[s].shape


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
def test_mostly_dry_ensembles_take_single_steps(storage):
    nr = nc = 512
    for wet, steps in ((0.1, 1), (1.0, 4)):
        cls = np.full((nc, nr), L.OBSTACLE, np.uint8)
        cls[1:int(wet * (nc - 2)), 1:nr - 1] = L.FLUID
        lats = [L.Lattice(cls, storage=storage, tau=0.8) for _ in range(6)]
        with L.Batch(lats) as b:
            assert b.steps_per_launch() == steps
        for lat in lats:
            lat.close()


@pytest.mark.parametrize("storage,nr,nc,psbb", [
    (L.F64, 100, 120, False), (L.F64, 300, 310, False), (L.F64, 9000, 4, False), (L.F32_SHIFTED, 200, 210, False),
    (L.F32_SHIFTED, 400, 410, False), (L.F16_SHIFTED, 300, 310, False), (L.F16_SHIFTED, 1230, 1240, False),
    (L.F64, 100, 120, True), (L.F64, 300, 310, True), (L.F64, 500, 510, True)])
def test_calls_of_few_steps(storage, nr, nc, psbb):
    """Runs that mix tile launches and single steps, fields and new values
    among them, against single steps throughout."""
    rng = np.random.default_rng(nr)
    cls = random_class(rng, nr, nc, 0.1)
    p0 = state(rng, nc, nr)
    lats = [make(cls, np.random.default_rng(1), storage, L.TRT, POLICIES[:2]) for _ in range(2)]
    k = len(lats[0].open_nodes(0))
    b = rng.random(int(lats[0].node_counts()[6]))
    for lat, flags in zip(lats, (0, L.STEP_NO_GRAPH)):
        if psbb:
            lat.set_partial_bounce_back(0.9, b)
        lat.upload_populations(p0)
        for n in (1, 1, 2, 1, 10, 1, 3, 2, 11, 73, 1):
            lat.step(n, flags | (L.STEP_MACRO if n % 2 else 0))
        for n in (1, 2, 1, 10):
            lat.set_open_values(0, ux=np.full(k, 0.001 * n))
            lat.step(n, flags)
            lat.step(1, flags | L.STEP_MACRO | L.STEP_CHECK)
    a, c = lats
    assert np.array_equal(a.populations(), c.populations())
    for x, y in zip(a.macro(), c.macro()):
        assert np.array_equal(x, y)
    for lat in lats:
        lat.close()


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
@pytest.mark.parametrize("options", [0, L.OPT_PLANAR_LAYOUT])
@pytest.mark.parametrize("nr,nc", [(57, 5301), (64, 4700), (33400, 9), (30100, 10), (27300, 11), (25100, 12), (23100, 13)])
def test_asked_for_where_the_rule_says_no(nr, nc, options, storage):
    """Several steps per launch on lattices that take single ones by
    themselves: narrow ones with many solid nodes, windows all at the
    perimeter."""
    rng = np.random.default_rng(nr)
    cls = random_class(rng, nr, nc, 0.4)
    p0 = state(rng, nc, nr)
    out = []
    for k in (1, 2, 3, 4):
        lat = L.Lattice(cls, tau=0.8, inlet_policy=L.ZOUHE_PRESSURE, outlet_policy=L.OPEN_NOOP, storage=storage,
                        options=options)
        lat.set_steps_per_launch(k)
        assert lat.steps_per_launch() == k
        lat.upload_populations(p0)
        lat.step(44, L.STEP_CHECK)
        out.append(lat.populations())
        lat.close()
    assert all(np.array_equal(out[0], x) for x in out[1:])
