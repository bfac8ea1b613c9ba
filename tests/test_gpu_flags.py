"""What LBM_STEP_CHECK reports from launches of several steps: a NaN that
appears in one of their inner steps, and nothing on a clean run.

Two opposite streams near the largest finite number meet two steps after the
upload: their sum overflows there, and infinities become NaN densities in the
steps after.  The first step of a run is a launch of its own, so what it finds
is ruled out by asking it."""
import numpy as np
import pytest

import lbm_amd as L
from test_gpu_march import POLICIES, make, random_class, state

pytestmark = pytest.mark.gpu

F32_MAX, F64_MAX = float(np.finfo(np.float32).max), float(np.finfo(np.float64).max)


def colliding(p, storage, i, j):
    """p with two nodes either side of (i, j) whose only content streams to it."""
    big = 0.68 * (F64_MAX if storage == L.F64 else F32_MAX)
    q = p.copy()
    q[:, j - 1, i] = q[:, j + 1, i] = 0.0
    q[1, j - 1, i] = q[3, j + 1, i] = big
    return q


def first_report(lat, p, flags, steps):
    """The number of steps after which the check of one call reports a NaN."""
    lat.init_equilibrium()      # earlier reports are forgotten here
    lat.upload_populations(p)
    for n in range(1, steps + 1):
        try:
            lat.step(1, flags | L.STEP_CHECK)
        except L.LbmError as e:
            assert e.code == L.ERR_NAN
            return n
    return None


def reports(lat, p, flags, n):
    lat.init_equilibrium()
    lat.upload_populations(p)
    try:
        lat.step(n, flags | L.STEP_CHECK)
    except L.LbmError as e:
        assert e.code == L.ERR_NAN
        return True
    return False


# tiles, marching waves in both layouts, the large lattices' kernels
CASES = [(150, 160, 0), (560, 541, 0), (560, 541, L.OPT_PLANAR_LAYOUT), (2060, 2040, 0)]


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
@pytest.mark.parametrize("nr,nc,options", CASES)
def test_nan_of_an_inner_step(nr, nc, options, storage):
    rng = np.random.default_rng(nr)
    cls = np.zeros((nc, nr), np.uint8)
    cls[0] = cls[-1] = cls[:, 0] = cls[:, -1] = L.BOUNDARY
    cls[1:-1, 0] = L.INLET                      # a wet first row: perimeter windows
    p = state(rng, nc, nr)
    lat = L.Lattice(cls, tau=1.0, storage=storage, options=options)
    assert lat.steps_per_launch() > 3
    assert not reports(lat, p, 0, 23)
    # an inner window, and one with perimeter nodes
    for i, j in ((nr // 2, nc // 2), (3, nc // 3)):
        q = colliding(p, storage, i, j)
        at = first_report(lat, q, L.STEP_NO_GRAPH, 12)
        assert at is not None and at > 1, at
        for n in range(1, 14):
            assert reports(lat, q, 0, n) == (n >= at), (i, j, n, at)
    lat.close()


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
def test_nan_of_an_inner_step_in_an_ensemble(storage):
    nr, nc = 300, 310
    p = state(np.random.default_rng(5), nc, nr)
    cls = np.zeros((nc, nr), np.uint8)
    cls[0] = cls[-1] = cls[:, 0] = cls[:, -1] = L.BOUNDARY
    q = colliding(p, storage, 140, 150)
    lats = [L.Lattice(cls, tau=1.0, storage=storage) for _ in range(3)]
    at = first_report(lats[0], q, L.STEP_NO_GRAPH, 12)
    assert at is not None and at > 1
    for n in (1, 3, 5, 9, 33):
        for bad in (False, True):
            with L.Batch(lats) as b:
                b.set_steps_per_launch(4)
                assert b.steps_per_launch() == 4
                for k, lat in enumerate(lats):
                    lat.upload_populations(q if bad and k == 1 else p)
                try:
                    b.step(n, L.STEP_CHECK)
                    assert not (bad and n >= at), n
                except L.LbmError as e:
                    assert e.code == L.ERR_NAN and bad and n >= at, n
                    assert "sample 1" in str(e)
    for lat in lats:
        lat.close()


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
@pytest.mark.parametrize("nr,nc", [(57, 5301), (113, 2670), (33400, 9), (30100, 10), (27300, 11), (560, 541)])
def test_clean_runs_report_nothing(nr, nc, storage):
    """Every kind of perimeter and obstacle; windows whose outer lanes hold
    values of no meaning."""
    rng = np.random.default_rng(nr)
    cls = random_class(rng, nr, nc, 0.15)
    lat = make(cls, rng, storage, L.TRT, POLICIES[:2])
    lat.set_steps_per_launch(4)
    lat.upload_populations(state(rng, nc, nr))
    lat.step(47, L.STEP_CHECK)
    lat.close()
