"""The marching launches of lattices of 2^22 nodes and more (5 steps in FP64, 4
in FP32 with two columns per turn of the loop) at the edges of their windows and
columns, against one launch per step: the same bits at every remainder of a
launch."""
import numpy as np
import pytest

import lbm_amd as L
from test_gpu_march import POLICIES, make, random_class, state

pytestmark = pytest.mark.gpu

# stored rows of a window: 54 (5 steps), 56 (4); columns that the first and last
# ones influence: 2 K + 3 = 13, 11; one stripe, two, three, four
SIZES = [(53, 79200), (54, 77700), (55, 76300), (57, 73600), (108, 38900), (109, 38500), (113, 37200), (163, 25800),
         (217, 19400), (381400, 11), (350000, 12), (323000, 13), (300000, 14), (210000, 20)]


@pytest.mark.parametrize("storage", [L.F64, L.F32_SHIFTED])
@pytest.mark.parametrize("nr,nc", SIZES)
def test_same_bits_as_single_steps(nr, nc, storage):
    assert nr * nc >= 1 << 22
    rng = np.random.default_rng(nr + nc)
    cls = random_class(rng, nr, nc, 0.1)
    p0 = state(rng, nc, nr)
    policies = (POLICIES[nr % 3], POLICIES[nc % 3])
    collision = (L.BGK, L.TRT)[nr % 2]
    lats = [make(cls, np.random.default_rng(7), storage, collision, policies) for _ in range(2)]
    lats[0].set_steps_per_launch(5)
    assert lats[0].steps_per_launch() == (5 if storage == L.F64 else 4)
    for lat in lats:
        lat.upload_populations(p0)
    del p0
    # remainders 0 .. 4 of whole launches after the first step
    for n in (6, 5, 6, 7, 8, 9):
        for lat, flags in zip(lats, (0, L.STEP_NO_GRAPH)):
            lat.step(n, flags | L.STEP_CHECK)
        a, b = (lat.populations() for lat in lats)
        assert np.array_equal(a, b), n
    for lat in lats:
        lat.close()
