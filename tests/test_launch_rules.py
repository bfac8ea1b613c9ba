"""The launch rules (csrc/lbm_plan.cpp), on the CPU: what they deal out covers
every node once, and which launch they choose."""
import os
import shutil
import subprocess

import pytest

from conftest import PKG, ROOT

F64, F32, F16 = range(3)


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = str(tmp_path_factory.mktemp("rules") / "launch_rules")
    r = subprocess.run(["g++", "-std=c++20", "-O1", "-g", os.path.join(ROOT, "tests", "cpp", "launch_rules.cpp"),
                        os.path.join(PKG, "csrc", "lbm_plan.cpp"), "-o", exe], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]

    def ask(*lines):
        r = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-3000:]
        return [[int(x) for x in ln.split()] for ln in r.stdout.splitlines()]

    return ask


def shape(storage, nr, nc, top=False, bottom=False, psbb=False, cus=256, wet=1.0, segments=1.0):
    """wet, segments: shares of the nodes that are wet, of the 64-row segments
    that hold a wet node."""
    return (f"shape {storage} {int(psbb)} {nr} {nc} {int(top)} {int(bottom)} {cus} {int(wet * nr * nc)} "
            f"{int(segments * ((nr + 63) // 64) * nc)}")


# rows at the windows' ends for every K (60, 58, 56 and 54 stored rows), columns
# around the ones that the first and last columns influence
ROWS = (1, 3, 53, 54, 55, 56, 57, 59, 60, 61, 64, 65, 108, 109, 112, 113, 161, 162, 163, 1100)
COLS = (3, 6, 7, 8, 9, 10, 11, 12, 13, 14, 20, 61, 700)


@pytest.mark.parametrize("K", [2, 3, 4, 5])
@pytest.mark.parametrize("storage", [F64, F32])
def test_waves_cover_the_lattice(rules, storage, K):
    asked, lines = [], []
    for nr in ROWS:
        for nc in COLS:
            for top, bottom in ((0, 0), (1, 0), (0, 1), (1, 1)):
                asked.append((nr, nc, top, bottom))
                lines += [shape(storage, nr, nc, top, bottom, cus=256 if nr % 2 else 32), f"cover {K}"]
    for case, (ok,) in zip(asked, rules(*lines)):
        assert ok, case


@pytest.mark.parametrize("cols", [64, 16, 6, 0])
def test_ensemble_waves_cover_the_samples(rules, cols):
    lines = []
    for k, (nr, nc) in enumerate([(3, 3), (5, 9), (57, 10), (56, 11), (64, 12), (113, 40), (300, 200), (129, 700)]):
        lines += [shape(F32, nr, nc, k % 2, k % 3 == 0), "add"]
    waves, ok, longest = rules(*lines, f"table 4 {cols}")[0]
    assert ok and waves > 0 and longest <= (cols or 64)


LIDS = [(3, 106666), (16, 62500), (30, 9999), (50, 8000), (50, 20000), (64, 15625), (120, 9000)]


@pytest.mark.parametrize("storage", [F64, F32])
def test_perimeter_waves_do_not_fill_the_chip_with_halo_columns(rules, storage):
    """A wave of a perimeter window computes 2 K columns beside those it
    stores: short ones only while they leave room on the chip."""
    chip = 256 * 4 * (2 if storage == F64 else 3)
    for nr, nc in LIDS:
        for bottom in (False, True):
            (_, _, _, _, edge_cols, edge_row_waves, _, _), = rules(shape(storage, nr, nc, True, bottom), "plan 4")
            assert edge_cols >= 2 and (edge_cols == 8 or edge_row_waves <= chip), (nr, nc, bottom)
    # the same for an ensemble's table: 300 lattices of two stripes, one on the perimeter
    waves, ok, _ = rules(*[shape(storage, 64, 64, True), "add"] * 300, "table 4 64")[0]
    assert ok and waves - 300 * 3 <= 300 * 8


def test_long_chunks_only_where_they_fill_the_chip(rules):
    """Perimeter waves take slots of the chip, but not for as long as a long
    chunk takes: they are no reason for one."""
    for nr, nc in ((200, 5000), (130, 7692)):
        (_, _, _, cols, _, _, edge_waves, waves), = rules(shape(F64, nr, nc, True), "plan 4")
        assert cols <= 40 or (waves - edge_waves) >= 2048 // 5, (nr, nc)
    for storage in (F64, F32):
        for n, size in ((20, 129), (10, 256), (30, 100)):
            _, ok, longest = rules(*[shape(storage, size, size, True, True), "add"] * n, "table 4 0")[0]
            assert ok and longest <= 16, (storage, n, size)
        # without perimeter rows, enough waves for long chunks
        _, ok, longest = rules(*[shape(storage, 1024, 1024), "add"] * 12, "table 4 0")[0]
        assert ok and longest == 64


@pytest.mark.parametrize("storage", [F64, F32])
def test_lattices_that_march(rules, storage):
    """Single steps where marching measured slower: mostly dry lattices below
    2^20 nodes, and lattices whose windows are all at the perimeter, of more
    windows than segments or with many solid nodes."""
    yes = [shape(storage, 560, 541), shape(storage, 600, 600, wet=0.7), shape(storage, 600, 600, wet=0.2, segments=0.55),
           shape(storage, 1100, 1100, wet=0.1, segments=0.1), shape(storage, 4096, 4096, wet=0.05, segments=0.05),
           shape(storage, 50, 8000, True), shape(storage, 80, 12500, True, True), shape(storage, 64, 15625, True),
           shape(storage, 33400, 9), shape(storage, 700, 700, True, True)]
    no = [shape(storage, 600, 600, wet=0.05, segments=0.06), shape(storage, 600, 600, wet=0.1, segments=0.32),
          shape(storage, 2000, 200, wet=0.3, segments=0.3), shape(storage, 64, 15625, True, True),
          shape(storage, 44000, 10, wet=0.6), shape(storage, 400000, 12, wet=0.7)]
    got = rules(*sum([[s, "pays"] for s in yes + no], []))
    assert [x for x, in got] == [1] * len(yes) + [0] * len(no)


@pytest.mark.parametrize("storage", [F64, F32])
def test_ensembles_that_march(rules, storage):
    """Single steps where the samples are mostly dry, whose one-step table
    holds only segments with wet nodes."""
    for n, size, wet, segments, march in ((32, 700, 0.7, 1.0, 1), (512, 400, 0.6, 1.0, 1), (16, 512, 1.0, 1.0, 1),
                                          (16, 512, 0.05, 0.05, 0), (12, 1024, 0.05, 0.16, 0), (12, 1024, 0.1, 0.27, 0),
                                          (64, 128, 0.05, 0.1, 0), (2, 1024, 0.2, 0.22, 0), (16, 512, 0.2, 0.22, 0)):
        one = shape(storage, size, size, wet=wet, segments=segments)
        assert rules(*[one, "add"] * n, "ensemble 4")[0] == [march], (n, size, wet)
    lids = shape(storage, 256, 256, True)
    assert rules(*[lids, "add"] * 10, "ensemble 4")[0] == [1]


def test_calls_of_few_steps_in_tiles(rules):
    """A tile launch of one or two steps only where it is the faster one: the
    smallest lattices, shallow ones, or with new values waiting."""
    want = {(F64, 129, 129): (1, 1, 1), (F64, 200, 200): (1, 2, 1), (F64, 545, 545): (1, 2, 1),
            (F32, 250, 250): (1, 1, 1), (F32, 300, 300): (1, 2, 1), (F32, 545, 545): (1, 2, 1),
            (F16, 310, 310): (1, 1, 1), (F16, 400, 400): (1, 2, 1), (F16, 600, 600): (1, 2, 1),
            (F16, 850, 850): (1, 2, 1), (F16, 1240, 1240): (1, 3, 1),
            (F64, 40, 96): (1, 1, 1), (F64, 96666, 3): (0, 3, 1), (F32, 40000, 5): (1, 3, 1),
            (F64, 20000, 3): (1, 2, 1), (F64, 10000, 3): (1, 2, 1), (F64, 36250, 8): (1, 2, 1)}
    got = rules(*sum([[shape(*k), "tiles"] for k in want], []))
    assert {k: tuple(x) for k, x in zip(want, got)} == want
    got = rules(*sum([[shape(F64, n, n, psbb=True), "tiles"] for n in (60, 129, 300, 400, 545)], []))
    assert [tuple(x) for x in got] == [(1, 2, 1)] * 3 + [(1, 3, 1)] * 2
    # a wet first row makes the one-step kernels slow
    got = rules(*sum([[shape(st, 3, 20000, True), "tiles"] for st in (F64, F32, F16)], []))
    assert [x[1] for x in got] == [1, 1, 1]
