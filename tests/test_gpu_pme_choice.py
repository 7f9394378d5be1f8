"""Both forms of a PME solve at every order and precision, with the form that runs asserted (pgm_pme_path).

Brick passes with more atom rows per plane (atoms x order / planes) than the x-plane passes take in either precision, with
a margin of 20%, on grids whose first dimension is at most 1.5 bricks; bricks of more than 8 points on a grid whose planes
do not fit the LDS; x-planes of more than 64 KiB of LDS, of a grid with 512 planes (256 threads per plane), of a batch with
more than 512, and of a batch of four million points (wide radices); a batch whose 512 planes have too many atoms for
them; stored and on-the-fly field passes mixed between an
evaluation and its backward.  Against the FP64 oracle with the bounds of test_gpu_edge.
"""

import dataclasses

import numpy as np
import pytest
from test_gpu_batch import _batch
from test_gpu_edge import _against_oracle, _tight, rel_rms

import oracle as O
from pgmhip import engine as E
from pgmhip import systems as S

pytestmark = pytest.mark.gpu

BOUNDS = {"double": (1e-11, 1e-9), "mixed": (1e-6, 5e-5)}


def _check(sy, precision, want):
    sy = _tight(dataclasses.replace(sy, settings=dict(sy.settings)))
    if precision == "mixed":
        sy.settings.update(tol=1e-6)
    eng, _ = _against_oracle(sy, precision, *BOUNDS[precision])
    assert eng.pme_path() - {"beside"} == want


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("order,grid", [(4, (6, 40, 42)), (5, (8, 45, 36)), (6, (9, 30, 49)), (7, (10, 48, 35)), (8, (12, 40, 36))])
def test_bricks_at_every_order(order, grid, precision):
    sy = S.water_box(1728, 3.73, 12, 4, 0.03, "w1728", S.base_settings(grid=grid, order=order))
    assert sy.n * order / grid[0] > 1.2 * 2600
    _check(sy, precision, set())


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("order", [4, 5, 6, 7, 8])
def test_large_bricks(order, precision):
    sy = S.water_box(216, 2.0, 6, 5, 0.03, "w216", S.base_settings(grid=(108, 125, 120), order=order))
    _check(sy, precision, set())


@pytest.mark.parametrize(
    "precision,order,grid",
    [("double", 6, (32, 75, 80)), ("mixed", 6, (20, 108, 96)), ("double", 8, (20, 80, 75)), ("mixed", 8, (16, 105, 98)),
     ("double", 6, (512, 9, 8)), ("mixed", 6, (512, 9, 8)), ("double", 4, (625, 5, 6)), ("mixed", 8, (576, 8, 10))],
)  # fmt: skip
def test_large_and_many_planes(precision, order, grid):
    sy = S.water_box(343, 2.2, 7, 3, 0.03, "w343", S.base_settings(grid=grid, order=order))
    _check(sy, precision, {"planes"})


def _batch_against_oracle(systems, precision, want):
    for sy in systems:
        _tight(sy)
        if precision == "mixed":
            sy.settings.update(tol=1e-6)
    eng, off, pos, boxes = _batch(systems, precision)
    terms, f = eng.compute_batch(pos, boxes)
    assert eng.pme_path() - {"beside"} == want
    e_tol, f_tol = BOUNDS[precision]
    for k, sy in enumerate(systems):
        eo, fo = O.Oracle(sy).compute(sy.pos, sy.box)
        assert abs(E.total_energy(terms[k]) / eo - 1) < e_tol, k
        assert rel_rms(f[off[k] : off[k + 1]], fo) < f_tol, k


@pytest.mark.parametrize("precision", ["double", "mixed"])
def test_batch_of_many_planes(precision):
    grids = [(32, 24, 27), (40, 30, 24), (36, 36, 36), (35, 21, 28)]
    systems = [
        S.water_box(m, 2.2, 7, m, 0.02, f"w{m}", S.base_settings(grid=grids[m % 4])) for m in range(85, 101)
    ]
    assert sum(sy.settings["grid"][0] for sy in systems) >= 512
    _batch_against_oracle(systems, precision, {"planes"})


@pytest.mark.parametrize("precision", ["double", "mixed"])
def test_batch_of_four_million_points(precision):
    systems = [
        S.water_box(m, 2.2, 7, m, 0.02, f"w{m}", S.base_settings(grid=g))
        for m, g in ((343, (168, 75, 80)), (300, (168, 80, 75)), (201, (168, 75, 80)), (256, (175, 72, 84)))
    ]
    assert sum(np.prod(sy.settings["grid"]) for sy in systems) >= 4000000
    _batch_against_oracle(systems, precision, {"planes", "wide"})


def test_batch_of_full_planes():
    """512 planes of 960 atom rows: each system alone takes the x-planes, the batch of the two the bricks."""
    st = S.base_settings(grid=(256, 20, 20), tol=1e-6, predictor=0, peek=0.0)
    systems = [S.water_box(13660, 7.43, 24, k, 0.02, f"w{k}", dict(st)) for k in (1, 2)]
    eng, off, pos, boxes = _batch(systems, "mixed")
    terms, f = eng.compute_batch(pos, boxes)
    assert "planes" not in eng.pme_path()
    for k, sy in enumerate(systems):
        single = E.Engine.for_system(sy, precision="mixed")
        t, fk, _ = single.compute(sy.pos, sy.box)
        assert "planes" in single.pme_path()
        assert abs(E.total_energy(terms[k]) / E.total_energy(t) - 1) < 1e-6, k
        assert rel_rms(f[off[k] : off[k + 1]], fk) < 5e-5, k


@pytest.mark.parametrize("first", [False, True])
def test_field_pass_changed_before_the_backward(first):
    """The on-the-fly field pass stores no pair kernels: a backward that reads them, after the choice has changed,
    gives the gradients of an engine that had it from the start."""
    sy = S.config0()
    sy.settings.update(tol=1e-8, predictor=0, peek=0.0)
    g = np.random.default_rng(2).normal(0.0, 1e-3, (sy.n, 3))
    out = []
    for begin in (first, not first):
        eng = E.Engine.for_system(sy, precision="mixed")
        eng.set_field_otf(begin)
        eng.compute(sy.pos, sy.box)
        eng.set_field_otf(not first)
        out.append(eng.backward(sy.pos, sy.box, g, 0.5))
    for k in out[0]:
        assert np.abs(out[0][k] - out[1][k]).max() <= 1e-6 * np.abs(out[1][k]).max(), k
