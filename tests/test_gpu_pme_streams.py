"""PME solves on a stream of their own and on the engine's stream: the same results, whatever the default is.

Both choices are set here (pgm_set_pme_overlap), and which one an engine then takes is asserted (pgm_pme_path), so a
missing dependency between the streams shows at every size: it would read half-written fields, errors of order one.  An
evaluation is the same bit for bit either way; the adjoint's tangent grids add floating-point numbers in any order, which
moves FP64 gradients by ulps and FP32 ones by their rounding (bounds 1e-12 and 1e-6 of the largest, as in
test_gpu_engine).
"""

import numpy as np
import pytest
from test_gpu_batch import _batch
from test_gpu_launch import Device, _same

from pgmhip import engine as E
from pgmhip import systems as S

pytestmark = pytest.mark.gpu

GRAD_TOL = {"double": 1e-12, "mixed": 1e-6}


@pytest.fixture(scope="module")
def torch():
    return pytest.importorskip("torch")


def _set(eng, beside):
    eng.set_pme_overlap(beside)
    return eng


def _is(eng, beside, planes=None):
    path = eng.pme_path()
    assert ("beside" in path) == beside
    if planes is not None:
        assert ("planes" in path) == planes


def _grads_close(a, b, precision):
    for k in a:
        assert np.abs(a[k] - b[k]).max() <= GRAD_TOL[precision] * np.abs(b[k]).max(), k


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("planes,grid", [(True, (32, 32, 32)), (False, (8, 45, 48))])
def test_evaluation_and_backward(precision, planes, grid):
    sy = S.water_box(1300, 3.4, 11, 3, 0.02, "w1300", S.base_settings(grid=grid, tol=1e-8, predictor=0, peek=0.0))
    g = np.random.default_rng(2).normal(0.0, 1e-3, (sy.n, 3))
    out = []
    for beside in (True, False, True):
        eng = _set(E.Engine.for_system(sy, precision=precision), beside)
        t, f, strain = eng.compute(sy.pos, sy.box, strain=True)
        _is(eng, beside, planes)
        out.append((t, f, strain, eng.induced_dipoles(), eng.iterations(), eng.backward(sy.pos, sy.box, g, 0.5)))
    t0, f0, s0, m0, i0, g0 = out[0]
    for t, f, strain, m, its, gr in out[1:]:
        assert t == t0 and its == i0
        for a, b in ((f, f0), (strain, s0), (m, m0)):
            np.testing.assert_array_equal(a, b)
        _grads_close(gr, g0, precision)


@pytest.mark.parametrize("precision", ["double", "mixed"])
def test_batch_backward(precision):
    systems = [S.config3_snapshot(k) for k in (41, 57, 18)]
    for sy in systems:
        sy.settings.update(tol=1e-8, predictor=0, peek=0.0)
    out = []
    for beside in (True, False):
        eng, _, pos, boxes = _batch(systems, precision)
        _set(eng, beside)
        terms, f = eng.compute_batch(pos, boxes)
        _is(eng, beside)
        g = np.random.default_rng(3).normal(0.0, 1e-3, pos.shape)
        out.append((terms, f, eng.backward_batch(pos, boxes, g, np.array([0.1, -0.2, 0.3]))))
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
    _grads_close(out[0][2], out[1][2], precision)


@pytest.mark.parametrize("beside", [True, False])
@pytest.mark.parametrize("precision", ["double", "mixed"])
def test_launch_stale_list_and_short_solve(torch, precision, beside):
    """Launches along a trajectory, one that finds its list stale and one whose solve falls short, each repeated:
    the results of evaluations with the other choice over the same positions."""
    sy = S.config0()
    dev = Device(torch, sy.n)
    eng = _set(E.Engine.for_system(sy, precision=precision), beside)
    ref = _set(E.Engine.for_system(sy, precision=precision), not beside)

    def step(pos, repeated):
        dev.load(pos)
        tr, fr = dev.compute(ref, sy.box)
        for k in range(2):
            dev.load(pos)
            dev.launch(eng, sy.box)
            t, valid = eng.finish_device()
            assert valid == (k == 1 or not repeated)
            if valid:
                break
        assert eng.iterations() == ref.iterations()
        _same(t, dev.forces(), tr, fr, precision)

    for pos in S.rigid_moves(sy, 6, 0.001, 6):
        step(pos, False)
    jump = pos.copy()
    jump[5] += [0.09, 0.0, 0.0]
    step(jump, True)   # one atom beyond the skin
    bad = np.random.default_rng(8).normal(0.0, 0.01, (4, sy.n, 3))   # |mu| is about 0.003 e nm
    for e in (eng, ref):
        e.set_history(bad)
    step(jump, True)   # more iterations than the solves before
    _is(eng, beside)
    _is(ref, not beside)


def test_default_is_in_line_where_the_field_pass_rides_in_the_planes():
    """Until it is set or tuned: in line on the x-planes of one system, also with many atoms, and on small bricks;
    beside for large systems on bricks."""
    for nmol, edge, grid, planes, beside in (
        (6000, 5.64, (72, 72, 72), True, False),
        (6000, 5.64, (24, 72, 72), False, False),
        (15200, 7.69, (24, 72, 72), False, True),
    ):
        sy = S.water_box(nmol, edge, 25, 3, 0.02, "w", S.base_settings(grid=grid, tol=1e-4))
        eng = E.Engine.for_system(sy, precision="mixed")
        eng.compute(sy.pos, sy.box, forces=False)
        _is(eng, beside, planes)
