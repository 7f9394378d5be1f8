"""The CG field pass carried by the x-plane spread's launch against the pass in a launch of its own.

A system of few planes with the PME in line runs the field pass's rows in further blocks of the spread's launch; with the
PME on its own stream (pgm_set_pme_overlap 1) the pass is a launch.  The rows are the same code in the same order, so the
results are equal bit for bit, for every lane count and kind of field pass, at atom counts that leave the last block of
1,024 threads ragged; and they match the FP64 oracle (bounds as in test_gpu_edge).
"""

import numpy as np
import pytest
from test_gpu_edge import _tight, rel_rms

import oracle as O
from pgmhip import engine as E
from pgmhip import systems as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [16, 32, 64])
@pytest.mark.parametrize("precision,otf", [("double", False), ("mixed", False), ("mixed", True)])
@pytest.mark.parametrize("nmol", [85, 343])
def test_beside_planes_equals_a_launch_of_its_own(lanes, precision, otf, nmol):
    sy = _tight(S.water_box(nmol, 2.2, 7, 3, 0.02, "w", S.base_settings(grid=(30, 25, 28))))
    if precision == "mixed":
        sy.settings.update(tol=1e-6)
    out = []
    for overlap in (False, True):
        eng = E.Engine.for_system(sy, precision=precision)
        eng.set_lanes(lanes)
        eng.set_field_otf(otf)
        eng.set_pme_overlap(overlap)
        t, f, _ = eng.compute(sy.pos, sy.box)
        out.append((t, f, eng.iterations()))
    assert out[0][2] == out[1][2]
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
    eo, fo = O.Oracle(sy).compute(sy.pos, sy.box)
    e_tol, f_tol = (1e-11, 1e-9) if precision == "double" else (1e-6, 5e-5)
    assert abs(E.total_energy(out[0][0]) / eo - 1) < e_tol
    assert rel_rms(out[0][1], fo) < f_tol
