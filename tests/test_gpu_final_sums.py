"""The solve's vector kernels and the final stage at the edges of their blocks, against the FP64 oracle.

Both run 256 atoms per block: systems of 255, 258, 768 and 771 atoms (one atom below a block, two above, exactly three
blocks, three above), each alone with its strain and all together as one batch, whose chunks end at the systems' ends.
Bounds as in test_gpu_edge: energy 1e-11, forces and strain 1e-9 relative in FP64.
"""

import numpy as np
import pytest
from test_gpu_batch import _batch
from test_gpu_edge import _tight, rel_rms

import oracle as O
from pgmhip import engine as E
from pgmhip import systems as S

pytestmark = pytest.mark.gpu


def _systems():
    return [
        _tight(S.water_box(m, 2.2, 7, m, 0.02, f"w{m}", S.base_settings(grid=(24, 24, 24)))) for m in (85, 86, 256, 257)
    ]


@pytest.mark.parametrize("case", [0, 1, 2, 3])
def test_single_with_strain(case):
    sy = _systems()[case]
    o = O.Oracle(sy)
    eo, fo = o.compute(sy.pos, sy.box)
    eng = E.Engine.for_system(sy, precision="double")
    for _ in range(2):   # the second with the solve enqueued ahead
        t, f, s = eng.compute(sy.pos, sy.box, strain=True)
        assert abs(E.total_energy(t) / eo - 1) < 1e-11
        assert rel_rms(f, fo) < 1e-9
        assert np.abs(s - o.strain()).max() < 1e-9 * np.abs(o.strain()).max()
        for k, v in o.terms().items():
            assert abs(t[k] - v) < 1e-9 * abs(eo), k


def test_batch_of_ragged_systems():
    systems = _systems()
    eng, off, pos, boxes = _batch(systems)
    terms, f = eng.compute_batch(pos, boxes)
    for k, sy in enumerate(systems):
        eo, fo = O.Oracle(sy).compute(sy.pos, sy.box)
        assert abs(E.total_energy(terms[k]) / eo - 1) < 1e-11, k
        assert rel_rms(f[off[k] : off[k + 1]], fo) < 1e-9, k
