"""The two forms of a PME solve against the FP64 oracle at the sizes where each can go wrong.

The x-plane passes (few atoms per plane, or many planes) spread, transform and gather one x-plane per workgroup;
the brick passes (many atoms per plane) spread and gather bricks of 8 to 14 points through LDS.  Which one runs
follows from atoms x order / planes; the cases sit on both sides of that line, with grids as small as the order (every
row and plane wraps), odd and unequal dimensions, every order, bricks larger than a dimension's remainder, and
a grid of four million points, where the transforms take their widest radices (90 = 10 x 9, 160 = 8 x 5 x 4,
280 = 8 x 7 x 5).  Bounds as in test_gpu_edge: FP64 round-off (energy 1e-11, forces 1e-9 relative), mixed 1e-6 and 5e-5.
"""

import dataclasses

import pytest
from test_gpu_edge import _against_oracle, _tight

from pgmhip import systems as S

pytestmark = pytest.mark.gpu

PLANES = [(4, (4, 25, 27)), (5, (15, 5, 21)), (6, (6, 6, 49)), (6, (32, 35, 8)), (7, (32, 7, 7)), (8, (20, 24, 9))]
BRICKS = [(4, (5, 30, 32)), (5, (6, 14, 45)), (6, (8, 10, 42)), (7, (9, 27, 16)), (8, (8, 35, 28)), (6, (6, 6, 6))]


def _both(sy):
    _against_oracle(sy)
    m = _tight(dataclasses.replace(sy))
    m.settings.update(tol=1e-6)
    _against_oracle(m, "mixed", 1e-6, 5e-5)


@pytest.mark.parametrize("order,grid", PLANES)
def test_x_plane_passes(order, grid):
    _both(_tight(S.water_box(343, 2.2, 7, 3, 0.03, "w343", S.base_settings(grid=grid, order=order))))


@pytest.mark.parametrize("order,grid", BRICKS)
def test_brick_passes(order, grid):
    _both(_tight(S.water_box(1000, 3.1, 10, 4, 0.03, "w1000", S.base_settings(grid=grid, order=order))))


def test_wide_radices():
    _both(_tight(S.water_box(216, 2.0, 6, 5, 0.03, "w216", S.base_settings(grid=(90, 160, 280)))))
