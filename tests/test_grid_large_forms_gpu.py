"""The grid kernels of large grids (from 2^20 cells the velocity and its
boundary in two launches, four rows to a thread) and the small ones at their
smallest side against the oracle: walls, sources, the relations of N and M on
which the right ghost column depends, cylindrical.  Tolerances as in
test_grid_forms_gpu: four steps of FP64 from the same random fields."""
import pytest

import test_grid_forms_gpu as forms

pytestmark = pytest.mark.gpu

SHAPES = ((1024, 1024), (1025, 1024), (1030, 1020), (1020, 1030))


@pytest.mark.parametrize("pml", range(16))
def test_walls_and_sources(brp, pml):
    for k, source in enumerate(forms.SOURCES):
        nx, ny = SHAPES[(k + pml) % 4]
        forms.check(brp, forms.config(brp, nx, ny, pml, source))


# every relation of N and M beside an x1 and a y1 wall
@pytest.mark.parametrize("nx,ny", SHAPES)
@pytest.mark.parametrize("pml", [0b0000, 0b0111, 0b1101])
def test_walls_and_shapes(brp, nx, ny, pml):
    forms.check(brp, forms.config(brp, nx, ny, pml, forms.SOURCES[5]))


@pytest.mark.parametrize("nx,ny", [(1025, 1026), (601, 557)])
@pytest.mark.parametrize("pml", [0b1111, 0b0110])
def test_cylindrical(brp, nx, ny, pml):
    forms.check(brp, forms.config(brp, nx, ny, pml, forms.SOURCES[1], cyl=1))


@pytest.mark.parametrize("pml", range(16))
def test_smallest_sides(brp, pml):
    for nx, ny in ((4, 4), (4, 5), (5, 4), (4, 130), (130, 4)):
        for source in forms.SOURCES:
            forms.check(brp, forms.config(brp, nx, ny, pml, source))
