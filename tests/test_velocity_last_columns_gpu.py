"""The velocity of the last column where it absorbs reads the pressure's ghost
column, whichever lane, wavefront or workgroup holds it: N + 1 of every
remainder by four (the cells of a thread), by 256 (of a wavefront's row), from a
random pressure, ghosts included, against the oracle (tolerances as in
test_grid_forms_gpu)."""
import pytest

import test_grid_forms_gpu as forms

pytestmark = pytest.mark.gpu


# four rows and cells to a thread (from 2^20 cells), one cell
@pytest.mark.parametrize("nx,ny", [(1023, 1030), (1024, 1025), (1025, 1026), (1026, 1024), (1027, 1025),
                                   (1279, 821), (1283, 822), (255, 300), (63, 40), (67, 40), (251, 33)])
@pytest.mark.parametrize("cyl", [0, 1])
def test_last_column(brp, nx, ny, cyl):
    for pml in (0b0010, 0b1111):
        forms.check(brp, forms.config(brp, nx, ny, pml, forms.SOURCES[2], cyl=cyl))
