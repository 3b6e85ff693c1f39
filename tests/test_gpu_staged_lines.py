"""The staged outer-k transforms of 8 orbitals on boxes without opposite offsets, lines past 128 units, against the
direct kernels."""
import pytest

import test_gpu_staged as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cut,kgrid,window", [
    ((-1, -1, -1), (2, 2, 48), 2.5),      # 4^3 box: every k of a line has bands
    ((None, None, -1), (3, 2, 64), 2.0),  # face 5 x 4
    (None, (2, 2, 64), 2.0)])             # the lane form
def test_long_lines_of_8_orbitals(backend, cut, kgrid, window):
    S.test_staged_against_direct(backend, 8, 1, 5, cut, kgrid, (1, 2, kgrid[2]), window)
