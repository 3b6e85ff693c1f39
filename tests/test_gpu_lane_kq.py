"""kR->kq with one lane per (mode, i) (lane_kq_kernel, 9 to 16 orbitals, 9 to 16 modes) against the direct kernels."""
import pytest

import test_gpu_staged as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw,atoms,box,kgrid,qgrid,window", [
    (9, 3, 5, (4, 5, 6), (4, 5, 6), 3.0),       # 9 modes; more entries in four lines than one part holds
    (10, 4, 5, (2, 3, 64), (2, 3, 64), 1.0),    # lines of 64 q, fewer than four lines
    (12, 4, 7, (6, 4, 5), (3, 4, 5), 0.8),      # q grid a divisor, last group of one line
    (13, 5, 5, (3, 7, 9), (3, 7, 9), 0.5),      # odd mode count, three of four waves' columns filled
    (15, 3, 7, (4, 4, 4), (4, 4, 4), 4.0),      # every band in the window
    (16, 5, 7, (4, 4, 2), (4, 4, 2), 3.0),
    (9, 3, 5, (1, 28, 28), (1, 28, 28), 4.0)])  # tables past what a workgroup holds: the other kernel
def test_lane_kq_against_direct(backend, nw, atoms, box, kgrid, qgrid, window):
    S.test_staged_against_direct(backend, nw, atoms, box, None, kgrid, qgrid, window)
