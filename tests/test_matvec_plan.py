"""Host-side choice of the vectors per wave of the float MatVecs (CPU only)."""
import ctypes
import os

import pytest

from qauntrunner_amd import _lib

F32, F16 = 0, 1


@pytest.mark.parametrize("fmt,rows,nq,vectors", [
    (F16, 4096, 8, 4),   # 23.1 us; one 30.6, two 28.2, three (a second round of workgroups) 33.9
    (F16, 5632, 5, 1),   # 15.7; 16.5, 18.9 and 18.7
    (F16, 2048, 16, 4),  # one round
    (F16, 4096, 2, 1),   # 12.2; 13.0
    (F32, 4096, 11, 4),
    (F32, 4096, 3, 2),   # 15.7; one 22.6 (bound by reads of the weights), three 17.9
    (F32, 8192, 12, 4),  # 49; 153, 83 and 62
    (F32, 1021, 29, 3),
    (F16, 1021, 15, 2),
    (F16, 64, 3, 1),
    (F16, 64, 1, 1),
])
def test_fp_vectors_of_measured_shapes(fmt, rows, nq, vectors):
    """No more workgroups than the LDS of that many vectors lets run at once, where a choice has that."""
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    f = getattr(ctypes.CDLL(_lib.LIB_PATH), "_ZN2qr17matvec_fp_vectorsEiii")
    assert f(fmt, (rows + 7) // 8, nq) == vectors
