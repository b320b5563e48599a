"""bench.py's algorithmic bytes of the update's kernel are those that the timed
launch moves: image in and out, gradient and (where a plan keeps one, n0 <= 1024)
reference iterate in, grid rows out.
"""
from types import SimpleNamespace

import pytest


@pytest.mark.parametrize("N0,N1,n0,n1", [(512, 512, 1024, 1024), (464, 464, 1024, 1024), (1024, 512, 2048, 1024),
                                         (1007, 1007, 2048, 2048)])
def test_row_fwd_bytes(N0, N1, n0, n1):
    import bench
    half = N0 & (N0 - 1) == 0
    got = bench.algorithmic_bytes(SimpleNamespace(M=41 * N0, n0=n0, n1=n1, N0=N0, N1=N1))["row_fwd"]
    rows = 8 * N0 * (n1 // 2 + 8 if half else n1)
    assert got == rows + (4 + 4 + 4 + (4 if n0 <= 1024 else 0)) * N0 * N1
