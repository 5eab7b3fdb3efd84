"""Planes of any size up to 128 x 128: both dense contractions in one launch
against the two launches (PLLC_DCT=gemm)."""
import numpy as np
import pytest

import pllcart3d_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["plain", "mixed"])
@pytest.mark.parametrize("plane", [(5, 4), (15, 17), (17, 16), (33, 120), (45, 39), (48, 80), (96, 96), (112, 128),
                                   (128, 7), (127, 113), (65, 128)])
def test_one_launch_equals_two(precision, plane, monkeypatch):
    """Two steps with either form: the same sums in the same order, so the
    same bits, at planes of one tile to 8 x 8 tiles, whole and ragged."""
    prm = P.make_params(5, *plane, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    c0 = P.ic_fill(prm, P.IC_NOISE, 3, 0.05)
    a = P.Sim(prm, precision)
    monkeypatch.setenv("PLLC_DCT", "gemm")
    b = P.Sim(prm, precision)
    for s in (a, b):
        s.init(c0)
        s.run(2)
    for f in ("PHI", "C_OLD", "U_OLD", "V_OLD", "W_OLD", "U_PG"):
        x, y = a.download(f), b.download(f)
        assert np.all(np.isfinite(x)) and np.array_equal(x, y), (precision, plane, f, np.abs(x - y).max())
