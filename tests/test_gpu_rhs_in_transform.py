"""The Poisson right-hand side made in the forward transform's load against
divergence and packing in launches of their own, for each transform that has
it: small planes, any planes up to 128 x 128, 128 x 128 and 256 x 256."""
import numpy as np
import pytest

import pllcart3d_amd as P

pytestmark = pytest.mark.gpu

SEQ = ["CONCENTRATION", "VISCOSITY", "XMOM", "YMOM", "ZMOM", "VELO_BOUNDARY", "DIVERGENCE", "PHISOLVER",
       "PHI_GHOSTS", "VELO_CORRECTION", "VELOGHOST", "PRESSURE_GRADIENT", "UPDATE_OLD"]


@pytest.mark.parametrize("precision", ["plain", "mixed"])
@pytest.mark.parametrize("shape", [(5, 16, 16), (70, 32, 32), (9, 48, 64), (600, 64, 48), (5, 96, 40), (7, 21, 100),
                                   (4, 128, 128), (3, 256, 256)])
def test_right_hand_side_in_transform(precision, shape, monkeypatch):
    """One step, every bit: the same expressions at every point.  (One thread
    per line in the sweeps: partitioned, the joint sweeps of three components
    solve x-lines of 3 rows otherwise than a component's own.)"""
    monkeypatch.setenv("PLLC_LINE_SOLVER", "thomas")
    prm = P.make_params(*shape, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    c0 = P.ic_fill(prm, P.IC_NOISE, 3, 0.05)
    a = P.Sim(prm, precision)
    b = P.Sim(prm, precision)
    a.init(c0)
    b.init(c0)
    a.run(1)
    dt = min(b.op("FIND_CFL"), b.timestep)
    for rk in range(3):
        vb = b.op("BULK_VELO", rk=rk)
        for op in SEQ:
            b.op(op, dt, rk, vb)
    for f in ("PHI", "U_OLD", "V_OLD", "W_OLD", "U_PG"):
        x, y = a.download(f), b.download(f)
        assert np.array_equal(x, y), (precision, shape, f, np.abs(x - y).max())
