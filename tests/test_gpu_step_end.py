"""The launch that ends a substage and starts the next (face sums, deficit,
stale values, bulk velocity) against the operators, each its own launches: rows
around its 16-column pieces, as many rows as it takes and more, stale values
that read the outlet face (ny + 1 or nz + 1 near nx + 2)."""
import numpy as np
import pytest

import pllcart3d_amd as P

pytestmark = pytest.mark.gpu

SEQ = ["CONCENTRATION", "VISCOSITY", "XMOM", "YMOM", "ZMOM", "VELO_BOUNDARY", "DIVERGENCE", "PHISOLVER",
       "PHI_GHOSTS", "VELO_CORRECTION", "VELOGHOST", "PRESSURE_GRADIENT", "UPDATE_OLD"]


@pytest.mark.parametrize("precision", ["plain", "mixed"])
@pytest.mark.parametrize("shape", [(12, 13, 16), (13, 12, 15), (14, 15, 17), (17, 5, 18), (9, 127, 33), (9, 128, 31),
                                   (9, 129, 17), (9, 16, 129)])
def test_step_end_equals_operators(precision, shape):
    """Two steps, every bit: the same sums in the same order."""
    prm = P.make_params(*shape, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    c0 = P.ic_fill(prm, P.IC_NOISE, 3, 0.05)
    a = P.Sim(prm, precision)
    b = P.Sim(prm, precision)
    a.init(c0)
    b.init(c0)
    t, dt = a.run(2)
    for _ in range(2):
        dt = min(b.op("FIND_CFL"), b.timestep)
        for rk in range(3):
            vb = b.op("BULK_VELO", rk=rk)
            for op in SEQ:
                b.op(op, dt, rk, vb)
    for f in ("C_OLD", "U_OLD", "V_OLD", "W_OLD", "PHI", "U_PG", "V_PG", "W_PG"):
        x, y = a.download(f), b.download(f)
        assert np.array_equal(x, y), (precision, shape, f, np.abs(x - y).max())
