"""The explicit parts' joint launch against one launch per field: the planes a
thread takes (1 to 8, by the number of points and fields in the launch), a
last group of fewer planes, odd and even rows, rows of more than one tile."""
import numpy as np
import pytest

import pllcart3d_amd as P

pytestmark = pytest.mark.gpu

SEQ = ["CONCENTRATION", "VISCOSITY", "XMOM", "YMOM", "ZMOM", "VELO_BOUNDARY", "DIVERGENCE", "PHISOLVER",
       "PHI_GHOSTS", "VELO_CORRECTION", "VELOGHOST", "PRESSURE_GRADIENT", "UPDATE_OLD"]


@pytest.mark.parametrize("precision", ["plain", "mixed"])
@pytest.mark.parametrize("shape, force", [((9, 5, 4), 0.0), ((41, 33, 37), 0.0), ((75, 70, 65), 0.3),
                                          ((101, 64, 131), 0.0), ((173, 97, 82), 0.0), ((169, 90, 129), 0.3)])
def test_joint_explicit_parts_equal_single_ones(precision, shape, force):
    """One step with the fields' explicit parts in one launch (u, v and w in
    one with a body force) against the operators, each its own launch: the
    same bits in every field (the same arithmetic at every point)."""
    prm = P.make_params(*shape, Vratio=3.0, Pe=300.0, Inf_thick=0.1, Fx=force, Fy=force)
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
    for f in ("C_OLD", "C_N", "U_OLD", "U_N", "V_OLD", "V_N", "W_OLD", "W_N", "PHI", "U_PG", "W_PG", "MUO_CELL"):
        x, y = a.download(f), b.download(f)
        assert np.array_equal(x, y), (precision, shape, f, np.abs(x - y).max())
