"""The joint launch of the explicit parts over several steps, eager and
replayed from a graph (whose launches keep the planes per thread that they were
captured with), against one launch per field."""
import numpy as np
import pytest

import pllcart3d_amd as P

pytestmark = pytest.mark.gpu

SEQ = ["CONCENTRATION", "VISCOSITY", "XMOM", "YMOM", "ZMOM", "VELO_BOUNDARY", "DIVERGENCE", "PHISOLVER",
       "PHI_GHOSTS", "VELO_CORRECTION", "VELOGHOST", "PRESSURE_GRADIENT", "UPDATE_OLD"]


@pytest.mark.parametrize("graph", ["1", "0"])
@pytest.mark.parametrize("precision", ["plain", "mixed"])
def test_steps_equal_single_launches(precision, graph, monkeypatch):
    """96x96x96, 16x16-mode front: after 3 and 7 fused steps every field has
    the bits of the operators called one by one."""
    prm = P.make_params(96, 96, 96, Vratio=3.0, Pe=2000.0, Inf_thick=0.05)
    c0 = P.ic_fill(prm, P.IC_MULTIMODE, 2, 0.01)
    monkeypatch.setenv("PLLC_GRAPH", graph)
    a = P.Sim(prm, precision)
    b = P.Sim(prm, precision)
    a.init(c0)
    b.init(c0)
    for steps in (3, 4):
        a.run(steps)
        for _ in range(steps):
            dt = min(b.op("FIND_CFL"), b.timestep)
            for rk in range(3):
                vb = b.op("BULK_VELO", rk=rk)
                for op in SEQ:
                    b.op(op, dt, rk, vb)
        for f in ("C_OLD", "C_N", "U_OLD", "U_N", "V_OLD", "V_N", "W_OLD", "W_N", "PHI", "U_PG", "W_PG", "MUO_CELL"):
            x, y = a.download(f), b.download(f)
            assert np.all(np.isfinite(x)) and np.array_equal(x, y), (precision, graph, steps, f, np.abs(x - y).max())
