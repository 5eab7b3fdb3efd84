"""The partitioned line solves at the edges of their chunks: lines of one row
more or less than a multiple of 16 in every direction, one chunk only, lines
whose chunks share a wave with other lines (z: up to 64 lanes per line), the
longest partitioned lines (1024 rows) and the first ones past them."""
import numpy as np
import pytest

import pllcart3d_amd as P

pytestmark = pytest.mark.gpu

SHAPES = [(16, 17, 31), (17, 32, 16), (33, 15, 48), (48, 49, 5), (5, 4, 65), (12, 130, 6), (12, 6, 257),
          (8, 5, 300), (8, 5, 530), (8, 530, 5), (1024, 5, 6), (1030, 6, 5)]


def _rel(parts, sim, orc):
    a = np.concatenate([sim.download(f).ravel() for f in parts])
    b = np.concatenate([orc.field(f).ravel() for f in parts])
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("shape", SHAPES)
def test_chunk_edges_track_oracle(oracle_mod, shape):
    """Two steps against the FP64 oracle: c and the velocity to 1e-11, phi to
    1e-11 or, on long lines, the condition of the x-lines' mean mode
    (16 n^2/pi^2) times the rounding unit."""
    prm = P.make_params(*shape, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    c0 = P.ic_fill(prm, P.IC_NOISE, 3, 0.05)
    orc = oracle_mod.Oracle(prm)
    orc.init(c0)
    sim = P.Sim(prm, "plain")
    sim.init(c0)
    orc.run(2)
    sim.run(2)
    c, v, phi = (_rel(f, sim, orc) for f in (["C_OLD"], ["U_OLD", "V_OLD", "W_OLD"], ["PHI"]))
    print("[chunk edges] %s c %.2e velocity %.2e phi %.2e" % ("x".join(map(str, shape)), c, v, phi), flush=True)
    assert c <= 1e-11 and v <= 1e-11
    assert phi <= max(1e-11, 16 * shape[0] ** 2 / np.pi ** 2 * np.finfo(float).eps)


@pytest.mark.parametrize("shape", SHAPES)
def test_mixed_chunk_edges_per_operator(oracle_mod, shape):
    """The implicit updates in FP32 from the oracle's state after two steps:
    the new values to 1e-6 plus the update's relative size times 8 rounding
    units and the lines' condition 1 + 4 k, k = dt mu / (2 Re h^2)."""
    prm = P.make_params(*shape, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    orc = oracle_mod.Oracle(prm)
    orc.init(P.ic_fill(prm, P.IC_NOISE, 3, 0.05))
    orc.run(2)
    sim = P.Sim(prm, "mixed")
    sim.init(None)
    for f in P.FIELDS:
        sim.upload(f, orc.field(f))
    dt = min(orc.op("FIND_CFL"), orc.timestep)
    vb = orc.op("BULK_VELO", rk=0)
    for op in ("CONCENTRATION", "VISCOSITY", "XMOM", "YMOM", "ZMOM"):
        orc.op(op, dt, 0, vb)
        sim.op(op, dt, 0, vb)
    h = min(4.0 / shape[0], 1.0 / shape[1], 1.0 / shape[2])
    cond = 1 + 4 * 0.5 * dt * np.exp(3.0) / h ** 2
    for new, old in ((["C_NEW"], ["C_OLD"]), (["U_NEW", "V_NEW", "W_NEW"], ["U_OLD", "V_OLD", "W_OLD"])):
        a, b, b0 = (np.concatenate([q(f).ravel() for f in fs])
                    for q, fs in ((sim.download, new), (orc.field, new), (orc.field, old)))
        n = np.linalg.norm(b)
        err, tol = np.linalg.norm(a - b) / n, 1e-6 + 8 * np.finfo(np.float32).eps * cond * np.linalg.norm(b - b0) / n
        print("[chunk edges mixed] %s %s %.2e (tolerance %.2e)" % ("x".join(map(str, shape)), new[0], err, tol),
              flush=True)
        assert err <= tol
