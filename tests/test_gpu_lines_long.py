"""Partitioned x-lines of more than 1024 rows (65 to 256 chunks, few lines a
block) and the first ones that take one thread per line again."""
import numpy as np
import pytest

import pllcart3d_amd as P

pytestmark = pytest.mark.gpu


def _rel(parts, sim, orc):
    a = np.concatenate([sim.download(f).ravel() for f in parts])
    b = np.concatenate([orc.field(f).ravel() for f in parts])
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("shape", [(1025, 5, 6), (1040, 4, 9), (2049, 4, 5), (4096, 5, 4), (4097, 4, 5)])
def test_long_lines_track_oracle(oracle_mod, shape):
    """One step against the FP64 oracle: c to 1e-11; phi, and the velocity that
    its gradient makes, to the condition of the x-lines' mean mode
    (16 n^2/pi^2) times the rounding unit."""
    prm = P.make_params(*shape, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    c0 = P.ic_fill(prm, P.IC_NOISE, 3, 0.05)
    orc = oracle_mod.Oracle(prm)
    orc.init(c0)
    sim = P.Sim(prm, "plain")
    sim.init(c0)
    orc.run(1)
    sim.run(1)
    c, v, phi = (_rel(f, sim, orc) for f in (["C_OLD"], ["U_OLD", "V_OLD", "W_OLD"], ["PHI"]))
    print("[long lines] %s c %.2e velocity %.2e phi %.2e" % ("x".join(map(str, shape)), c, v, phi), flush=True)
    assert c <= 1e-11
    assert max(v, phi) <= 16 * shape[0] ** 2 / np.pi ** 2 * np.finfo(float).eps
