"""The default arithmetic against the reference's over many steps of an
unstable front: what differs in the last bits of the plateau ahead of the front
is amplified when the front reaches it."""
import numpy as np
import pytest

import pllcart3d_amd as P
from pllcart3d_amd.configs import CONFIGS, config_params

pytestmark = pytest.mark.gpu


def test_200_steps_stay_at_rounding_of_the_reference_arithmetic(monkeypatch):
    """front_256x128x128 in FP64 with the default solver and stencils against
    PLLC_LINE_SOLVER=thomas (the reference's operations): c and the velocity
    after 50, 100 and 200 steps differ by at most a rounding per substage, all of
    one sign (3 n 2^-53), the velocity by ten of them."""
    c = CONFIGS["front_256x128x128"]
    prm = config_params("front_256x128x128")
    c0 = P.ic_fill(prm, c["ic"], c["seed"], c["amp"])
    a = P.Sim(prm, "plain")
    monkeypatch.setenv("PLLC_LINE_SOLVER", "thomas")
    b = P.Sim(prm, "plain")
    for s in (a, b):
        s.init(c0)
    done = 0
    for n in (50, 100, 200):
        for s in (a, b):
            s.run(n - done)
        done = n
        for name, fields, most in (("c", ("C_OLD",), 1), ("velocity", ("U_OLD", "V_OLD", "W_OLD"), 10)):
            x, y = (np.concatenate([s.download(f).ravel() for f in fields]) for s in (a, b))
            err = np.linalg.norm(x - y) / np.linalg.norm(y)
            print("[long run] step %d %s %.2e" % (n, name, err), flush=True)
            assert err <= most * 3 * n * 2.0 ** -53, (n, name, err)
