"""Uploads, downloads, field copies and the CFL reduction over the fields'
pitched rows: rows that end one value before, at and after a 128-byte line in
either precision, and rows at the limits of the launches' row split."""
import numpy as np
import pytest

import pllcart3d_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [4, 13, 14, 15, 16, 29, 30, 31, 32, 61, 62, 63, 127, 128, 129, 257])
def test_rows_round_trip(oracle_mod, nz):
    """Every point of every state field comes back as uploaded (mixed: rounded
    to FP32 once), the old fields take the new ones, and the CFL maximum has
    the oracle's value (FP64: 1e-14 relative; FP32: 3 roundings, 1e-6)."""
    prm = P.make_params(7, 6, nz, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    rng = np.random.default_rng(nz)
    orc = oracle_mod.Oracle(prm)
    orc.init(None)
    shape = orc.field("C_OLD").shape
    data = {f: rng.standard_normal(shape) for f in P.FIELDS}
    for f in P.FIELDS:
        orc.field(f)[...] = data[f]
    want = orc.op("FIND_CFL")
    for precision, tol in (("plain", 1e-14), ("mixed", 1e-6)):
        sim = P.Sim(prm, precision)
        sim.init(None)
        for f in P.FIELDS:
            sim.upload(f, data[f])
        seen = {f: data[f] if precision == "plain" else data[f].astype(np.float32).astype(float) for f in P.FIELDS}
        for f in P.FIELDS:
            assert np.array_equal(sim.download(f), seen[f]), (precision, f)
        assert abs(sim.op("FIND_CFL") - want) <= tol * want
        sim.op("UPDATE_OLD")
        for q in "CUVW":
            assert np.array_equal(sim.download(q + "_OLD"), seen[q + "_NEW"]), (precision, q)
