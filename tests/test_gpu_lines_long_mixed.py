"""Partitioned x-lines of 1025 to 4096 rows in FP32, the Poisson lines among
them, and the first size past them."""
import numpy as np
import pytest

import pllcart3d_amd as P

pytestmark = pytest.mark.gpu

SEQ = ["CONCENTRATION", "VISCOSITY", "XMOM", "YMOM", "ZMOM", "VELO_BOUNDARY", "DIVERGENCE", "PHISOLVER",
       "PHI_GHOSTS", "VELO_CORRECTION", "VELOGHOST", "PRESSURE_GRADIENT"]
READ = {"CONCENTRATION": [("C_NEW",)], "ZMOM": [("U_NEW", "V_NEW", "W_NEW")], "PHISOLVER": [("PHI",)],
        "PRESSURE_GRADIENT": [("U_NEW", "V_NEW", "W_NEW"), ("U_PG", "V_PG", "W_PG")]}


@pytest.mark.parametrize("shape", [(1025, 6, 5), (1040, 33, 20), (2049, 4, 5), (4096, 5, 4), (4096, 16, 16), (4097, 4, 5)])
def test_long_lines_no_worse_than_thomas(oracle_mod, shape, monkeypatch):
    """One substage in FP32 from the oracle's state after two steps: what each
    solve leaves is no further from the FP64 oracle than with one thread per
    line (PLLC_LINE_SOLVER=thomas), or within two roundings of FP32."""
    prm = P.make_params(*shape, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    orc = oracle_mod.Oracle(prm)
    orc.init(P.ic_fill(prm, P.IC_NOISE, 3, 0.05))
    orc.run(2)
    sims = []
    for solver in (None, "thomas"):
        if solver:
            monkeypatch.setenv("PLLC_LINE_SOLVER", solver)
        sims.append(P.Sim(prm, "mixed"))
        sims[-1].init(None)
        for f in P.FIELDS:
            sims[-1].upload(f, orc.field(f))
    dt = min(orc.op("FIND_CFL"), orc.timestep)
    vb = orc.op("BULK_VELO", rk=0)
    for op in SEQ:
        orc.op(op, dt, 0, vb)
        for s in sims:
            s.op(op, dt, 0, vb)
        for fields in READ.get(op, ()):
            b = np.concatenate([orc.field(f).ravel() for f in fields])
            part, thomas = (np.linalg.norm(np.concatenate([s.download(f).ravel() for f in fields]) - b) /
                            np.linalg.norm(b) for s in sims)
            print("[long lines mixed] %s %s %s %.2e (thomas %.2e)" % ("x".join(map(str, shape)), op, fields[0], part,
                                                                     thomas), flush=True)
            assert part <= max(thomas, 2.0 ** -23)


def test_batched_long_lines_equal_standalone_runs():
    """Members whose x-lines have 65 chunks form a batch and keep the bits of
    the same simulations run alone."""
    prm = [P.make_params(1040, 16, 32, Vratio=3.0 - i, Pe=300.0 + 100 * i, Inf_thick=0.1) for i in range(2)]
    c0 = [P.ic_fill(p, P.IC_NOISE, 3 + i, 0.05) for i, p in enumerate(prm)]
    ens = P.Ensemble(prm, "mixed")
    assert ens.batches() == 1
    alone = [P.Sim(p, "mixed") for p in prm]
    for m, s, c in zip(ens.members, alone, c0):
        m.init(c)
        s.init(c)
    ens.run(3)
    for m, s in zip(ens.members, alone):
        s.run(3)
        for f in ("C_OLD", "U_OLD", "V_OLD", "W_OLD", "PHI", "U_PG"):
            assert np.array_equal(m.download(f), s.download(f)), f
    ens.close()
