"""Large fields (from 1.5 million points and 64 points a row on), whose rows are
pitched to whole 128-byte lines: rows one value longer than a line, one shorter
than two and of whole lines, through uploads, downloads and a step."""
import os

import numpy as np
import pytest

import pllcart3d_amd as P

pytestmark = pytest.mark.gpu

SEQ = ["CONCENTRATION", "VISCOSITY", "XMOM", "YMOM", "ZMOM", "VELO_BOUNDARY", "DIVERGENCE", "PHISOLVER",
       "PHI_GHOSTS", "VELO_CORRECTION", "VELOGHOST", "PRESSURE_GRADIENT", "UPDATE_OLD"]


@pytest.mark.parametrize("precision", ["plain", "mixed"])
@pytest.mark.parametrize("shape", [(520, 82, 81), (206, 129, 127), (214, 127, 126)])
def test_rows_round_trip(precision, shape):
    """Every point comes back as uploaded (mixed: rounded to FP32 once), the
    old fields take the new ones and the untouched ones stay."""
    prm = P.make_params(*shape, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    rng = np.random.default_rng(shape[2])
    sim = P.Sim(prm, precision)
    sim.init(None)
    assert np.prod(sim.shape) >= 3.5e6
    data = {f: rng.standard_normal(sim.shape) for f in ("C_NEW", "W_NEW", "C_NM1")}
    for f, a in data.items():
        sim.upload(f, a)
    seen = {f: a if precision == "plain" else a.astype(np.float32).astype(float) for f, a in data.items()}
    for f, a in seen.items():
        assert np.array_equal(sim.download(f), a), f
    sim.op("UPDATE_OLD")
    assert np.array_equal(sim.download("C_OLD"), seen["C_NEW"])
    assert np.array_equal(sim.download("W_OLD"), seen["W_NEW"])
    assert not sim.download("V_OLD").any()


def test_step_tracks_oracle(oracle_mod):
    """One step against the FP64 oracle: c and the velocity to 1e-11, phi to
    the condition of the x-lines' mean mode (16 n^2/pi^2) times the rounding
    unit."""
    oracle_mod.set_threads(min(16, len(os.sched_getaffinity(0))))
    prm = P.make_params(520, 82, 81, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    c0 = P.ic_fill(prm, P.IC_NOISE, 3, 0.05)
    orc = oracle_mod.Oracle(prm)
    orc.init(c0)
    sim = P.Sim(prm, "plain")
    sim.init(c0)
    orc.run(1)
    sim.run(1)
    for fields, tol in ((["C_OLD"], 1e-11), (["U_OLD", "V_OLD", "W_OLD"], 1e-11),
                        (["PHI"], 16 * 520 ** 2 / np.pi ** 2 * np.finfo(float).eps)):
        a = np.concatenate([sim.download(f).ravel() for f in fields])
        b = np.concatenate([orc.field(f).ravel() for f in fields])
        err = np.linalg.norm(a - b) / np.linalg.norm(b)
        print("[pitched] %s %.2e" % (fields[0], err), flush=True)
        assert err <= tol


@pytest.mark.parametrize("precision", ["plain", "mixed"])
def test_fused_step_equals_operators(precision):
    prm = P.make_params(520, 82, 81, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
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
    for f in ("C_OLD", "U_OLD", "V_OLD", "W_OLD", "PHI", "U_PG", "W_PG", "MUO_CELL"):
        x, y = a.download(f), b.download(f)
        assert np.array_equal(x, y), (precision, f, np.abs(x - y).max())


def test_batched_members_equal_standalone_runs():
    """Two members of 200x64x64, pitched as the batch has 1.8 million points,
    keep the bits of the same simulations run alone, whose rows are packed."""
    prm = [P.make_params(200, 64, 64, Vratio=3.0 - i, Pe=300.0 + 100 * i, Inf_thick=0.1) for i in range(2)]
    c0 = [P.ic_fill(p, P.IC_NOISE, 3 + i, 0.05) for i, p in enumerate(prm)]
    ens = P.Ensemble(prm, "mixed")
    assert ens.batches() == 1
    alone = [P.Sim(p, "mixed") for p in prm]
    for m, s, c in zip(ens.members, alone, c0):
        m.init(c)
        s.init(c)
    w = np.random.default_rng(1).standard_normal(alone[0].shape)
    for steps in (2, 3):
        ens.run(steps)
        for m, s in zip(ens.members, alone):
            s.run(steps)
            for f in ("C_OLD", "U_OLD", "V_OLD", "W_OLD", "PHI", "U_PG"):
                assert np.array_equal(m.download(f), s.download(f)), (steps, f)
            m.upload("DIV", w)
            assert np.array_equal(m.download("DIV"), w.astype(np.float32).astype(float))
    ens.close()
