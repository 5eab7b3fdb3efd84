"""Launch shapes that follow from sizes alone.  Launches of long thin grids stay
within 65535 blocks along z: the rule on the host, over its range, and on the
GPU the first sizes at which the joint explicit launch reaches the limit.  The
autotuner's candidates."""
import os
import subprocess

import numpy as np
import pytest

import pllcart3d_amd as P

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pllcart3d_amd", "csrc")

SEQ = ["CONCENTRATION", "VISCOSITY", "XMOM", "YMOM", "ZMOM", "VELO_BOUNDARY", "DIVERGENCE", "PHISOLVER",
       "PHI_GHOSTS", "VELO_CORRECTION", "VELOGHOST", "PRESSURE_GRADIENT", "UPDATE_OLD"]


@pytest.mark.parametrize("what", ["blocks along z", "z-sweep block shapes tuned"])
def test_rules_on_the_host(tmp_path, what):
    exe = tmp_path / "grid_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, "-o", str(exe),
                    os.path.join(HERE, "native", "grid_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    assert int(out.split()[["blocks along z", "z-sweep block shapes tuned"].index(what)]) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["plain", "mixed"])
def test_long_thin_grid_joint_launch_equals_single_ones(precision):
    """One fused step of 16389x2x2 against the operators, each its own launch:
    the same bits.  (With 3 points across, w's z-lines have two rows, so the
    three components' common launch takes one thread per line where u's and
    v's own launches take the partitioned solve: equal to rounding only.)"""
    prm = P.make_params(16389, 2, 2, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
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
    for f in ("C_OLD", "C_N", "U_OLD", "V_OLD", "W_OLD", "W_N", "PHI", "U_PG"):
        x, y = a.download(f), b.download(f)
        assert np.all(np.isfinite(x)) and np.array_equal(x, y), (precision, f, np.abs(x - y).max())


@pytest.mark.gpu
def test_long_thin_grid_tracks_oracle(oracle_mod):
    """One step of 16389x3x3 in FP64 against the oracle: c to 1e-11; phi, and
    the velocity that its gradient makes, to the condition of the x-lines'
    mean mode (16 n^2/pi^2) times the rounding unit."""
    prm = P.make_params(16389, 3, 3, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    c0 = P.ic_fill(prm, P.IC_NOISE, 3, 0.05)
    orc = oracle_mod.Oracle(prm)
    orc.init(c0)
    sim = P.Sim(prm, "plain")
    sim.init(c0)
    orc.run(1)
    sim.run(1)
    err = {}
    for name, fields in (("c", ["C_OLD"]), ("velocity", ["U_OLD", "V_OLD", "W_OLD"]), ("phi", ["PHI"])):
        x = np.concatenate([sim.download(f).ravel() for f in fields])
        y = np.concatenate([orc.field(f).ravel() for f in fields])
        err[name] = np.linalg.norm(x - y) / np.linalg.norm(y)
    print("[long thin grid]", {k: "%.2e" % v for k, v in err.items()}, flush=True)
    assert err["c"] <= 1e-11
    assert max(err["velocity"], err["phi"]) <= 16 * 16389 ** 2 / np.pi ** 2 * np.finfo(float).eps


@pytest.mark.gpu
@pytest.mark.parametrize("nz", [12, 24, 40])
def test_tuned_shapes_leave_the_bits(nz):
    """A handle with the shapes that the autotuner kept for its grid gives the
    bits of one created before; the z-lines are those of 1, 2 or 4 waves."""
    prm = P.make_params(40, 20, nz, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    c0 = P.ic_fill(prm, P.IC_NOISE, 3, 0.05)
    a = P.Sim(prm, "mixed")
    lines = P.Sim(prm, "mixed").autotune(2)
    print("[autotune] nz %d lines per block x/y/z %s" % (nz, lines), flush=True)
    assert lines[2] in [w * {12: 64, 24: 32, 40: 16}[nz] for w in (1, 2, 4)]
    b = P.Sim(prm, "mixed")
    for s in (a, b):
        s.init(c0)
        s.run(3)
    for f in ("C_OLD", "U_OLD", "V_OLD", "W_OLD", "PHI"):
        assert np.array_equal(a.download(f), b.download(f)), f
