"""Uploads and downloads by every route: packed FP64 fields as they are, FP32
ones converted on the host or (from 50000 points on where the host memory is
page-locked, from 1.5 million on where not) on the device in several pieces,
pitched FP64 ones through the device."""
import ctypes

import numpy as np
import pytest
import torch

import pllcart3d_amd as P
from pllcart3d_amd._lib import FIELD_ID

pytestmark = pytest.mark.gpu


def _host(shape, locked):
    return torch.empty(shape, dtype=torch.float64, pin_memory=locked).numpy()


def _call(fn, sim, field, a):
    assert fn(sim.h, FIELD_ID[field], a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))) == 0, P.last_error()


@pytest.mark.parametrize("locked", [False, True])
@pytest.mark.parametrize("precision", ["plain", "mixed"])
@pytest.mark.parametrize("shape", [(7, 6, 4), (30, 38, 32), (31, 40, 32), (129, 40, 39), (130, 41, 43), (250, 90, 78), (520, 82, 81)])
def test_round_trip(shape, precision, locked):
    """Every value comes back as uploaded (mixed: rounded to FP32 once), from
    and to host memory of either kind, before and after fused steps (whose
    swapped pairs a transfer sets right)."""
    sim = P.Sim(P.make_params(*shape, Vratio=3.0, Pe=300.0, Inf_thick=0.1), precision)
    sim.init(None)
    rng = np.random.default_rng(shape[2])
    a, back = _host(sim.shape, locked), _host(sim.shape, not locked)
    for steps in (0, 3):
        if steps:
            sim.init(None)
            sim.run(steps)
        kept = sim.download("U_OLD")
        assert kept.any()
        a[...] = rng.standard_normal(sim.shape)
        want = a if precision == "plain" else a.astype(np.float32).astype(float)
        _call(sim.L.pllc_sim_upload, sim, "W_NM1", a)
        _call(sim.L.pllc_sim_download, sim, "W_NM1", back)
        assert np.array_equal(back, want)
        back[...] = 0.0
        _call(sim.L.pllc_sim_download, sim, "U_OLD", a)
        assert np.array_equal(a, kept)
        assert np.array_equal(sim.download("U_NEW"), kept)
