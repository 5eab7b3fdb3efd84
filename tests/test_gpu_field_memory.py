"""The fields' pitched rows take at most half as much again as packed ones."""
import pytest
import torch

import pllcart3d_amd as P

pytestmark = pytest.mark.gpu


def _used(shape, precision):
    torch.cuda.init()
    free = torch.cuda.mem_get_info()[0]
    sim = P.Sim(P.make_params(*shape, Vratio=2.0, Pe=1000.0, Inf_thick=0.1), precision)
    used = free - torch.cuda.mem_get_info()[0]
    sim.close()
    return used


@pytest.mark.parametrize("shape", [(400, 400, 4), (400, 400, 9), (128, 256, 32), (128, 256, 64), (64, 256, 128)])
def test_fields_take_at_most_half_more_than_packed_ones(shape):
    """Against 39 packed fields of the precision (36 of the state and the
    sweeps, the transform's three blocks), 32 MB aside for tables
    and the allocator's pages."""
    points = (shape[0] + 6) * (shape[1] + 2) * (shape[2] + 2)
    for precision, size in (("plain", 8), ("mixed", 4)):
        used = _used(shape, precision)
        print("[memory] %s %s %.0f MB, packed field %.2f MB" % (shape, precision, used / 1e6, points * size / 1e6),
              flush=True)
        assert used <= 1.5 * 39 * points * size + 32e6, (precision, used)
