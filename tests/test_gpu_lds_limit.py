"""The dynamic LDS limit of the plane transforms belongs to the kernel, which
every handle of the process shares: a handle of small planes must leave it at
what a living handle of larger planes launches with."""
import ctypes as C

import numpy as np
import pytest

import pllcart3d_amd as P
from pllcart3d_amd._lib import load

pytestmark = pytest.mark.gpu

WIDE = "_ZN4pllc10k_dct_wideI%sLb%dEEEviiPT_PKS1_S4_NS_6PhiOutIS1_EENS_5DivInIS1_EE"
PLANES = "_ZN4pllc12k_dct_planesI%sLb%dELi0EEEviiiiPT_PKS1_S4_NS_6PhiOutIS1_EENS_5DivInIS1_EENS_2BtE"


class _Attributes(C.Structure):   # hipFuncAttributes
    _fields_ = [("binary", C.c_int), ("cache", C.c_int), ("constant", C.c_size_t), ("local", C.c_size_t),
                ("dynamic", C.c_int), ("rest", C.c_char * 128)]


def _limit(name):
    a = _Attributes()
    kernel = C.c_void_p.in_dll(load(), name)
    assert C.CDLL("libamdhip64.so").hipFuncGetAttributes(C.byref(a), C.c_void_p(C.addressof(kernel))) == 0
    return a.dynamic


@pytest.mark.parametrize("precision", ["plain", "mixed"])
@pytest.mark.parametrize("kernel, large, small", [(WIDE, (127, 113), (17, 13)), (PLANES, (48, 64), (16, 32))])
def test_small_planes_leave_the_limit_of_larger_ones(precision, kernel, large, small):
    t, size = ("d", 8) if precision == "plain" else ("f", 4)
    prm = P.make_params(6, *large, Vratio=3.0, Pe=300.0, Inf_thick=0.1)
    a = P.Sim(prm, precision)
    a.init(None)
    a.run(1)
    want = a.download("PHI")
    b = P.Sim(P.make_params(6, *small, Vratio=3.0, Pe=300.0, Inf_thick=0.1), precision)
    for inverse in (0, 1):
        # a launch of a holds its plane in LDS at least
        assert _limit(kernel % (t, inverse)) >= large[0] * large[1] * size
    b.init(None)
    b.run(1)
    a.init(None)
    a.run(1)
    assert np.array_equal(a.download("PHI"), want)
