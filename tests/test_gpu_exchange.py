"""Fields in and out in the reference's order against the device order: the
transposes move values, so every comparison is exact.  Shapes: tile
remainders in r and theta, one tile, and (30, 9, 3), whose columns do not fit
the staging array at once."""
import numpy as np
import pytest

from helpers import small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(30, 9, 3), (27, 20, 13), (64, 27, 31), (8, 4, 5), (100, 3, 96)])
def test_fortran_order_is_the_device_order_transposed(tc, shape):
    p = small_params(tc, *shape)
    s = tc.Solver(p)
    rng = np.random.default_rng(1)
    a = np.asfortranarray(rng.standard_normal(s.shape))
    s.set("qz", a)
    dev = np.empty(s.shape)
    tc._check(tc.lib().tc_download_field(s.h, tc.FIELDS["qz"], tc._dp(dev), tc.LAYOUT_DEVICE))
    assert np.array_equal(dev, a)
    b = rng.standard_normal(s.shape)
    tc._check(tc.lib().tc_upload_field(s.h, tc.FIELDS["ru1"], tc._dp(b), tc.LAYOUT_DEVICE))
    assert np.array_equal(s.get("ru1"), b)
    assert np.array_equal(s.get("qz"), a)
