"""The explicit terms of even theta sizes, computed in theta pairs, against
the oracle: the smallest grids, where both neighbours of a pair wrap onto
it, and planes of a few pairs less than a block of 256, of one block, and a
few pairs more.  Tolerance: the 1e-12 relative L2 of the routine tests (FP64
stencils that differ by FMA contraction)."""
import pytest

from helpers import load_both, random_state, rel_l2, small_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 2, 3), (4, 3, 3), (6, 5, 4), (20, 25, 3), (32, 16, 4), (54, 10, 5)])
def test_explicit_terms_in_pairs(tc, oracle, shape):
    nrm = shape[2]
    p = small_params(tc, *shape)
    dev, orc = tc.Solver(p), oracle.Oracle(p)
    load_both(dev, orc, random_state(p, 5))
    for s in (dev, orc):
        s.set_time(0.3, 1e-3)
        s.begin_step()
        s.set_substep(2)
    for name in ("QT", "QR", "QZ"):
        getattr(dev, "ExplicitTerms" + name)()
        orc.call("explicit_terms_" + name.lower())
    for f, first in (("dq", 0), ("dph", 1), ("qcap", 0)):
        assert rel_l2(dev.get(f)[first:nrm], orc.get(f)[first:nrm]) <= 1e-12, f
