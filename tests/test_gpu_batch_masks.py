"""Free-slip patterns set on the members of a batch: the grouped kernels with
wall masks and their serial solve, against the oracle marched routine by
routine under the same masks.  Tolerance: the 1e-10 relative L2 of the
workload contract."""
import numpy as np
import pytest

from helpers import load_both, random_state, rel_l2, small_params

pytestmark = pytest.mark.gpu

FIELDS = ("qt", "qr", "qz")
EXPLICIT = tuple("explicit_terms_" + f for f in FIELDS)
IMPLICIT = tuple("implicit_and_update_" + f for f in FIELDS)


def _masks(p, seed, outer):
    rng = np.random.default_rng(seed)
    shape = (p["nzm"], p["nthm"])
    inner = rng.integers(0, 2, shape).astype(np.int32)
    return inner, rng.integers(0, 2, shape).astype(np.int32) if outer else np.ones(shape, np.int32)


def _march(orc, p, masks, n0, n1):
    for n in range(n0, n1):
        orc.set_time(n * p["dtmax"], p["dtmax"])
        orc.begin_step()
        orc.set_masks(*masks)
        for ns in (1, 2, 3):
            orc.set_substep(ns)
            for r in EXPLICIT + IMPLICIT:
                orc.call(r)
            for f in FIELDS:
                orc.update_halo(f)
            orc.call("calc_local_divergence")
            orc.call("solve_pressure_correction")
            orc.update_halo("dph")
            orc.call("correct_velocity")
            orc.call("correct_pressure")
            for f in FIELDS + ("pr",):
                orc.update_halo(f)


def _compare(batch, ids, orcs, nrm):
    for i, o in zip(ids, orcs):
        for f, m in (("qt", nrm), ("qr", nrm + 1), ("qz", nrm), ("pr", nrm)):
            assert rel_l2(batch.solver(i).get(f)[:m], o.get(f)[:m]) <= 1e-10, (i, f)


def _batch(tc, oracle, p, b, seeds, tuning=None):
    ids, orcs = [], []
    for seed in seeds:
        ids.append(b.add(p, tuning))
        orcs.append(oracle.Oracle(p))
        load_both(b.solver(ids[-1]), orcs[-1], random_state(p, seed))
    return ids, orcs


@pytest.mark.parametrize("graph", [False, True])
def test_masks_set_between_advances(tc, oracle, graph):
    """The launches follow the masks that a member has at each advance: none,
    then grooves, then rows exchanged by a free-slip outer wall, then none."""
    p = small_params(tc, 20, 9, 33, idtv=0, ntst=1000, ren=50.0, dtmin=0.1, dtmax=0.1, limitcfl=1e30)
    ones = np.ones((p["nzm"], p["nthm"]), np.int32)
    with tc.Batch() as b:
        ids, orcs = _batch(tc, oracle, p, b, (3, 4))
        am = tc.grid_vector(p, "am1j")[32]
        assert am * 0.5 * p["dtmax"] / p["ren"] * 8.0 / 15.0 > 1.0
        for n, masks in enumerate(((ones, ones), _masks(p, 1, False), _masks(p, 2, True), (ones, ones))):
            for i in ids[1:]:
                b.solver(i).set_masks(*masks)
            b.advance(1, graph=graph)
            _march(orcs[0], p, (ones, ones), n, n + 1)
            _march(orcs[1], p, masks, n, n + 1)
            _compare(b, ids, orcs, p["nrm"])


@pytest.mark.parametrize("lpt,defer", [(1, -1), (2, -1), (1, 2), (2, 2)])
@pytest.mark.parametrize("shape", [(20, 9, 29), (27, 10, 29), (20, 9, 101), (20, 9, 300), (16, 6, 810)])
def test_grouped_kernels_with_masks(tc, oracle, shape, lpt, defer):
    """Masks of their own on each member, on both walls, through every row
    capacity; odd theta sizes have no deferred correction."""
    p = small_params(tc, *shape, idtv=0, ntst=1000, ren=500.0, dtmin=1e-4, dtmax=1e-4, limitcfl=1e30)
    with tc.Batch() as b:
        ids, orcs = _batch(tc, oracle, p, b, (3, 4), dict(helm_lpt=lpt, defer=defer))
        masks = [_masks(p, 5 + i, True) for i in ids]
        for i, m in zip(ids, masks):
            b.solver(i).set_masks(*m)
        b.advance(2)
        for o, m in zip(orcs, masks):
            _march(o, p, m, 0, 2)
        _compare(b, ids, orcs, p["nrm"])
