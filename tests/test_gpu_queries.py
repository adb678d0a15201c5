"""The grid queries in front of the searches and of the swept tests: the pairs they
hand on, counted, against all pairs of boxes, near the origin and far from it."""
import numpy as np
import pytest

from fastipc_amd import _lib
from fastipc_amd import scene as S
from fastipc_amd.newton import NewtonIPC
from oracle import lib as O

pytestmark = pytest.mark.gpu

CROWDS = [(2, 1, 1.0), (2, 3, 0.3), (3, 2, 0.2), (4, 3, 0.5), (2, 20, 0.8)]
OFFSETS = [0.0, 1e4]  # at 1e4 single precision resolves a thousandth, a hundredth of an edge


def _crowd(n, copies, spread, offset):
    """copies of an n^3 lattice thrown into a box of size spread over a fixed ground"""
    rng = np.random.default_rng(1000 * n + copies)
    xc, tc = S.lattice(n)
    xs = [xc + rng.uniform(0, spread, 3) + [0, 0.05, 0] for _ in range(copies)]
    gx, gt = S.box([-1, -0.1, -1], [2, 0.0, 2])
    x = np.concatenate(xs + [gx]) + offset * np.array([1.0, -2.0, 0.3])
    tets = np.concatenate([tc + k * len(xc) for k in range(copies)] + [gt + copies * len(xc)]).astype(np.int32)
    one = np.ones(len(tets))
    sc = S.Scene(name="crowd", x=x, tets=tets, density=1000 * one, youngs=1e5 * one, poisson=0.4 * one,
                 dirichlet_mask=np.arange(len(x)) >= copies * len(xc), dt=0.01, dhat_rel=1e-2)
    return sc, rng


def _overlaps(alo, ahi, blo, bhi, dhat):
    """The swept tests' box test, in its operations: a's box below b's plus dhat and b's less dhat below a's."""
    return ((alo[:, None] < bhi[None] + dhat) & (blo[None] - dhat < ahi[:, None])).all(2)


def _swept_candidates(x, p, sc, dhat, eta):
    """point-triangle and edge-edge pairs without a common vertex whose swept boxes
    overlap within dhat and whose distance could be closed: the lower bound of
    the time of impact is below one"""
    bp, be, bt = sc.boundary

    def box(v):
        q = np.concatenate([x[v], x[v] + p[v]], 1)
        return q.min(1), q.max(1)

    def bound(d2, a, b):
        size = [np.sqrt(max((p[v] ** 2).sum() for v in ids)) for ids in (a, b)]
        return sum(size) != 0 and (1 - eta) * np.sqrt(d2) / sum(size) < 1

    pt = _overlaps(*box(bp[:, None]), *box(bt), dhat) & (bp[:, None, None] != bt[None]).all(2)
    n_pt = 0
    for i, j in zip(*np.nonzero(pt)):
        q = [O.dptr(O.f64(x[v])) for v in (bp[i], *bt[j])]
        n_pt += bound(O.lib().orc_PT_dist2(*q, O.lib().orc_PT_type(*q)), [bp[i]], bt[j])
    ee = np.triu(_overlaps(*box(be), *box(be), dhat), 1) & (be[:, None, :, None] != be[None, :, None, :]).all((2, 3))
    n_ee = 0
    for i, j in zip(*np.nonzero(ee)):
        q = [O.dptr(O.f64(x[v])) for v in (*be[i], *be[j])]
        n_ee += bound(O.lib().orc_EE_dist2(*q, O.lib().orc_EE_type(*q)), be[i], be[j])
    return n_pt, n_ee


def _near(x, sc, dhat):
    """point-triangle and edge-edge pairs whose boxes overlap within dhat, without a common vertex"""
    bp, be, bt = sc.boundary
    t, e = x[bt], x[be]
    pt = _overlaps(x[bp], x[bp], t.min(1), t.max(1), dhat) & (bp[:, None, None] != bt[None]).all(2)
    ee = np.triu(_overlaps(e.min(1), e.max(1), e.min(1), e.max(1), dhat), 1)
    ee &= (be[:, None, :, None] != be[None, :, None, :]).all((2, 3))
    return int(pt.sum()), int(ee.sum())


@pytest.mark.parametrize("offset", OFFSETS)
@pytest.mark.parametrize("n,copies,spread", CROWDS)
def test_swept_candidates_and_searches_along_the_step(n, copies, spread, offset):
    """The candidates of the step bound; then, at the end of the step, where the
    searches reuse its grids of swept boxes, the pairs that they test."""
    sc, rng = _crowd(n, copies, spread, offset)
    sim = NewtonIPC(sc)
    dhat, eta = sim.setup.dHat, sim.setup.eta
    x = sc.x + rng.normal(0, 0.01, sc.x.shape)
    p = rng.normal(0, 0.03, sc.x.shape)
    sim.set_state(x, np.zeros_like(x))
    sim.set_vector(1, p)
    sim.save_xPrev()
    sim.compute_intersection_free_step_size()
    pairs = np.zeros(2, np.int32)
    _lib.call("fipc_ccd_counts", sim.ctx, _lib.iptr(pairs))
    assert tuple(pairs) == _swept_candidates(x, p, sc, dhat, eta)
    sim.search_stats(True)
    for alpha in (0.5, 1.0):
        sim.apply_sol(alpha)
        sim.find_constraints()
        assert tuple(sim.search_counts()) == _near(sim.x, sc, dhat), alpha
    sim.close()


@pytest.mark.parametrize("factor", [0.3, 3.0])
def test_cell_size_changed_between_searches(factor):
    """Grids of the former cell size are not reused at the same positions."""
    sc, rng = _crowd(3, 2, 0.2, 0.0)
    sim = NewtonIPC(sc)
    s = sim.setup
    x = sc.x + rng.normal(0, 0.01, sc.x.shape)
    sim.set_state(x, np.zeros_like(x))
    sim.set_vector(1, rng.normal(0, 0.03, sc.x.shape))
    sim.save_xPrev()
    sim.search_stats(True)
    want = _near(x, sc, s.dHat)
    for inv_dx in (s.inv_dx, factor * s.inv_dx):
        _lib.call("fipc_set_params", sim.ctx, s.dt, s.dHat, s.kappa, inv_dx, s.gravity)
        sim.find_constraints()
        assert tuple(sim.search_counts()) == want
    # the same with the step bound's grids of swept boxes
    sim.compute_intersection_free_step_size()
    sim.apply_sol(1.0)
    want = _near(sim.x, sc, s.dHat)
    for inv_dx in (factor * s.inv_dx, s.inv_dx):
        _lib.call("fipc_set_params", sim.ctx, s.dt, s.dHat, s.kappa, inv_dx, s.gravity)
        sim.find_constraints()
        assert tuple(sim.search_counts()) == want
    sim.close()


def test_previous_positions_set_before_a_step():
    """A step from positions that the caller set is not on the segment that the
    step bound's grids sweep."""
    sc, rng = _crowd(3, 2, 0.2, 0.0)
    sim = NewtonIPC(sc)
    x = sc.x + rng.normal(0, 0.01, sc.x.shape)
    sim.set_state(x, np.zeros_like(x))
    sim.set_vector(1, rng.normal(0, 0.03, sc.x.shape))
    sim.save_xPrev()
    sim.compute_intersection_free_step_size()
    sim.set_vector(5, x + rng.normal(0, 0.2, sc.x.shape))
    sim.apply_sol(0.5)
    sim.search_stats(True)
    sim.find_constraints()
    assert tuple(sim.search_counts()) == _near(sim.x, sc, sim.setup.dHat)
    sim.close()
