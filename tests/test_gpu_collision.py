"""The collision check against all pairs of surface edges and triangles."""
import numpy as np
import pytest

from fastipc_amd import scene as S
from fastipc_amd.newton import NewtonIPC

pytestmark = pytest.mark.gpu


def _crowd(n, copies, spread):
    """copies of an n^3 lattice thrown into a box of size spread over a fixed ground"""
    rng = np.random.default_rng(1000 * n + copies)
    xc, tc = S.lattice(n)
    xs = [xc + rng.uniform(0, spread, 3) + [0, 0.05, 0] for _ in range(copies)]
    gx, gt = S.box([-1, -0.1, -1], [2, 0.0, 2])
    x = np.concatenate(xs + [gx])
    tets = np.concatenate([tc + k * len(xc) for k in range(copies)] + [gt + copies * len(xc)]).astype(np.int32)
    one = np.ones(len(tets))
    sc = S.Scene(name="crowd", x=x, tets=tets, density=1000 * one, youngs=1e5 * one, poisson=0.4 * one,
                 dirichlet_mask=np.arange(len(x)) >= copies * len(xc), dt=0.01, dhat_rel=2e-2)
    return sc, rng


def _seg_tri_pairs(x, sc, infl, inv_dx):
    """How many pairs of surface edge and triangle, without a common vertex and with
    a common grid cell (the triangle's box widened by infl), pass the
    segment-triangle test, in the operations and the order of the oracle's."""
    _, be, bt = sc.boundary

    def cells(v, w):
        return np.floor((v.min(1) - w) * inv_dx), np.floor((v.max(1) + w) * inv_dx)

    (elo, ehi), (tlo, thi) = cells(x[be], 0.0), cells(x[bt], infl)
    near = ((elo[:, None] <= thi[None]) & (tlo[None] <= ehi[:, None])).all(2)
    near &= (be[:, None, :, None] != bt[None, :, None, :]).all((2, 3))
    i, j = np.nonzero(near)

    def dot(a, b):
        return a[:, 0] * b[:, 0] + a[:, 1] * b[:, 1] + a[:, 2] * b[:, 2]

    def cross(a, b):
        return np.stack([a[:, k - 2] * b[:, k - 1] - a[:, k - 1] * b[:, k - 2] for k in range(3)], 1)

    P, Q, (A, B, C) = x[be[i, 0]], x[be[i, 1]], (x[bt[j, k]] for k in range(3))
    R = Q - P
    length = np.sqrt(dot(R, R))
    R = R / length[:, None]
    E1, E2, AO = B - A, C - A, P - A
    N, DAO = cross(E1, E2), cross(AO, R)
    det = -dot(R, N)
    with np.errstate(divide="ignore", invalid="ignore"):
        inv = 1.0 / det
        u, v, t = dot(E2, DAO) * inv, -dot(E1, DAO) * inv, dot(AO, N) * inv
        return int(((det >= 1e-12) & (t >= 0) & (u >= 0) & (v >= 0) & (u + v <= 1) & (t <= length)).sum())


@pytest.mark.parametrize("size", [0.01, 1.0, 100.0, 1000.0])
def test_collision_check_of_coplanar_faces(size):
    """Two boxes apart by a third of their edge with their faces in common planes,
    turned at random: with long edges the rounding error of the segment-triangle
    test passes some pairs, and the check reports what that test says of every
    pair with a common grid cell."""
    found = 0
    for seed in range(12):
        bx, bt = S.box([0, 0, 0], [size, size, size])
        q = np.linalg.qr(np.random.default_rng(seed).normal(size=(3, 3)))[0]
        x = np.concatenate([bx, bx + [1.3 * size, 0, 0]]) @ (q * np.linalg.det(q)).T
        tets = np.concatenate([bt, bt + 8]).astype(np.int32)
        one = np.ones(len(tets))
        sc = S.Scene(name="boxes", x=x, tets=tets, density=1000 * one, youngs=1e5 * one, poisson=0.4 * one,
                     dirichlet_mask=np.zeros(16, bool), dt=0.01)
        sim = NewtonIPC(sc)
        want = _seg_tri_pairs(x, sc, sim.setup.dHat, sim.setup.inv_dx) > 0
        assert sim.check_collision() == want, seed
        found += want
        sim.close()
    assert (found > 0) == (size >= 100)


@pytest.mark.parametrize("n,copies,spread", [(2, 3, 0.3), (3, 2, 0.2), (4, 9, 0.9), (2, 40, 4.0), (2, 40, 0.5)])
def test_collision_check_against_all_pairs(n, copies, spread):
    """Bodies thrown together and bodies apart, against all pairs."""
    sc, rng = _crowd(n, copies, spread)
    sim = NewtonIPC(sc)
    apart = sc.x + 3.0 * np.repeat(np.arange(copies + 1), [n ** 3] * copies + [8])[:, None]
    for x in (sc.x + rng.normal(0, 0.002, sc.x.shape), apart):
        sim.set_state(x, np.zeros_like(x))
        want = _seg_tri_pairs(x, sc, sim.setup.dHat, sim.setup.inv_dx)
        assert sim.check_collision() == (want > 0), want
        assert x is not apart or want == 0
    sim.close()
