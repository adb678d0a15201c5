"""Sizes at which a kernel's launch shape could go wrong: remainders of waves,
blocks and tiles, the smallest sizes and the first past a boundary."""
import numpy as np
import pytest

from fastipc_amd import _lib

pytestmark = pytest.mark.gpu

NPTS = (2, 3, 4, 4, 4, 4, 4)


def _constraints(kind, X, X0, project=1):
    n, nd = len(X), 3 * NPTS[kind]
    E, g, H = np.zeros(n), np.zeros((n, nd)), np.zeros((n, nd, nd))
    _lib.call("fipc_batch_constraint", kind, n, _lib.dptr(X), _lib.dptr(X0), 1e-2, 1.0, project, _lib.dptr(E),
              _lib.dptr(g), _lib.dptr(H))
    return E, g, H


@pytest.mark.parametrize("kind", range(7))
def test_contact_rows_do_not_depend_on_their_number(kind):
    """A row's gradient and projected Hessian are the same bits whether it is
    alone, in a partial group of lanes, or in the last block (4 or 8 rows per
    wave, 16 or 32 per block of the projection)."""
    rng = np.random.default_rng(kind)
    X = np.ascontiguousarray(rng.normal(0, 0.03, (70, NPTS[kind], 3)))
    if kind >= 4:  # nearly parallel edges, so that the mollifier acts
        X[:, 3] = X[:, 2] + (X[:, 1] - X[:, 0]) + rng.normal(0, 1e-3, (70, 3))
    X0 = np.ascontiguousarray(X + rng.normal(0, 0.01, X.shape))
    whole = _constraints(kind, X, X0)
    # projected: positive semi-definite up to the projection's rounding
    for H in whole[2]:
        assert np.linalg.eigvalsh(H)[0] >= -1e-9 * max(np.abs(H).max(), 1e-300)
    for n in (1, 3, 4, 5, 8, 9, 16, 17, 33, 64, 65):
        part = _constraints(kind, X[:n].copy(), X0[:n].copy())
        for a, b in zip(part, whole):
            assert np.array_equal(a, b[:n], equal_nan=True), n


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(1, 1, 3), (2, 3, 5), (3, 4, 9)])  # contact slots in one, many, and more blocks than surface vertices fill
def test_product_and_solve_with_contacts(shape, precision):
    """The product's contact part and the solver on piles whose contact blocks
    fit one partial per thread, and on one whose slots would fill more blocks
    than its surface vertices: the solution's residual by the product itself."""
    import ctypes as C
    from fastipc_amd import scene as S
    from fastipc_amd.newton import NewtonIPC
    m, layers, n = shape
    xc, tc = S.lattice(n)
    edge = (n - 1) * S.LATTICE_SPACING
    xs, ts, nv = [], [], 0
    for layer in range(layers):
        for i in range(m):
            for k in range(m):
                off = [(1.06 * i + 0.31 * (layer % 2)) * edge, layer * (edge + 1e-3) + 1e-3, (1.06 * k + 0.17 * (layer % 2)) * edge]
                xs.append(xc + off)
                ts.append(tc + nv)
                nv += len(xc)
    gx, gt = S.box([-edge, -0.1, -edge], [(m + 2) * edge, 0.0, (m + 2) * edge])
    x, tets = np.concatenate(xs + [gx]), np.concatenate(ts + [gt + nv]).astype(np.int32)
    one = np.ones(len(tets))
    sc = S.Scene(name="pile", x=x, tets=tets, density=1000 * one, youngs=1e5 * one, poisson=0.4 * one,
                 dirichlet_mask=np.arange(len(x)) >= nv, dt=0.01)
    sim = NewtonIPC(sc, precision=precision)
    rng = np.random.default_rng(n)
    state = sc.x.copy()
    state[:nv] += rng.uniform(-1e-4, 1e-4, (nv, 3))
    sim.set_state(state, np.zeros_like(state))
    sim.compute_xn_and_xTilde(0.0)
    counts = sim.find_constraints()
    assert sum(counts) > 0 and sim.check_collision() == 0
    sim.compute_hessian_and_gradient()
    tol = 1e-6
    sim.solve_system(tol=tol)
    assert sim.last_solve_converged
    p, b, y = sim.vector(1), sim.vector(2), np.zeros((sim.nv, 3))
    _lib.call("fipc_spmv", sim.ctx, _lib.dptr(p), _lib.dptr(y))
    # the recurrence's residual met the tolerance; the true one is near it
    assert np.linalg.norm(b - y) <= 2 * tol * np.linalg.norm(b)
    # symmetric: u.(A v) = v.(A u) up to the rounding of sums of some thousand terms
    u, v = rng.standard_normal((2, sim.nv, 3))
    u[nv:] = v[nv:] = 0
    yu, yv = np.zeros_like(y), np.zeros_like(y)
    _lib.call("fipc_spmv", sim.ctx, _lib.dptr(u), _lib.dptr(yu))
    _lib.call("fipc_spmv", sim.ctx, _lib.dptr(v), _lib.dptr(yv))
    assert abs(np.vdot(u, yv) - np.vdot(v, yu)) <= 1e-9 * np.linalg.norm(u) * np.linalg.norm(yv)
    sim.close()


def _brute_pairs(x, sc, dhat):
    """point-triangle and edge-edge pairs whose boxes overlap within dhat, without a common vertex"""
    bp, be, bt = sc.boundary
    lo, hi = x[bt].min(1), x[bt].max(1)
    pt = ((x[bp][:, None] < hi[None] + dhat) & (lo[None] - dhat < x[bp][:, None])).all(2)
    pt &= (bp[:, None, None] != bt[None]).all(2)
    lo, hi = x[be].min(1), x[be].max(1)
    ee = ((lo[:, None] < hi[None] + dhat) & (lo[None] - dhat < hi[:, None])).all(2)
    ee &= (be[:, None, :, None] != be[None, :, None, :]).all((2, 3))
    return int(pt.sum()), int(np.triu(ee, 1).sum())


@pytest.mark.parametrize("n,copies,spread", [(2, 1, 1.0), (2, 3, 0.3), (3, 2, 0.2), (4, 9, 0.9), (5, 4, 0.4), (2, 40, 0.5)])
def test_grid_queries_visit_every_pair_once(n, copies, spread):
    """The pairs that the searches' queries visit, counted, against all pairs of
    boxes: one wave's pairs, several blocks of queries, crowded and nearly empty
    buckets, and the few large boxes of the ground among them."""
    import ctypes as C
    from fastipc_amd import scene as S
    from fastipc_amd.newton import NewtonIPC
    rng = np.random.default_rng(1000 * n + copies)
    xc, tc = S.lattice(n)
    xs = [xc + rng.uniform(0, spread, 3) + [0, 0.05, 0] for _ in range(copies)]
    gx, gt = S.box([-1, -0.1, -1], [2, 0.0, 2])
    x = np.concatenate(xs + [gx])
    tets = np.concatenate([tc + k * len(xc) for k in range(copies)] + [gt + copies * len(xc)]).astype(np.int32)
    one = np.ones(len(tets))
    sc = S.Scene(name="crowd", x=x, tets=tets, density=1000 * one, youngs=1e5 * one, poisson=0.4 * one,
                 dirichlet_mask=np.arange(len(x)) >= copies * len(xc), dt=0.01, dhat_rel=2e-2)
    sim = NewtonIPC(sc)
    moved = sc.x + rng.normal(0, 0.01, sc.x.shape)
    sim.set_state(moved, np.zeros_like(moved))
    sim.search_stats(True)
    sim.find_constraints()
    assert tuple(sim.search_counts()) == _brute_pairs(moved, sc, sc.dhat)
    sim.close()


@pytest.mark.parametrize("rows", [1, 31, 32, 33, 63, 64, 65, 511, 512, 513, 1100])
def test_network_gradient_over_row_remainders(rows):
    """Loss and gradient of the warm-start shape at the edges of its 32-row blocks
    and row slices, against the same network in float64 with inputs of every
    product rounded to BF16 (8 bits): each rounding moves a product by at most
    2^-9 of its size, and 10 of them follow one another."""
    from fastipc_amd.warmstart import WarmStartMLP
    rng = np.random.default_rng(rows)
    net = WarmStartMLP(seed=rows)
    X = rng.standard_normal((rows, 16)).astype(np.float32)
    T = rng.standard_normal((rows, 3)).astype(np.float32)
    loss, grad = net.grad(X, T)
    w = net.params().astype(np.float64)

    def bf(a):
        u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
        return ((((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32)).view(np.float32).astype(np.float64)

    dims, o, Ws, bs = [16, 256, 256, 256, 256, 3], 0, [], []
    for a, b in zip(dims, dims[1:]):
        Ws.append(w[o:o + a * b].reshape(a, b))
        bs.append(w[o + a * b:o + a * b + b])
        o += a * b + b
    A, Z, h = [], [], X.astype(np.float64)
    for k, (W, b) in enumerate(zip(Ws, bs)):
        A.append(bf(h))
        z = A[-1] @ bf(W) + b
        Z.append(z)
        h = z / (1 + np.exp(-z)) if k < 4 else z
    d = h - T
    assert abs(loss - (d ** 2).mean()) <= 1e-3 * (d ** 2).mean()
    G, want = 2 * d / d.size, [None] * 5
    for k in range(4, -1, -1):
        want[k] = np.concatenate([(A[k].T @ bf(G)).ravel(), G.sum(0)])
        if k:
            s = 1 / (1 + np.exp(-Z[k - 1]))
            G = (bf(G) @ bf(Ws[k]).T) * (s * (1 + Z[k - 1] * (1 - s)))
    o = 0
    for g in want:
        got = grad[o:o + g.size]
        assert np.linalg.norm(got - g) <= 10 * 2.0 ** -9 * np.linalg.norm(g), np.linalg.norm(got - g) / np.linalg.norm(g)
        o += g.size
    net.close()


@pytest.mark.parametrize("shape", [(16, 256, 4, 3), (9, 40, 2, 5)])  # on the chip, and layer by layer
@pytest.mark.parametrize("rows", [1024, 1025, 3001, 16401])
def test_network_gradient_over_row_slices(shape, rows):
    """Loss and gradient with one row slice, two, several, and with short and empty
    slices at the end, close enough to notice one row that is left out.  The
    reference rounds the same values to BF16 in float64.  What remains are float32
    sums and the few values that these move across a rounding to BF16; the same
    network in float32 NumPy, with 2e-7 of noise after every layer, differs from the
    reference by at most 7e-8 in the loss, 6e-4 in a layer's weights and 1.6e-4 in
    its biases, over these sizes, where one row of 16,401 makes 4e-5, 6e-4 and
    6e-4 at least.  Allowed: 1e-6, 3e-3 and 5e-4."""
    import ctypes as C
    n_in, width, depth, n_out = shape
    net, count = C.c_void_p(), C.c_long()
    _lib.call("fipc_mlp_create", C.byref(net), n_in, width, depth, n_out, 7)
    _lib.call("fipc_mlp_nparams", net, C.byref(count))
    w, grad, loss = np.zeros(count.value, np.float32), np.zeros(count.value, np.float32), C.c_float()
    rng = np.random.default_rng(rows)
    X = rng.standard_normal((rows, n_in)).astype(np.float32)
    T = rng.standard_normal((rows, n_out)).astype(np.float32)
    _lib.call("fipc_mlp_get_params", net, _lib.fptr(w))
    _lib.call("fipc_mlp_grad", net, rows, _lib.fptr(X), _lib.fptr(T), C.byref(loss), _lib.fptr(grad))
    _lib.call("fipc_mlp_destroy", net)

    def bf(a):
        u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
        return ((((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32)).view(np.float32).astype(np.float64)

    dims, o, Ws, bs = [n_in] + [width] * depth + [n_out], 0, [], []
    for a, b in zip(dims, dims[1:]):
        Ws.append(w[o:o + a * b].reshape(a, b))
        bs.append(w[o + a * b:o + a * b + b].astype(np.float64))
        o += a * b + b
    A, Z, h = [], [], X
    for k, (W, b) in enumerate(zip(Ws, bs)):
        A.append(bf(h))
        Z.append(A[-1] @ bf(W) + b)
        h = Z[-1] / (1 + np.exp(-Z[-1])) if k < depth else Z[-1]
    d = h - T
    assert abs(loss.value - (d ** 2).mean()) <= 1e-6 * (d ** 2).mean()
    G, end = 2 * d / d.size, grad.size
    for k in range(depth, -1, -1):
        for want, tol in ((G.sum(0), 5e-4), ((A[k].T @ bf(G)).ravel(), 3e-3)):
            got, end = grad[end - want.size:end], end - want.size
            assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want), (k, np.linalg.norm(got - want) / np.linalg.norm(want))
        if k:
            s = 1 / (1 + np.exp(-Z[k - 1]))
            G = (bf(G) @ bf(Ws[k]).T) * (s * (1 + Z[k - 1] * (1 - s)))


@pytest.mark.parametrize("rows", [1, 2, 4, 8, 16, 64])
def test_network_gradient_ignores_the_rows_past_the_last(rows):
    """The rows that fill up a block of 32 add nothing, also where the biases alone
    overflow: here a row of zeros gives 2^66 in the first layer and infinity in the
    second, while the rows themselves give zero.  All rows are alike, so the mean's
    gradient is that of one full block; with powers of two every product scales
    exactly, which leaves the rounding of FP32 sums of up to 64 equal terms."""
    from fastipc_amd.warmstart import WarmStartMLP
    net = WarmStartMLP(seed=1)
    big, w = 2.0 ** 66, net.params()
    W0 = w[:16 * 256].reshape(16, 256)
    W0[:], W0[0] = 0, -big
    w[16 * 256:17 * 256] = big
    w[17 * 256:17 * 256 + 256 * 256] = big
    net.set_params(w)

    def grad(n):
        X = np.zeros((n, 16), np.float32)
        X[:, 0] = 1
        return net.grad(X, np.ones((n, 3), np.float32))

    loss, g = grad(rows)
    loss32, g32 = grad(32)
    assert np.isfinite(g).all() and np.abs(g32).max() > 0
    assert abs(loss - loss32) <= 64 * 2.0 ** -24 * loss32
    assert np.linalg.norm(g - g32) <= 64 * 2.0 ** -24 * np.linalg.norm(g32)
    net.close()


@pytest.mark.parametrize("kind", [0, 1])
def test_batch_ccd_does_not_depend_on_the_number_of_pairs(kind):
    """A pair's time is the same bits alone and in full and partial blocks of 64."""
    rng = np.random.default_rng(kind)
    P = rng.uniform(-1, 1, (200, 12))
    D = rng.normal(0, 1, (200, 12))
    d2 = np.full(200, 1e-4)
    toc = np.zeros(200)
    _lib.call("fipc_batch_ccd", kind, 200, _lib.dptr(P), _lib.dptr(D), 0.2, _lib.dptr(d2), _lib.dptr(toc))
    assert ((toc >= 0) & (toc <= 1)).all() and (toc < 1).any() and (toc == 1).any()
    for n in (1, 63, 64, 65, 128, 129):
        t = np.zeros(n)
        _lib.call("fipc_batch_ccd", kind, n, _lib.dptr(P[:n].copy()), _lib.dptr(D[:n].copy()), 0.2,
                  _lib.dptr(d2[:n].copy()), _lib.dptr(t))
        assert np.array_equal(t, toc[:n]), n


@pytest.mark.parametrize("n,m,layers", [(3, 1, 2), (6, 2, 2), (9, 2, 2), (12, 2, 2), (12, 2, 3)])
def test_row_sets_on_both_sides_of_the_one_launch_sort(n, m, layers):
    """Constraint rows, in np.unique order, against the oracle's search: sets below
    and above 1,024 rows, after one another on one context."""
    from fastipc_amd import scene as S
    from fastipc_amd.newton import NewtonIPC
    from oracle.newton import OracleIPC
    xc, tc = S.lattice(n)
    edge = (n - 1) * S.LATTICE_SPACING
    xs, ts, nv = [], [], 0
    for layer in range(layers):
        for i in range(m):
            for k in range(m):
                xs.append(xc + [(1.06 * i + 0.31 * (layer % 2)) * edge, layer * (edge + 1e-3) + 1e-3,
                                (1.06 * k + 0.17 * (layer % 2)) * edge])
                ts.append(tc + nv)
                nv += len(xc)
    gx, gt = S.box([-edge, -0.1, -edge], [(m + 2) * edge, 0.0, (m + 2) * edge])
    x, tets = np.concatenate(xs + [gx]), np.concatenate(ts + [gt + nv]).astype(np.int32)
    one = np.ones(len(tets))
    sc = S.Scene(name="pile", x=x, tets=tets, density=1000 * one, youngs=1e5 * one, poisson=0.4 * one,
                 dirichlet_mask=np.arange(len(x)) >= nv, dt=0.01)
    sim, orc = NewtonIPC(sc), OracleIPC(sc)
    rng = np.random.default_rng(n)
    for lift in (0.0, 2.0, 0.0):  # all in contact, the bodies apart, in contact again
        state = sc.x.copy()
        state[:nv] += rng.uniform(-1e-4, 1e-4, (nv, 3))
        state[:nv, 1] += lift * edge * (sc.x[:nv, 1] > 0.5 * edge)
        sim.set_state(state, np.zeros_like(state))
        sim.find_constraints()
        orc.x = np.ascontiguousarray(state)
        orc.find_constraints()
        got = sim.constraints(sort=False)
        for k, rows in orc.constraints().items():
            assert np.array_equal(got[k], rows), (k, len(got[k]), len(rows))
    sim.close()
