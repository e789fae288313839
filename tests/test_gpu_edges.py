"""Values at the edge of the number range and calls at the edge of what the
engine takes: infinities, zeros and NaN in networks, captured streams, several
streams and contexts, networks with very many vertices."""
import math

import numpy as np
import pytest

from helpers import oracle_eval, rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.fixture(scope="module")
def eng(q):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return q.engine_context()


def _chain(q, L, bond, dims=1):
    return q.continuous_siteinds(q.named_grid((L * dims, 1)), map_dimension=dims)


def _comb(q, teeth, digits):
    return q.continuous_siteinds(q.named_comb_tree((teeth, digits)),
                                 [[(i, j) for j in range(1, digits + 1)] for i in range(1, teeth + 1)])


def _overflowing(q, s, bond, rng, scale):
    """Positive cores whose digit-1 slices are `scale` times larger, the root
    negative: points with many 1 digits have the value -inf."""
    f = q.random_itn(s, link_space=bond, rng=rng)
    cores = [rng.uniform(0.5, 1.5, c.shape) / math.sqrt(c[0].size) for c in f.cores]
    for c in cores:
        if c.shape[1] == 2:
            c[:, 1] *= scale
    cores[0] = -cores[0]
    f.set_cores(cores)
    return f


def _same_with_infinities(y, ref):
    # sums of numbers of one sign: relative per value; infinite where the reference is
    inf = np.isinf(ref)
    assert inf.any() and not inf.all()
    assert np.array_equal(y[inf], ref[inf])
    assert np.max(np.abs(y[~inf] / ref[~inf] - 1.0)) < TOL


# ------------------------------------------------------------------ infinite values
@pytest.mark.parametrize("bond,npts", [(1, 7), (2, 1000), (3, 1000), (4, 64), (5, 100), (8, 16384), (9, 1000),
                                       (12, 500), (15, 12288), (16, 1000), (17, 100), (31, 1000), (32, 1000)])
def test_few_points_infinite(q, po, eng, rng, bond, npts):
    # a value that overflows is infinite, not NaN: the lanes past the bond stay zero
    f = _overflowing(q, _chain(q, 13, bond), bond, rng, 1e40)
    xs = rng.uniform(0, 1, (npts, 1))
    xs[:4, 0] = [0.0, 0.25, 0.5, 1.0]
    _same_with_infinities(q.evaluate(f, xs), oracle_eval(po, f, xs))


def _tree(q, kind):
    if kind == "comb":
        return _comb(q, 3, 5)
    # one vertex without a digit and four branches: three input legs wherever the tree is cut
    verts = [(0, 0)] + [(i, j) for i in range(1, 5) for j in range(1, 4)]
    edges = [((0, 0), (i, 1)) for i in range(1, 5)] + [((i, j), (i, j + 1)) for i in range(1, 5) for j in range(1, 3)]
    return q.continuous_siteinds(q.NamedGraph(verts, edges), [[(i, j) for j in range(1, 4)] for i in range(1, 5)])


@pytest.mark.parametrize("kind", ["comb", "star"])
@pytest.mark.parametrize("bond,npts", [(3, 1), (5, 40), (16, 300), (20, 3000)])
def test_tree_infinite(q, po, eng, rng, kind, bond, npts):
    # bonds that are padded in the matrix products, points as rows and as table
    # entries; branches that overflow by themselves, beside others that do not
    if kind == "star":
        bond = min(bond, 6)
    f = _overflowing(q, _tree(q, kind), bond, rng, 1e110 if kind == "star" else 1e80)
    xs = rng.uniform(0, 1, (max(npts, 2), f.dimension()))
    xs[0], xs[1] = 0.0, 1.0
    _same_with_infinities(q.evaluate(f, xs), oracle_eval(po, f, xs))


@pytest.mark.parametrize("kind", ["comb", "star"])
@pytest.mark.parametrize("npts", [2, 3000])
def test_tree_zero_blocks_beside_infinite(q, po, eng, rng, kind, npts):
    # a sum of two functions has zero blocks: where one of them overflows the sum is
    # infinite, and with that one's block of the root zero it is the other's value
    s = _tree(q, kind)
    f1, f2 = _overflowing(q, s, 3, rng, 1e110 if kind == "star" else 1e80), _overflowing(q, s, 2, rng, 1.0)
    f = q.builders.add_host(f1, f2)
    xs = rng.uniform(0, 1, (npts, f.dimension()))
    xs[0], xs[1] = 0.0, 1.0
    y1, y2 = oracle_eval(po, f1, xs), oracle_eval(po, f2, xs)
    _same_with_infinities(q.evaluate(f, xs), y1 + y2)
    cores = [c.copy() for c in f.cores]
    cores[0][(slice(None), slice(None)) + (slice(0, 3),) * len(f.topo.children[0])] = 0.0
    f.set_cores(cores)
    assert np.max(np.abs(q.evaluate(f, xs) / y2 - 1.0)) < TOL


@pytest.mark.parametrize("bond,npts", [(1, 3), (5, 4), (5, 3000), (16, 300), (20, 9), (33, 2000)])
def test_gradient_infinite_weight(q, po, eng, rng, bond, npts):
    # one sample with an infinite weight: the entries that its digits select are
    # infinite, all others are the gradient of the other samples
    L = 11
    f = _overflowing(q, _chain(q, L, bond), bond, rng, 1.0)
    f.set_cores([np.abs(c) for c in f.cores])
    xs, yb = rng.uniform(0, 1, (npts, 1)), rng.uniform(0.5, 1.5, npts)
    t = f.topo
    j = npts // 2
    rest = np.arange(npts) != j
    ref = po.eval_grad(t.parent, t.sdim, f.cores, t.vcoord, t.vdigit, t.Lc, xs[rest], yb[rest])
    yb[j] = np.inf
    for v, (g, r) in enumerate(zip(q.eval_grad(f, xs, yb), ref)):
        d = int(xs[j, 0] * 2.0 ** t.vdigit[v]) & 1
        assert np.all(g[:, d] == np.inf)
        assert rel_l2(g[:, 1 - d], r[:, 1 - d]) < TOL


@pytest.mark.parametrize("bond", [3, 5, 16, 17, 40, 53])
@pytest.mark.parametrize("npts", [1, 7, 300, 5000])
def test_gradient_infinite_weight_signs(q, po, eng, rng, bond, npts):
    # cores of both signs: a weight is the last factor of its sample's term, so one
    # infinite weight gives infinities of the term's sign and no NaN
    f = q.random_itn(_chain(q, 13, 2), link_space=bond, rng=rng)
    xs, yb = rng.uniform(0, 1, (npts, 1)), rng.uniform(-1.5, 1.5, npts)
    yb[npts // 2] = -np.inf
    t = f.topo
    ref = po.eval_grad(t.parent, t.sdim, f.cores, t.vcoord, t.vdigit, t.Lc, xs, yb)
    for g, r in zip(q.eval_grad(f, xs, yb), ref):
        inf = np.isinf(r)
        assert inf.any() and not np.isnan(r).any()
        assert np.array_equal(g[inf], r[inf])
        if not inf.all():
            assert rel_l2(g[~inf], r[~inf]) < TOL
    # the calls after it are what they were
    yb[npts // 2] = 0.5
    ref = po.eval_grad(t.parent, t.sdim, f.cores, t.vcoord, t.vdigit, t.Lc, xs, yb)
    for g, r in zip(q.eval_grad(f, xs, yb), ref):
        assert rel_l2(g, r) < TOL


# ------------------------------------------------------------------ NaN
@pytest.mark.parametrize("bond,cutoff,maxdim", [(6, 1e-10, 1 << 30), (24, 1e-10, 20), (40, 0.0, 16), (80, 1e-8, 64),
                                                (110, 0.0, 60)])
@pytest.mark.parametrize("where", ["first", "middle", "last"])
def test_truncate_nan(q, eng, rng, bond, cutoff, maxdim, where):
    # a network with a NaN entry: rows whose norm is NaN still have a place in the
    # order of the singular values (moves in LDS, on the global workspace, with
    # helper workgroups); the calls after it are what they were
    s = _chain(q, 13, bond)
    good = q.random_itn(s, link_space=bond, rng=rng)
    op = q.second_derivative_operator(s)
    def values():
        g = q.truncate(good, cutoff=cutoff, maxdim=maxdim)
        return q.evaluate(g, np.linspace(0, 1, 50)[:, None]), g.bonds()
    before = values()
    cores = [c.copy() for c in good.cores]
    v = {"first": 0, "middle": 6, "last": 12}[where]
    cores[v].reshape(-1)[cores[v].size // 2] = np.nan
    bad = q.ITensorNetworkFunction(s, cores)
    for g in (q.truncate(bad, cutoff=cutoff, maxdim=maxdim), q.operate(op, bad, cutoff=cutoff, maxdim=maxdim)):
        b = g.bonds()
        assert np.all(b >= 1) and np.all(b <= min(maxdim, 64))
        assert np.isnan(q.integrate(g))
    after = values()
    assert np.array_equal(before[0], after[0]) and np.array_equal(before[1], after[1])


# ------------------------------------------------------------------ very many vertices
@pytest.mark.parametrize("extra,bond,maxdim", [(1300, 128, 128), (17000, 48, 20), (19500, 24, 10)])
def test_truncate_very_many_vertices(q, po, eng, rng, extra, bond, maxdim):
    # the vertices' bonds take the LDS that moves beyond it use otherwise: no room
    # for the blocked path (with a product that helper workgroups share), then none
    # for the tiles of a gather either
    nd = 16
    g = q.named_grid((extra + nd, 1))
    f0 = [(extra + i, 1) for i in range(1, nd + 1)]
    s = q.continuous_siteinds(g, [f0])
    cap = [1] * (extra + 1) + [min(bond, 2 ** min(j, nd - j)) for j in range(1, nd)] + [1]
    cores = [np.ones((1, 1, 1)) for _ in range(extra)]
    for j in range(nd):
        a, b = cap[extra + j], cap[extra + j + 1]
        shape = (a, 2, b) if j + 1 < nd else (a, 2)
        cores.append(rng.standard_normal(shape) * (0.8 ** np.arange(a)).reshape((-1,) + (1,) * (len(shape) - 1)))
    f = q.ITensorNetworkFunction(s, cores)
    t = f.topo
    for cutoff in (0.0, 1e-10):
        got = q.truncate(f, cutoff=cutoff, maxdim=maxdim)
        ref, err = po.truncate(t.parent, t.sdim, f.cores, cutoff, maxdim)
        assert np.array_equal(got.bonds(), [c.shape[0] for c in ref])
        xs = rng.uniform(0, 1, (200, 1))
        yr = po.evaluate(t.parent, t.sdim, ref, t.vcoord, t.vdigit, t.Lc, xs)[0]
        assert rel_l2(q.evaluate(got, xs), yr) < 1e-10


# ------------------------------------------------------------------ captured streams
@pytest.mark.parametrize("bond,npts,warm", [(5, 20000, 0), (5, 20000, 3), (16, 20000, 3), (16, 20000, 20000),
                                            (16, 40000, 3), (16, 40000, 40000), (31, 13000, 1), (32, 5, 0),
                                            (33, 700, 0), (33, 700, 700), (96, 300, 5), (160, 65, 65)])
def test_evaluate_captured(q, po, eng, rng, bond, npts, warm):
    # a captured evaluate, the network fresh or used with `warm` points before: the
    # capture makes nothing for the network, replays give the values of eager calls,
    # and so do the eager calls before the first replay
    import torch
    L = 30 if bond <= 32 else 12
    s = _chain(q, L, bond)
    f = q.random_itn(s, link_space=bond, rng=rng, std=1.0 / math.sqrt(bond))
    xs = rng.uniform(0, 1, (npts, 1))
    xd = torch.tensor(xs, device="cuda")
    out = torch.zeros(npts, dtype=torch.float64, device="cuda")
    if warm:
        q.evaluate(f, xd[:warm].contiguous())
    else:
        q.api.device_network(f)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        q.evaluate(f, xd, out=out)
    y = q.evaluate(f, xd)
    eng.sync()
    assert rel_l2(y.cpu().numpy(), oracle_eval(po, f, xs)) < TOL
    for r in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert rel_l2(out.cpu().numpy(), y.cpu().numpy()) < TOL
        assert torch.equal(q.evaluate(f, xd), y)
        xd.copy_(torch.flip(xd, (0,)))  # other points in the same buffer
        y = q.evaluate(f, xd)
        eng.sync()


def test_evaluate_tree_captured_refused(q, po, eng, rng):
    # a tree needs its plan made: refused on a captured stream, without harm to the
    # calls after it
    import torch
    f = q.random_itn(_comb(q, 3, 4), link_space=5, rng=rng)
    xs = rng.uniform(0, 1, (50, 3))
    xd = torch.tensor(xs, device="cuda")
    q.evaluate(f, xd)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    other = torch.zeros(8, device="cuda")
    with torch.cuda.graph(graph):
        other += 1.0
        with pytest.raises(q.api._capi.EngineError):
            q.evaluate(f, xd)
    graph.replay()
    torch.cuda.synchronize()
    assert float(other.sum()) == 8.0
    assert rel_l2(q.evaluate(f, xd).cpu().numpy(), oracle_eval(po, f, xs)) < TOL


# ------------------------------------------------------------------ calls of changing size, streams, contexts
@pytest.mark.parametrize("kind", ["wide", "comb"])
def test_tables_serve_other_sizes(q, po, eng, rng, kind):
    # point counts up and down on one network, evaluate and gradient: the same bits as
    # a fresh network's first call of that size
    s = _chain(q, 18, 40) if kind == "wide" else _comb(q, 3, 9)
    f = q.random_itn(s, link_space=40 if kind == "wide" else 9, rng=rng, std=0.3)
    xs = rng.uniform(0, 1, (70000, f.dimension()))
    yb = rng.standard_normal(70000)
    def fresh():
        return q.ITensorNetworkFunction(s, f.cores)
    for n in (300, 70000, 1, 9, 70000, 2000, 300):
        assert np.array_equal(q.evaluate(f, xs[:n]), q.evaluate(fresh(), xs[:n]))
        if kind == "wide" and n in (300, 2000):
            g = q.eval_grad(f, xs[:n], yb[:n])
            assert all(np.array_equal(a, b) for a, b in zip(g, q.eval_grad(fresh(), xs[:n], yb[:n])))
    assert rel_l2(q.evaluate(f, xs[:500]), oracle_eval(po, f, xs[:500])) < TOL
    # and after the cores changed
    h = q.truncate(f, cutoff=0.0, maxdim=6)
    for n in (2000, 10, 2000):
        assert rel_l2(q.evaluate(h, xs[:n]), oracle_eval(po, h, xs[:n])) < TOL


@pytest.mark.parametrize("kind", ["wide", "comb"])
def test_tree_evaluate_on_streams(q, po, eng, rng, kind):
    # one network used on two streams and through a second context, nothing waited for
    # in between: what the first call makes is there for the second, and the scratch
    # that both use is taken in turn
    import ctypes
    import torch
    s = _chain(q, 20, 40) if kind == "wide" else _comb(q, 3, 10)
    bond = 150 if kind == "wide" else 40
    n = 30000
    xs = rng.uniform(0, 1, (n, 1 if kind == "wide" else 3))
    xd = torch.tensor(xs, device="cuda")
    other = q.api._capi.Context(0)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for rep in range(3):
        f = q.random_itn(s, link_space=bond, rng=rng, std=1.0 / math.sqrt(bond))
        g = q.random_itn(s, link_space=bond, rng=rng, std=1.0 / math.sqrt(bond))
        dn = q.api.device_network(f)
        q.api.device_network(g)
        out = [torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(4)]
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            q.evaluate(f, xd, out=out[0])
        with torch.cuda.stream(b):
            q.evaluate(f, xd, out=out[1])
            q.evaluate(g, xd, out=out[2])
        other.check(q.api._capi.lib().qtt_eval(other.handle, dn.handle, ctypes.c_void_p(xd.data_ptr()), n,
                                               ctypes.c_void_p(out[3].data_ptr()), 0))
        other.sync()
        torch.cuda.synchronize()
        yf, yg = oracle_eval(po, f, xs[:300]), oracle_eval(po, g, xs[:300])
        assert rel_l2(out[0][:300].cpu().numpy(), yf) < TOL
        assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[3])
        assert rel_l2(out[2][:300].cpu().numpy(), yg) < TOL
    other.close()


# ------------------------------------------------------------------ more points than one pass takes
@pytest.mark.parametrize("nc", [1, 3])
def test_evaluate_in_passes(q, po, eng, rng, nc):
    # more point rows than the scratch holds at once: 40 sites of bond 160 are some
    # 2200 doubles per point beyond the tables, so a pass takes 30 thousand points; the
    # backbone of a comb of bond 64 is 192, 350 thousand points
    s = _chain(q, 40, 160) if nc == 1 else _comb(q, 3, 14)
    f = q.random_itn(s, link_space=160 if nc == 1 else 64, rng=rng, std=0.1)
    n = 45007 if nc == 1 else 400003
    xs = rng.uniform(0, 1, (n, nc))
    y = q.evaluate(f, xs)
    sel = np.concatenate([np.arange(0, n, n // 200), [n - 1]])
    assert rel_l2(y[sel], oracle_eval(po, f, np.ascontiguousarray(xs[sel]))) < TOL


@pytest.mark.parametrize("bond,L,n", [(53, 50, 30011), (20, 60, 60001)])
def test_gradient_in_passes(q, po, eng, rng, bond, L, n):
    # several passes of points add into the cores' gradient: against the sum of the
    # gradients of pieces that one pass takes
    f = q.random_itn(_chain(q, L, bond), link_space=bond, rng=rng, std=1.0 / math.sqrt(bond))
    xs, yb = rng.uniform(0, 1, (n, 1)), rng.standard_normal(n)
    g = q.eval_grad(f, xs, yb)
    parts = [q.eval_grad(f, xs[i:i + 5000], yb[i:i + 5000]) for i in range(0, n, 5000)]
    for v, a in enumerate(g):
        assert rel_l2(a, sum(p[v] for p in parts)) < TOL
    t = f.topo
    ref = po.eval_grad(t.parent, t.sdim, f.cores, t.vcoord, t.vdigit, t.Lc, xs[:300], yb[:300])
    assert all(rel_l2(a, b) < TOL for a, b in zip(q.eval_grad(f, xs[:300], yb[:300]), ref))


# ------------------------------------------------------------------ singular values around the cutoff's level
def _level_matrix(n, b, cut, seed):
    """n x b with singular values 1, two between, and the others within a factor of
    some 3 of the level below which rows are not rotated against each other."""
    rng = np.random.default_rng(seed)
    k = min(n, b)
    lev = np.sqrt(cut / k)
    S = np.concatenate([[1.0], 0.1 ** rng.uniform(0.3, 3, 2), lev * np.exp(rng.uniform(np.log(0.2), np.log(3), k - 3))])
    U = np.linalg.qr(rng.standard_normal((n, k)))[0]
    V = np.linalg.qr(rng.standard_normal((b, k)))[0]
    return (U * S) @ V.T, S


# (moves of one wavefront, in LDS, preconditioned, tall, on the global workspace,
# with helper workgroups; seeds that do not converge while the rule holds)
@pytest.mark.parametrize("n,b,seed", [(12, 24, 25), (12, 24, 31), (20, 40, 2), (20, 40, 19), (32, 64, 4), (32, 64, 17),
                                      (34, 30, 18), (64, 96, 0), (64, 96, 9), (110, 140, 0), (150, 260, 0),
                                      (200, 260, 1)])
def test_truncate_values_at_noise_level(q, po, eng, n, b, seed):
    import ctypes
    from types import SimpleNamespace
    cut = 1e-8
    M, S = _level_matrix(n, b, cut, seed)
    topo = SimpleNamespace(nv=2, parent=np.array([-1, 0]), sdim=np.array([b, n]), vcoord=np.array([-1, -1]),
                           vdigit=np.array([0, 0]), Lc=np.zeros(0), ncoord=0,
                           core_shape=lambda v, bond: (1, b, int(bond[1])) if v == 0 else (int(bond[1]), n))
    cores = [np.eye(b).reshape(1, b, b), np.ascontiguousarray(M.T)]
    capi = q.api._capi
    net = capi.DeviceNetwork.upload(eng, topo, cores)
    err = ctypes.c_double()
    eng.check(capi.lib().qtt_truncate(eng.handle, net.handle, cut, 1 << 40, ctypes.byref(err)))
    c0, c1 = net.download()
    s2 = np.sort(S ** 2)
    drop = int(np.sum(np.cumsum(s2) <= cut * s2.sum()))
    assert c1.shape[0] == len(S) - drop
    lost = s2[:drop].sum()
    assert abs(err.value - lost / s2.sum()) <= 1e-6 * lost / s2.sum()
    assert abs(np.sum((c0[0] @ c1 - M.T) ** 2) - lost) <= 1e-6 * lost
    # the oracle as well
    ref, e = po.truncate(topo.parent, topo.sdim, cores, cut, 1 << 40)
    assert ref[1].shape[0] == c1.shape[0] and abs(e - err.value) <= 1e-6 * err.value


# ------------------------------------------------------------------ table sizes of large calls
@pytest.mark.parametrize("bond,n", [(11, (1 << 21) - 1), (11, 1 << 21), (9, (1 << 21) + 333), (8, 1 << 18),
                                    (3, (1 << 19) - 1), (8, 1 << 20), (7, 1 << 21), (20, 1 << 18), (21, 1 << 18)])
def test_evaluate_table_sizes(q, po, eng, rng, bond, n):
    # the default table size changes with the points; larger and smaller calls in turn
    import torch
    f = q.random_itn(_chain(q, 17, bond, dims=2), link_space=bond, rng=rng, std=1.0 / math.sqrt(bond))
    xd = torch.rand(n, 2, dtype=torch.float64, device="cuda")
    for m in (n, 40000, n):
        y = q.evaluate(f, xd[:m]).cpu().numpy()
        sel = np.concatenate([np.arange(0, m, m // 500), [m - 1]])
        assert rel_l2(y[sel], oracle_eval(po, f, xd.cpu().numpy()[sel])) < TOL


@pytest.mark.parametrize("bond,npts", [(1, 1), (2, 50), (3, 12288), (4, 12289), (4, 7)])
def test_few_points_small_bonds_repeated(q, po, eng, rng, bond, npts):
    # up to bond 4 a network's first call of few points reads the cores, the next ones
    # the packed copy: the same bits, also after the cores changed
    f = q.random_itn(_chain(q, 12, bond), link_space=bond, rng=rng)
    xs = rng.uniform(0, 1, (npts, 1))
    y = q.evaluate(f, xs)
    assert rel_l2(y, oracle_eval(po, f, xs)) < TOL
    assert all(np.array_equal(q.evaluate(f, xs), y) for _ in range(3))
    g = q.truncate(f, cutoff=0.0, maxdim=max(1, bond - 1))
    z = q.evaluate(g, xs)
    assert rel_l2(z, oracle_eval(po, g, xs)) < TOL
    assert np.array_equal(q.evaluate(g, xs), z)


# ------------------------------------------------------------------ tall and wide moves of few columns or rows
@pytest.mark.parametrize("s0,b,s1", [(257, 1, 3), (300, 4, 5), (257, 15, 40), (257, 16, 40), (1000, 12, 12), (3, 300, 7),
                                     (4, 300, 300), (15, 15, 300), (16, 16, 300), (17, 17, 900), (300, 300, 2),
                                     (260, 260, 3), (700, 20, 600)])
@pytest.mark.parametrize("maxdim", [1 << 40, 3])
def test_truncate_thin_moves(q, eng, rng, s0, b, s1, maxdim):
    # two vertices, so that the moves' matrices are s0 x b (QR) and s1 x min(s0, b)
    # (SVD): around the lines at 256 rows and at 16 columns or 4 rows
    import ctypes
    from types import SimpleNamespace
    topo = SimpleNamespace(nv=2, parent=np.array([-1, 0]), sdim=np.array([s0, s1]), vcoord=np.array([-1, -1]),
                           vdigit=np.array([0, 0]), Lc=np.zeros(0), ncoord=0,
                           core_shape=lambda v, bond: (1, s0, int(bond[1])) if v == 0 else (int(bond[1]), s1))
    a, c = rng.standard_normal((s0, b)) * 0.8 ** np.arange(b), rng.standard_normal((b, s1))
    capi = q.api._capi
    net = capi.DeviceNetwork.upload(eng, topo, [a.reshape(1, s0, b), c])
    err = ctypes.c_double()
    eng.check(capi.lib().qtt_truncate(eng.handle, net.handle, 0.0, maxdim, ctypes.byref(err)))
    c0, c1 = net.download()
    m = min(s0, b, s1, maxdim)
    assert c1.shape[0] == m
    M = a @ c
    U, S, V = np.linalg.svd(M, full_matrices=False)
    assert np.linalg.norm(c0[0] @ c1 - (U[:, :m] * S[:m]) @ V[:m]) < 1e-11 * np.linalg.norm(M)
    lost = np.sum(S[m:] ** 2) / np.sum(S ** 2)
    assert abs(err.value - lost) <= 1e-11


# ------------------------------------------------------------------ small gradients and inner products
@pytest.mark.parametrize("bond", [1, 2, 3, 8, 9, 16])
@pytest.mark.parametrize("dims,L,npts", [(1, 4, 1), (1, 4, 255), (2, 4, 256), (3, 3, 257), (2, 12, 64), (1, 16, 65),
                                         (2, 20, 700)])
def test_gradient_small(q, po, eng, rng, bond, dims, L, npts):
    # a lane per point (small calls) and rows of digit strings, on both sides of the
    # line between them, with tiles that the points do not fill
    f = q.random_itn(_chain(q, L, bond, dims), link_space=bond, rng=rng, std=1.0 / math.sqrt(bond))
    xs, yb = rng.uniform(0, 1, (npts, dims)), rng.standard_normal(npts)
    xs[0] = 1.0
    t = f.topo
    ref = po.eval_grad(t.parent, t.sdim, f.cores, t.vcoord, t.vdigit, t.Lc, xs, yb)
    g = q.eval_grad(f, xs, yb)
    num = math.sqrt(sum(np.sum((a - b) ** 2) for a, b in zip(g, ref)))
    assert num <= TOL * math.sqrt(sum(np.sum(b ** 2) for b in ref))
    assert all(np.array_equal(a, b) for a, b in zip(g, q.eval_grad(f, xs, yb)))


@pytest.mark.parametrize("kind,ba,bb", [("chain", 1, 1), ("chain", 2, 3), ("chain", 8, 7), ("chain", 11, 9),
                                        ("chain", 12, 12), ("comb", 2, 2), ("comb", 6, 4), ("comb", 4, 9), ("star", 2, 3),
                                        ("star", 4, 4), ("single", 1, 1)])
def test_inner_small(q, po, eng, rng, kind, ba, bb):
    # one workgroup (small networks) and a launch per height, around the line between them
    s = _chain(q, 1 if kind == "single" else 13, 2) if kind in ("chain", "single") else _tree(q, kind)
    f, g = (q.random_itn(s, link_space=b, rng=rng, std=1.0 / b) for b in (ba, bb))
    t = f.topo
    ref = po.inner(t.parent, t.sdim, f.cores, g.cores)
    na, nb = (po.inner(t.parent, t.sdim, h.cores, h.cores) for h in (f, g))
    assert abs(q.inner(f, g) - ref) <= TOL * math.sqrt(na * nb)
