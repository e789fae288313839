"""Performance cases of the quantics engine: what a program using it waits for.

Each case is one call (or one operate followed by an evaluate of its result)
through the package's Python API or, where the API's host arrays would hide
the device path (the gradient), through the C entry point that takes device
pointers.  A truncated network is returned by its values at points and its
bond dimensions: its cores are fixed only up to a change of basis on every
bond.
"""
import ctypes
import math

import numpy as np
import torch

import __graft_entry__

q = __graft_entry__._load_package()


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one value on the host: a probe inside a solver's control loop
        {"name": "point_host", "kind": "evaluate", "layout": "chain", "dims": 2, "digits": 20, "bond": 16,
         "npts": 1, "precision": 0, "host": True},
        # a plot or a quadrature rule over a 2D field: many points, network resident
        {"name": "points_2d", "kind": "evaluate", "layout": "chain", "dims": 2, "digits": 20, "bond": 16,
         "npts": 1_000_000, "precision": 0, "host": False},
        # the same through the float32 hi/lo split option
        {"name": "points_2d_split", "kind": "evaluate", "layout": "chain", "dims": 2, "digits": 20, "bond": 15,
         "npts": 200_003, "precision": 1, "host": False},
        # a network before compression: bonds beyond the register kernels
        {"name": "points_wide", "kind": "evaluate", "layout": "chain", "dims": 1, "digits": 24, "bond": 96,
         "npts": 100_003, "precision": 0, "host": False},
        # a function on a comb tree (one tooth per coordinate)
        {"name": "points_comb", "kind": "evaluate", "layout": "comb", "dims": 3, "digits": 16, "bond": 32,
         "npts": 20_011, "precision": 0, "host": False},
        # the smallest differential operator call: second derivative of a 1D function
        {"name": "operate_1d", "kind": "operate", "layout": "chain", "dims": 1, "digits": 12, "terms": 1,
         "cutoff": 1e-12, "maxdim": 0, "npts": 100_000},
        # the 2D Laplacian, truncated, then looked at
        {"name": "operate_2d", "kind": "operate", "layout": "chain", "dims": 2, "digits": 20, "terms": 8,
         "cutoff": 1e-10, "maxdim": 128, "npts": 100_000},
        # d/dx of a dense comb of bond 128, recompressed: the largest single network
        {"name": "operate_comb", "kind": "operate_comb", "teeth": 3, "digits": 16, "bond": 128, "npts": 256},
        # one step of a batch of integral-equation solves at a bounded bond dimension
        {"name": "batch_fredholm", "kind": "batch", "nfun": 512, "digits_max": 24, "bond_max": 96, "maxdim": 32,
         "npts": 4096},
        # the gradient of a fit to 2^20 samples
        {"name": "gradient_2d", "kind": "gradient", "layout": "chain", "dims": 2, "digits": 14, "bond": 32,
         "npts": 1 << 20},
        # overlap of two functions on a comb
        {"name": "inner_comb", "kind": "inner", "layout": "comb", "dims": 3, "digits": 16, "bond": 64,
         "bond2": 48, "operator": False},
        # integral of a 45 MB comb
        {"name": "integral_comb", "kind": "integrate", "layout": "comb", "dims": 3, "digits": 16, "bond": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "chain", "wide", "split", "tree", "operate", "operate_comb", "batch", "gradient",
                       "gradient_comb", "inner", "integrate"])
    if kind == "host":
        return {"kind": "evaluate", "layout": "chain", "dims": rng.randint(1, 3), "digits": rng.randint(6, 13),
                "bond": rng.randint(2, 32), "npts": _log(rng, 1, 500), "precision": 0, "host": True}
    if kind in ("chain", "split"):
        d = rng.randint(1, 2)
        return {"kind": "evaluate", "layout": "chain", "dims": d, "digits": rng.randint(8, 40 // d),
                "bond": rng.randint(2, 32), "npts": _log(rng, 100, 1_000_000 if kind == "chain" else 200_000),
                "precision": 0 if kind == "chain" else rng.choice([1, 2]), "host": False}
    if kind == "wide":
        return {"kind": "evaluate", "layout": "chain", "dims": 1, "digits": rng.randint(8, 24),
                "bond": rng.randint(33, 128), "npts": _log(rng, 100, 100_000), "precision": 0, "host": False}
    if kind == "tree":
        return {"kind": "evaluate", "layout": "comb", "dims": rng.randint(2, 3), "digits": rng.randint(4, 16),
                "bond": rng.randint(2, 32), "npts": _log(rng, 1, 20_000), "precision": 0, "host": False}
    if kind == "operate":
        if rng.random() < 0.5:
            return {"kind": "operate", "layout": "chain", "dims": 1, "digits": rng.randint(8, 16), "terms": 1,
                    "cutoff": rng.choice([1e-10, 1e-12]), "maxdim": 0, "npts": _log(rng, 100, 100_000)}
        return {"kind": "operate", "layout": "chain", "dims": 2, "digits": rng.randint(8, 20),
                "terms": rng.randint(2, 8), "cutoff": 1e-10, "maxdim": 128, "npts": _log(rng, 100, 100_000)}
    if kind == "operate_comb":
        return {"kind": "operate_comb", "teeth": rng.randint(2, 3), "digits": rng.randint(6, 16),
                "bond": rng.randint(8, 112), "npts": _log(rng, 1, 256)}
    if kind == "batch":
        return {"kind": "batch", "nfun": _log(rng, 1, 256), "digits_max": rng.randint(10, 24),
                "bond_max": rng.randint(8, 96), "maxdim": rng.randint(16, 32), "npts": _log(rng, 100, 4096)}
    if kind == "gradient":
        d = rng.randint(1, 2)
        return {"kind": "gradient", "layout": "chain", "dims": d, "digits": rng.randint(8, 28 // d),
                "bond": rng.randint(2, 64 if rng.random() < 0.3 else 32), "npts": _log(rng, 100, 1 << 18)}
    if kind == "gradient_comb":
        return {"kind": "gradient", "layout": "comb", "dims": 2, "digits": rng.randint(4, 10),
                "bond": rng.randint(2, 12), "npts": _log(rng, 100, 20_000)}
    layout = rng.choice(["chain", "comb"])
    if kind == "inner":
        op = layout == "chain" and rng.random() < 0.5
        return {"kind": "inner", "layout": layout, "dims": 1 if op else rng.randint(1, 2) if layout == "chain" else 3,
                "digits": rng.randint(6, 16), "bond": rng.randint(4, 64), "bond2": rng.randint(4, 48),
                "operator": op}
    return {"kind": "integrate", "layout": layout, "dims": 2, "digits": rng.randint(6, 16),
            "bond": _log(rng, 2, 128)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _siteinds(case):
    if case.get("layout", "comb") == "chain":
        return q.continuous_siteinds(q.named_grid((case["dims"] * case["digits"], 1)), map_dimension=case["dims"])
    teeth, digits = case.get("dims", case.get("teeth")), case["digits"]
    return q.continuous_siteinds(q.named_comb_tree((teeth, digits)),
                                 [[(i, j) for j in range(1, digits + 1)] for i in range(1, teeth + 1)])


def _random_network(s, bond, rng):
    """Dense normal cores, each of unit norm times sqrt(its parent bond times
    its site): values stay of order one whatever the size."""
    f = q.random_itn(s, link_space=bond, rng=rng, normalize_cores=True)
    f.set_cores([c * math.sqrt(c.shape[0] * c.shape[1]) for c in f.cores])
    return f


def _field_terms(case, rng):
    n = case["terms"]
    return rng.standard_normal(n), rng.uniform(1.0, 40.0, n), rng.uniform(0.0, 3.0, n)


def _field(s, case, rng):
    """1D: sin + cos + exp (bond 5); 2D: sum of separable sin(w x) exp(-b y)."""
    if case["dims"] == 1:
        w = 2 * math.pi * rng.uniform(0.5, 1.5)
        return (q.sin_itn(s, k=w), q.cos_itn(s, k=3 * w, c=0.5), q.exp_itn(s, k=-rng.uniform(0.5, 1.5)))
    a, w, b = _field_terms(case, rng)
    return tuple(q.builders.multiply_host(q.sin_itn(s, k=w[k], c=a[k], dim=1), q.exp_itn(s, k=-b[k], dim=2))
                 for k in range(len(a)))


def _points(case, rng, edges=False):
    """Uniform points; with edges the grid's boundary lines too, where a
    Dirichlet derivative has its largest values."""
    nd = case.get("dims", case.get("teeth", 1))
    xs = rng.uniform(0.0, 1.0, (case["npts"], nd))
    if edges:
        n = min(64, case["npts"])
        last = 1.0 - 2.0 ** -case["digits"]
        for c in range(nd):
            sel = xs[c * 2 * n:(c + 1) * 2 * n, c]
            sel[0::2] = 0.0
            sel[1::2] = last
    return xs


def _inputs(case, seed):
    """Networks and operators of a case, from its seed."""
    rng = np.random.default_rng([seed, 17])
    kind = case["kind"]
    if kind == "batch":
        ops, nets, xs = {}, [], []
        for _ in range(case["nfun"]):
            L = int(rng.integers(8, case["digits_max"] + 1))
            s = q.continuous_siteinds(q.named_grid((L, 1)))
            if L not in ops:
                ops[L] = q.fredholm_operator(s)
            chi = int(rng.integers(4, case["bond_max"] + 1))
            nets.append((ops[L], q.random_itn(s, link_space=chi, rng=rng)))
            xs.append(rng.uniform(0.0, 1.0, (case["npts"], 1)))
        return {"op": [o for o, _ in nets], "f": [f for _, f in nets], "xs": xs}
    s = _siteinds(case)
    if kind == "operate":
        f = None
        for t in _field(s, case, rng):
            f = t if f is None else q.builders.add_host(f, t)
        op = q.second_derivative_operator(s) if case["dims"] == 1 else q.laplacian_operator(s)
        return {"op": op, "f": f, "xs": _points(case, rng, edges=True)}
    if kind == "operate_comb":
        return {"op": q.first_derivative_operator(s, dim=1), "xs": _points(case, rng),
                "f": q.random_itn(s, link_space=case["bond"], rng=rng, normalize_cores=True)}
    if kind == "inner":
        op = q.second_derivative_operator(s) if case["operator"] else None
        return {"op": op, "f": _random_network(s, case["bond"], rng), "g": _random_network(s, case["bond2"], rng)}
    if kind == "integrate":
        return {"f": _random_network(s, case["bond"], rng)}
    st = {"f": _random_network(s, case["bond"], rng), "xs": _points(case, rng)}
    if kind == "gradient":  # residuals of a least-squares fit
        st["ybar"] = rng.standard_normal(case["npts"]) * (2.0 / case["npts"])
    return st


def prepare(case, seed):
    st = _inputs(case, seed)
    st["case"] = case
    fs = st["f"] if isinstance(st["f"], list) else [st["f"]]
    for f in fs + [st[k] for k in ("g",) if k in st]:
        q.api.device_network(f)
    ops = st.get("op") if isinstance(st.get("op"), list) else [st.get("op")]
    for op in ops:
        if op is not None:
            q.api.device_operator(op)
    if "xs" in st and not case.get("host"):
        xs = st["xs"]
        st["xs"] = [torch.tensor(x, device="cuda") for x in xs] if isinstance(xs, list) else \
            torch.tensor(xs, device="cuda")
    if "ybar" in st:
        st["ybar"] = torch.tensor(st["ybar"], device="cuda")
        st["grad"] = torch.empty(q.api.device_network(st["f"]).size(), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    f = state["f"]
    if kind == "evaluate":
        return q.evaluate(f, state["xs"], precision=case["precision"])
    if kind == "operate":
        g = q.operate(state["op"], f, cutoff=case["cutoff"], maxdim=case["maxdim"] or None)
        return q.evaluate(g, state["xs"]), g.bonds()
    if kind == "operate_comb":
        g = q.operate(state["op"], f, cutoff=0.0, maxdim=case["bond"])
        return q.evaluate(g, state["xs"]), g.bonds()
    if kind == "batch":
        # (the discarded weights it reports too are 1e-14 of the norm: round-off of the rest)
        _, _, integrals, values = q.operate_batch_pipeline(state["op"], f, state["xs"], maxdim=case["maxdim"])
        return {"integrals": integrals, "values": torch.stack(values)}
    if kind == "gradient":
        ctx = q.engine_context()
        ctx.check(q.api._capi.lib().qtt_eval_grad(
            ctx.handle, q.api.device_network(f).handle, ctypes.c_void_p(state["xs"].data_ptr()),
            ctypes.c_void_p(state["ybar"].data_ptr()), state["xs"].shape[0],
            ctypes.c_void_p(state["grad"].data_ptr()), 0))
        return state["grad"]
    if kind == "inner":
        return q.inner(f, state["g"], op=state["op"])
    return q.integrate(f)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _bonds(t, bond):
    b = np.full(t.nv, bond, dtype=np.int64)
    b[0] = 1
    return b


def _core_elems(t, b):
    return [int(b[v]) * int(t.sdim[v]) * int(np.prod([b[c] for c in t.children[v]], dtype=np.int64))
            for v in range(t.nv)]


def _chain_flops(b, npts):
    """Values of a chain at many points by the cheapest sharing: products of
    the first and last digits formed once per distinct value, the rest per
    point."""
    n = len(b)
    e = [int(x) for x in b] + [1]
    site = [2.0 * e[k] * e[k + 1] for k in range(n)]
    best = npts * sum(site)
    for tb in range(1, min(n // 2, 20) + 1):
        tables = sum(2.0 ** (k + 1) * (site[k] + site[n - 1 - k]) for k in range(tb))
        best = min(best, tables + npts * (sum(site[tb:n - tb]) + 2.0 * e[tb]))
    return best


def _tree_flops(t, b, npts):
    """Values on a comb: the teeth are chains shared by their digits, the
    backbone is contracted per point."""
    elems = _core_elems(t, b)
    total = 0.0
    for v in range(t.nv):
        kids = len(t.children[v])
        if kids > 1 or v == 0:
            total += npts * 2.0 * elems[v] / t.sdim[v]
        else:  # below the backbone: at most one value per distinct digit string
            depth, u = 0, v
            while t.children[u]:
                u = t.children[u][0]
                depth += 1
            total += min(npts, 2 ** (depth + 1)) * 2.0 * elems[v] / t.sdim[v]
    return total


def _sweep_flops(t, b, out_cap):
    """Householder QR of every product core toward a neighbour and the SVD of
    its triangle on the way back, with bonds at most what the digits allow."""
    sub = np.ones(t.nv)
    for v in range(t.nv - 1, -1, -1):
        sub[v] = t.sdim[v] * np.prod([sub[c] for c in t.children[v]])
    total = 2.0 ** min(60, t.nv)
    flops = 0.0
    for v in range(1, t.nv):
        rows = float(t.sdim[v] * np.prod([min(b[c], sub[c]) for c in t.children[v]]))
        cols = float(min(b[v], total / sub[v]))
        m, n = max(rows, cols), min(rows, cols)
        r = min(n, out_cap)
        flops += 2 * m * n * n - 2 * n ** 3 / 3 + 22.0 * r ** 3
    return flops


def work(case):
    kind = case["kind"]
    if kind == "batch":
        n, L, chi = case["nfun"], 0.5 * (8 + case["digits_max"]), 0.5 * (4 + case["bond_max"])
        core = 2 * chi * chi * L * 1.2
        s = q.continuous_siteinds(q.named_grid((int(L), 1)))
        t = q.Topology(s)
        fl = _sweep_flops(t, _bonds(t, int(3 * chi)), 16)
        return {"bytes": n * 8.0 * (core + case["npts"] * 2), "flops": n * (fl + 6 * core * 4)}
    t = q.Topology(_siteinds(case))
    if kind == "operate":
        chi = 5 if case["dims"] == 1 else 2 * case["terms"]
        w = 3 if case["dims"] == 1 else 5
        b = _bonds(t, chi)
        pts = case["npts"]
        fl = _sweep_flops(t, w * b, 15) + 4.0 * w * w * sum(_core_elems(t, b))
        return {"bytes": 8.0 * (2 * sum(_core_elems(t, b)) + pts * (case["dims"] + 1)),
                "flops": fl + _chain_flops(np.minimum(b, 15), pts)}
    b = _bonds(t, case["bond"])
    elems = sum(_core_elems(t, b))
    if kind == "operate_comb":
        wb = b.copy()
        tooth = [v for v in range(t.nv) if t.vcoord[v] == 0]
        wb[[v for v in tooth if v != 0]] *= 3
        return {"bytes": 8.0 * (2 * elems + case["npts"] * (case["teeth"] + 1)),
                "flops": _sweep_flops(t, wb, case["bond"]) + _tree_flops(t, b, case["npts"])}
    if kind == "integrate":
        return {"bytes": 8.0 * elems, "flops": 2.0 * elems}
    if kind == "inner":
        b2 = _bonds(t, case["bond2"])
        fl = 0.0
        for v in range(t.nv):
            ax = 2.0 * b2[v] * t.sdim[v]
            kids = t.children[v]
            rest = float(np.prod([b2[c] for c in kids]))
            for c in kids:
                fl += ax * rest * b[c]
                rest = rest / b2[c] * b[c]
            fl += ax * rest * b[v]
        return {"bytes": 8.0 * (elems + sum(_core_elems(t, b2))), "flops": fl}
    pts, nd = case["npts"], case["dims"]
    fl = _chain_flops(b, pts) if case["layout"] == "chain" else _tree_flops(t, b, pts)
    if kind == "gradient":
        return {"bytes": 8.0 * (2 * elems + pts * (nd + 1)), "flops": 3 * fl}
    return {"bytes": 8.0 * (elems + pts * (nd + 1)), "flops": fl}


# ---------------------------------------------------------------------------
# the same outputs from plain torch and numpy in 64 bits
# ---------------------------------------------------------------------------
_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _digits(t, xs):
    """[nv][npts] digit values: bit (msb first) of floor(x 2^L), saturated at x >= 1."""
    out = np.zeros((t.nv, xs.shape[0]), dtype=np.int64)
    for v in range(t.nv):
        c = int(t.vcoord[v])
        if c >= 0:
            L = int(t.Lc[c])
            k = np.minimum(np.floor(np.ldexp(xs[:, c], L)), 2.0 ** L - 1).astype(np.int64)
            out[v] = (k >> (L - int(t.vdigit[v]))) & 1
    return out


def _gpu(a):
    return torch.tensor(np.ascontiguousarray(a), device=_DEV)


def _subtrees(t, cores, dig, keep=False):
    """Vectors over every parent bond, per point (children before parents)."""
    vec = [None] * t.nv
    for v in range(t.nv - 1, -1, -1):
        A = cores[v]
        n = dig.shape[1]
        out = torch.zeros((n, A.shape[0]), dtype=torch.float64, device=_DEV)
        for d in range(A.shape[1]):
            sel = torch.nonzero(dig[v] == d).reshape(-1)
            for part in torch.split(sel, max(1, (1 << 26) // max(1, A[:, d].numel() // max(1, A.shape[-1])))):
                T = A[:, d].unsqueeze(0)
                first = True
                for c in reversed(t.children[v]):
                    x = vec[c][part]
                    if first:
                        flat = A[:, d].reshape(-1, A.shape[-1]).contiguous()
                        T = (x @ flat.t().contiguous()).reshape((len(part),) + tuple(A[:, d].shape[:-1]))
                        first = False
                    else:
                        sh = (len(part),) + (1,) * (T.dim() - 2) + (x.shape[1],)
                        T = (T * x.reshape(sh)).sum(-1)
                out[part] = T.expand(len(part), A.shape[0]) if first else T
        vec[v] = out
        if not keep:
            for c in t.children[v]:
                vec[c] = None
    return vec


def _values(t, cores, xs):
    cores = [_gpu(c) for c in cores]
    res = []
    for i in range(0, xs.shape[0], 1 << 17):
        x = xs[i:i + (1 << 17)]
        res.append(_subtrees(t, cores, _gpu(_digits(t, x)))[0][:, 0].cpu().numpy())
    return np.concatenate(res)


def _gradient(t, cores, xs, ybar):
    cores = [_gpu(c) for c in cores]
    grads = [torch.zeros_like(c) for c in cores]
    for i in range(0, xs.shape[0], 1 << 16):
        x = xs[i:i + (1 << 16)]
        n = x.shape[0]
        dig = _gpu(_digits(t, x))
        up = _subtrees(t, cores, dig, keep=True)
        env = [None] * t.nv
        env[0] = _gpu(ybar[i:i + (1 << 16)]).reshape(n, 1)
        for v in range(t.nv):
            A, kids = cores[v], t.children[v]
            e = env[v]
            outer = torch.ones((n, 1), dtype=torch.float64, device=_DEV)
            for c in kids:
                outer = (outer.unsqueeze(2) * up[c].unsqueeze(1)).reshape(n, -1)
                env[c] = torch.zeros((n, A.shape[2 + kids.index(c)]), dtype=torch.float64, device=_DEV)
            for d in range(A.shape[1]):
                sel = torch.nonzero(dig[v] == d).reshape(-1)
                if not len(sel):
                    continue
                es = e[sel]
                grads[v][:, d] += (es.t().contiguous() @ outer[sel]).reshape(A[:, d].shape)
                if not kids:
                    continue
                E = (es @ A[:, d].reshape(A.shape[0], -1)).reshape((len(sel),) + tuple(A.shape[2:]))
                for k, c in enumerate(kids):
                    T = E
                    for j in range(len(kids) - 1, -1, -1):
                        if j != k:
                            sh = [len(sel)] + [1] * (T.dim() - 1)
                            sh[1 + j] = T.shape[1 + j]
                            T = (T * up[kids[j]][sel].reshape(sh)).sum(1 + j, keepdim=True)
                    env[c][sel] = T.reshape(len(sel), -1)
            env[v] = None
    return torch.cat([g.reshape(-1) for g in grads]).cpu().numpy()


def _product(t, W, f):
    """Exact operator product: O[p, si, so, c..] f[q, si, e..] -> [(p q), so, (c e)..]."""
    out = []
    for v in range(t.nv):
        m = len(t.children[v])
        la, lb = "abcd"[:m], "ijkl"[:m]
        C = np.einsum("Pst%s,Qs%s->PQt%s" % (la, lb, "".join(x + y for x, y in zip(la, lb))), W[v], f[v])
        sh = [W[v].shape[0] * f[v].shape[0], W[v].shape[2]] + \
            [W[v].shape[3 + k] * f[v].shape[2 + k] for k in range(m)]
        out.append(C.reshape(sh))
    return out


def _axis(t, x, u):
    return 0 if t.parent[x] == u else 2 + t.children[x].index(u)


def _move(t, cores, x, u, cut):
    """Orthogonalise x toward u; cut = (cutoff, maxdim) truncates the edge."""
    ax, au = _axis(t, x, u), _axis(t, u, x)
    M = np.moveaxis(cores[x], ax, -1)
    sh = M.shape
    M = M.reshape(-1, sh[-1])
    if cut is None:
        U, R = np.linalg.qr(M)
    else:
        U, S, Vh = np.linalg.svd(M, full_matrices=False)
        p = S * S
        tot, m, err = p.sum() or 1.0, len(p), 0.0
        while m > cut[1]:
            m -= 1
            err += p[m]
        while m > 1 and err + p[m - 1] <= cut[0] * tot:
            m -= 1
            err += p[m]
        U, R = U[:, :m], S[:m, None] * Vh[:m]
    cores[x] = np.moveaxis(U.reshape(sh[:-1] + (U.shape[1],)), -1, ax)
    cores[u] = np.moveaxis(np.tensordot(R, cores[u], (1, au)), 0, au)


def _truncated(t, cores, cutoff, maxdim):
    """The truncation sweep: every edge in post-order from vertex 0, the
    orthogonality centre moved to its lower vertex, the edge cut by the rule on
    squared singular values."""
    cores, post = list(cores), []

    def visit(v):
        for c in t.children[v]:
            visit(c)
        if v:
            post.append(v)
    visit(0)
    seen, order, via = {post[0]}, [post[0]], {}
    for v in order:
        for u in ([int(t.parent[v])] if v else []) + list(t.children[v]):
            if u not in seen:
                seen.add(u)
                via[u] = v
                order.append(u)
    for v in reversed(order[1:]):
        _move(t, cores, v, via[v], None)
    centre = post[0]
    for c in post:
        while centre != c:
            x = c
            while x != 0 and t.parent[x] != centre:
                x = int(t.parent[x])
            step = x if x != 0 else int(t.parent[centre])
            _move(t, cores, centre, step, None)
            centre = step
        _move(t, cores, c, int(t.parent[c]), (cutoff, maxdim))
        centre = int(t.parent[c])
    return cores


def _integral(t, cores):
    vec = [None] * t.nv
    for v in range(t.nv - 1, -1, -1):
        T = cores[v].sum(1) * (0.5 if cores[v].shape[1] == 2 else 1.0)
        for c in reversed(t.children[v]):
            T = T @ vec[c]
        vec[v] = T
    return float(vec[0][0])


def _overlap(t, a, b):
    E = [None] * t.nv
    for v in range(t.nv - 1, -1, -1):
        Y = b[v]
        for k, c in enumerate(t.children[v]):
            Y = np.moveaxis(np.tensordot(E[c], Y, (1, 2 + k)), 0, 2 + k)
        E[v] = a[v].reshape(a[v].shape[0], -1) @ Y.reshape(Y.shape[0], -1).T
    return float(E[0][0, 0])


def exact(case, seed):
    kind = case["kind"]
    w = work(case)
    if kind == "batch" and w["flops"] > 1e9:
        return None  # minutes of small factorizations on the host
    st = _inputs(case, seed)
    if kind == "batch":
        ints, vals = [], []
        for op, f, xs in zip(st["op"], st["f"], st["xs"]):
            cores = _truncated(f.topo, _product(f.topo, op.cores, f.cores), 0.0, case["maxdim"])
            ints.append(_integral(f.topo, cores))
            vals.append(_values(f.topo, cores, xs))
        return {"integrals": np.array(ints), "values": np.stack(vals)}
    f = st["f"]
    t, cores = f.topo, f.cores
    if kind == "evaluate":
        y = _values(t, cores, st["xs"])
        return y
    if kind in ("operate", "operate_comb"):
        cut = (case["cutoff"], case["maxdim"] or 1 << 40) if kind == "operate" else (0.0, case["bond"])
        g = _truncated(t, _product(t, st["op"].cores, cores), *cut)
        return _values(t, g, st["xs"]), np.array([c.shape[0] for c in g], dtype=np.int64)
    if kind == "gradient":
        return _gradient(t, cores, st["xs"], st["ybar"])
    if kind == "inner":
        b = st["g"].cores if st["op"] is None else _product(t, st["op"].cores, st["g"].cores)
        return _overlap(t, cores, b)
    return _integral(t, cores)
