"""Performance cases: the work a user's program has this package do, over its range of sizes.

A case is a dict of plain values; ``prepare`` makes the context (operator, tile plan) and the
device vectors a program holds before the call, ``run`` makes one call sequence through
``pned_amd.gpu``, ``exact`` states the same results in 64-bit torch without this package.

kind     what a program does with it
hv       one H.v, p_mltply_v3 (v0 += H v1 with <v1|H|v1>): the call every Krylov method makes
         (complex64: with the mTPQ operator L - H in the place of H)
lanczos  lnc1 for a fixed number of steps from a normalised vector: ground-state runs
sector   the same in a fixed-S^z basis (the Heisenberg point, which conserves S^z)
batch    lanczos_batch_steps with one operator per column: what a serving pool runs between two
         convergence checks
tps      fused mTPQ on R interleaved random vectors, launch by launch or from a captured graph
dsf      S^z(q) excitation, DSF Lanczos, continued fraction on 2000 frequencies, and the
         shifted solve (H - e0 + i eta) x = b that cross-checks it
"""
import math

import numpy as np
import torch

# L1 x L2 honeycomb tori, N = 2 L1 L2 sites
_A1 = np.array([0.5, 0.5 / math.sqrt(3.0)])
_A2 = np.array([0.5, -0.5 / math.sqrt(3.0)])
_A3 = np.array([0.0, 1.0 / math.sqrt(3.0)])


def listed():
    return [
        # the smallest call: a 2x3 cluster, where launches and the host round trip are the cost
        {"name": "hv-12", "kind": "hv", "l1": 2, "l2": 3, "q": 2, "phi": 126.0, "field": 0.1, "cols": 1, "dtype": "c128"},
        # the ordinary single-vector product: 24 sites in a [111] field
        {"name": "hv-24", "kind": "hv", "l1": 3, "l2": 4, "q": 2, "phi": 126.0, "field": 0.1, "cols": 1, "dtype": "c128"},
        # complex64 storage at 28 sites: the mTPQ operator L - H, which is what runs in complex64
        {"name": "hv-28-c64", "kind": "hv", "l1": 2, "l2": 7, "q": 2, "phi": 54.0, "field": 0.0, "cols": 1, "dtype": "c64"},
        # the largest: 30 sites in a field, 16 GiB a vector
        {"name": "hv-30", "kind": "hv", "l1": 3, "l2": 5, "q": 2, "phi": 126.0, "field": 0.1, "cols": 1, "dtype": "c128"},
        # spin 1, 16 sites (3^16 states)
        {"name": "hv-spin1-16", "kind": "hv", "l1": 2, "l2": 4, "q": 3, "phi": 108.0, "field": 0.0, "cols": 1, "dtype": "c128"},
        # a small ground-state run: launch bound
        {"name": "lanczos-16", "kind": "lanczos", "l1": 2, "l2": 4, "q": 2, "phi": 126.0, "field": 0.1, "dtype": "c128", "steps": 40},
        # the 24-site ground-state run
        {"name": "lanczos-24", "kind": "lanczos", "l1": 3, "l2": 4, "q": 2, "phi": 54.0, "field": 0.0, "dtype": "c128", "steps": 40},
        # the S^z = 0 sector of 24 sites (2704156 states: a ragged length)
        {"name": "sector-24", "kind": "sector", "l1": 3, "l2": 4, "down": 12, "phi": 180.0, "steps": 20},
        # a serving pool of eight 20-site requests between two convergence checks
        {"name": "batch-20x8", "kind": "batch", "l1": 2, "l2": 5, "phi": 200.0, "field": 0.2, "cols": 8, "steps": 5},
        # small mTPQ ensemble from captured graphs
        {"name": "tps-16x8", "kind": "tps", "l1": 2, "l2": 4, "phi": 90.0, "cols": 8, "dtype": "c128", "steps": 31, "graph": True},
        # the 24-site ensemble of 64 samples in complex64
        {"name": "tps-24x64-c64", "kind": "tps", "l1": 3, "l2": 4, "phi": 90.0, "cols": 64, "dtype": "c64", "steps": 4, "graph": False},
        # spin-1 dynamics on 12 sites (3^12 states)
        {"name": "dsf-spin1-12", "kind": "dsf", "l1": 2, "l2": 3, "q": 3, "phi": 108.0, "steps": 28, "e0": -14.0, "eta": 1.0},
    ]


def draw(rng):
    phi = round(rng.uniform(0.0, 360.0), 2)
    field = round(rng.uniform(0.02, 0.5), 3) if rng.random() < 0.6 else 0.0
    kind = rng.choice(["hv", "hv", "hv", "spin", "lanczos", "lanczos", "sector", "batch", "tps", "tps", "dsf"])
    half = [(2, 2), (2, 3), (2, 4), (3, 3), (2, 5), (3, 4), (2, 7), (3, 5)]
    if kind == "hv":
        l1, l2 = rng.choice(half)
        n = 2 * l1 * l2
        cols = rng.choice([1, 1, 1, 2, 4, 16]) if n <= 20 else 1
        dtype = rng.choice(["c128", "c128", "c64"])
        return {"kind": "hv", "l1": l1, "l2": l2, "q": 2, "phi": phi, "field": field, "cols": cols, "dtype": dtype}
    if kind == "spin":
        q, l1, l2 = rng.choice([(3, 2, 2), (3, 2, 3), (3, 2, 4), (4, 2, 2), (4, 2, 3), (5, 2, 2), (6, 2, 2)])
        return {"kind": "hv", "l1": l1, "l2": l2, "q": q, "phi": phi, "field": field, "cols": 1, "dtype": "c128"}
    if kind == "lanczos":
        q, l1, l2 = rng.choice([(2, 2, 4), (2, 3, 3), (2, 2, 5), (2, 3, 4), (3, 2, 3)])
        return {"kind": "lanczos", "l1": l1, "l2": l2, "q": q, "phi": phi, "field": field, "dtype": "c128",
                "steps": rng.randint(18, 32)}
    if kind == "sector":
        l1, l2 = rng.choice([(2, 4), (3, 3), (2, 5), (3, 4)])
        return {"kind": "sector", "l1": l1, "l2": l2, "down": l1 * l2 - rng.randint(0, 3), "phi": rng.choice([0.0, 180.0]),
                "steps": rng.randint(10, 20)}
    if kind == "batch":
        l1, l2 = rng.choice([(2, 3), (2, 4), (3, 3), (2, 5)])
        return {"kind": "batch", "l1": l1, "l2": l2, "phi": phi, "field": round(rng.uniform(0.05, 0.5), 3),
                "cols": rng.choice([2, 4, 8, 8]), "steps": 5}
    if kind == "tps":
        l1, l2 = rng.choice([(2, 3), (2, 4), (3, 3), (2, 5), (3, 4)])
        n = 2 * l1 * l2
        cols = rng.choice([1, 2, 8, 32, 64]) if n <= 20 else rng.choice([4, 16])
        graph = n <= 18 and rng.random() < 0.6
        return {"kind": "tps", "l1": l1, "l2": l2, "phi": phi, "cols": cols, "dtype": rng.choice(["c64", "c64", "c128"]),
                "steps": 31 if graph else rng.randint(3, 8), "graph": graph}
    q, l1, l2 = rng.choice([(3, 2, 3), (2, 2, 4), (2, 3, 3)])
    return {"kind": "dsf", "l1": l1, "l2": l2, "q": q, "phi": rng.choice([54.0, 72.0, 108.0]), "steps": rng.randint(18, 28),
            "e0": -14.0 if q == 3 else -5.0, "eta": 1.0}


# ---- the model: sum over bonds of J S.S + 2 sin(phi) S^g S^g, J = cos(phi), and h (Sx + Sy + Sz) ----

def _bonds(l1, l2):
    """(site, site, spin component of the Kitaev term) of every bond, sites from 0."""
    out = []
    for j in range(l2):
        for i in range(l1):
            s = 2 * (j * l1 + i)
            out.append((s, s + 1, 0))
            out.append((s, 2 * (j * l1 + (i - 1) % l1) + 1, 1))
            out.append((s, 2 * (((j - 1) % l2) * l1 + i) + 1, 2))
    return out


def _sites(l1, l2):
    pos = []
    for j in range(l2):
        for i in range(l1):
            p = 0.5 * _A3 + (_A1 + _A2) * i + (_A1 + _A3) * j
            pos += [p, p + _A1]
    return np.array(pos)


def _momenta(l1, l2):
    b = 2.0 * math.pi * np.linalg.inv(np.array([_A1 + _A2, _A1 + _A3])).T
    return np.array([(m1 / l1) * b[0] + (m2 / l2) * b[1] for m2 in range(l2) for m1 in range(l1)])


def _spin(q):
    """Sx, Sy, Sz; digit d has m = d - S, for S = 1/2 bit 0 is up."""
    s = 0.5 * (q - 1)
    up = np.zeros((q, q), dtype=complex)
    for d in range(q - 1):
        m = d - s
        up[d + 1, d] = math.sqrt((s - m) * (s + m + 1.0))
    sz = np.diag(np.arange(q) - s).astype(complex)
    if q == 2:
        up, sz = up.T.copy(), -sz
    dn = up.conj().T
    return 0.5 * (up + dn), -0.5j * (up - dn), sz


def _bond_matrix(q, phi, g):
    s = _spin(q)
    c, k = math.cos(math.radians(phi)), 2.0 * math.sin(math.radians(phi))
    return sum((c + (k if a == g else 0.0)) * np.kron(s[a], s[a]) for a in range(3))


def _lb(case):
    """Per-bond shift of the mTPQ operator: 1.2 times the largest bond norm."""
    return 1.2 * max(float(np.linalg.norm(_bond_matrix(2, case["phi"], g), 2)) for g in range(3))


def _add(y, x, z):
    z = complex(z)
    if z != 0.0:
        y.add_(x, alpha=z.real if z.imag == 0.0 else z)


def _apply(case, x, n, q, phi, field):
    """H x for x of shape (q^n, columns)."""
    y = torch.zeros_like(x)
    r = x.shape[1]
    for a, b, g in _bonds(case["l1"], case["l2"]):
        lo, hi = min(a, b), max(a, b)
        shape = (q ** (n - 1 - hi), q, q ** (hi - lo - 1), q, q ** lo * r)
        xv, yv, m = x.view(shape), y.view(shape), _bond_matrix(q, phi, g)
        for o in range(q * q):
            for i in range(q * q):
                if abs(m[o, i]) > 1e-14:
                    _add(yv[:, o // q, :, o % q], xv[:, i // q, :, i % q], m[o, i])
    if field:
        f = field * sum(_spin(q))
        for a in range(n):
            xv, yv = x.view(q ** (n - 1 - a), q, q ** a * r), y.view(q ** (n - 1 - a), q, q ** a * r)
            for o in range(q):
                for i in range(q):
                    _add(yv[:, o], xv[:, i], f[o, i])
    return y


# ---- inputs ------------------------------------------------------------------------------

_TORCH = {"c128": torch.complex128, "c64": torch.complex64}


def _n(case):
    return 2 * case["l1"] * case["l2"]


def _random(dim, cols, dtype, seed):
    """Normalised Gaussian columns (dim, cols), as every Krylov run starts from."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.empty(dim, cols, dtype=dtype, device="cuda")
    torch.view_as_real(x).normal_(generator=gen)
    for c in range(cols):
        x[:, c] /= torch.linalg.vector_norm(x[:, c])
    return x


def _phis(case):
    return [(case["phi"] + 23.0 * c, case["field"] + 0.01 * c) for c in range(case["cols"])]


def _sector_dim(case):
    return math.comb(_n(case), case["down"])


class _Memory:
    """A device vector's memory, for torch."""

    def __init__(self, vec, dim, cols):
        self.vec = vec   # keeps the memory while a tensor uses it
        self.__cuda_array_interface__ = {"shape": (dim, cols), "typestr": "<c16" if vec.np_dtype == np.complex128 else "<c8",
                                         "data": (vec.data_ptr(), False), "version": 2}


def _tensor(ctx, vec, full):
    """The vector as a tensor in the order of the basis (a view; the context may keep its sites
    in another order in memory)."""
    t = torch.as_tensor(_Memory(vec, ctx.dim, vec.nvec), device="cuda")
    if not full:
        return t
    n, bit = ctx.n, ctx.layout()
    t = t.view([2] * n + [vec.nvec])
    return t.permute([n - 1 - int(bit[k]) for k in reversed(range(n))] + [n])


def prepare(case, seed):
    from pned_amd import gpu, lattice, model

    kind, n, q = case["kind"], _n(case), case.get("q", 2)
    cl = lattice.torus(case["l1"], case["l2"])
    dt = gpu.C64 if case.get("dtype") == "c64" else gpu.C128
    cols = case.get("cols", 1)
    if kind == "batch":
        ops = [model.build_operator(cl, 20, p, field=f) for p, f in _phis(case)]
        ctx = gpu.Context(ops[0], batch_ops=ops)
    elif kind == "tps":
        ctx = gpu.Context(model.build_operator(cl, 20, case["phi"], tps=True, tps_lb=_lb(case)))
        ctx.tps_set_observables(cl.site_vec, _momenta(case["l1"], case["l2"])[:5])
    elif kind == "hv" and dt == gpu.C64:
        ctx = gpu.Context(model.build_operator(cl, 20, case["phi"], field=case["field"], tps=True, tps_lb=_lb(case)))
    else:
        ctx = gpu.Context(model.build_operator(cl, 20, case["phi"], q=q, field=case.get("field", 0.0)))
    if kind == "sector":
        ctx.sz_sector(case["down"])
    full = q == 2 and kind != "sector"
    v = [ctx.vector(cols, dt) for _ in range({"tps": 4, "dsf": 7}.get(kind, 2))]
    t = [_tensor(ctx, u, full) for u in v]
    ctx.hv_fresh(v[0], v[1])   # builds the tile plan, which a program keeps
    x = _random(ctx.dim, cols, _TORCH[case.get("dtype", "c128")], 2 * seed)
    t[0].copy_(x.view(t[0].shape))
    if kind == "hv":
        t[1].copy_(_random(ctx.dim, cols, x.dtype, 2 * seed + 1).view(t[1].shape))
    del x
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    state = {"case": case, "ctx": ctx, "v": v, "t": t}
    if kind == "dsf":
        state["q"] = _momenta(case["l1"], case["l2"])[1]
        state["site_vec"] = cl.site_vec
    return state


def run(state):
    case, ctx, v, t = state["case"], state["ctx"], state["v"], state["t"]
    kind = case["kind"]
    if kind == "hv":
        pr = ctx.p_mltply_v3(v[0], v[1])
        return {"v0": t[1], "prdct": pr}
    if kind in ("lanczos", "sector"):
        itr, alpha, beta, ene = ctx.lnc1(v[0], v[1], fixed_steps=case["steps"], nvec=1)
        return {"alpha": alpha, "beta": beta, "ene": ene, "v1": t[0], "v0": t[1]}
    if kind == "batch":
        cols = case["cols"]
        a, b = ctx.lanczos_batch_steps(v[0], v[1], np.ones(cols, dtype=np.int32), np.zeros(cols), np.zeros(cols), case["steps"])
        return {"alpha": a, "beta": b, "v1": t[0], "v0": t[1]}
    if kind == "tps":
        v[1].copy_from(v[0])   # the start columns are kept; the run works in the other three
        a, b, c = ctx.tps_fused(v[1], v[2], v[3], _n(case) * 1.5 * _lb(case), case["steps"], graph_steps=0 if case["graph"] else None)
        return {"alpha": a, "beta": b, "coef": c}
    cnorm = ctx.intalv_zz(v[0], v[1], state["q"], state["site_vec"])
    v[2].copy_from(v[1])
    sa, sb = ctx.dsflnc1z(v[1], v[3], cnorm, case["steps"])
    w, dsf, conv = ctx.renbun(sa, sb, case["e0"], 0.1, 2000, 4.0 / 2000, sq=cnorm)
    ctx.cocg(case["e0"], case["eta"], v[2], v[3], v[4], v[5], v[6], tol=1e-11)
    return {"cnorm": cnorm, "alpha": sa, "beta": sb, "w": w, "dsf": dsf, "conv": conv, "x": t[3]}


# ---- what a pass cannot do without -------------------------------------------------------------

def work(case):
    kind, n, q = case["kind"], _n(case), case.get("q", 2)
    cols, size = case.get("cols", 1), 8 if case.get("dtype") == "c64" else 16
    elems = (_sector_dim(case) if kind == "sector" else q ** n) * cols
    # per element of an H.v: the diagonal, one real term a bond, one complex term a site in a field
    offdiag = 1 if q == 2 else 4
    hv = elems * (4 + 4 * offdiag * 3 * n // 2 + (8 * n if case.get("field") else 0))
    if kind == "hv":
        return {"bytes": 3 * size * elems, "flops": hv}
    if kind in ("lanczos", "sector"):
        return {"bytes": case["steps"] * 3 * size * elems, "flops": case["steps"] * (hv + 8 * elems)}
    if kind == "batch":
        return {"bytes": case["steps"] * 3 * size * elems, "flops": case["steps"] * (hv + 8 * elems)}
    if kind == "tps":
        return {"bytes": case["steps"] * 3 * size * elems, "flops": case["steps"] * (hv + 60 * elems)}
    # about 100 iterations of the shifted solve (p, x, r read and written, y kept) beside the Lanczos
    steps = case["steps"] - 1
    return {"bytes": (3 * steps + 6 * 100) * size * elems, "flops": (steps + 100) * (hv + 16 * elems)}


# ---- the same in 64 bits -----------------------------------------------------------------------

def _dots(x, y):
    return torch.stack([torch.vdot(x[:, c], y[:, c]) for c in range(x.shape[1])])


def _lanczos(h, v, steps):
    """alpha, beta of lnc1 and its loop vectors after the last step (v1, H v1 - beta v_prev)."""
    prev, alpha, beta = None, [], []
    for k in range(steps):
        w = h(v)
        if prev is not None:
            w -= beta[-1] * prev
        a = torch.vdot(v[:, 0], w[:, 0])
        b = torch.linalg.vector_norm(w - a * v).item()
        alpha.append(a.real.item())
        beta.append(b)
        if k + 1 < steps:
            prev, v = v, (w - a.real * v) / b
    return np.array(alpha), np.array(beta), v, w


def _exact_tps(case, x, n):
    lb, nb = _lb(case), 3 * n // 2
    lmax, shift = n * 1.5 * lb, nb * lb
    dim, steps, cols = x.shape[0], case["steps"], case["cols"]
    s = torch.arange(dim, device="cuda")
    site, mom = _sites(case["l1"], case["l2"]), _momenta(case["l1"], case["l2"])[:5]
    nsq = len(mom)
    zz = torch.zeros(dim, dtype=torch.float64, device="cuda")
    for a, b, g in _bonds(case["l1"], case["l2"]):
        if g == 2:   # the reference reads the bit one above each site's, and none past the last
            z1 = (s >> (a + 1) & 1) - 0.5 if a + 1 < n else -0.5
            z2 = (s >> (b + 1) & 1) - 0.5 if b + 1 < n else -0.5
            zz += z1 * z2
    b0 = s & 1
    weights = []
    for k in range(nsq):
        acc = torch.zeros(dim, dtype=torch.complex128, device="cuda")
        for j in range(n):
            bj = s >> j & 1
            wt = (bj.double() - 0.5) * (b0.double() - 0.5) if k % 4 < 2 else (bj ^ b0).double() * 0.25
            ph = float(mom[k // 4] @ site[j])
            acc += wt * complex(math.cos(ph), math.sin(ph))
        weights.append(acc)
    alpha, beta, coef = np.zeros((steps, cols)), np.zeros((steps, cols)), np.zeros((steps, cols, 7 + nsq))
    for c in range(cols):   # a column at a time: it fits beside the inputs
        u, up = x[:, c: c + 1].to(torch.complex128).contiguous(), None
        for i in range(1, steps + 1):
            w = shift * u - _apply(case, u, n, 2, case["phi"], 0.0)
            a1, b1 = torch.vdot(u[:, 0], w[:, 0]).real.item(), torch.linalg.vector_norm(w).item()
            row = coef[i - 1, c]
            row[:4] = 2 * i / a1, lmax, b1, lmax - a1
            g = torch.zeros_like(u) if up is None else up
            row[4] = (lmax * torch.vdot(g[:, 0], u[:, 0]) - torch.vdot(g[:, 0], w[:, 0])).real.item()
            zu = zz * u[:, 0]
            row[5], row[6] = torch.vdot(u[:, 0], zu).real.item(), torch.vdot(g[:, 0], zu).real.item()
            for k in range(nsq):
                row[7 + k] = torch.vdot((g if k % 2 else u)[:, 0], weights[k] * u[:, 0]).real.item()
            alpha[i - 1, c], beta[i - 1, c] = lmax - a1, b1
            up, u = u, w / b1
    return {"alpha": alpha, "beta": beta, "coef": coef}


def _exact_dsf(case, x, n, q):
    s = torch.arange(x.shape[0], device="cuda")
    site, mom = _sites(case["l1"], case["l2"]), _momenta(case["l1"], case["l2"])[1]
    f = torch.zeros(x.shape[0], dtype=torch.complex128, device="cuda")
    for j in range(n):
        ph = float(mom @ site[j])
        f += ((torch.div(s, q ** j, rounding_mode="floor") % q).double() - 0.5 * (q - 1)) * complex(math.cos(ph), math.sin(ph))
    b = f[:, None] * x
    nn = torch.linalg.vector_norm(b).item() ** 2
    b /= math.sqrt(nn)
    cnorm = nn / n

    def h(v):
        return _apply(case, v, n, q, case["phi"], 0.0)

    steps = case["steps"]
    alpha, bt, _, _ = _lanczos(h, b, steps - 1)
    beta = np.concatenate([[cnorm], bt])
    w = np.arange(2000) * (4.0 / 2000)
    z = w + case["e0"] + 0.1j
    cf = np.zeros(2000, dtype=complex)
    for m in reversed(range(steps - 1)):
        cf = -beta[m] ** 2 / (z - alpha[m] + cf)
    dsf = cf.imag
    dsf = cnorm / (0.5 * (4.0 / 2000) * (dsf[1:] + dsf[:-1]).sum()) * dsf
    # conjugate orthogonal conjugate gradients, well past the tolerance of the call
    xs, r, p = torch.zeros_like(b), b.clone(), b.clone()
    rho = (r * r).sum()
    for _ in range(5000):
        y = h(p) + (1j * case["eta"] - case["e0"]) * p
        al = rho / (p * y).sum()
        xs += al * p
        r -= al * y
        if torch.linalg.vector_norm(r).item() < 1e-14:
            break
        new = (r * r).sum()
        p = r + (new / rho) * p
        rho = new
    return {"cnorm": cnorm, "alpha": np.append(alpha, 0.0), "beta": np.append(beta, 0.0), "w": w, "dsf": dsf, "conv": None, "x": xs}


def exact(case, seed):
    kind, n, q = case["kind"], _n(case), case.get("q", 2)
    cols, dtype = case.get("cols", 1), _TORCH[case.get("dtype", "c128")]
    shape = [2] * n + [cols] if q == 2 and kind != "sector" else None

    def out(v):
        return v.view(shape) if shape else v

    x = _random(_sector_dim(case) if kind == "sector" else q ** n, cols, dtype, 2 * seed)
    if kind == "tps":
        return _exact_tps(case, x, n)
    x = x.to(torch.complex128)
    if kind == "hv":
        y = _apply(case, x, n, q, case["phi"], case["field"])
        if dtype == torch.complex64:
            y = y.neg_().add_(x, alpha=1.5 * n * _lb(case))
        pr = _dots(x, y).cpu().numpy()
        y += _random(q ** n, cols, dtype, 2 * seed + 1)
        return {"v0": out(y), "prdct": pr if cols > 1 else pr[0]}
    if kind == "dsf":
        return {k: (out(v) if k == "x" else v) for k, v in _exact_dsf(case, x, n, q).items()}
    if kind == "batch":
        res = [_lanczos(lambda v, p=p, f=f: _apply(case, v, n, 2, p, f), x[:, c: c + 1].contiguous(), case["steps"])
               for c, (p, f) in enumerate(_phis(case))]
        return {"alpha": np.stack([r[0] for r in res], 1), "beta": np.stack([r[1] for r in res], 1),
                "v1": out(torch.cat([r[2] for r in res], 1)), "v0": out(torch.cat([r[3] for r in res], 1))}
    if kind == "sector":
        s = torch.arange(2 ** n, device="cuda")
        pop = sum((s >> j & 1) for j in range(n))
        states = torch.nonzero(pop == case["down"])[:, 0]   # ascending, as the sector's basis

        def h(v):
            full = torch.zeros(2 ** n, 1, dtype=torch.complex128, device="cuda")
            full[states] = v
            return _apply(case, full, n, 2, case["phi"], 0.0)[states]
    else:
        def h(v):
            return _apply(case, v, n, q, case["phi"], case["field"])
    alpha, beta, v1, v0 = _lanczos(h, x, case["steps"])
    t = np.diag(alpha) + np.diag(beta[:-1], 1) + np.diag(beta[:-1], -1)
    return {"alpha": alpha, "beta": beta, "ene": np.linalg.eigvalsh(t)[:1], "v1": out(v1), "v0": out(v0)}
