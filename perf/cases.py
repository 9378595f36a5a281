"""Performance cases: what a program that uses this library has it do.

A case is a dict of plain values; ``prepare`` makes what such a program has in
hand before the call (fields on the GPU, the library's context, weights),
``run`` is one pass through the public entry points, ``work`` the bytes and
operations that the pass cannot do without and ``exact`` its result in 64-bit
arithmetic from plain torch.  Kinds of case:

* ``dslash``: the one-parity hopping term on the multi-RHS layout, the operation
  a caller's own solver is built on (bare, or fused with out = x + c D in);
* ``operator``: mat_Qcu, the full operator on per-RHS vectors in the caller's
  precision, through the reference's call protocol;
* ``solve``: one gauge configuration's propagator solve: load the field, choose
  the operator, queue the sources, invert;
* ``groups``: the same for several groups of sources of different sizes at once;
* ``network``: one application of the learned preconditioner (inference);
* ``gradient``: one training pass of the network (loss and weight gradients).

Links are exp(i eps H) with H a traceless Hermitian Gaussian matrix, sources
complex Gaussian, as in the benchmark.
"""
import functools
import math

import numpy as np
import torch

from qcu_mrhs_amd import api, lgnn

PREC = {"half": 0, "single": 1, "double": 2, "bf16": 4}
COMPLEX_BYTES = {"half": 4, "bf16": 4, "single": 8, "double": 16}
CHANNELS = 8  # hidden channels of the learned preconditioner


# ------------------------------------------------------------------- the cases
def _dslash(lattice, nc, rhs, prec, dagger=False, xpay=False, eps=0.5):
    return {"kind": "dslash", "lattice": lattice, "nc": nc, "rhs": rhs, "prec": prec, "dagger": dagger, "xpay": xpay,
            "eps": eps}


def _operator(lattice, nc, rhs, user, inner, clover=False, dagger=False, kappa=0.12, eps=0.5):
    return {"kind": "operator", "lattice": lattice, "nc": nc, "rhs": rhs, "user": user, "inner": inner,
            "clover": clover, "dagger": dagger, "kappa": kappa, "eps": eps}


def _solve(lattice, nc, rhs, user, inner, kappa, eps, clover=False):
    return {"kind": "solve", "lattice": lattice, "nc": nc, "rhs": rhs, "user": user, "inner": inner,
            "clover": clover, "kappa": kappa, "eps": eps, "tol": 1e-10}


def _groups(lattice, nc, sizes, kappa, eps):
    return {"kind": "groups", "lattice": lattice, "nc": nc, "sizes": sizes, "inner": "single", "kappa": kappa,
            "eps": eps, "tol": 1e-10}


def _network(lattice, nc, rhs, prec, projected, kappa=0.1355, eps=0.5):
    return {"kind": "network", "lattice": lattice, "nc": nc, "rhs": rhs, "prec": prec, "projected": projected,
            "kappa": kappa, "eps": eps}


def _gradient(lattice, nc, rhs, power, kappa=0.1355, eps=0.5):
    return {"kind": "gradient", "lattice": lattice, "nc": nc, "rhs": rhs, "power": power, "kappa": kappa, "eps": eps}


def listed():
    named = {
        # the inner solver's hop at the benchmark's size: the second hop of the Schur operator, x + c D in
        "dslash half 24c48 r16": _dslash("24x24x24x48", 3, 16, "half", xpay=True),
        # a caller's own double-precision solver, 12 sources (one point source's spin-colours)
        "dslash double 16c32 r12": _dslash("16x16x16x32", 3, 12, "double"),
        # a single-precision adjoint hop, SU(4), an odd number of right-hand sides
        "dslash single su4 r17": _dslash("16x16x16x16", 4, 17, "single", dagger=True),
        # the smallest call: one application of M on a test lattice, where launches and latency count
        "operator double 8c8 r4": _operator("8x8x8x8", 3, 4, "double", "double"),
        # the operator with the clover term on single-precision vectors, ragged extents
        "operator clover ragged r5": _operator("20x14x10x18", 3, 5, "single", "single", clover=True, dagger=True),
        # a small system solved in plain double precision: many short steps
        "solve double 8c8 r4": _solve("8x8x8x8", 3, 4, "double", "double", 0.12, 1.0),
        # the benchmark's system with the fastest inner precision
        "solve half 24c48 r16": _solve("24x24x24x48", 3, 16, "double", "half", 0.1355, 0.5),
        # an intermediate volume, single-precision inner solve, 12 sources
        "solve single 16c32 r12": _solve("16x16x16x32", 3, 12, "double", "single", 0.13, 0.4),
        # an improved-action configuration: clover term built, then solved for one point source
        "solve clover half 16c32 r12": _solve("16x16x16x32", 3, 12, "double", "half", 0.12, 0.5, clover=True),
        # sources that arrive in uneven groups, SU(4) (the batched benchmark)
        "groups su4 16c16": _groups("16x16x16x16", 4, "3,8,17,32", 0.12, 1.0),
        # inference of the learned preconditioner inside the half-precision solve
        "network half 24c48 r16": _network("24x24x24x48", 3, 16, "half", True),
        # a training step's forward and backward pass at the training lattice
        "gradient 16c32 r16": _gradient("16x16x16x32", 3, 16, 3),
    }
    return [dict(c, name=name) for name, c in named.items()]


def _extents(rng, lo, hi):
    """An even x even x even x even lattice whose volume lies in [lo, hi] (spread over its logarithm)."""
    target = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    sizes = [4, 6, 8, 10, 12, 14, 16, 18, 20, 24, 28, 32, 48]
    best = None
    for _ in range(200):
        e = [rng.choice(sizes[:10]) for _ in range(3)] + [rng.choice(sizes)]
        v = math.prod(e)
        if lo <= v <= hi and (best is None or abs(math.log(v / target)) < abs(math.log(math.prod(best) / target))):
            best = e
    return "x".join(str(n) for n in (best or [4, 4, 4, 4]))


def draw(rng):
    kind = rng.choice(["dslash", "dslash", "operator", "solve", "solve", "groups", "network", "gradient"])
    eps = round(rng.uniform(0.4, 1.2), 2)
    kappa = round(rng.uniform(0.11, 0.13), 4)
    nc = rng.choice([2, 3, 3, 3, 3, 4, 8])
    rhs = rng.choice([1, 2, 3, 4, 5, 7, 8, 11, 12, 12, 13, 16, 16, 17, 24, 32])

    def volume(values):  # sites for at most `values` complex numbers in a full vector
        return _extents(rng, 256, max(512, values // (4 * nc * rhs)))

    if kind == "dslash":
        prec = rng.choice(["half", "bf16", "single", "double"])
        return _dslash(volume(2 ** 31 // COMPLEX_BYTES[prec] // 4), nc, rhs, prec, rng.random() < 0.3,
                       rng.random() < 0.5, eps)
    if kind == "operator":
        user, inner = rng.choice(["single", "double"]), rng.choice(["half", "bf16", "single", "double"])
        return _operator(volume(2 ** 25), nc, rhs, user, inner, rng.random() < 0.3, rng.random() < 0.3, kappa, eps)
    if kind == "solve":
        user, inner = rng.choice(["single", "double"]), rng.choice(["half", "half", "bf16", "single", "double"])
        return _solve(volume(2 ** 24), nc, rhs, user, inner, kappa, eps, rng.random() < 0.3)
    if kind == "groups":
        nc = rng.choice([2, 3, 4, 8])
        sizes = [rng.choice([1, 2, 3, 4, 6, 8, 12, 16, 17, 32]) for _ in range(rng.choice([2, 3, 4]))]
        rhs = sum(sizes)
        return _groups(volume(2 ** 23), nc, ",".join(str(s) for s in sizes), min(kappa, 0.12), eps)
    nc = rng.choice([2, 3, 3, 3, 4])
    rhs = max(rhs, 4)
    if kind == "network":
        prec = rng.choice(["half", "half", "bf16", "single"])
        return _network(volume(2 ** 26), nc, rhs, prec, rng.random() < 0.5, kappa, eps)
    return _gradient(volume(2 ** 23), nc, rhs, rng.choice([1, 2, 3]), kappa, eps)


# ----------------------------------------------------------------------- fields
def _shape(case):
    lattice = tuple(int(n) for n in case["lattice"].split("x"))
    return lattice, case["nc"], math.prod(lattice) // 2


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _gaussian(gen, *shape):
    return torch.view_as_complex(torch.randn(*shape, 2, dtype=torch.float64, device="cuda", generator=gen))


def _matmul(a, b):
    """Products of small matrices, element by element."""
    n = a.shape[-1]
    return sum(a[..., :, k, None] * b[..., None, k, :] for k in range(n))


def _links(case, gen):
    """Even/odd gauge field [4][2][Vh][Nc][Nc], complex128: exp(i eps H), by Taylor's series and squaring."""
    _, nc, vh = _shape(case)
    a = _gaussian(gen, 4, 2, vh, nc, nc)
    h = 0.5 * (a + a.conj().transpose(-1, -2))
    one = torch.eye(nc, dtype=torch.complex128, device="cuda")
    h = h - (torch.diagonal(h, dim1=-2, dim2=-1).sum(-1) / nc)[..., None, None] * one
    x = h * (1j * case["eps"] / 32)
    u = one + x / 12
    for k in range(11, 0, -1):
        u = one + _matmul(x, u) / k
    for _ in range(5):
        u = _matmul(u, u)
    return u.contiguous()


def _store(z, prec):
    """A complex128 tensor in the library's storage of a precision (16-bit: a trailing (re, im) pair)."""
    if prec == "double":
        return z.clone()
    if prec == "single":
        return z.to(torch.complex64)
    return torch.view_as_real(z).to(torch.float16 if prec == "half" else torch.bfloat16).contiguous()


def _wide(z):
    """A stored tensor as complex128."""
    return z.to(torch.complex128) if z.is_complex() else torch.view_as_complex(z.to(torch.float64).contiguous())


def _fields(case, seed):
    """The inputs of a case, from the seed alone: (gauge complex128, sources in the caller's storage)."""
    lattice, nc, vh = _shape(case)
    kind = case["kind"]
    # an operator, a network and its training work on the configuration that the context holds
    # through many calls; a solve and a stateless hop are given theirs
    gauge = _links(case, _gen(seed if kind in ("dslash", "solve", "groups") else 77))
    gen = _gen(1000003 * (int(seed) % 1000000) + 1)
    if kind == "dslash":
        n = case["rhs"]
        fields = [_store(_gaussian(gen, vh, 4, nc, n), case["prec"]) for _ in range(2 if case["xpay"] else 1)]
        return _store(gauge, case["prec"]), fields
    if kind in ("operator", "solve"):
        return gauge, [_store(_gaussian(gen, case["rhs"], 2, vh, 4, nc), case["user"])]
    if kind == "groups":
        return gauge, [_gaussian(gen, int(s), 2, vh, 4, nc) for s in case["sizes"].split(",")]
    return gauge, [_store(_gaussian(gen, vh, 4, nc, case["rhs"]), case.get("prec", "single"))]


def _weights(case):
    """The network's weights: the first Neumann term and a training's starting noise."""
    w1, w2 = lgnn.neumann_weights(case["kappa"], channels=CHANNELS, noise=0.01, seed=11)
    return w1, (lgnn.project_w2(w2) if case.get("projected") else w2)


# --------------------------------------------------------------------- the passes
_held = {"context": None}  # the library has one context a process: what it was made for


def _context(case):
    lattice, nc, _ = _shape(case)
    inner = case.get("inner", case.get("prec", "single"))
    key = (lattice, nc, case.get("rhs", 4), PREC[case.get("user", "double")], PREC[inner])
    if _held["context"] != key:
        api.initGridSize(*key)
        _held["context"] = key
    api.set_solver_options(key[4], 0.0, False)
    _choose(case)


def _choose(case):
    api.getDslash(api.DSLASH_CLOVER if case.get("clover") else api.DSLASH_WILSON, 1.0 / (2 * case["kappa"]) - 4.0)


def prepare(case, seed):
    gauge, fields = _fields(case, seed)
    state = {"case": case, "gauge": gauge, "in": fields, "out": [torch.empty_like(f) for f in fields[:1]]}
    torch.cuda.synchronize()
    kind = case["kind"]
    if kind == "groups":
        state["out"] = [torch.empty_like(f) for f in fields]
    if kind != "dslash":
        _context(case)
    if kind in ("operator", "network", "gradient"):
        api.loadQcuGauge(gauge.data_ptr(), PREC["double"])
    if kind in ("network", "gradient"):
        lgnn.set_projected(case.get("projected", False))
        lgnn.set_weights(*_weights(case))
    torch.cuda.synchronize()
    return state


def _queue(x, b):
    for r in range(b.shape[0]):
        api.pushBackFermions(x[r].data_ptr(), b[r].data_ptr())


def run(state):
    case, out, fields = state["case"], state["out"], state["in"]
    kind = case["kind"]
    if kind == "dslash":
        lattice, nc, _ = _shape(case)
        xpay = fields[1].data_ptr() if case["xpay"] else None
        api.dslash_mrhs(out[0].data_ptr(), fields[0].data_ptr(), state["gauge"].data_ptr(), lattice, nc, case["rhs"], 1,
                        int(case["dagger"]), PREC[case["prec"]], xpay, -0.0184 if case["xpay"] else 1.0)
        return out
    if kind == "operator":
        _queue(out[0], fields[0])
        api.mat_Qcu(int(case["dagger"]))
        return out
    if kind in ("solve", "groups"):
        api.loadQcuGauge(state["gauge"].data_ptr(), PREC["double"])
        _choose(case)
        if kind == "solve":
            _queue(out[0], fields[0])
            api.qcuInvertEx(1000, case["tol"], raise_on_nonconvergence=True)
        else:
            api.invert_groups([([x[r].data_ptr() for r in range(len(x))], [b[r].data_ptr() for r in range(len(b))])
                               for x, b in zip(out, fields)], 1000, case["tol"], raise_on_nonconvergence=True)
        return out
    if kind == "network":
        lgnn.apply(out[0].data_ptr(), fields[0].data_ptr(), PREC[case["prec"]])
        return out
    loss, g1, g2 = lgnn.power_loss_grad(fields[0].data_ptr(), case["power"], CHANNELS)
    # the passes run in single precision, and the program keeps their result so
    return {"loss": np.float32(loss), "g1": g1.astype(np.complex64), "g2": g2.astype(np.complex64)}


def work(case):
    """Inputs read once, outputs written once; the operations of the hops that the definition names (a solve: those of
    its right-hand side, one operator application and the even half of its solution)."""
    _, nc, vh = _shape(case)
    kind = case["kind"]
    rhs = sum(int(s) for s in case["sizes"].split(",")) if kind == "groups" else case["rhs"]
    hop = vh * rhs * (8 * 2 * (8 * nc - 2) * nc + 8 * 2 * 2 * nc + 7 * 8 * nc)
    half = vh * 4 * nc * rhs
    links = 8 * vh * nc * nc
    if kind == "dslash":
        return {"bytes": COMPLEX_BYTES[case["prec"]] * (links + half * (3 if case["xpay"] else 2)), "flops": hop}
    if kind == "operator":
        c = COMPLEX_BYTES[case["inner"]]
        return {"bytes": links * c + 4 * half * COMPLEX_BYTES[case["user"]], "flops": 2 * hop}
    if kind in ("solve", "groups"):
        c = COMPLEX_BYTES[case.get("user", "double")]
        return {"bytes": links * 16 + 4 * half * c, "flops": 4 * hop}
    # eight transports each way of four spins and the (hop, spin) mixing between them
    net = vh * rhs * nc * (2 * 8 * 4 * 8 * nc + 8 * 32 * 32)
    if kind == "network":
        return {"bytes": COMPLEX_BYTES[case["prec"]] * (links + 2 * half), "flops": net}
    return {"bytes": 8 * (links + half), "flops": case["power"] * (3 * net + 4 * hop)}


# ------------------------------------------------------------ the same in 64 bits
_G = torch.tensor(lgnn.GAMMA)  # chiral gamma matrices: one entry a row


@functools.lru_cache(maxsize=2)
def _neighbours(lattice):
    """Full-lattice (parity-major) neighbour sites [8][2 Vh], hop 2 mu + (0 forward, 1 backward)."""
    lx, ly, lz, lt = lattice
    vh = math.prod(lattice) // 2
    cb = np.arange(vh)
    xh, y, z, t = cb % (lx // 2), cb // (lx // 2) % ly, cb // (lx // 2 * ly) % lz, cb // (lx // 2 * ly * lz)
    coords = [np.concatenate([2 * xh + ((y + z + t + p) & 1) for p in (0, 1)])] + [np.tile(v, 2) for v in (y, z, t)]
    rows = []
    for mu in range(4):
        for step in (1, -1):
            c = [(v + step) % n if k == mu else v for k, (v, n) in enumerate(zip(coords, lattice))]
            rows.append(((c[0] + c[1] + c[2] + c[3]) & 1) * vh + ((c[3] * lz + c[2]) * ly + c[1]) * (lx // 2) + c[0] // 2)
    return torch.tensor(np.stack(rows), device="cuda")


class _Lattice:
    """Transports and operators on complex128 fields [sites of one parity][4][Nc][R]."""

    def __init__(self, lattice, gauge):
        self.nb = _neighbours(lattice)
        self.vh = gauge.shape[2]
        self.nc = gauge.shape[-1]
        self.gauge = gauge.reshape(4, 2 * self.vh, self.nc, self.nc)

    def link(self, k, p):
        """Transport matrices of hop k to the sites of parity p, and the neighbours (on parity 1 - p)."""
        s = slice(p * self.vh, (p + 1) * self.vh)
        nb = self.nb[k, s]
        u = self.gauge[k >> 1, s] if k & 1 == 0 else self.gauge[k >> 1, nb].conj().transpose(-1, -2)
        return u, nb - (1 - p) * self.vh

    def rotate(self, u, f):
        return torch.stack([sum(u[:, a, b, None, None] * f[:, :, b] for b in range(self.nc)) for a in range(self.nc)], 2)

    def transport(self, k, f, p):
        u, nb = self.link(k, p)
        return self.rotate(u, f[nb])

    def hop(self, f, p, dagger=False):
        """D f on parity p: sum over hops of (1 -+ gamma) U f(neighbour), two spins at a time."""
        out = torch.zeros_like(f)
        for k in range(8):
            u, nb = self.link(k, p)
            g, sign = _G[k >> 1], (-1.0 if (k & 1 == 0) != dagger else 1.0)
            v = f[nb]
            pair = [int(g[s].abs().argmax()) for s in range(4)]
            h = torch.stack([v[:, s] + sign * complex(g[s, pair[s]]) * v[:, pair[s]] for s in range(2)], 1)
            h = self.rotate(u, h)
            out[:, :2] += h
            for s in (2, 3):
                out[:, s] += sign * complex(g[s, pair[s]]) * h[:, pair[s]]
        return out

    def schur(self, f, kappa, dagger=False):
        return f - kappa ** 2 * self.hop(self.hop(f, 0, dagger), 1, dagger)

    def clover(self, kappa):
        """A - 1 = -kappa sum_{mu<nu} sigma_{mu nu} F_{mu nu} for every site, [2 Vh][4 Nc][4 Nc]."""
        n = 2 * self.vh
        eye = torch.eye(self.nc, dtype=torch.complex128, device="cuda")
        a = torch.zeros(n, 4, self.nc, 4, self.nc, dtype=torch.complex128, device="cuda")
        at = lambda k, s: self.nb[k][s]  # noqa: E731
        here = torch.arange(n, device="cuda")
        dag = lambda m: m.conj().transpose(-1, -2)  # noqa: E731
        for mu in range(4):
            for nu in range(mu + 1, 4):
                U, V = self.gauge[mu], self.gauge[nu]
                f, b, F, B = 2 * mu, 2 * mu + 1, 2 * nu, 2 * nu + 1
                leaves = (
                    (U[here], V[at(f, here)], dag(U[at(F, here)]), dag(V[here])),
                    (V[here], dag(U[at(F, at(b, here))]), dag(V[at(b, here)]), U[at(b, here)]),
                    (dag(U[at(b, here)]), dag(V[at(b, at(B, here))]), U[at(b, at(B, here))], V[at(B, here)]),
                    (dag(V[at(B, here)]), U[at(B, here)], V[at(f, at(B, here))], dag(U[here])),
                )
                q = sum(functools.reduce(_matmul, leaf) for leaf in leaves)
                q = q - dag(q)
                q = (q - (torch.diagonal(q, dim1=-2, dim2=-1).sum(-1) / self.nc)[:, None, None] * eye) / 8j
                sigma = 0.5j * (_G[mu] @ _G[nu] - _G[nu] @ _G[mu])
                for s in range(4):
                    for t in range(4):
                        if sigma[s, t] != 0:
                            a[:, s, :, t] -= kappa * complex(sigma[s, t]) * q
        return a.reshape(n, 4 * self.nc, 4 * self.nc)

    def full(self, f, kappa, dagger, clover):
        """M f on a full field [2][Vh][4][Nc][R]."""
        out = torch.stack([f[p] - kappa * self.hop(f[1 - p], p, dagger) for p in (0, 1)])
        if clover is not None:
            v, m = f.reshape(2 * self.vh, 4 * self.nc, -1), 4 * self.nc
            out += torch.stack([sum(clover[:, i, j, None] * v[:, j] for j in range(m) if clover[0, i, j] != 0)
                                for i in range(m)], 1).reshape(f.shape)
        return out


def _bicgstab(apply, b):
    """apply(x) = b for every right-hand side (the last index) to the rounding of 64 bits."""
    dims = tuple(range(b.dim() - 1))
    dot = lambda u, v: (u.conj() * v).sum(dims)  # noqa: E731
    over = lambda u, v: torch.where(v.abs() > 0, u / v, torch.zeros_like(u))  # noqa: E731
    x, target = torch.zeros_like(b), 2e-14 * dot(b, b).real.sqrt()
    for _ in range(3):  # restarted from its true residual
        r = b - apply(x)
        if (dot(r, r).real.sqrt() <= target).all():
            break
        r0, p, rho = r.clone(), r.clone(), dot(r, r)
        for _ in range(400):
            v = apply(p)
            alpha = over(rho, dot(r0, v))
            s = r - alpha * v
            t = apply(s)
            omega = over(dot(t, s), dot(t, t))
            x += alpha * p + omega * s
            r = s - omega * t
            if (dot(r, r).real.sqrt() <= target).all():
                break
            new = dot(r0, r)
            p = r + over(new * alpha, rho * omega) * (p - omega * v)
            rho = new
    return x


def _network_forward(lat, psi, w1, w2):
    """The two layers on an odd field, as their definition has them: every hop of every channel."""
    spin = lambda w, f: torch.stack([sum(w[s, t] * f[:, t] for t in range(4)) for s in range(4)], 1)  # noqa: E731
    hops = [lat.transport(k, psi, 0) for k in range(8)]  # on the even sites
    out = 0
    even = [sum(spin(w1[o, k + 1], hops[k]) for k in range(8)) for o in range(CHANNELS)]
    odd = [spin(w1[o, 0], psi) for o in range(CHANNELS)]
    for o in range(CHANNELS):
        out = out + spin(w2[o, 0], odd[o])
    for k in range(8):
        out = out + lat.transport(k, sum(spin(w2[o, k + 1], even[o]) for o in range(CHANNELS)), 1)
    return out


def exact(case, seed):
    lattice, nc, vh = _shape(case)
    gauge, fields = _fields(case, seed)
    kind = case["kind"]
    lat = _Lattice(lattice, _wide(gauge))
    wide = [_wide(f) for f in fields]
    kappa = case.get("kappa")
    if kind == "dslash":
        out = lat.hop(wide[0], 1, case["dagger"])
        out = wide[1] - 0.0184 * out if case["xpay"] else out
        return [out if fields[0].is_complex() else torch.view_as_real(out)]
    clover = lat.clover(kappa) if case.get("clover") else None
    if kind == "operator":
        f = wide[0].permute(1, 2, 3, 4, 0)
        return [lat.full(f, kappa, case["dagger"], clover).permute(4, 0, 1, 2, 3).contiguous()]
    if kind in ("solve", "groups"):
        found = []
        for w in wide:
            b = w.permute(1, 2, 3, 4, 0).contiguous()
            if clover is None:
                xo = _bicgstab(lambda f: lat.schur(f, kappa), b[1] + kappa * lat.hop(b[0], 1))
                x = torch.stack([b[0] + kappa * lat.hop(xo, 0), xo])
            else:
                x = _bicgstab(lambda f: lat.full(f, kappa, False, clover), b)
            found.append(x.permute(4, 0, 1, 2, 3).contiguous())
        return found
    w1, w2 = (torch.tensor(w, device="cuda") for w in _weights(case))
    if kind == "network":
        out = _network_forward(lat, wide[0], w1, w2)
        return [out if fields[0].is_complex() else torch.view_as_real(out)]
    w1.requires_grad_(True)
    w2.requires_grad_(True)
    v = wide[0]
    w = v / (v.conj() * v).real.sum((0, 1, 2)).sqrt()
    for _ in range(case["power"]):
        w = w - lat.schur(_network_forward(lat, w, w1, w2), kappa)
    loss = (w.conj() * w).real.sum()
    loss.backward()
    return {"loss": np.float64(loss.item()), "g1": w1.grad.cpu().numpy(), "g2": w2.grad.cpu().numpy()}
