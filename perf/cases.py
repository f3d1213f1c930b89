"""Measured workloads of the Kohn-Sham eigensolver path.

Every case goes through the public entry points (the classes of `dfx`) on a
structured finite-element mesh built here in plain torch: tensor-product
elements of order p on cubes of edge h, Gauss-Lobatto nodes numbered by first
appearance, smeared Coulomb centres, optional Slater-type enrichment (five
functions per atom, support radius 6 bohr), zero Dirichlet values on the
boundary, or (`periodic`) opposite x faces tied together.  The operators depend
on the case alone; vectors come from the seed.

Kinds:
  apply           Y = A X, one operator apply (Lanczos, Cholesky-Gram-Schmidt,
                  Rayleigh-Ritz, residuals)
  inverse         Y = H M^-1 X, the composite apply of the Chebyshev filter
  cg              batched Jacobi-preconditioned Poisson solve
  orthonormalize  Cholesky-Gram-Schmidt of a subspace
  ritz            Rayleigh-Ritz step on an orthonormal-like subspace
  chfsi           passes of the Chebyshev-filtered subspace iteration with the
                  residual norms of every state
  density         electron density at the quadrature points
"""
import json
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "dft-efe_amd"))
import dfx  # noqa: E402

SUPPORT, FUNCS = 6.0, 5   # enrichment support radius (bohr) and functions per atom


def _case(kind, name=None, **kw):
    c = dict(kind=kind, p=3, nx=8, ny=8, nz=8, h=1.5, atoms=4, enriched=False, op="H",
             columns=8, dtype="f64", periodic=False, degree=0, block=0, mixed=False,
             graph=False, passes=1)
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one vector on a serving-sized mesh (6^3 cells): a Lanczos step, all latency
        _case("apply", "apply_lanczos", nx=6, ny=6, nz=6, h=3.0, columns=1),
        # a caller's own ragged block: odd column count, uneven mesh, a constraint
        # set with parents
        _case("apply", "apply_ragged", nx=11, ny=7, nz=9, atoms=3, enriched=True, op="M",
              columns=13, periodic=True),
        # all states at once in FP64, the apply inside orthonormalization and Ritz
        _case("apply", "apply_all_states", p=4, nx=24, ny=24, nz=24, h=1.25, atoms=14,
              enriched=True, columns=200),
        # one filter step's operator on the 4-atom enriched mesh (16^3 cells, 40 states)
        _case("inverse", "filter_apply_16", nx=16, ny=16, nz=16, enriched=True, columns=40,
              dtype="f32"),
        # the same on the 32-atom mesh (32^3 cells at p = 4) for one filter batch
        _case("inverse", "filter_apply_32", p=4, nx=32, ny=32, nz=32, h=1.25, atoms=32,
              enriched=True, columns=128, dtype="f32"),
        # electrostatics: 8 Gaussian charge right-hand sides, 16^3 cells
        _case("cg", "poisson_16", nx=16, ny=16, nz=16, h=1.25, atoms=0, op="K", columns=8),
        # orthonormalization of 200 filtered states
        _case("orthonormalize", "cholesky_gs", p=4, nx=20, ny=20, nz=20, h=1.25, atoms=8,
              enriched=True, op="M", columns=200),
        # Rayleigh-Ritz with an uneven number of states
        _case("ritz", "rayleigh_ritz", p=4, nx=13, ny=14, nz=15, h=1.25, atoms=3, columns=101),
        # a serving request's solver passes: 10^3 cells, 20 states, replayed degree loop
        _case("chfsi", "chfsi_serving", nx=10, ny=10, nz=10, h=2.0, atoms=3, enriched=True,
              columns=20, degree=24, mixed=True, graph=True, passes=2),
        # double-precision passes of the 4-atom mesh, one block
        _case("chfsi", "chfsi_fp64", nx=16, ny=16, nz=16, enriched=True, columns=40, degree=24,
              passes=2),
        # the 32-atom mesh: 200 states in batches of 64, degree 30, FP32 filter
        _case("chfsi", "chfsi_32", p=4, nx=32, ny=32, nz=32, h=1.25, atoms=32, enriched=True,
              columns=200, degree=30, block=64, mixed=True, passes=2),
        # the density of 40 states
        _case("density", "density_16", nx=16, ny=16, nz=16, columns=40),
    ]


def _spread(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """Any kind, over the mesh sizes, orders, widths and options of the listed cases."""
    kind = rng.choice(["apply", "apply", "inverse", "inverse", "cg", "orthonormalize", "ritz",
                       "chfsi", "chfsi", "density"])
    p = rng.choice([2, 3, 4])
    n = _spread(rng, 5, 24 if kind in ("apply", "inverse") else 16)
    c = _case(kind, p=p, h=rng.choice([1.25, 1.5, 2.0]), atoms=rng.randint(1, 6),
              enriched=rng.random() < 0.6)
    for d in ("nx", "ny", "nz"):
        c[d] = max(4, n + rng.randint(-2, 2))
    if kind == "apply":
        c.update(op=rng.choice(["H", "M", "K"]), columns=_spread(rng, 1, 200),
                 dtype=rng.choice(["f64", "f32"]), periodic=rng.random() < 0.3)
    elif kind == "inverse":
        c.update(columns=_spread(rng, 4, 128), dtype=rng.choice(["f64", "f32", "f32"]))
    elif kind == "cg":
        c.update(op="K", atoms=0, enriched=False, columns=_spread(rng, 1, 16))
    elif kind in ("orthonormalize", "ritz"):
        c.update(op="M" if kind == "orthonormalize" else "H", columns=_spread(rng, 8, 160))
    elif kind == "chfsi":
        c.update(p=max(p, 3), columns=_spread(rng, 5, 64), degree=rng.randint(8, 20),
                 mixed=rng.random() < 0.6, graph=rng.random() < 0.5, passes=2)
    else:
        c.update(enriched=False, columns=_spread(rng, 4, 80))
    return c


# ------------------------------------------------------------------ mesh
def _boxes(case):
    return (np.array([case["nx"], case["ny"], case["nz"]]),
            -0.5 * case["h"] * np.array([case["nx"], case["ny"], case["nz"]], dtype=float))


def _atoms(case):
    """Seeded positions of unit charges, at least 1.2 bohr apart and 6 bohr (or a quarter
    of the box) from the boundary."""
    cells, lo = _boxes(case)
    length = case["h"] * cells
    rng, out = random.Random(100 * case["atoms"] + int(cells.sum())), []
    while len(out) < case["atoms"]:
        m = np.minimum(SUPPORT, length / 4)
        x = [rng.uniform(lo[d] + m[d], lo[d] + length[d] - m[d]) for d in range(3)]
        if all(np.linalg.norm(np.subtract(x, a[:3])) >= 1.2 for a in out):
            out.append((*map(float, x), 1))
    return out


def _cell_atoms(case):
    """Per cell (x fastest) the atoms whose support box meets it: (counts, lists)."""
    cells, lo = _boxes(case)
    nc = int(cells.prod())
    hit = np.zeros((nc, case["atoms"] if case["enriched"] else 0), dtype=bool)
    i = np.arange(nc)
    idx = np.stack([i % cells[0], i // cells[0] % cells[1], i // (cells[0] * cells[1])], axis=1)
    a0 = lo + case["h"] * idx
    if case["enriched"]:
        for a, at in enumerate(_atoms(case)):
            x = np.array(at[:3])
            hit[:, a] = ((x + SUPPORT >= a0) & (x - SUPPORT <= a0 + case["h"])).all(axis=1)
    return hit.sum(axis=1), hit, a0


def _sizes(case):
    """(dofs, per-cell dof counts)."""
    cells, _ = _boxes(case)
    count, _, _ = _cell_atoms(case)
    nd = (case["p"] + 1) ** 3 + FUNCS * count
    nodes = int((case["p"] * cells + 1).prod())
    return nodes + (FUNCS * case["atoms"] if case["enriched"] else 0), nd.astype(np.int64)


def _rules(p, nq):
    """Gauss-Lobatto nodes / weights and the Lagrange basis and its slopes (nq x p+1) at
    nq Gauss points."""
    leg = np.polynomial.legendre.Legendre.basis(p)
    x = np.concatenate([[-1.0], np.sort(leg.deriv().roots().real), [1.0]])
    wl = 2.0 / (p * (p + 1) * leg(x) ** 2)
    xq, wq = np.polynomial.legendre.leggauss(nq)
    L, D = np.ones((nq, p + 1)), np.zeros((nq, p + 1))
    for a in range(p + 1):
        others = [b for b in range(p + 1) if b != a]
        for b in others:
            L[:, a] *= (xq - x[b]) / (x[a] - x[b])
            t = np.ones(nq) / (x[a] - x[b])
            for k in others:
                if k != b:
                    t *= (xq - x[k]) / (x[a] - x[k])
            D[:, a] += t
    return x, wl, xq, wq, L, D


class _Mesh:
    """Numbering, constraints, lumped mass and (on demand) cell matrices of a case."""

    def __init__(self, case):
        p, h = case["p"], case["h"]
        self.case, self.n1 = case, p + 1
        cells, lo = _boxes(case)
        self.count, self.hit, self.a0 = _cell_atoms(case)
        self.N, self.nd = _sizes(case)
        nc, n1 = len(self.nd), p + 1
        pts = p * cells + 1
        i = np.arange(nc)
        ci = [i % cells[0], i // cells[0] % cells[1], i // (cells[0] * cells[1])]
        loc = np.arange(n1 ** 3)
        lex = sum((p * ci[d][:, None] + (loc // n1 ** d % n1)[None]) * int(np.prod(pts[:d]))
                  for d in range(3))
        _, first = np.unique(lex.ravel(), return_index=True)
        order = np.argsort(first, kind="stable")          # node number -> lexicographic node
        rank = np.empty(len(order), dtype=np.int64)
        rank[order] = np.arange(len(order))
        self.classical = rank[lex]                        # (cells, n1^3)
        self.nC = len(order)
        self.off = np.concatenate([[0], np.cumsum(self.nd)])
        self.moff = np.concatenate([[0], np.cumsum(self.nd ** 2)])
        self.map = np.empty(int(self.off[-1]), dtype=np.int64)
        self.groups = []                                  # (cells, their map) of one size
        for k in np.unique(self.count):
            e = np.nonzero(self.count == k)[0]
            atoms = np.nonzero(self.hit[e])[1].reshape(len(e), k)
            enr = self.nC + (FUNCS * atoms[:, :, None] + np.arange(FUNCS)).reshape(len(e), -1)
            m = np.concatenate([self.classical[e], enr.astype(np.int64)], axis=1)
            self.map[self.off[e][:, None] + np.arange(m.shape[1])] = m
            self.groups.append((e, atoms, m))
        # node coordinates and constraints
        x, wl = _rules(p, p + 1)[:2]
        at = [order // int(np.prod(pts[:d])) % pts[d] for d in range(3)]
        self.xyz = np.stack([lo[d] + h * (np.minimum(at[d] // p, cells[d] - 1) + 0.5 *
                                          (1 + x[at[d] - p * np.minimum(at[d] // p, cells[d] - 1)]))
                             for d in range(3)], axis=1)
        edge = [(at[d] == 0) | (at[d] == pts[d] - 1) for d in range(3)]
        tied = np.zeros(self.nC, dtype=bool)
        if case["periodic"]:
            dirichlet = edge[1] | edge[2]
            tied = (at[0] == pts[0] - 1) & ~dirichlet
        else:
            dirichlet = edge[0] | edge[1] | edge[2]
        self.rows = np.nonzero(dirichlet | tied)[0]
        self.child = np.nonzero(tied)[0]
        self.parent = rank[order[self.child] - (pts[0] - 1)]
        self.size = tied[self.rows].astype(np.int64)      # entries per row
        w3 = np.kron(wl, np.kron(wl, wl)) * (0.5 * h) ** 3
        self.lumped = np.bincount(self.classical.ravel(), minlength=self.nC,
                                  weights=np.tile(w3, nc))

    def matrices(self, names):
        """Concatenated cell blocks of each name in "HMK" on the GPU, in cell order."""
        case, dev = self.case, "cuda"
        p, h, nq = case["p"], case["h"], case["p"] + 2
        _, _, xq, wq, L, D = _rules(p, nq)
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
        kron = lambda a, b, c: t(np.kron(c, np.kron(b, a)))              # noqa: E731
        B0 = kron(L, L, L)
        G0 = [kron(D, L, L) * (2 / h), kron(L, D, L) * (2 / h), kron(L, L, D) * (2 / h)]
        w = t(np.kron(wq, np.kron(wq, wq)) * (0.5 * h) ** 3)
        q = np.arange(nq ** 3)
        xyz = t(0.5 * h * (1 + np.stack([xq[q % nq], xq[q // nq % nq], xq[q // nq ** 2]], axis=1)))
        at = t(np.array(_atoms(case), dtype=float).reshape(-1, 4))
        out = {k: torch.empty(int(self.moff[-1]), dtype=torch.float64, device=dev) for k in names}
        for e, atoms, _ in self.groups:
            n = (p + 1) ** 3 + FUNCS * atoms.shape[1]
            step = max(1, (1 << 27) // (n * nq ** 3))
            for s in range(0, len(e), step):
                x = t(self.a0[e[s:s + step]])[:, None, :] + xyz        # cells, points, 3
                c = x.shape[0]
                B = B0.expand(c, -1, -1)
                G = [g.expand(c, -1, -1) for g in G0]
                if atoms.shape[1]:
                    val, grad = self._enrichment(x, at[t(atoms[s:s + step])])
                    B = torch.cat([B, val], dim=2)
                    G = [torch.cat([G[d], grad[d]], dim=2) for d in range(3)]
                prod = lambda A, ww: torch.bmm(A.transpose(1, 2).contiguous(),  # noqa: E731
                                               (A * ww[..., None]).contiguous())
                put = t(self.moff[e[s:s + step]])[:, None] + torch.arange(n * n, device=dev)
                wc = w.expand(c, -1)
                K = sum(prod(g, wc) for g in G) if "H" in names or "K" in names else None
                if "K" in names:
                    out["K"][put] = K.reshape(c, -1)
                if "M" in names:
                    out["M"][put] = prod(B, wc).reshape(c, -1)
                if "H" in names:
                    v = torch.zeros_like(wc)
                    for a in range(at.shape[0]):
                        r = (x - at[a, :3]).norm(dim=2).clamp_min(1e-9)
                        v = v - at[a, 3] * torch.erf(2 * r) / r
                    out["H"][put] = (0.5 * K + prod(B, wc * v)).reshape(c, -1)
        return out

    @staticmethod
    def _enrichment(x, atoms):
        """Five Slater-type functions per atom with a smooth cutoff from 4 to 6 bohr:
        values (cells, points, 5k) and the three gradient arrays."""
        d = x[:, None] - atoms[:, :, None, :3]                   # cells, k, points, 3
        r = d.norm(dim=3).clamp_min(1e-9)
        z = (1 + 0.1 * atoms[:, :, 3])[:, :, None]
        u = ((r - 4) / 2).clamp(0, 1)
        fc, dfc = 1 - u ** 3 * (10 - 15 * u + 6 * u * u), -15 * u * u * (1 - u) ** 2
        e1, e2 = torch.exp(-z * r), torch.exp(-0.5 * z * r)
        radial = [(e1, -z * e1), (r * e2, (1 - 0.5 * z * r) * e2), (e2, -0.5 * z * e2)]
        radial = [(f * fc, g * fc + f * dfc) for f, g in radial]
        val = [radial[0][0], radial[1][0]] + [radial[2][0] * d[..., i] for i in range(3)]
        grad = []
        for j in range(3):
            unit = d[..., j] / r
            g = [radial[0][1] * unit, radial[1][1] * unit]
            g += [radial[2][1] * unit * d[..., i] + (radial[2][0] if i == j else 0)
                  for i in range(3)]
            grad.append(torch.stack(g, dim=2))
        flat = lambda a: a.permute(0, 3, 1, 2).reshape(x.shape[0], x.shape[1], -1)  # noqa: E731
        return flat(torch.stack(val, dim=2)), [flat(g) for g in grad]

    def enriched_mass(self, M):
        """Assembled enriched block of the consistent mass (cell order)."""
        nE, n0 = self.N - self.nC, (self.case["p"] + 1) ** 3
        out = np.zeros(nE * nE)
        for e, atoms, m in self.groups:
            if not atoms.shape[1]:
                continue
            n = m.shape[1]
            ij = torch.from_numpy((np.arange(n0, n)[:, None] * n + np.arange(n0, n)).ravel())
            at = torch.from_numpy(self.moff[e])[:, None] + ij
            blocks = M[at.to(M.device)].cpu().numpy()
            g = m[:, n0:] - self.nC
            out += np.bincount((g[:, :, None] * nE + g[:, None, :]).ravel(),
                               weights=blocks.ravel(), minlength=nE * nE)
        return out.reshape(nE, nE)

    def inverse_mass(self, M):
        """(diagonal, enriched block) of the approximate inverse overlap."""
        d = np.zeros(self.N)
        d[:self.nC] = 1 / self.lumped
        d[self.rows] = 0
        nE = self.N - self.nC
        return d, np.linalg.inv(self.enriched_mass(M)) if nE else np.zeros((0, 0))


# ------------------------------------------------- plain 64-bit arithmetic
class _Plain:
    """The same operators as dense per-cell products in torch, FP64."""

    def __init__(self, mesh, mats):
        self.mesh, self.mats = mesh, mats
        dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
        self.rows, self.child, self.parent = dev(mesh.rows), dev(mesh.child), dev(mesh.parent)

    def to_child(self, X):
        X[self.rows] = 0
        X[self.child] = X[self.parent]
        return X

    def to_parent(self, Y):
        Y[self.parent] += Y[self.child]
        Y[self.rows] = 0
        return Y

    def apply(self, name, X):
        X, A, B = self.to_child(X), self.mats[name], X.shape[1]
        Y = torch.zeros_like(X)
        for e, _, m in self.mesh.groups:
            n = m.shape[1]
            step = max(1, (1 << 27) // (n * max(B, n)))
            for s in range(0, len(e), step):
                i = torch.from_numpy(m[s:s + step]).cuda()
                at = torch.from_numpy(self.mesh.moff[e[s:s + step]]).cuda()
                blocks = A[at[:, None] + torch.arange(n * n, device="cuda")].reshape(-1, n, n)
                y = torch.bmm(blocks, X[i.reshape(-1)].reshape(-1, n, B))
                Y.index_add_(0, i.reshape(-1), y.reshape(-1, B))
        return self.to_parent(Y)

    def inverse(self, X):
        if not hasattr(self, "dinv"):
            d, E = self.mesh.inverse_mass(self.mats["M"])
            self.dinv, self.E = torch.from_numpy(d).cuda()[:, None], torch.from_numpy(E).cuda()
        Y = self.dinv * X
        if len(self.E):
            Y[self.mesh.nC:] = self.E @ X[self.mesh.nC:]
        Y[self.rows] = 0
        return Y

    def top(self):
        """Upper bound of the spectrum of M^-1 H (power iteration, with a margin), rounded."""
        g = torch.Generator(device="cuda").manual_seed(7)
        x = torch.rand(self.mesh.N, 1, generator=g, device="cuda", dtype=torch.float64) - 0.5
        lam = 0.0
        for _ in range(60):
            x = self.inverse(self.apply("H", x / x.norm()))
            lam = float(x.norm())
        scale = 10.0 ** math.floor(math.log10(lam)) / 10
        return math.ceil(1.1 * lam / scale) * scale

    def orthonormalize(self, X):
        X = self.to_child(X)
        L = torch.linalg.cholesky(X.T @ self.apply("M", X))
        return X @ torch.linalg.inv(L).T

    def ritz(self, X):
        ev, Q = torch.linalg.eigh(X.T @ self.apply("H", X))
        return ev, X @ Q

    def filtered(self, X, lam, m, a, b, c):
        """Residual form of the degree-m Chebyshev filter of M^-1 H on (a, b, c)."""
        e, c0 = 0.5 * (c - b), 0.5 * (c + b)
        s1 = e / (a - c0)
        r0 = self.apply("H", X) - lam * self.apply("M", X)
        al1, s = s1 / e, s1
        r, old = al1 * r0, torch.zeros_like(r0)
        mu, mu_old = al1 * (lam - c0), torch.ones_like(lam)
        for _ in range(2, m + 1):
            s2 = 1 / (2 / s1 - s)
            al1, al2, s = 2 * s2 / e, -s * s2, s2
            r, old = (al1 * (self.apply("H", self.inverse(r)) - c0 * r) + al2 * old +
                      al1 * mu * r0), r
            mu, mu_old = al1 * (lam - c0) * mu + al2 * mu_old, mu
        return self.inverse(r) + mu * X


# ---------------------------------------------------------------- states
class _Shared:
    """What a program keeps from call to call: the context, and the operators of the
    case at hand."""
    ctx, key, kept = None, None, None


def _context():
    if _Shared.ctx is None:
        _Shared.ctx = dfx.Context(0)
    return _Shared.ctx


def _needs(case):
    return {"apply": case["op"], "inverse": "HM", "cg": "K", "orthonormalize": "M", "ritz": "H",
            "chfsi": "HM", "density": ""}[case["kind"]]


def _operators(case):
    key = json.dumps({k: v for k, v in case.items() if k not in ("name", "degree", "passes")},
                     sort_keys=True)
    if _Shared.key == key:
        return _Shared.kept
    _Shared.key = _Shared.kept = None
    ctx, mesh, kept = _context(), _Mesh(case), {}
    kept["mesh"] = mesh
    if case["kind"] == "density":
        cells, lo = _boxes(case)
        kept["problem"] = dfx.Problem(ctx, p=case["p"], n=tuple(int(v) for v in cells),
                                      lo=tuple(lo), hi=tuple(-lo), atoms=_atoms(case))
    else:
        mats = mesh.matrices(_needs(case))
        start = np.concatenate([[0], np.cumsum(mesh.size)])[:-1]
        cons = dfx.Constraints(ctx, mesh.N, mesh.rows, mesh.size, start, mesh.parent,
                               np.ones(len(mesh.parent)))
        for k, v in mats.items():
            kept[k] = dfx.CellOperator(ctx, mesh.nd, mesh.map, v.cpu().numpy(), mesh.N, mesh.nC,
                                       cons, keep_fp32=case["dtype"] == "f32" or case["mixed"])
        if case["kind"] in ("inverse", "chfsi"):
            d, E = mesh.inverse_mass(mats["M"])
            kept["Minv"] = dfx.DiagonalOperator(ctx, d, mesh.N - mesh.nC, E.ravel(), cons)
        if case["kind"] == "cg":
            kept["pc"] = dfx.DiagonalOperator(ctx, _jacobi(mesh, mats["K"]))
        if case["kind"] == "chfsi":
            kept["top"] = _Plain(mesh, mats).top()
        del mats
        torch.cuda.empty_cache()
    _Shared.key, _Shared.kept = key, kept
    return kept


def _jacobi(mesh, K):
    diag = np.zeros(mesh.N)
    for e, _, m in mesh.groups:
        n = m.shape[1]
        at = torch.from_numpy(mesh.moff[e][:, None] + np.arange(n) * (n + 1)).cuda()
        diag += np.bincount(m.ravel(), weights=K[at].cpu().numpy().ravel(), minlength=mesh.N)
    diag[mesh.rows] = 1
    return 1 / diag


class _Memory:
    """Device memory of a multivector, for torch to look at without a copy."""

    def __init__(self, mv):
        self.mv = mv
        self.__cuda_array_interface__ = {
            "shape": (mv.N, mv.B), "typestr": "<f8" if mv.dtype == dfx.F64 else "<f4",
            "data": (mv.device_ptr, False), "version": 2}


def _tensor(mv):
    return torch.as_tensor(_Memory(mv), device="cuda")


def _random(seed, shape):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return 2 * torch.rand(shape, generator=g, device="cuda", dtype=torch.float64) - 1


def _modes(case, mesh, seed, out):
    """Subspace guess written to `out`: the box's lowest standing waves, roughened by the
    seed, and their free energies."""
    n = out.shape[1]
    cells, lo = _boxes(case)
    length = case["h"] * cells
    ks = np.stack(np.meshgrid(*[np.arange(1, 13)] * 3, indexing="ij")).reshape(3, -1)
    en = 0.5 * ((np.pi * ks / length[:, None]) ** 2).sum(axis=0)
    pick = np.argsort(en, kind="stable")[:n]
    pos = torch.from_numpy((mesh.xyz - lo) / length).cuda()
    rows = torch.from_numpy(mesh.rows).cuda()
    for j in range(0, n, 32):
        k = torch.from_numpy(ks[:, pick[j:j + 32]].astype(float)).cuda()
        w = 0.05 * _random(1000 * seed + j, (mesh.N, k.shape[1]))
        s = [torch.sin(math.pi * pos[:, d:d + 1] * k[d]) for d in range(3)]
        w[:mesh.nC] += s[0] * s[1] * s[2]
        w[rows] = 0
        out[:, j:j + 32] = w
    return en[pick]


def _charges(case, mesh, seed):
    """Right-hand sides: lumped integrals of four Gaussian charges each."""
    g = np.random.RandomState(seed % (1 << 31))
    _, lo = _boxes(case)
    b = np.zeros((mesh.N, case["columns"]))
    for j in range(case["columns"]):
        for _ in range(4):
            c, q = 0.8 * lo * g.uniform(-1, 1, 3), g.randint(1, 7)
            r2 = ((mesh.xyz - c) ** 2).sum(axis=1)
            b[:mesh.nC, j] += 4 * math.pi * q * np.exp(-r2 / 0.5) / (0.5 * math.pi) ** 1.5
    b[:mesh.nC] *= mesh.lumped[:, None]
    b[mesh.rows] = 0
    return b


def _occupation(n):
    return np.where(np.arange(n) < (n + 1) // 2, 1.0, 0.25)


def prepare(case, seed):
    ctx, kept = _context(), _operators(case)
    mesh, kind, n = kept["mesh"], case["kind"], case["columns"]
    dt = dfx.F32 if case["dtype"] == "f32" else dfx.F64
    s = dict(kept, case=case, ctx=ctx)
    mv = lambda d=dfx.F64: dfx.MultiVector(ctx, mesh.N, n, d)  # noqa: E731
    if kind in ("apply", "inverse"):
        s["X"], s["Y"] = mv(dt), mv(dt)
        _tensor(s["X"]).copy_(_random(seed, (mesh.N, n)))
        s["out"] = _tensor(s["Y"])
    elif kind == "cg":
        s["b"], s["x"] = dfx.MultiVector.from_numpy(ctx, _charges(case, mesh, seed)), mv()
        s["cg"] = dfx.CGLinearSolver(ctx, 10000, 1e-30, 1e-10, 1e10)
        s["out"] = _tensor(s["x"])
    elif kind == "density":
        s["X"], s["occ"] = mv(), _occupation(n)
        _modes(case, mesh, seed, _tensor(s["X"]))
    else:
        s["X"], s["Y"] = mv(), mv()
        en = _modes(case, mesh, seed, _tensor(s["X"]))
        s["out"] = _tensor(s["Y"])
        if kind == "chfsi":
            s["G"], s["en"] = mv(), en
            s["solver"] = dfx.ChebyshevFilteredEigenSolver(
                ctx, en[0], en[-1], kept["top"], case["degree"], 1e-14, s["G"], True,
                case["block"], dfx.PREC_MIXED if case["mixed"] else dfx.PREC_FP64, case["graph"])
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "apply":
        s[case["op"]].apply(s["X"], s["Y"])
        return s["out"]
    if kind == "inverse":
        s["H"].apply_after_inverse(s["Minv"], s["X"], s["Y"])
        return s["out"]
    if kind == "cg":
        s["x"].set(0.0)
        rc = s["cg"].solve(s["K"], s["pc"], s["b"], s["x"])
        return {"code": rc, "x": s["out"]}
    if kind == "orthonormalize":
        rc = dfx.cholesky_gram_schmidt(s["ctx"], s["X"], s["Y"], s["M"])
        return {"code": rc, "x": s["out"]}
    if kind == "ritz":
        rc, ev = dfx.rayleigh_ritz(s["ctx"], s["H"], s["X"], s["Y"])
        return {"code": rc, "values": ev, "vectors": s["out"]}
    if kind == "density":
        return _tensor(s["problem"].density(s["occ"], s["X"]))
    # passes of the eigensolver from the same guess, each with its convergence test
    ev, solver = s["en"].copy(), s["solver"]
    s["G"].copy_from(s["X"])
    solver.reinit(ev[0], ev[-1], s["top"], case["degree"], 1e-14, s["G"])
    for k in range(case["passes"]):
        if k:
            s["G"].copy_from(s["Y"])
            solver.reinit(ev[0], ev[-1], s["top"], case["degree"], 1e-14, s["G"])
        rc = solver.solve(s["H"], ev, s["Y"], True, s["M"], s["Minv"])
        res = solver.residual_norms(s["H"], s["M"], s["Y"], ev)
    return {"code": rc, "values": ev, "vectors": s["out"], "residuals": res}


def exact(case, seed):
    """Ritz vectors have no value of their own (signs), and an iterate no better one than
    the solution that it approaches."""
    mesh, kind, n = _Mesh(case), case["kind"], case["columns"]
    if kind == "density":
        x, _, _, _, L, _ = _rules(case["p"], case["p"] + 1)
        B = torch.from_numpy(np.kron(L, np.kron(L, L))).cuda()
        X = torch.empty(mesh.N, n, dtype=torch.float64, device="cuda")
        _modes(case, mesh, seed, X)
        f, m, rho = torch.from_numpy(2 * _occupation(n)).cuda(), mesh.classical, []
        for c in range(0, len(m), 1024):
            i = torch.from_numpy(m[c:c + 1024]).cuda()
            rho.append(((B @ X[i]) ** 2 @ f).reshape(-1))
        return torch.cat(rho)[:, None]
    plain = _Plain(mesh, mesh.matrices(_needs(case)))
    if kind in ("apply", "inverse"):
        X = _random(seed, (mesh.N, n))
        X = X.float().double() if case["dtype"] == "f32" else X
        return plain.apply(case["op"] if kind == "apply" else "H",
                           plain.inverse(plain.to_child(X)) if kind == "inverse" else X)
    if kind == "cg":
        b = torch.from_numpy(_charges(case, mesh, seed)).cuda()
        d = torch.from_numpy(_jacobi(mesh, plain.mats["K"])).cuda()[:, None]
        x, r = torch.zeros_like(b), b.clone()
        z = d * r
        q, rz = z.clone(), (r * z).sum(dim=0)
        for _ in range(2000):
            w = plain.apply("K", q)
            a = rz / (q * w).sum(dim=0)
            x, r = x + a * q, r - a * w
            if bool((r.norm(dim=0) < 1e-13 * b.norm(dim=0)).all()):
                break
            z = d * r
            rz, last = (r * z).sum(dim=0), rz
            q = z + (rz / last) * q
        return {"code": None, "x": x}
    X = torch.empty(mesh.N, n, dtype=torch.float64, device="cuda")
    en = _modes(case, mesh, seed, X)
    if kind == "orthonormalize":
        return {"code": None, "x": plain.orthonormalize(X)}
    if kind == "ritz":
        return {"code": None, "values": plain.ritz(X)[0], "vectors": None}
    ev, top = torch.from_numpy(en).cuda(), plain.top()
    for _ in range(case["passes"]):
        a, b = float(ev[0]), float(ev[-1])
        wide = [plain.filtered(X[:, j:j + 100].contiguous(), ev[j:j + 100], case["degree"], a, b,
                               top) for j in range(0, n, 100)]
        ev, X = plain.ritz(plain.orthonormalize(torch.cat(wide, dim=1)))
    res = (plain.apply("H", X) - ev * plain.apply("M", X)).norm(dim=0)
    return {"code": None, "values": ev, "vectors": None, "residuals": res}


# ---------------------------------------------------------- work and limits
def work(case):
    N, nd = _sizes(case)
    n, kind, s = case["columns"], case["kind"], 4 if case["dtype"] == "f32" else 8
    n2, n1 = float((nd ** 2).sum()), float(nd.sum())
    one = lambda s, n: (s * n2 + 4 * n1 + 2.0 * s * N * n, 2.0 * n * n2)  # noqa: E731
    by, fl = one(s, n)
    if kind == "inverse":
        by += 8.0 * N
    elif kind == "cg":
        # about 10 iterations per cell edge
        its = 10 * max(case["nx"], case["ny"], case["nz"])
        by, fl = its * (by + 8 * 8.0 * N * n), its * (fl + 12.0 * N * n)
    elif kind == "orthonormalize":
        fl += N * float(n) * n * 3
        by += 8.0 * N * n
    elif kind == "ritz":
        fl += N * float(n) * n * 3
        by += 8.0 * N * n
    elif kind == "density":
        q = float(len(nd)) * (case["p"] + 1) ** 3
        by, fl = 8.0 * (N * n + q), 2.0 * q * n * (case["p"] + 1) ** 3
    elif kind == "chfsi":
        f = 4 if case["mixed"] else 8
        step = (f * n2 + 4 * n1 + 4.0 * f * N * n, 2.0 * n * n2)
        full = one(8, n)
        dense = (6 * 8.0 * N * n, 3 * 3.0 * N * n * n)
        by = case["passes"] * ((case["degree"] - 1) * step[0] + 2 * full[0] + dense[0])
        fl = case["passes"] * ((case["degree"] - 1) * step[1] + 2 * full[1] + dense[1])
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """About four times what is seen between this path, `exact` and the same sums in
    another order."""
    if case["kind"] == "chfsi":
        # vectors after two passes, FP32 filter against FP64 filter: up to 1.7e-4; the FP64
        # filter amplifies rounding by its growth over the occupied part: 3e-11 seen, and
        # ten times that is allowed for steeper spectra
        return {"rel": 8e-4} if case["mixed"] else {"rel": 1e-9}
    if case["kind"] == "cg":
        return {"rel": 1e-9}    # stopped at 1e-10 of the right-hand side
    if case["kind"] == "ritz":
        return {"rel": 1e-10}   # vectors of close values mix
    if case["dtype"] == "f32":
        return {"rel": 8e-7}
    return {"rel": 1e-13}
