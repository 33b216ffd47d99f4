"""Timed workloads of the gis solver library on one GPU.

Every case is one call sequence a user's program runs per time step (or per
training step) through the public entry points of ``cufoam_amd``:

* ``foam``: what an OpenFOAM wrapper does per time step, from host arrays: new
  coefficients (``set_values``), then ``foam_solve`` with psi and source;
* ``cg`` / ``mixed``: a device-resident FP64 or mixed-precision CG solve;
* ``gamg``: new device coefficients, then GAMG-preconditioned CG (the hierarchy of
  the mesh is kept, its values follow the coefficients);
* ``multi``: the velocity components of one momentum matrix in one BiCG solve;
* ``batch``: many independent systems of uneven size in one batched CG solve;
* ``adjoint``: a differentiable solve, forward and backward, in torch.

The systems are the 7-point Laplacians of ``cufoam_amd.mesh`` (same mesh, same
coefficient distributions), drawn on the GPU from the seed.  ``numbering`` is the
cell order: the structured mesh's own (``lexicographic``), or ``cuthill_mckee``,
the level-by-level order OpenFOAM's renumberMesh gives unstructured meshes.
"""
from __future__ import annotations

import numpy as np
import torch

from cufoam_amd import autograd
from cufoam_amd.gis import Gis
from cufoam_amd.mesh import LduSystem

DEVICE = "cuda:0"

FOAM_TOLERANCE = 1e-8      # on the NormFactor-scaled residual, as the drop-in solves run
REL_TOL = 1e-10            # ||b - A x||_2 / ||b||_2 of the device solves
BATCH_REL_TOL = 1e-8
MAX_ITER = 20000


def listed() -> list[dict]:
    return [
        # a small case's pressure step: call latency and launches are all of it
        _foam("foam_cg_16", "CG", 16, 16, 16),
        # a mid-size unstructured-style numbering, odd edge: no offset tables that fit
        _foam("foam_cg_renumbered_63", "CG", 63, 63, 63, numbering="cuthill_mckee"),
        # the drop-in pressure system (symmetric) at its usual benchmark size
        _foam("foam_cg_128", "CG", 128, 128, 128),
        # the drop-in transport system (nonsymmetric), odd edge
        _foam("foam_bicg_101", "BiCG", 101, 101, 101),
        # OpenFOAM's customary symmetric choice, PCG with DIC
        _foam("foam_pcg_dic_64", "PCG", 64, 64, 64, precond="DIC"),
        # and its customary asymmetric one, PBiCG with DILU
        _foam("foam_pbicg_dilu_45", "PBiCG", 45, 45, 45, precond="DILU"),
        # the headline system, FP64 and mixed precision: bound by memory bandwidth
        _device("cg_256", "cg", 256, 256, 256, shift=1e-4),
        _device("mixed_256", "mixed", 256, 256, 256, shift=1e-4),
        # multigrid pressure solve
        _device("gamg_128", "gamg", 128, 128, 128, precond="GAMG"),
        # momentum predictor: three components share one nonsymmetric matrix
        _device("multi3_bicg_128", "multi", 128, 128, 128, shift=0.1, nrhs=3),
        # a batch of independent sub-domain systems, edges 16 to 64
        {"name": "batch_64", "kind": "batch", "count": 64, "lo": 16, "hi": 64, "edges_seed": 0,
         "shift": 1e-3},
        # gradient of a loss through the solve (adjoint), at the size its checks use
        _device("adjoint_64", "adjoint", 64, 64, 64),
    ]


def draw(rng) -> dict:
    """A box of cells about as large as a cube of an edge spread over the kind's range."""
    def box(lo, hi):
        e = lo * (hi / lo) ** rng.random()
        f, g = rng.uniform(0.7, 1.4), rng.uniform(0.7, 1.4)
        nx, ny = max(3, round(e * f)), max(3, round(e * g))
        return nx, ny, max(3, int(e ** 3 / (nx * ny)))

    kind = rng.choice(["foam_cg", "foam_cg", "foam_renumbered", "foam_bicg", "foam_dic",
                       "foam_dilu", "cg", "mixed", "gamg", "multi", "batch", "adjoint"])
    if kind == "foam_cg":
        case = _foam(None, "CG", *box(10, 160))
    elif kind == "foam_renumbered":
        case = _foam(None, "CG", *box(10, 128), numbering="cuthill_mckee")
    elif kind == "foam_bicg":
        case = _foam(None, "BiCG", *box(10, 128))
    elif kind == "foam_dic":
        case = _foam(None, "PCG", *box(8, 80), precond="DIC",
                     numbering=rng.choice(["lexicographic", "cuthill_mckee"]))
    elif kind == "foam_dilu":
        case = _foam(None, "PBiCG", *box(8, 64), precond="DILU")
    elif kind in ("cg", "mixed"):
        case = _device(None, kind, *box(24, 240), shift=1e-4)
    elif kind == "gamg":
        case = _device(None, kind, *box(24, 160), precond=rng.choice(["GAMG", "GAMG32"]))
    elif kind == "multi":
        case = _device(None, kind, *box(24, 128), shift=0.1, nrhs=rng.choice([2, 3]))
    elif kind == "adjoint":
        case = _device(None, kind, *box(8, 80))
    else:
        lo = rng.randint(8, 24)
        case = {"kind": "batch", "count": round(4 * 16 ** rng.random()), "lo": lo,
                "hi": rng.randint(lo + 8, 64), "edges_seed": rng.randint(0, 10 ** 6),
                "shift": 1e-3}
    case.pop("name", None)
    return case


def _foam(name, method, nx, ny, nz, precond="none", numbering="lexicographic") -> dict:
    nonsym = method in ("BiCG", "PBiCG")
    return {"name": name, "kind": "foam", "method": method, "nx": nx, "ny": ny, "nz": nz,
            "precond": precond, "numbering": numbering, "shift": 0.1 if nonsym else 1e-3}


def _device(name, kind, nx, ny, nz, shift=1e-3, **more) -> dict:
    return {"name": name, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "shift": shift, **more}


# -- systems ---------------------------------------------------------------------
class _Hex:
    """7-point system on a box of cells, on the GPU: per cell the coefficients of the
    faces towards +x, +y, +z (``up``: A(c, c + d); ``lo``: A(c + d, c); zero where the
    mesh ends) and the diagonal, all in the lexicographic cell order."""

    def __init__(self, dims, shift: float, symmetric: bool, gen: torch.Generator):
        nx, ny, nz = dims
        self.N = nx * ny * nz
        self.steps = (1, nx, nx * ny)
        c = torch.arange(self.N, device=DEVICE)
        self.ijk = (c % nx, (c // nx) % ny, c // (nx * ny))
        self.ok = torch.stack([i < n - 1 for i, n in zip(self.ijk, dims)], 1)
        up = -(1.0 + 0.5 * _rand((self.N, 3), gen)) * self.ok
        lo = up if symmetric else up * (1.0 + 0.5 * _rand((self.N, 3), gen))
        self.up, self.lo = up, lo
        diag = -up.sum(1)
        for d, s in enumerate(self.steps):
            diag[s:] -= lo[:-s, d]
        self.diag = diag + shift

    def matvec(self, x, transpose=False):
        up, lo = (self.lo, self.up) if transpose else (self.up, self.lo)
        y = self.diag * x
        for d, s in enumerate(self.steps):
            y[:-s] += up[:-s, d] * x[s:]
            y[s:] += lo[:-s, d] * x[:-s]
        return y

    def order(self, numbering: str):
        """rank[c]: the place of lexicographic cell c in the numbering."""
        if numbering == "lexicographic":
            return torch.arange(self.N, device=DEVICE)
        i, j, k = self.ijk
        key = (i + j + k) * self.N + torch.arange(self.N, device=DEVICE)
        rank = torch.empty_like(key)
        rank[torch.argsort(key)] = torch.arange(self.N, device=DEVICE)
        return rank

    def ldu(self, rank):
        """(lower_addr, upper_addr, diag, lower, upper) in the numbering `rank`, faces
        in upper-triangular order."""
        c = torch.arange(self.N, device=DEVICE)
        a = rank[c.unsqueeze(1).expand(-1, 3)[self.ok]]
        b = rank[torch.stack([c + s for s in self.steps], 1)[self.ok].clamp_(max=self.N - 1)]
        up, lo = self.up[self.ok], self.lo[self.ok]
        flip = a > b
        own, nbr = torch.where(flip, b, a), torch.where(flip, a, b)
        upper, lower = torch.where(flip, lo, up), torch.where(flip, up, lo)
        order = torch.argsort(own * self.N + nbr)
        diag = torch.empty_like(self.diag)
        diag[rank] = self.diag
        return (own[order].int().contiguous(), nbr[order].int().contiguous(), diag,
                lower[order].contiguous(), upper[order].contiguous())


def _rand(shape, gen):
    return torch.rand(shape, generator=gen, device=DEVICE, dtype=torch.float64)


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _system(case: dict, seed: int):
    """The case's matrix, right-hand sides (k, N) and start vector, lexicographic."""
    gen = _gen(seed)
    symmetric = case.get("method") not in ("BiCG", "PBiCG") and case["kind"] != "multi"
    h = _Hex((case["nx"], case["ny"], case["nz"]), case["shift"], symmetric, gen)
    b = 2.0 * _rand((case.get("nrhs", 1), h.N), gen) - 1.0
    x0 = 0.2 * _rand((h.N,), gen) - 0.1      # a time step starts from the last one's field
    return h, b, x0


def _edges(case: dict) -> list[int]:
    rng = np.random.default_rng(case["edges_seed"])
    return rng.integers(case["lo"], case["hi"] + 1, size=case["count"]).tolist()


def _batch_systems(case: dict, seed: int):
    gen = _gen(seed)
    out = []
    for n in _edges(case):
        h = _Hex((n, n, n), case["shift"], True, gen)
        out.append((h, 2.0 * _rand((h.N,), gen) - 1.0))
    return out


# -- what a user's program holds, and one pass --------------------------------------
def prepare(case: dict, seed: int):
    kind = case["kind"]
    g = Gis(0)
    if kind == "batch":
        systems, b = [], []
        for h, rhs in _batch_systems(case, seed):
            la, ua, diag, lower, upper = (t.cpu().numpy() for t in h.ldu(h.order("lexicographic")))
            systems.append(LduSystem(h.N, la, ua, diag, lower, upper, rhs.cpu().numpy(),
                                     np.zeros(h.N)))
            b.append(rhs)
        g.batch_set_systems(systems)
        error = np.array([BATCH_REL_TOL * float(torch.linalg.vector_norm(v)) for v in b])
        return {"case": case, "gis": g, "b": torch.cat(b), "error": error}

    h, b, x0 = _system(case, seed)
    rank = h.order(case.get("numbering", "lexicographic"))
    la, ua, diag, lower, upper = h.ldu(rank)
    if kind == "foam":
        src, psi = torch.empty_like(b[0]), torch.empty_like(x0)
        src[rank], psi[rank] = b[0], x0
        host = {k: t.cpu().numpy() for k, t in
                {"la": la, "ua": ua, "diag": diag, "lower": lower, "upper": upper,
                 "source": src, "psi": psi}.items()}
        g.set_pattern(h.N, host["la"], host["ua"])
        return {"case": case, "gis": g, **host}

    g.set_pattern(h.N, la, ua)
    state = {"case": case, "gis": g, "diag": diag, "lower": lower, "upper": upper,
             "b": b if kind == "multi" else b[0],
             "error": REL_TOL * float(torch.linalg.vector_norm(b[0]))}
    if kind == "adjoint":
        for k in ("diag", "lower", "upper", "b"):
            state[k].requires_grad_(True)
        state["w"] = x0
        return state
    g.set_values(diag, lower, upper)
    if kind == "gamg":
        g.gamg_levels()      # the mesh's hierarchy, kept over the time steps
    return state


def run(state):
    case, g = state["case"], state["gis"]
    kind = case["kind"]
    if kind == "foam":
        g.set_values(state["diag"], state["lower"], state["upper"])
        psi = state["psi"].copy()
        if case["precond"] == "none":
            perf = g.foam_solve(case["method"], psi, state["source"], FOAM_TOLERANCE, MAX_ITER)
        else:
            perf = g.foam_solve(case["method"], psi, state["source"], FOAM_TOLERANCE, MAX_ITER,
                                preconditioner=case["precond"])
        return {"psi": psi, "initial_residual": perf.initial_residual,
                "n_iterations": perf.n_iterations}
    if kind == "batch":
        x, it, _, _ = g.batch_solve(state["b"], torch.zeros_like(state["b"]), state["error"],
                                    MAX_ITER)
        return {"x": x, "iterations": it}
    if kind == "adjoint":
        x = autograd.solve(g, state["diag"], state["lower"], state["upper"], state["b"],
                           error=state["error"], max_steps=MAX_ITER)
        grads = torch.autograd.grad(
            x, (state["diag"], state["lower"], state["upper"], state["b"]), state["w"])
        return {"x": x.detach(), "diag": grads[0], "lower": grads[1], "upper": grads[2],
                "b": grads[3]}
    b = state["b"]
    x = torch.zeros_like(b)
    if kind == "cg":
        x, hist, _ = g.solve("CG", b, x, error=state["error"], max_steps=MAX_ITER)
        return {"x": x, "iterations": len(hist) - 1}
    if kind == "mixed":
        x, hist, it, _, _ = g.solve_mixed(b, x, REL_TOL, 1e-2, MAX_ITER, 0)
        return {"x": x, "iterations": it}
    if kind == "gamg":
        g.set_values(state["diag"], state["lower"], state["upper"])
        x, hist, _ = g.solve_pcg(case["precond"], b, x, error=state["error"], max_steps=2000)
        return {"x": x, "iterations": len(hist) - 1}
    if kind == "multi":
        x, it, _, _ = g.solve_multi("BiCG", b, x, error=state["error"], max_steps=MAX_ITER)
        return {"x": x, "iterations": it}
    raise ValueError(kind)


# -- necessary work --------------------------------------------------------------
def _iterations(case: dict, e: float) -> float:
    """Krylov iterations at an edge of e cells, as the systems were measured to take."""
    kind, precond = case["kind"], case.get("precond")
    if kind == "gamg":
        return 20.0 + 0.12 * e
    if precond == "DIC":
        return 2.2 * e + 10.0
    if precond == "DILU":
        return 0.7 * e + 12.0
    if case.get("method") == "BiCG" or kind == "multi":
        return 2.0 * e + 10.0
    if kind in ("cg", "mixed"):
        return 7.2 * e
    return 4.9 * e + 70.0


def work(case: dict) -> dict:
    """Bytes: the matrix coefficients and the vectors in, the results out, once each.
    Flops: the matrix products and vector operations of the iterations."""
    kind = case["kind"]
    if kind == "batch":
        e = np.array(_edges(case), dtype=np.float64)
        return {"bytes": float((8.0 * (1 + 6 + 2) * e ** 3).sum()),
                "flops": float((e ** 3 * 24.0 * (4.9 * e + 70.0)).sum())}
    N = case["nx"] * case["ny"] * case["nz"]
    nnz = 7 * N
    k = case.get("nrhs", 1)
    nonsym = case.get("method") in ("BiCG", "PBiCG") or kind == "multi"
    products = 2 if nonsym or kind == "adjoint" else 1
    vectors = 3 * N if kind == "foam" else 2 * k * N     # foam: psi goes in as well
    bytes_ = 8.0 * (nnz + vectors)
    if kind == "adjoint":
        bytes_ += 8.0 * (3 * N + nnz)                    # the cotangent in, the gradients out
    it = _iterations(case, N ** (1.0 / 3.0))
    return {"bytes": bytes_, "flops": k * it * (products * 2.0 * nnz + 10.0 * N)}


# -- accuracy --------------------------------------------------------------------
def tolerance(case: dict):
    """About four times the largest distance from the exact solution at which the
    stopping rule of each kind of solve left it, over sizes and seeds: 4e-7 (foam),
    3e-8 (batch, cg, mixed), 7e-9 (adjoint), 5e-10 (gamg, multi)."""
    return {"rel": {"foam": 1.6e-6, "batch": 1.3e-7, "cg": 1.1e-7, "mixed": 1.1e-7,
                    "adjoint": 2.6e-8, "gamg": 2e-9, "multi": 2e-9}[case["kind"]]}


def _cg(A, b, tol=1e-15, cap=30000):
    """Conjugate gradients in 64 bits with restarts from the true residual."""
    x = torch.zeros_like(b)
    bn = torch.linalg.vector_norm(b)
    for _ in range(4):
        r = b - A(x)
        if torch.linalg.vector_norm(r) <= 1e-14 * bn:
            break
        p, rho = r.clone(), torch.dot(r, r)
        target = float((tol * bn) ** 2)
        for k in range(cap):
            q = A(p)
            alpha = rho / torch.dot(p, q)
            x += alpha * p
            r -= alpha * q
            new = torch.dot(r, r)
            p = r + (new / rho) * p
            rho = new
            if k % 20 == 19 and float(rho) <= target:
                break
    return x


def _bicgstab(A, b, tol=1e-15, cap=5000):
    x = torch.zeros_like(b)
    bn = torch.linalg.vector_norm(b)
    for _ in range(6):
        r = b - A(x)
        if torch.linalg.vector_norm(r) <= 1e-14 * bn:
            break
        rs, p, rho = r.clone(), r.clone(), torch.dot(r, r)
        target = float((tol * bn) ** 2)
        for k in range(cap):
            v = A(p)
            alpha = rho / torch.dot(rs, v)
            s = r - alpha * v
            t = A(s)
            omega = torch.dot(t, s) / torch.dot(t, t)
            x += alpha * p + omega * s
            r = s - omega * t
            if float(torch.dot(r, r)) <= target:
                break
            new = torch.dot(rs, r)
            p = r + (new / rho) * (alpha / omega) * (p - omega * v)
            rho = new
    return x


def exact(case: dict, seed: int):
    """The systems' solutions (and gradients) in plain 64-bit torch."""
    kind = case["kind"]
    if kind == "batch":
        x = torch.cat([_cg(h.matvec, b) for h, b in _batch_systems(case, seed)])
        return {"x": x, "iterations": None}
    h, b, x0 = _system(case, seed)
    solve = _cg if h.lo is h.up else _bicgstab
    if kind == "multi":
        return {"x": torch.stack([solve(h.matvec, v) for v in b]), "iterations": None}
    x = solve(h.matvec, b[0])
    if kind == "foam":
        psi = torch.empty_like(x)
        psi[h.order(case["numbering"])] = x
        initial = float(torch.linalg.vector_norm(b[0] - h.matvec(x0)))
        return {"psi": psi.cpu().numpy(), "initial_residual": initial, "n_iterations": None}
    if kind == "adjoint":
        lam = solve(h.matvec, x0)
        c = torch.arange(h.N, device=DEVICE)
        own = c.unsqueeze(1).expand(-1, 3)[h.ok]
        nbr = torch.stack([c + s for s in h.steps], 1)[h.ok]
        return {"x": x, "diag": -lam * x, "lower": -lam[nbr] * x[own],
                "upper": -lam[own] * x[nbr], "b": lam}
    return {"x": x, "iterations": None}
