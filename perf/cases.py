"""The work that users of this package have it do, as measurable cases.

Each case is one pass through the package's public entry points:

  call       one drop-in chunk call NLSEmagic{1,2,3}D_Take_Steps_GPU on host arrays
  solver     a resident Solver: `frames` chunks of `chunk` RK4 steps, the
             diagnostics of every chunk, then the state
  group      resident 2D solvers of several sizes advanced together (Group)
  batch      many uneven 2D problems advanced together (Batch)
  vorticity  the vorticity of a resident 3D state into device arrays

Sizes follow the package's own workloads: 1D 400-65536 points (N = 2048 with
MSD walls), 2D 64-1024 per side (1024^2 with MSD walls; batches of sides
64-512), 3D 48-256 per side (256^3 Dirichlet); CD and 2SHOC; double (2),
single (1) and compensated single (3) precision; Dirichlet (1), MSD (2) and
Lap0 (3) boundaries; V = 0 or a harmonic trap V = -omega^2 |x|^2.  Time steps
are the reference drivers' k = 0.8 klin.

exact() restates the equations in plain 64-bit torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import nlsemagic_amd as nm

VEPS = 1e-3  # the vorticity's division guard


def _solver(name, shape, method, precision, BC, frames, chunk, omega=0.0):
    n = tuple(shape) + (1, 1)
    return {"name": name, "kind": "solver", "dim": len(shape), "n0": n[0], "n1": n[1], "n2": n[2], "method": method,
            "precision": precision, "BC": BC, "omega": omega, "frames": frames, "chunk": chunk}


def _call(name, shape, method, precision, BC, chunk, omega=0.0):
    c = _solver(name, shape, method, precision, BC, 1, chunk, omega)
    c["kind"] = "call"
    return c


def _many(kind, name, count, lo, hi, sizes, method, precision, BC, chunk):
    return {"name": name, "kind": kind, "dim": 2, "count": count, "lo": lo, "hi": hi, "sizes": sizes,
            "method": method, "precision": precision, "BC": BC, "frames": 1, "chunk": chunk}


def _vort(name, shape, precision):
    return {"name": name, "kind": "vorticity", "dim": 3, "n0": shape[0], "n1": shape[1], "n2": shape[2], "method": 1,
            "precision": precision, "BC": 1, "omega": 0.0, "frames": 0, "chunk": 0}


def listed():
    return [
        _call("1d-call-401-cd", (401,), 1, 2, 3, 25),
        _solver("1d-2048-cd-msd", (2048,), 1, 2, 2, 5, 100),
        _solver("1d-50021-2shoc-f32c", (50021,), 2, 3, 1, 4, 100, 0.0018),
        _call("2d-call-131x150-cd-lap0", (131, 150), 1, 2, 3, 20),
        _solver("2d-1024-2shoc-msd", (1024, 1024), 2, 2, 2, 10, 50),
        _solver("2d-901x1013-cd-msd-f32", (901, 1013), 1, 1, 2, 10, 50),
        _many("group", "2d-group-5-2shoc", 5, 128, 700, 7, 2, 2, 2, 100),
        _many("batch", "2d-batch-96-2shoc-f32c", 96, 64, 512, 1, 2, 3, 1, 100),
        _solver("3d-256-2shoc", (256, 256, 256), 2, 2, 1, 4, 50),
        _solver("3d-157x149x163-cd-msd", (157, 149, 163), 1, 2, 2, 5, 50),
        _solver("3d-97x120x111-2shoc-msd-f32c", (97, 120, 111), 2, 3, 2, 4, 100, 0.08),
        _vort("3d-vorticity-201x180x190", (201, 180, 190), 2),
    ]


def _lu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["1d", "1d", "2d", "2d", "2d", "3d", "3d", "3d", "call", "call", "group", "batch", "vorticity"])
    method, precision, BC = rng.choice([1, 2]), rng.choice([1, 2, 3]), rng.choice([1, 2, 3])

    def omega(shape):  # no trap, or one of depth |V| <= 20 at the corners
        r = _h(len(shape)) * math.hypot(*shape) / 2
        return rng.choice([0.0, round(min(rng.uniform(0.05, 0.1), math.sqrt(20.0) / r), 6)])

    if kind == "1d":
        shape = (_lu(rng, 400, 65536),)
        c = _solver("", shape, method, precision, BC, rng.randint(1, 5), rng.randint(50, 100), omega(shape))
    elif kind == "2d":
        shape = (_lu(rng, 64, 1024), _lu(rng, 64, 1024))
        c = _solver("", shape, method, precision, BC, rng.randint(1, 10), rng.randint(20, 50), omega(shape))
    elif kind == "3d":
        shape = tuple(_lu(rng, 48, 192) for _ in range(3))
        c = _solver("", shape, method, precision, BC, rng.randint(1, 4), rng.randint(20, 50), omega(shape))
    elif kind == "call":
        dim = rng.choice([1, 2, 3])
        shape = tuple(_lu(rng, *((400, 65536), (64, 1024), (48, 160))[dim - 1]) for _ in range(dim))
        c = _call("", shape, method, rng.choice([1, 2]), BC, _lu(rng, 10, 100), omega(shape))
    elif kind == "group":
        c = _many("group", "", rng.randint(2, 8), 128, 700, rng.randint(2, 1 << 20), method, rng.choice([2, 3]), BC,
                  rng.randint(50, 100))
    elif kind == "batch":
        c = _many("batch", "", _lu(rng, 8, 96), 64, 512, rng.randint(2, 1 << 20), method, rng.choice([2, 3]),
                  BC, rng.randint(50, 100))
    else:
        c = _vort("", tuple(_lu(rng, 48, 256) for _ in range(3)), rng.choice([1, 2, 3]))
    del c["name"]
    return c


# ---- shapes, steps and initial states

def _shape(case):
    return tuple(case[k] for k in ("n0", "n1", "n2")[:case["dim"]])


def _problems(case):
    """Per problem of a group or batch: shape, s, a, omega."""
    rng = np.random.default_rng(case["sizes"])
    out = []
    for _ in range(case["count"]):
        n = np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]), 2)).round().astype(int)
        shape = (int(n[0]), int(n[0])) if case["kind"] == "batch" else (int(n[0]), int(n[1]))
        out.append((shape, float(rng.choice([-1.0, 1.0])), float(rng.uniform(0.5, 1.0)),
                    float(rng.uniform(0.05, 0.2)) if case["kind"] == "batch" else 0.0))
    return out


def _h(dim):
    return 0.2 if dim == 3 else 0.1


def _k(dim, method, a):
    return 0.8 * (1.0 if method == 1 else 0.75) * _h(dim) ** 2 / (dim * math.sqrt(2) * a)


def _axes(shape):
    h, dim = _h(len(shape)), len(shape)
    ax = [h * (torch.arange(n, dtype=torch.float64, device="cuda") - (n - 1) / 2) for n in shape]
    return [x.reshape([-1 if d == e else 1 for e in range(dim)]) for d, x in enumerate(ax)]


def _field(shape, s, omega, g):
    """(U, V) on the GPU: dark solitons, vortices or vortex rings on a uniform
    background (s < 0) or a bright Gaussian (s > 0), plus complex uniform
    noise of amplitude 1e-3; V = -omega^2 |x|^2."""
    X = _axes(shape)
    dim = len(shape)
    r = lambda: 2.0 * torch.rand((), dtype=torch.float64, generator=g, device="cuda") - 1.0  # noqa: E731
    size = [_h(dim) * n / 2 for n in shape]
    r2 = sum(x * x for x in X)
    if s > 0:
        U = torch.exp(-r2 / 2) * torch.exp(1j * 0.1 * r() * X[0])
    elif dim == 1:
        U = torch.tanh((X[0] - 0.25 * size[0] * r()) / math.sqrt(2)) + 0j
    elif dim == 2:
        U = torch.ones(shape, dtype=torch.complex128, device="cuda")
        for m in (1, -1):
            x, y = X[0] - 0.5 * size[0] * r(), X[1] - 0.5 * size[1] * r()
            U = U * torch.tanh(torch.hypot(x, y)) * torch.exp(1j * m * torch.atan2(y, x))
    else:
        U = torch.ones(shape, dtype=torch.complex128, device="cuda")
        for m in (1, -1):
            x, y, z = X[0] - 0.2 * size[0] * r(), X[1] - 0.2 * size[1] * r(), X[2] - 0.2 * size[2] * r()
            rho = torch.hypot(y, z) - 0.5 * min(size)
            U = U * torch.tanh(torch.hypot(x, rho) / math.sqrt(2)) * torch.exp(1j * m * torch.atan2(x, rho))
    U = U + 1e-3 * torch.complex(2 * torch.rand(shape, dtype=torch.float64, generator=g, device="cuda") - 1,
                                 2 * torch.rand(shape, dtype=torch.float64, generator=g, device="cuda") - 1)
    V = (-omega * omega * r2).expand(shape) if omega else torch.zeros(shape, dtype=torch.float64, device="cuda")
    return U, V


def _inputs(case, seed):
    """[(shape, s, a, U, V)] of a case's problems, on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    if case["kind"] in ("group", "batch"):
        return [(sh, s, a, *_field(sh, s, om, g)) for sh, s, a, om in _problems(case)]
    return [(_shape(case), -1.0, 1.0, *_field(_shape(case), -1.0, case["omega"], g))]


def prepare(case, seed):
    dim, method, prec, BC = case["dim"], case["method"], case["precision"], case["BC"]
    h2 = _h(dim) ** 2
    probs = [(sh, s, a, U.cpu().numpy(), V.contiguous().cpu().numpy()) for sh, s, a, U, V in _inputs(case, seed)]
    st = {"case": case}
    if case["kind"] == "call":
        sh, s, a, U, V = probs[0]
        gateway = getattr(nm, f"NLSEmagic{dim}D_Take_Steps_GPU")
        st["call"] = lambda: gateway(U, V, s, a, h2, BC, case["chunk"], _k(dim, method, a), prec, method)
    elif case["kind"] == "batch":
        st["batch"] = nm.Batch([p[0] for p in probs], [p[1] for p in probs], [p[2] for p in probs], h2,
                               [_k(dim, method, p[2]) for p in probs], method=method, precision=prec, BC=BC)
        for i, p in enumerate(probs):
            st["batch"].set_state(i, p[3], p[4])
    else:
        st["solvers"] = []
        for sh, s, a, U, V in probs:
            S = nm.Solver(sh, method, prec, BC, s, a, h2, _k(dim, method, a))
            S.set_state(U, V)
            st["solvers"].append(S)
        if case["kind"] == "vorticity":
            st["out"] = [torch.empty(_shape(case), dtype=torch.float64, device="cuda") for _ in range(4)]
            torch.cuda.synchronize()
    return st


def run(st):
    case = st["case"]
    if case["kind"] == "call":
        return {"U": st["call"]()}
    if case["kind"] == "solver":
        S, diag = st["solvers"][0], []
        for _ in range(case["frames"]):
            S.step(case["chunk"])
            diag.append(S.diagnostics())
        return {"diagnostics": diag, "U": S.state()}
    if case["kind"] == "group":
        G = nm.Group(st["solvers"])
        G.step(case["chunk"])
        G.sync()
        G.close()
        return {"U": [S.state() for S in st["solvers"]]}
    if case["kind"] == "batch":
        B = st["batch"]
        B.step(case["chunk"])
        return {"diagnostics": B.diagnostics(), "U": np.concatenate([B.state(i).ravel() for i in range(case["count"])])}
    S = st["solvers"][0]
    S.vorticity_device(1 / (2 * _h(3)), VEPS, *[t.data_ptr() for t in st["out"]])
    S.sync()
    return {"w": st["out"]}


# real operations of one point and one RK4 step: four right-hand sides (the
# stencil, the nonlinear term) and stage updates
_FLOPS = {(1, 1): 92, (1, 2): 132, (2, 1): 108, (2, 2): 196, (3, 1): 124, (3, 2): 292}


def work(case):
    if case["kind"] in ("group", "batch"):
        n = sum(sh[0] * sh[1] for sh, *_ in _problems(case))
    else:
        n = math.prod(_shape(case))
    c = {1: 8, 2: 16, 3: 16}[case["precision"]]  # a resident point (compensated: two floats per part)
    v = 8 if case["precision"] == 2 else 4
    if case["kind"] == "vorticity":
        return {"bytes": (c + 32) * n, "flops": 60 * n}
    steps = case["frames"] * case["chunk"]
    return {"bytes": (2 * c + v) * n, "flops": _FLOPS[case["dim"], case["method"]] * n * steps}


# ---- the same results in plain 64-bit torch

def _sl(dim, off):
    """The slice of an array at `off` from its interior points."""
    return tuple(slice(1 + o, None if o == 1 else o - 1) for o in off)


def _units(dim):
    return [tuple(sg if e == d else 0 for e in range(dim)) for d in range(dim) for sg in (1, -1)]


def _diagonals(dim):
    return [tuple({d: p, e: q}.get(f, 0) for f in range(dim)) for d in range(dim) for e in range(d + 1, dim)
            for p in (1, -1) for q in (1, -1)]


class _Rhs:
    """F(U) = i (a Lap U + (s|U|^2 - V) U) with the scheme and the boundary rules."""

    def __init__(self, shape, V, s, a, h2, method, BC):
        self.dim, self.V, self.s, self.a, self.h2, self.method, self.BC = len(shape), V, s, a, h2, method, BC
        self.inner = _sl(self.dim, (0,) * self.dim)
        if BC == 2:  # each boundary point and its partner: the coordinates clamped into the interior
            mask = torch.ones(shape, dtype=torch.bool, device=V.device)
            mask[self.inner] = False
            at = mask.nonzero(as_tuple=True)
            self.at = at
            self.to = tuple(x.clamp(1, n - 2) for x, n in zip(at, shape))

    def lap(self, U):
        out = (-2.0 * self.dim) * U[self.inner]
        for o in _units(self.dim):
            out += U[_sl(self.dim, o)]
        return out.div_(self.h2)

    def __call__(self, U):
        a, dim, inner = self.a, self.dim, self.inner
        N = self.s * (U.real * U.real + U.imag * U.imag) - self.V
        if self.method == 1:
            L = a * self.lap(U)
        else:
            if self.BC == 1:
                D = (-1.0 / a) * N * U
            else:
                D = torch.zeros_like(U)
            D[inner] = self.lap(U)
            if self.BC == 2:
                uq, ub = U[self.to], U[self.at]
                A = (D[self.to] * uq.conj()).real / (uq * uq.conj()).real
                D[self.at] = (A + (N[self.to] - N[self.at]) / a) * ub
            L = (a * {1: 7.0 / 6.0, 2: 1.0, 3: 10.0 / 12.0}[dim]) * D[inner]
            for o in _units(dim):
                L -= (a / 12.0) * D[_sl(dim, o)]
            if dim > 1:
                E = (-4.0 if dim == 2 else -12.0) * U[inner]
                for o in _diagonals(dim):
                    E += U[_sl(dim, o)]
                L += (a / (6.0 * self.h2)) * E
        if self.BC == 3:
            F = 1j * (N * U)
        else:
            F = torch.zeros_like(U)
        F[inner] = 1j * (L + N[inner] * U[inner])
        if self.BC == 2:
            F[self.at] = 1j * (F[self.to] / U[self.to]).imag * U[self.at]
        return F


def _advance(U, rhs, k, steps):
    for _ in range(steps):
        K = rhs(U)
        acc = K.clone()
        K = rhs(U + (k / 2) * K)
        acc += 2 * K
        K = rhs(U + (k / 2) * K)
        acc += 2 * K
        K = rhs(U + k * K)
        acc += K
        U = U + (k / 6) * acc
    return U


def _diag(U):
    return float((U.real ** 2 + U.imag ** 2).sum()), float(U.real.max()), int((~torch.isfinite(U.abs())).sum())


def _grad(A, lh2):
    """Differences of A along the three axes: central inside, one-sided on
    the faces (the second and third axes' faces take the first axis'
    difference forward), 0 on edges and corners."""
    out = []
    for d in range(3):
        G = torch.zeros_like(A)
        up = tuple(1 if e == d else 0 for e in range(3))
        dn = tuple(-u for u in up)
        G[_sl(3, (0, 0, 0))] = lh2 * (A[_sl(3, up)] - A[_sl(3, dn)])
        for f in range(3):
            for end in (0, -1):
                face = lambda o: tuple((end + (o if end == 0 else -o) if e == f else slice(1, -1)) for e in range(3))  # noqa: E731
                if d == f:
                    G[face(0)] = 2 * lh2 * ((A[face(1)] - A[face(0)]) if end == 0 else (A[face(0)] - A[face(1)]))
                else:
                    sh = lambda o: tuple(end if e == f else (slice(1 + o, None if o == 1 else o - 1) if e == d else slice(1, -1))  # noqa: E731
                                         for e in range(3))
                    G[face(0)] = 2 * lh2 * (A[sh(1)] - A[sh(0)]) if d == 0 else lh2 * (A[sh(1)] - A[sh(-1)])
        out.append(G)
    return out


def _vorticity(U, lh2, veps):
    q = 2 * U.real ** 2 + 2 * U.imag ** 2 + veps
    vx, vy, vz = [(U.real * gi - U.imag * gr) / q for gr, gi in zip(_grad(U.real, lh2), _grad(U.imag, lh2))]
    (_, xy, xz), (yx, _, yz), (zx, zy, _) = _grad(vx, lh2), _grad(vy, lh2), _grad(vz, lh2)
    w = [zy - yz, xz - zx, yx - xy]
    return w + [torch.sqrt(w[0] ** 2 + w[1] ** 2 + w[2] ** 2)]


def exact(case, seed):
    dim, method = case["dim"], case["method"]
    h2 = _h(dim) ** 2
    inputs = _inputs(case, seed)
    if case["kind"] == "vorticity":
        return {"w": _vorticity(inputs[0][3], 1 / (2 * _h(3)), VEPS)}
    diag, states = [], []
    for sh, s, a, U, V in inputs:
        rhs = _Rhs(sh, V, s, a, h2, method, case["BC"])
        for _ in range(case["frames"]):
            U = _advance(U, rhs, _k(dim, method, a), case["chunk"])
            diag.append(_diag(U))
        states.append(U)
    if case["kind"] == "call":
        return {"U": states[0]}
    if case["kind"] == "solver":
        return {"diagnostics": diag, "U": states[0]}
    if case["kind"] == "group":
        return {"U": states}
    return {"diagnostics": np.array(diag, dtype=float), "U": torch.cat([u.reshape(-1) for u in states])}
