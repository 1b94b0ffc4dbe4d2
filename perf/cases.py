"""The work that programs built on this library give it, as measurable cases.

A case is one call, or the few calls that belong together, through
solver_cpp_amd's public entry points on device tensors: a product with a
sparse matrix, the vector operations around it, a whole Krylov solve, or a
differentiable solve with its backward pass.  The matrices are the ones that
the benchmark and the tests solve (5- and 7-point stencils, a log-normal
anisotropic Laplacian, random rows of Zipf length), assembled here with torch
so that their coefficients and right-hand sides come from a seed.
"""
import math

import torch

from solver_cpp_amd import api, autograd

F64 = torch.float64
_CTX = None


def _context():
    """The process's one solver context, as a program keeps it."""
    global _CTX
    if _CTX is None:
        _CTX = api.Context(0)
    return _CTX


def listed():
    return [
        # the vector operations a caller's own iteration makes, at a length that is a multiple of nothing
        dict(name="blas_100003", op="blas", n=100003),
        # the smallest product in use: one residual check on a 256 x 256 grid
        dict(name="spmv_poisson2d_256", op="spmv", matrix="poisson", dim=2, nx=256, ny=256, nz=1, precision=64,
             trans=False),
        # the pair of products of a two-sided method, on a grid of odd edges
        dict(name="spmv_pair_131x127x125", op="spmv", matrix="convdiff", dim=3, nx=131, ny=127, nz=125, precision=64,
             trans=True),
        # the product of a mixed solver's inner level on the largest grid in use
        dict(name="spmv_fp32_192", op="spmv", matrix="convdiff", dim=3, nx=192, ny=192, nz=192, precision=32,
             trans=False),
        # rows of very different length with columns from all over: graphs, networks
        dict(name="spmv_zipf_4m", op="spmv", matrix="zipf", n=4000000, cap=4096, precision=64, trans=False),
        # a small symmetric solve, many short iterations
        dict(name="cg_poisson2d_256", op="solve", matrix="poisson", dim=2, nx=256, ny=256, nz=1, solver="cg"),
        # nonsymmetric solves of a medium grid: two-sided, and restarted with a long basis
        dict(name="bicg_convdiff3d_128", op="solve", matrix="convdiff", dim=3, nx=128, ny=128, nz=128, solver="bicg"),
        dict(name="gmres_convdiff3d_128", op="solve", matrix="convdiff", dim=3, nx=128, ny=128, nz=128,
             solver="gmres"),
        # the communication-avoiding solve: matrix powers and Gram products
        dict(name="kskipcg_poisson3d_96", op="solve", matrix="poisson", dim=3, nx=96, ny=96, nz=96, solver="kskipcg"),
        # the mixed-precision solve that the benchmark is about: FP64 outside, ten FP32 steps inside
        dict(name="vpgmres_poisson3d_160", op="solve", matrix="poisson", dim=3, nx=160, ny=160, nz=160,
             solver="vpgmres"),
        # learning the coefficients of a diffusion problem: solve, and the gradient by the symmetric adjoint
        dict(name="grad_aniso2d_300", op="grad", matrix="aniso", dim=2, nx=300, ny=300, nz=1, solver="vpcg"),
        # the same through a random matrix with rows scaled, adjoint on the explicit transpose
        dict(name="grad_zipf_1m", op="grad", matrix="zipf", n=1000000, cap=4096, solver="vpgmres"),
    ]


def _edge(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, dim, lo, hi):
    """A box of about e^dim points, e spread over [lo, hi] by its logarithm, its edges near e but seldom equal."""
    e = _edge(rng, lo, hi)
    near = [max(4, min(hi, int(e * rng.uniform(0.85, 1.15)))) for _ in range(dim)]
    return dict(dim=dim, nx=near[0], ny=near[1], nz=near[2] if dim == 3 else 1)


def draw(rng):
    kind = rng.choice(["blas", "spmv2", "spmv3", "spmv3", "zipf", "cg", "bicg", "gmres", "kskipcg", "vpgmres", "aniso",
                       "gradzipf"])
    if kind == "blas":
        return dict(op="blas", n=_edge(rng, 1000, 4000000))
    if kind in ("spmv2", "spmv3"):
        g = _grid(rng, 2, 64, 1024) if kind == "spmv2" else _grid(rng, 3, 16, 192)
        return dict(op="spmv", matrix=rng.choice(["poisson", "convdiff"]), precision=rng.choice([64, 32]),
                    trans=rng.random() < 0.5, **g)
    if kind == "zipf":
        return dict(op="spmv", matrix="zipf", n=_edge(rng, 3000, 3000000), cap=rng.choice([300, 4096]),
                    precision=rng.choice([64, 32]), trans=rng.random() < 0.5)
    if kind == "cg":
        g = _grid(rng, 2, 64, 512) if rng.random() < 0.5 else _grid(rng, 3, 16, 128)
        return dict(op="solve", matrix="poisson", solver="cg", **g)
    if kind in ("bicg", "gmres"):
        return dict(op="solve", matrix="convdiff", solver=kind, **_grid(rng, 3, 16, 128))
    if kind == "kskipcg":
        return dict(op="solve", matrix="poisson", solver="kskipcg", **_grid(rng, 3, 24, 112))
    if kind == "vpgmres":
        return dict(op="solve", matrix=rng.choice(["poisson", "convdiff"]), solver="vpgmres", **_grid(rng, 3, 32, 150))
    if kind == "aniso":
        return dict(op="grad", matrix="aniso", solver="vpcg", **_grid(rng, 2, 48, 340))
    return dict(op="grad", matrix="zipf", n=_edge(rng, 20000, 1000000), cap=rng.choice([300, 4096]), solver="vpgmres")


# ---------------------------------------------------------------- matrices --
def _rows(case):
    return case["n"] if "n" in case else case["nx"] * case["ny"] * case["nz"]


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(1000003 * (int(seed) % (1 << 40)) + salt)


def _from_bands(n, bands):
    """CSR of a matrix given as (column offset, present, value) per band, offsets ascending; values broadcast over n."""
    has = torch.stack([h for _, h, _ in bands], 1)
    row = torch.arange(n, device="cuda")
    ptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    ptr[1:] = torch.cumsum(has.sum(1), 0)
    col = torch.stack([row + o for o, _, _ in bands], 1)[has]
    val = torch.stack([v.to(F64).expand(n) for _, _, v in bands], 1)[has]
    return ptr.int(), col.int(), val.contiguous()


def _stencil(case, seed):
    """5- / 7-point Laplacian, or first-order upwind convection-diffusion with a flow whose direction comes from the
    seed (Peclet number 0.5)."""
    dim, e = case["dim"], [case["nx"], case["ny"], case["nz"]]
    n = _rows(case)
    at = torch.arange(n, device="cuda")
    pos, step = [], []
    s = 1
    for d in range(dim):
        pos.append(at // s % e[d])
        step.append(s)
        s *= e[d]
    c = torch.zeros(3, dtype=F64, device="cuda")
    if case["matrix"] == "convdiff":
        vel = 0.25 + 0.75 * torch.rand(3, generator=_gen(seed, 1), dtype=F64, device="cuda")
        c = vel / vel.max()  # 2 Pe v_d / max v
    low = [(-step[d], pos[d] > 0, -1 - c[d]) for d in reversed(range(dim))]
    high = [(step[d], pos[d] < e[d] - 1, -torch.ones((), dtype=F64, device="cuda")) for d in range(dim)]
    mid = (0, torch.ones(n, dtype=torch.bool, device="cuda"), 2 * dim + c[:dim].sum())
    return _from_bands(n, low + [mid] + high)


def _aniso(case, seed):
    """Graph Laplacian on a grid with log-normal conductivities on its edges, the boundary's included."""
    nx, ny = case["nx"], case["ny"]
    kx = torch.randn(ny, nx + 1, generator=_gen(seed, 2), dtype=F64, device="cuda").exp()
    ky = torch.randn(ny + 1, nx, generator=_gen(seed, 3), dtype=F64, device="cuda").exp()
    w, e, s, t = kx[:, :-1].reshape(-1), kx[:, 1:].reshape(-1), ky[:-1].reshape(-1), ky[1:].reshape(-1)
    at = torch.arange(nx * ny, device="cuda")
    x, y = at % nx, at // nx
    yes = torch.ones_like(x, dtype=torch.bool)
    return _from_bands(nx * ny, [(-nx, y > 0, -s), (-1, x > 0, -w), (0, yes, w + e + s + t), (1, x < nx - 1, -e),
                                 (nx, y < ny - 1, -t)])


def _zipf(case, seed):
    """Random rows of Zipf(1.5) length up to cap (the same lengths for every seed, in another order), columns anywhere,
    the diagonal 1.1 times the row's other entries."""
    n, g = case["n"], _gen(seed, 4)
    p = torch.arange(1, min(case["cap"], n) + 1, dtype=F64, device="cuda").pow(-1.5)
    cdf = torch.cumsum(p, 0) / p.sum()
    at = (torch.arange(n, dtype=F64, device="cuda") + 0.5) / n
    cnt = (torch.searchsorted(cdf, at) + 1).clamp(max=len(p))[torch.randperm(n, generator=g, device="cuda")]
    ptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    ptr[1:] = torch.cumsum(cnt, 0)
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), cnt)
    col = torch.randint(0, n - 1, row.shape, generator=g, device="cuda")
    col += col >= row  # not the diagonal ...
    col[ptr[:-1]] = torch.arange(n, device="cuda")  # ... which each row's first entry is, before the sort
    col = torch.sort(row * n + col)[0] % n
    val = torch.randn(row.shape, generator=g, dtype=F64, device="cuda")
    diag = col == row
    other = torch.segment_reduce(val.abs().masked_fill_(diag, 0), "sum", lengths=cnt)
    val[diag] = torch.where(cnt > 1, 1.1 * other, torch.ones_like(other))
    return ptr.int(), col.int(), val


def _matrix(case, seed):
    return {"poisson": _stencil, "convdiff": _stencil, "aniso": _aniso, "zipf": _zipf}[case["matrix"]](case, seed)


def _vector(case, seed, salt, normal=False):
    n = _rows(case)
    if normal:
        return torch.randn(n, generator=_gen(seed, salt), dtype=F64, device="cuda")
    return 2 * torch.rand(n, generator=_gen(seed, salt), dtype=F64, device="cuda") - 1


# ------------------------------------------------------------------- cases --
# solver settings: the benchmark's, at tolerances between its 1e-10 and 1e-14
_MIXED = dict(outer_restart=21, outer_maxloop=5000, inner_maxloop=11, inner_restart=12, inner_eps=0.0,
              inner_precision=32)
_SOLVE = {
    "cg": dict(outer_eps=1e-12, outer_maxloop=20000),
    "bicg": dict(outer_eps=1e-12, outer_maxloop=20000),
    "gmres": dict(outer_eps=1e-12, outer_maxloop=20000, outer_restart=31),
    "kskipcg": dict(outer_eps=1e-12, outer_maxloop=20000, outer_kskip=2),
    "vpgmres": dict(outer_eps=1e-12, **_MIXED),
}


def prepare(case, seed):
    ctx = _context()
    if case["op"] == "blas":
        return dict(case=case, ctx=ctx, x=_vector(case, seed, 5), y=_vector(case, seed, 6, True))
    ptr, col, val = _matrix(case, seed)
    if case["op"] == "grad":
        sym = case["matrix"] == "aniso"
        tight = dict(outer_eps=1e-12 if sym else 1e-14, outer_maxloop=20000)
        system = autograd.SparseSystem(
            ctx, ptr.cpu().numpy(), col.cpu().numpy(), spd=sym, row_scale=not sym, fp32=True, solver=case["solver"],
            inner="cg" if sym else "gmres",
            params=dict(tight, inner_maxloop=10, inner_precision=32) if sym else dict(_MIXED, **tight),
            adjoint_solver="cg" if sym else "gmres", adjoint_inner="NO",
            adjoint_params=tight if sym else dict(tight, outer_restart=21))
        return dict(case=case, system=system, val=val.requires_grad_(), b=_vector(case, seed, 5).requires_grad_(),
                    target=_vector(case, seed, 6, True))
    two = case["op"] == "spmv" and case["trans"] or case.get("solver") == "bicg"
    single = case.get("precision") == 32 or case.get("solver") == "vpgmres"
    A = api.Matrix(ctx, ptr, col, val, transpose=two, fp32=single)
    if case["op"] == "solve":
        return dict(case=case, ctx=ctx, A=A, b=_vector(case, seed, 5))
    x = _vector(case, seed, 6, True)
    y = _vector(case, seed, 7, True) if case["trans"] else None
    if case["precision"] == 32:
        x, y = x.float(), None if y is None else y.float()
    return dict(case=case, A=A, x=x, y=y)


def run(s):
    case = s["case"]
    if case["op"] == "blas":
        ctx, x, y = s["ctx"], s["x"], s["y"]
        return ctx.dot(x, y), ctx.norm2(x), ctx.axpy(0.75, x, y)
    if case["op"] == "spmv":
        p = case["precision"]
        out = [s["A"].spmv(s["x"], precision=p)]
        if case["trans"]:
            out.append(s["A"].spmv(s["y"], trans=True, precision=p))
        return out
    if case["op"] == "solve":
        inner = "gmres" if case["solver"] == "vpgmres" else "NO"
        return api.solve(s["ctx"], s["A"], s["b"], case["solver"], inner, history=False, **_SOLVE[case["solver"]])[0]
    x = s["system"].solve(s["val"], s["b"])
    loss = 0.5 * ((x - s["target"]) ** 2).sum()
    gv, gb = torch.autograd.grad(loss, (s["val"], s["b"]))
    return x.detach(), gv, gb


# ------------------------------------------------------------- what it takes --
# Krylov steps to 1e-12 per grid edge (for the random matrix: in all), as these problems take them
_STEPS = {"cg": 3.8, "bicg": 4.3, "gmres": 4.6, "kskipcg": 4.8, "vpgmres": 0.75, "vpcg": 2.7}


def work(case):
    n = _rows(case)
    if case["op"] == "blas":
        return {"bytes": 8.0 * 6 * n, "flops": 6.0 * n}
    if case["matrix"] == "zipf":
        p = [k ** -1.5 for k in range(1, min(case["cap"], n) + 1)]
        nnz = n * sum(k * q for k, q in enumerate(p, 1)) / sum(p)
        edge = 1
    else:
        e = [case["nx"], case["ny"], case["nz"]][:case["dim"]]
        nnz = n * (2 * len(e) + 1) - 2 * sum(n / d for d in e)
        edge = n ** (1 / case["dim"])

    def product(size):
        return (size + 4) * nnz + (4 + 2 * size) * n

    if case["op"] == "spmv":
        k = 2 if case["trans"] else 1
        return {"bytes": k * product(case["precision"] // 8), "flops": k * 2.0 * nnz}
    # one step: its products, and each of its vectors read or written once per update
    inner32 = 10 * (product(4) + 4 * n * 14)
    step = {"cg": (product(8) + 8 * n * 8, 2 * nnz + 10 * n),
            "bicg": (2 * product(8) + 8 * n * 14, 4 * nnz + 18 * n),
            "gmres": (product(8) + 8 * n * 18, 2 * nnz + 64 * n),
            "kskipcg": (product(8) + 8 * n * 8, 2 * nnz + 10 * n),
            "vpcg": (product(8) + 8 * n * 8 + 10 * (product(4) + 4 * n * 8), 22 * nnz + 110 * n),
            "vpgmres": (product(8) + 8 * n * 13 + inner32, 22 * nnz + 280 * n)}
    steps = {k: v * edge for k, v in _STEPS.items()}
    if case["op"] == "solve":
        k = steps[case["solver"]]
        return {"bytes": k * step[case["solver"]][0], "flops": k * step[case["solver"]][1]}
    if case["matrix"] == "zipf":
        fwd, adj, back = 5, 39, "gmres"
    else:
        fwd, adj, back = steps["vpcg"], 4.7 * steps["cg"], "cg"
    outer = 12.0 * nnz  # the gradient of the values
    return {"bytes": fwd * step[case["solver"]][0] + adj * step[back][0] + outer,
            "flops": fwd * step[case["solver"]][1] + adj * step[back][1] + nnz}


# ------------------------------------------------------------- in 64 bits --
class _Csr:
    """A x and A^T x with torch's own operations."""

    def __init__(self, ptr, col, val):
        self.n = len(ptr) - 1
        self.col, self.val = col.long(), val
        self.row = torch.repeat_interleave(torch.arange(self.n, device="cuda"), (ptr[1:] - ptr[:-1]).long())
        self.order = None

    @staticmethod
    def _sum(idx, w, n):
        return torch.segment_reduce(w, "sum", lengths=torch.bincount(idx, minlength=n))

    def mul(self, x):
        return self._sum(self.row, self.val * x[self.col], self.n)

    def tmul(self, x):
        if self.order is None:
            self.order = torch.sort(self.col, stable=True)[1]
        o = self.order
        return self._sum(self.col, (self.val * x[self.row])[o], self.n)

    def diag(self):
        on = self.row == self.col
        return self.val[on]


def _bicgstab(mul, d, b, tol, most):
    """Right-preconditioned by the diagonal d; returns x and the residual it reached, relative."""
    x, r = torch.zeros_like(b), b.clone()
    r0, p, rho = r.clone(), r.clone(), torch.dot(r, r)
    top = b.norm()
    for i in range(most):
        y = p / d
        v = mul(y)
        a = rho / torch.dot(r0, v)
        s = r - a * v
        z = s / d
        t = mul(z)
        w = torch.dot(t, s) / torch.dot(t, t)
        x += a * y + w * z
        r = s - w * t
        new = torch.dot(r0, r)
        p = r + (new / rho) * (a / w) * (p - w * v)
        rho = new
        if i % 10 == 9 and not float(r.norm() / top) > tol:
            break
    return x


def _cg(mul, d, b, tol, most):
    x, r = torch.zeros_like(b), b.clone()
    z = r / d
    p, rho, top = z.clone(), torch.dot(r, z), b.norm()
    for i in range(most):
        q = mul(p)
        a = rho / torch.dot(p, q)
        x += a * p
        r -= a * q
        z = r / d
        new = torch.dot(r, z)
        p = z + (new / rho) * p
        rho = new
        if i % 20 == 19 and not float(r.norm() / top) > tol:
            break
    return x


def _solve64(mul, d, b, sym):
    """x of A x = b, corrected until its residual no longer falls."""
    method = _cg if sym else _bicgstab
    x, best = torch.zeros_like(b), math.inf
    for _ in range(6):
        r = b - mul(x)
        off = float(r.norm() / b.norm())
        if not off < 0.5 * best:
            break
        best = off
        x = x + method(mul, d, r, 1e-9, 4000)
    return x


def exact(case, seed):
    if case["op"] == "blas":
        x, y = _vector(case, seed, 5), _vector(case, seed, 6, True)
        return float(torch.dot(x, y)), float(x.norm()), 0.75 * x + y
    A = _Csr(*_matrix(case, seed))
    if case["op"] == "spmv":
        x, y = _vector(case, seed, 6, True), _vector(case, seed, 7, True)
        if case["precision"] == 32:
            x, y = x.float().to(F64), y.float().to(F64)
        return [A.mul(x)] + ([A.tmul(y)] if case["trans"] else [])
    sym, b, d = case["matrix"] in ("poisson", "aniso"), _vector(case, seed, 5), A.diag()
    x = _solve64(A.mul, d, b, sym)
    if case["op"] == "solve":
        return x
    lam = _solve64(A.mul if sym else A.tmul, d, x - _vector(case, seed, 6, True), sym)
    return x, -lam[A.row] * x[A.col], lam
