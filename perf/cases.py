"""Performance cases of the framework: the calls a user's program makes, over the range of sizes,
value types and options that it makes them with.

Families (the ``op`` of a case)
-------------------------------
``matvec``   ``L2GMap.update`` (when the rank has ghost columns) and ``Matrix.mult``: the loop of
             a matvec program, on stencils and on irregular matrices, FP64, FP32 and BF16 values
``complex``  ``Matrix.mult`` and ``Matrix.transpmult`` of complex values (restriction and
             prolongation of a complex field)
``transp``   ``Matrix.transpmult`` of a rectangular incidence matrix (the gradient of assembled
             matrix values with respect to the edge conductivities)
``cg``       ``cg`` in FP64 to a relative residual
``ir``       ``ir_cg``: FP64 refinement around an FP32 inner solve on FP32 or BF16 values
``batch``    ``Batch.solve``: many uneven SPD systems, several right-hand sides each
``adjoint``  ``DiffusionOperator``: assemble, solve, loss, and the backward pass

Matrices are built on the GPU (torch) and handed over as the host CSR arrays that ``Matrix``
takes.  ``exact`` repeats a case in float64 torch operations: shifted slices for the stencils,
torch's own sparse product for the others, and a plain conjugate gradient with one restart to
about 1e-14 where a solve is needed.
"""
import math

import numpy as np
import torch

import spmv_amd as S
from spmv_amd import adjoint as AD

DEV = "cuda:0"
VALUE_BYTES = {"f64": 8, "f32": 4, "bf16": 2, "c64": 16, "c32": 8}
VECTOR_BYTES = {"f64": 8, "f32": 4, "bf16": 4, "c64": 16, "c32": 8}
VECTOR_DTYPE = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.float32,
                "c64": torch.complex128, "c32": torch.complex64}
DIAG = {5: 4.0, 7: 6.0, 27: 26.0}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one application in the loop of the reference demo's own CPU configuration: a 5-point
        # operator whose arrays stay in the caches, so that launches and latency count
        dict(name="matvec_5pt_512", op="matvec", kind=5, nx=512, ny=512, nz=1, ghost=0, dtype="f64"),
        # one rank's share of a large 27-point problem with a ghost plane to update: the headline
        dict(name="matvec_27pt_160_ghost", op="matvec", kind=27, nx=160, ny=160, nz=160, ghost=1,
             dtype="f64"),
        # an irregular matrix (power-law rows, columns anywhere): circuits, graphs, reordered meshes
        dict(name="matvec_random_300k", op="matvec", kind=0, n=300007, dtype="f64"),
        # a complex field on an odd-sized grid, one product and one transposed product
        dict(name="complex_7pt_63", op="complex", kind=7, nx=63, ny=65, nz=61, dtype="c64"),
        # the gradient through the assembly of a 1024 x 1024 diffusion operator
        dict(name="transp_diffusion_1024", op="transp", n=1024),
        # the smallest solves: a few hundred iterations of a system that a few CUs could hold
        dict(name="cg_5pt_64", op="cg", kind=5, nx=64, ny=64, nz=1, ghost=0, rtol=1e-8),
        # the reference's own CPU configuration, solved to 1e-8
        dict(name="cg_5pt_512", op="cg", kind=5, nx=512, ny=512, nz=1, ghost=0, rtol=1e-8),
        # a rank's share of a 27-point problem solved in FP64, the ghosts of the direction updated
        # in every iteration
        dict(name="cg_27pt_112_ghost", op="cg", kind=27, nx=112, ny=112, nz=112, ghost=1, rtol=1e-10),
        # mixed precision on the large 3D Poisson system, CSR arrays, FP32 values, to two digits
        # more than FP64 CG is asked for (one more inner solve)
        dict(name="ir_f32_7pt_256", op="ir", kind=7, nx=256, ny=256, nz=256, low="f32",
             sliced=False, adaptive=False, rtol=1e-12),
        # mixed precision with the options a tuned program sets: BF16 values in the sliced layout
        # and the adaptive inner tolerance
        dict(name="ir_bf16_sliced_7pt_160", op="ir", kind=7, nx=160, ny=160, nz=160, low="bf16",
             sliced=True, adaptive=True, rtol=1e-12),
        # many uneven systems at once, four right-hand sides each
        dict(name="batch_256", op="batch", nsys=256, lo=1000, hi=50000, sizes=17,
             nrhs=4, rtol=1e-6),
        # one training step through a diffusion solve: forward, and gradients of both inputs
        dict(name="adjoint_512", op="adjoint", n=512, rtol=1e-13),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def grid(kind, lo, hi):
        """A box of lo..hi rows whose sides differ."""
        rows = size(lo, hi)
        if kind == 5:
            nx = max(2, int(math.sqrt(rows) * rng.uniform(0.6, 1.6)))
            return dict(nx=nx, ny=max(2, rows // nx), nz=1)
        side = rows ** (1.0 / 3.0)
        nx, ny = max(2, int(side * rng.uniform(0.7, 1.4))), max(2, int(side * rng.uniform(0.7, 1.4)))
        return dict(nx=nx, ny=ny, nz=max(2, rows // (nx * ny)))

    op = rng.choice(["matvec", "matvec", "matvec", "random", "complex", "transp", "cg", "cg", "ir",
                     "batch", "adjoint"])
    if op == "matvec":
        kind = rng.choice([5, 7, 27])
        top = {5: 12e6, 7: 9e6, 27: 3.2e6}[kind]
        return dict(op=op, kind=kind, **grid(kind, 2e3, top), ghost=rng.choice([0, 1]) if kind != 5 else 0,
                    dtype=rng.choice(["f64", "f64", "f32", "bf16"]))
    if op == "random":
        return dict(op="matvec", kind=0, n=size(1000, 400000), dtype=rng.choice(["f64", "f64", "f32"]))
    if op == "complex":
        return dict(op=op, kind=7, **grid(7, 2e3, 5e5), dtype=rng.choice(["c64", "c32"]))
    if op == "transp":
        return dict(op=op, n=size(32, 1024))
    if op == "cg":
        kind = rng.choice([5, 7, 27])
        return dict(op=op, kind=kind, **grid(kind, 1e3, {5: 4e5, 7: 2e6, 27: 1e6}[kind]),
                    ghost=rng.choice([0, 1]) if kind != 5 else 0, rtol=1e-8 if kind == 5 else 1e-10)
    if op == "ir":
        return dict(op=op, kind=7, **grid(7, 1e5, 4e6), low=rng.choice(["f32", "bf16"]),
                    sliced=rng.choice([False, True]), adaptive=rng.choice([False, True]), rtol=1e-12)
    if op == "batch":
        return dict(op=op, nsys=size(16, 256), lo=1000, hi=size(4000, 50000), sizes=rng.randrange(1000),
                    nrhs=rng.choice([1, 2, 4]), rtol=1e-6)
    return dict(op=op, n=size(48, 512), rtol=1e-13)


# ---------------------------------------------------------------- matrices (torch, on the GPU)
def _rng(seed, stream):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + stream) % (1 << 62))


def _uniform(seed, stream, n, lo=-1.0, hi=1.0):
    return torch.rand(n, generator=_rng(seed, stream), device=DEV, dtype=torch.float64) * (hi - lo) + lo


def _offsets(kind):
    """(di, dj, dk) of a stencil's entries, in ascending column order."""
    r = (-1, 0, 1)
    offs = [(i, j, k) for k in r for j in r for i in r]
    if kind == 27:
        return offs
    return [o for o in offs if sum(map(abs, o)) <= 1 and (kind == 7 or o[2] == 0)]


class Csr:
    """CSR arrays on the GPU (rowptr int64, colidx int64, val float64)."""

    def __init__(self, nrows, ncols, rowptr, colidx, val):
        self.nrows, self.ncols, self.rowptr, self.colidx, self.val = nrows, ncols, rowptr, colidx, val

    def host(self):
        return (self.rowptr.to(torch.int32).cpu().numpy(), self.colidx.to(torch.int32).cpu().numpy(),
                self.val.cpu().numpy())

    def torch64(self):
        return torch.sparse_csr_tensor(self.rowptr, self.colidx, self.val, (self.nrows, self.ncols))


def _stencil(c):
    """Box stencil with Dirichlet boundaries; a ghost plane above the top holds further columns."""
    nx, ny, nz, g = c["nx"], c["ny"], c["nz"], c.get("ghost", 0)
    n = nx * ny * nz
    row = torch.arange(n, device=DEV, dtype=torch.int32)
    i, j, k = row % nx, (row // nx) % ny, row // (nx * ny)
    offs = _offsets(c["kind"])
    ok = torch.empty((n, len(offs)), dtype=torch.bool, device=DEV)
    col = torch.empty((n, len(offs)), dtype=torch.int32, device=DEV)
    for s, (di, dj, dk) in enumerate(offs):
        ok[:, s] = ((i + di >= 0) & (i + di < nx) & (j + dj >= 0) & (j + dj < ny) & (k + dk >= 0)
                    & (k + dk < nz + g))
        col[:, s] = row + (di + nx * dj + nx * ny * dk)
    rowptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(ok.sum(1), 0, out=rowptr[1:])
    colidx = col[ok]
    del col
    line = torch.tensor([DIAG[c["kind"]] if o == (0, 0, 0) else -1.0 for o in offs],
                        dtype=torch.float64, device=DEV)
    return Csr(n, n + nx * ny * g, rowptr, colidx, line.expand(n, -1)[ok])


def _apply_stencil(c, v):
    """The same operator on a float64 vector (owned entries, then the ghost plane) by slices."""
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    planes = v.numel() // (nx * ny)
    box = torch.zeros((nz + 2, ny + 2, nx + 2), dtype=v.dtype, device=DEV)
    box[1:1 + min(planes, nz + 1), 1:-1, 1:-1] = v.view(planes, ny, nx)
    out = torch.zeros((nz, ny, nx), dtype=v.dtype, device=DEV)
    for di, dj, dk in _offsets(c["kind"]):
        w = DIAG[c["kind"]] if (di, dj, dk) == (0, 0, 0) else -1.0
        out += w * box[1 + dk:1 + dk + nz, 1 + dj:1 + dj + ny, 1 + di:1 + di + nx]
    return out.reshape(-1)


def _random_spd(sizes, seed):
    """Block-diagonal SPD matrix: per system a random symmetric pattern with power-law row lengths
    in [3, 64], off-diagonal values uniform in [-1, 0], the diagonal 1.1 times their sum."""
    sizes = torch.tensor(sizes, dtype=torch.int64, device=DEV)
    first = torch.cumsum(sizes, 0) - sizes
    n = int(sizes.sum())
    base = torch.repeat_interleave(first, sizes)
    span = torch.repeat_interleave(sizes, sizes)
    u = _uniform(seed, 1, n, 0.0, 1.0)
    deg = (1.0 / (1.0 / 3 + u * (1.0 / 64 - 1.0 / 3))).long().clamp(3, 64)
    src = torch.repeat_interleave(torch.arange(n, device=DEV), (deg // 2).clamp(min=1))
    dst = base[src] + (_uniform(seed, 2, src.numel(), 0.0, 1.0) * span[src]).long()
    keep = src != dst
    src, dst = src[keep], dst[keep]
    key = torch.unique(torch.minimum(src, dst) * n + torch.maximum(src, dst))
    lo, hi = key // n, key % n
    # multiples of 2^-20, so that the sums of the diagonal are exact in any order
    w = -(torch.floor(_uniform(seed, 3, key.numel(), 0.0, 1.0) * 2.0 ** 20) + 1) * 2.0 ** -20
    me = torch.arange(n, device=DEV)
    key2, order = torch.sort(torch.cat([lo * n + hi, hi * n + lo, me * n + me]))
    rows, cols = key2 // n, key2 % n
    val = torch.cat([w, w, torch.zeros(n, dtype=torch.float64, device=DEV)])[order]
    counts = torch.bincount(rows, minlength=n)
    rowptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(counts, 0, out=rowptr[1:])
    run = torch.zeros(val.numel() + 1, dtype=torch.float64, device=DEV)
    torch.cumsum(-val, 0, out=run[1:])
    total = run[rowptr[1:]] - run[rowptr[:-1]]
    diag = torch.where(counts == 1, torch.ones_like(total), 1.1 * total)
    val = torch.where(rows == cols, diag[rows], val)
    return Csr(n, n, rowptr, cols, val)


def _general(c, seed):
    """The case's matrix as GPU CSR arrays."""
    if c["kind"] == 0:
        return _random_spd([c["n"]], seed)
    return _stencil(c)


def _matrix(A, dtype="f64", col_map=None, values=None):
    rowptr, colidx, val = A.host()
    return S.Matrix(rowptr, colidx, val if values is None else values, ncols=A.ncols,
                    col_map=col_map, dtype=dtype)


def _slab_map(c):
    """The exchange plan of the lower of two z-slabs: the upper one's first plane is ghosted here,
    and this one's last plane there."""
    n, plane = c["nx"] * c["ny"] * c["nz"], c["nx"] * c["ny"]
    return S.L2GMap(n, np.arange(n, n + plane), local_sizes=[n, n], rank=0,
                    remote_ghosts={1: np.arange(n - plane, n)})


def _batch_sizes(c):
    """Rows of the systems, log-uniform in [lo, hi]: the case's own, whatever the seed."""
    u = _uniform(c["sizes"], 4, c["nsys"], 0.0, 1.0).cpu().numpy()
    return np.exp(np.log(c["lo"]) + u * (np.log(c["hi"]) - np.log(c["lo"]))).astype(np.int64).tolist()


# ---------------------------------------------------------------- inputs from the seed
def _owned(c):
    return c["nx"] * c["ny"] * c["nz"]


def _matvec_inputs(c, seed):
    """x (owned entries) and the halo that the neighbour sends, rounded to the vector type."""
    dt = VECTOR_DTYPE[c["dtype"]]
    if c["kind"] == 0:
        return _uniform(seed, 11, c["n"]).to(dt), None
    halo = _uniform(seed, 12, c["nx"] * c["ny"]).to(dt) if c.get("ghost") else None
    return _uniform(seed, 11, _owned(c)).to(dt), halo


def _complex_inputs(c, seed, nnz):
    """Values, x and the transposed product's x."""
    n = _owned(c)
    pair = lambda k, m: torch.complex(_uniform(seed, k, m), _uniform(seed, k + 1, m))  # noqa: E731
    dt = VECTOR_DTYPE[c["dtype"]]
    return pair(21, nnz), pair(23, n).to(dt), pair(25, n).to(dt)


def _cg_rhs(c, seed):
    """The reference's 5-point configuration solves for a known x; the others take b as it comes."""
    x = _uniform(seed, 31, _owned(c))
    return _apply_stencil(c, x) if c["kind"] == 5 else x


def _batch_rhs(n, nrhs, seed):
    return _uniform(seed, 41, n * nrhs).float().view(n, nrhs)


def _diffusion_inputs(c, seed):
    """Log-normal edge conductivities, b in [0, 1], a normal target."""
    n = c["n"]
    ne = 2 * n * (n - 1) + 4 * n
    z = torch.randn(ne, generator=_rng(seed, 51), device=DEV, dtype=torch.float64)
    xt = torch.randn(n * n, generator=_rng(seed, 53), device=DEV, dtype=torch.float64)
    return torch.exp(0.5 * z), _uniform(seed, 52, n * n, 0.0, 1.0), xt


# ---------------------------------------------------------------- a pass
def prepare(case, seed):
    c, op = case, case["op"]
    if op == "matvec":
        x, halo = _matvec_inputs(c, seed)
        m = None
        if halo is not None:
            m = _slab_map(c)
            m.set_halo(halo.cpu().numpy(), dtype=S.F64 if c["dtype"] == "f64" else S.F32)
            x = torch.cat([x, torch.zeros_like(halo)])
        M = _matrix(_general(c, seed), c["dtype"], m)
        return dict(op=op, M=M, map=m, x=x, y=torch.empty(M.nrows, dtype=x.dtype, device=DEV))
    if op == "complex":
        A = _stencil(c)
        v, x, xt = _complex_inputs(c, seed, A.val.numel())
        M = _matrix(A, c["dtype"], values=v.cpu().numpy())
        M.transpmult(xt)  # the transposed copy is kept with the matrix
        return dict(op=op, M=M, x=x, xt=xt)
    if op == "transp":
        M = AD.DiffusionOperator(c["n"]).Pm
        g = _uniform(seed, 61, M.nrows)
        M.transpmult(g)
        return dict(op=op, M=M, g=g)
    if op == "cg":
        m = _slab_map(c) if c.get("ghost") else None  # zero halo for the direction
        return dict(op=op, M=_matrix(_stencil(c), "f64", m), b=_cg_rhs(c, seed), rtol=c["rtol"])
    if op == "ir":
        M = _matrix(_stencil(c))
        L = M.like(c["low"])
        if c["sliced"]:
            M.set_kernel(S.SLICED_VARIANT)
            L.set_kernel(S.SLICED_VARIANT)
        return dict(op=op, M=M, L=L, b=_cg_rhs(c, seed), rtol=c["rtol"], adaptive=c["adaptive"])
    if op == "batch":
        sizes = _batch_sizes(c)
        A = _random_spd(sizes, seed)
        rowptr, colidx, val = A.host()
        systems, r0 = [], 0
        for n in sizes:
            e0, e1 = int(rowptr[r0]), int(rowptr[r0 + n])
            systems.append(System(n, rowptr[r0:r0 + n + 1] - e0, colidx[e0:e1] - r0, val[e0:e1]))
            r0 += n
        return dict(op=op, B=S.Batch(systems, nrhs=c["nrhs"]), b=_batch_rhs(A.nrows, c["nrhs"], seed),
                    rtol=c["rtol"])
    theta, b, xt = _diffusion_inputs(c, seed)
    return dict(op=op, D=AD.DiffusionOperator(c["n"]), theta=theta.requires_grad_(True),
                b=b.requires_grad_(True), xt=xt, rtol=c["rtol"])


class System:
    """One host CSR system, as ``Batch`` takes them."""

    def __init__(self, nrows, rowptr, colidx, val):
        self.nrows, self.rowptr, self.colidx, self.val = nrows, rowptr, colidx, val


def run(state):
    s, op = state, state["op"]
    if op == "matvec":
        if s["map"] is not None:
            s["map"].update(s["x"])
        return s["M"].mult(s["x"], out=s["y"])
    if op == "complex":
        return s["M"] @ s["x"], s["M"].transpmult(s["xt"])
    if op == "transp":
        return s["M"].transpmult(s["g"])
    if op == "cg":
        return S.cg(s["M"], s["b"], 100000, s["rtol"])
    if op == "ir":
        # the reported statistics count FP32 iterations, which a rounding moves by a few
        x, _ = S.ir_cg(s["M"], s["L"], s["b"], rtol=s["rtol"], adaptive_inner=s["adaptive"])
        return x
    if op == "batch":
        return s["B"].solve(s["b"], max_its=20000, rtol=s["rtol"], iterations=False)
    x = s["D"].solve(s["theta"], s["b"], rtol=s["rtol"])
    loss = 0.5 * torch.sum((x - s["xt"]) ** 2)
    gtheta, gb = torch.autograd.grad(loss, (s["theta"], s["b"]))
    return x.detach(), gtheta, gb


# ---------------------------------------------------------------- what a pass cannot do without
def _stencil_nnz(c):
    nx, ny, nz, g = c["nx"], c["ny"], c["nz"], c.get("ghost", 0)
    along = lambda d, n: n - abs(d)  # noqa: E731
    return sum(along(o[0], nx) * along(o[1], ny) * (nz - 1 + (g if o[2] > 0 else 0) if o[2] else nz)
               for o in _offsets(c["kind"]))


def _product_bytes(nnz, nrows, ncols, dtype):
    """CSR arrays with 4-byte indices, x read once, y written once."""
    return nnz * (VALUE_BYTES[dtype] + 4) + 4 * (nrows + 1) + VECTOR_BYTES[dtype] * (ncols + nrows)


def _cg_iteration(nnz, n, values, vec):
    """Bytes and operations of one iteration: the matrix once, x, r and p read and written."""
    return nnz * (values + 4) + 4 * (n + 1) + 6 * vec * n, 2 * nnz + 10 * n


def _iterations(c, rtol):
    """About what these systems take (1043 for the 7-point operator on 256^3 to 1e-10)."""
    side = max(c["nx"], c["ny"], c["nz"])
    return max(1.0, {5: 0.102, 7: 0.177, 27: 0.104}[c["kind"]] * side * math.log(1 / rtol))


def work(case):
    c, op = case, case["op"]
    if op == "matvec":
        n = c["n"] if c["kind"] == 0 else _owned(c)
        plane = c["nx"] * c["ny"] if c.get("ghost") else 0
        nnz = int(9.5 * n) if c["kind"] == 0 else _stencil_nnz(c)
        vec = VECTOR_BYTES[c["dtype"]]
        return dict(bytes=_product_bytes(nnz, n, n + plane, c["dtype"]) + plane * (4 + 4 * vec),
                    flops=2 * nnz)
    if op == "complex":
        n, nnz = _owned(c), _stencil_nnz(c)
        return dict(bytes=2 * _product_bytes(nnz, n, n, c["dtype"]), flops=16 * nnz)
    if op == "transp":
        n = c["n"]
        nnz, rows, edges = 8 * n * n - 4 * n, 5 * n * n - 4 * n, 2 * n * (n - 1) + 4 * n
        return dict(bytes=_product_bytes(nnz, rows, edges, "f64"), flops=2 * nnz)
    if op == "cg":
        b, f = _cg_iteration(_stencil_nnz(c), _owned(c), 8, 8)
        k = _iterations(c, c["rtol"])
        return dict(bytes=k * b, flops=k * f)
    if op == "ir":
        # about one and a half times the FP64 iterations, in FP32
        b, f = _cg_iteration(_stencil_nnz(c), _owned(c), VALUE_BYTES[c["low"]], 4)
        k = (1.24 if c["adaptive"] else 1.49) * _iterations(c, c["rtol"])
        return dict(bytes=k * b, flops=k * f)
    if op == "batch":
        # about 60 iterations of each system
        n = c["nsys"] * (c["hi"] - c["lo"]) / math.log(c["hi"] / c["lo"])
        b, f = 9.5 * n * 8 + 4 * n + 6 * 4 * n * c["nrhs"], (2 * 9.5 + 10) * n * c["nrhs"]
        return dict(bytes=60 * b, flops=60 * f)
    # the two solves, the assembly and its transpose, and the product of the two solutions
    n = c["n"] * c["n"]
    b, f = _cg_iteration(5 * n - 4 * c["n"], n, 8, 8)
    k = 2 * 4.4 * c["n"]
    return dict(bytes=k * b + 2 * 8 * n * 12, flops=k * f)


# ---------------------------------------------------------------- the same in float64 torch
def _solve64(apply, b):
    """A^{-1} b by conjugate gradient, column by column, restarted once from the true residual."""
    b = b if b.dim() == 2 else b.view(-1, 1)
    x, scale = torch.zeros_like(b), b.square().sum(0)
    for _ in range(3):
        r = b - apply(x)
        d, p, rr = torch.zeros_like(b), r.clone(), r.square().sum(0)
        goal = torch.maximum(rr * 1e-26, scale * 1e-31)
        for k in range(20000):
            y = apply(p)
            live = rr > goal
            alpha = torch.where(live, rr / (p * y).sum(0), torch.zeros_like(rr))
            d += alpha * p
            r -= alpha * y
            new = r.square().sum(0)
            beta = torch.where(live, new / rr, torch.zeros_like(rr))
            rr = torch.where(live, new, rr)
            p = r + beta * p
            if k % 25 == 24 and not bool((rr > goal).any()):
                break
        x = x + d
    return x


def exact(case, seed):
    c, op = case, case["op"]
    if op == "matvec":
        x, halo = _matvec_inputs(c, seed)
        x = (x if halo is None else torch.cat([x, halo])).double()
        if c["kind"]:
            return _apply_stencil(c, x)  # the entries are small whole numbers in every type
        A = _general(c, seed)
        A.val = A.val.to({"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}[c["dtype"]]).double()
        return A.torch64() @ x
    if op == "complex":
        A = _stencil(c)
        v, x, xt = _complex_inputs(c, seed, A.val.numel())
        v, x, xt = v.to(VECTOR_DTYPE[c["dtype"]]).to(torch.complex128), x.to(torch.complex128), xt.to(torch.complex128)
        rows = torch.repeat_interleave(torch.arange(A.nrows, device=DEV), A.rowptr.diff())
        cols = A.colidx.long()
        parts = lambda t, at, w: torch.view_as_complex(  # noqa: E731
            torch.zeros((A.nrows, 2), dtype=torch.float64, device=DEV).index_add_(0, at, torch.view_as_real(v * t[w])))
        return parts(x, rows, cols), parts(xt, cols, rows)
    if op == "transp":
        rowptr, colidx, val = _incidence(c["n"])
        g = _uniform(seed, 61, rowptr.numel() - 1)
        rows = torch.repeat_interleave(torch.arange(rowptr.numel() - 1, device=DEV), rowptr.diff())
        ne = 2 * c["n"] * (c["n"] - 1) + 4 * c["n"]
        return torch.zeros(ne, dtype=torch.float64, device=DEV).index_add_(0, colidx, val * g[rows])
    if op in ("cg", "ir"):
        x = _solve64(lambda t: _apply_stencil(c, t.reshape(-1)).view(-1, 1), _cg_rhs(c, seed)).view(-1)
        if op == "ir":
            return x
        return torch.cat([x, torch.zeros(c["nx"] * c["ny"] * c.get("ghost", 0), dtype=x.dtype, device=DEV)]), None
    if op == "batch":
        A = _random_spd(_batch_sizes(c), seed)
        b = _batch_rhs(A.nrows, c["nrhs"], seed).double()
        A.val = A.val.float().double()
        M = A.torch64()
        return _solve64(lambda t: M @ t, b)
    theta, b, xt = _diffusion_inputs(c, seed)
    n = c["n"]
    nh, nn = n * (n - 1), 2 * n * (n - 1)
    east, north = theta[:nh].view(n, n - 1), theta[nh:nn].view(n - 1, n)
    sides = theta[nn:].view(4, n)  # j = 0, j = n-1, i = 0, i = n-1

    def apply(t):
        f = t.reshape(n, n)
        out = torch.zeros_like(f)
        fe, fn = east * (f[:, :-1] - f[:, 1:]), north * (f[:-1] - f[1:])
        out[:, :-1] += fe
        out[:, 1:] -= fe
        out[:-1] += fn
        out[1:] -= fn
        out[0] += sides[0] * f[0]
        out[-1] += sides[1] * f[-1]
        out[:, 0] += sides[2] * f[:, 0]
        out[:, -1] += sides[3] * f[:, -1]
        return out.reshape(-1, 1)

    x = _solve64(apply, b).view(-1)
    lam = _solve64(apply, x - xt).view(-1)
    u, w = lam.view(n, n), x.view(n, n)
    de = (u[:, :-1] - u[:, 1:]) * (w[:, :-1] - w[:, 1:])
    dn = (u[:-1] - u[1:]) * (w[:-1] - w[1:])
    edge = [u[0] * w[0], u[-1] * w[-1], u[:, 0] * w[:, 0], u[:, -1] * w[:, -1]]
    return x, -torch.cat([de.reshape(-1), dn.reshape(-1), *edge]), lam


def _incidence(n):
    """The (stored entry of A) x (edge) matrix of the n x n diffusion operator."""
    nh, nn = n * (n - 1), 2 * n * (n - 1)
    row = torch.arange(n * n, device=DEV)
    i, j = row % n, row // n
    none = torch.full_like(row, -1)
    at = lambda ok, e: torch.where(ok, e, none)  # noqa: E731
    south, west = at(j > 0, nh + (j - 1) * n + i), at(i > 0, j * (n - 1) + i - 1)
    east, north = at(i < n - 1, j * (n - 1) + i), at(j < n - 1, nh + j * n + i)
    border = [at(j == 0, nn + i), at(j == n - 1, nn + n + i), at(i == 0, nn + 2 * n + j),
              at(i == n - 1, nn + 3 * n + j)]
    # per grid point: the entries south, west, diagonal, east, north, each with its edges
    edges = torch.full((n * n, 5, 8), -1, dtype=torch.int64, device=DEV)
    for s, e in ((0, south), (1, west), (3, east), (4, north)):
        edges[:, s, 0] = e
    edges[:, 2] = torch.stack([south, west, east, north, *border], 1)
    sign = torch.full((n * n, 5, 8), -1.0, dtype=torch.float64, device=DEV)
    sign[:, 2] = 1.0
    has = edges >= 0
    stored = has.any(2)
    per = has.sum(2)[stored]
    rowptr = torch.zeros(per.numel() + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(per, 0, out=rowptr[1:])
    return rowptr, edges[has], sign[has]
