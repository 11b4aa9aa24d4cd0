"""The work this framework is measured on: sparse products, preconditioner
applies, refactorisations and whole solves, each through the entry points a
program calls.

A case is a dict of plain values. Its "path" names what is called, "nx", "ny"
and "nz" (or "rows") the operator's size, and the other keys the options:

  spmv        y = A x, y = b - A x ("residual") or y = A^T x ("transpose")
  apply       z = M^-1 r with an IC(0) / ILU(k) factor
  refactor    new matrix values, numeric factorisation on the device, apply
  fgmres      x after a fixed number of ILU(0)-FGMRES iterations
  adjoint     x = A(v)^-1 b by IC(0)-PCG, and the gradients of a data misfit

Operators: "five"/"seven"/"box" are grid stencils of 5, 7 and 27 points with
lognormal coefficients, "mesh" an irregular triangulation, "scattered" rows of
lognormal length whose columns lie anywhere (the graph-like case). They are
assembled in a row-wise padded form (columns, values), from which the CSR
arrays are cut.
"""
import numpy as np
import torch

import linearalgebra_amd as la

_DTYPE = {"f64": la.F64, "f32": la.F32, "bf16": la.BF16}
_BYTES = {"f64": 8, "f32": 4, "bf16": 2}
_FGMRES_STEPS = 25
_ADJOINT_TOL = 1e-10


def listed():
    return [
        # the smallest product: a 2-D Poisson-like operator, one call's latency
        {"name": "spmv_2d_small_f64", "path": "spmv", "op": "five", "nx": 256, "ny": 256, "nz": 1,
         "order": "rows", "val": "f64", "form": "plain"},
        # the headline product: a 7-point operator on 128^3 cells in a
        # bandwidth-reducing (Cuthill-McKee-like) order, FP64
        {"name": "spmv_3d_f64", "path": "spmv", "op": "seven", "nx": 128, "ny": 128, "nz": 128,
         "order": "planes", "val": "f64", "form": "plain"},
        # the residual of a mixed-precision refinement step on an anisotropic
        # 27-point operator
        {"name": "spmv_box_residual_f32", "path": "spmv", "op": "box", "nx": 101, "ny": 104,
         "nz": 99, "order": "rows", "val": "f32", "form": "residual"},
        # a graph-like operator whose x is larger than an L2 cache
        {"name": "spmv_scattered_f64", "path": "spmv", "op": "scattered", "rows": 2000000,
         "val": "f64", "form": "plain"},
        # the transposed product (adjoints, normal equations) of a smaller one
        {"name": "spmv_scattered_transpose_f32", "path": "spmv", "op": "scattered",
         "rows": 250007, "val": "f32", "form": "transpose"},
        # the exact IC(0) apply that dominates a PCG iteration on 128^3 cells
        {"name": "apply_ic0_3d_f64", "path": "apply", "op": "seven", "nx": 128, "ny": 128,
         "nz": 128, "order": "planes", "fill": 0, "kind": "ic", "val": "f64", "mode": "exact"},
        # its approximate form in mixed-precision PCG: three sweeps, BF16 factors
        {"name": "apply_ic0_3d_sweeps_bf16", "path": "apply", "op": "seven",
         "nx": 128, "ny": 125, "nz": 120, "order": "rows", "fill": 0, "kind": "ic", "val": "bf16",
         "mode": "sweeps"},
        # the ILU(1) apply of a mixed-precision FGMRES on a 27-point operator
        {"name": "apply_ilu1_box_f32", "path": "apply", "op": "box", "nx": 56, "ny": 56, "nz": 56,
         "order": "rows", "fill": 1, "kind": "ilu", "val": "f32", "mode": "exact"},
        # ILU(0) on an unstructured mesh, swept in one direction
        {"name": "apply_ilu0_mesh_f64", "path": "apply", "op": "mesh", "nx": 400, "ny": 380,
         "nz": 1, "order": "rows", "fill": 0, "kind": "ilu", "val": "f64", "mode": "exact"},
        # an implicit time step's set-up: new coefficients on a known pattern
        {"name": "refactor_ilu1_box", "path": "refactor", "op": "box", "nx": 48, "ny": 48, "nz": 48,
         "order": "rows", "fill": 1, "kind": "ilu", "val": "f64"},
        # a whole FGMRES cycle with a fixed budget of iterations
        {"name": "fgmres_ilu0_3d_f64", "path": "fgmres", "op": "seven", "nx": 100, "ny": 96,
         "nz": 90, "order": "rows", "fill": 0, "kind": "ilu", "val": "f64"},
        # training / inversion: forward solve and adjoint gradients on a 2-D grid
        {"name": "adjoint_2d_f64", "path": "adjoint", "op": "five", "nx": 128, "ny": 128, "nz": 1,
         "order": "rows", "fill": 0, "kind": "ic", "val": "f64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case of the same ranges."""
    def edges(lo, hi, dims=3):
        e = _log_int(rng, lo, hi)
        g = [max(lo, min(hi, int(round(e * rng.uniform(0.8, 1.2))))) for _ in range(dims)]
        return dict(zip(("nx", "ny", "nz"), g + [1] * (3 - dims)))

    kind = rng.choice(["spmv_grid", "spmv_grid", "spmv_scattered", "spmv_scattered", "apply_7",
                       "apply_2d", "apply_box", "apply_mesh", "apply_sweeps", "refactor",
                       "fgmres", "adjoint"])
    if kind == "spmv_grid":
        op = rng.choice(["five", "seven", "box"])
        grid = {"five": lambda: edges(200, 1000, 2), "seven": lambda: edges(32, 128),
                "box": lambda: edges(24, 99)}[op]()
        return {"path": "spmv", "op": op, **grid,
                "order": rng.choice(["rows", "planes"]) if op != "box" else "rows",
                "val": rng.choice(["f64", "f32", "bf16"]),
                "form": rng.choice(["plain", "residual", "transpose"])}
    if kind == "spmv_scattered":
        form = rng.choice(["plain", "residual", "transpose"])
        return {"path": "spmv", "op": "scattered",
                "rows": _log_int(rng, 50000, 250000 if form == "transpose" else 2000000),
                "val": rng.choice(["f64", "f32", "bf16"]), "form": form}
    case = {"path": "apply", "order": "rows", "mode": "exact",
            "val": rng.choice(["f64", "f32"])}
    if kind == "apply_7":
        case.update(op="seven", **edges(40, 128), fill=0, kind="ic",
                    order=rng.choice(["rows", "planes"]))
    elif kind == "apply_2d":
        case.update(op="five", **edges(128, 512, 2), fill=0, kind=rng.choice(["ic", "ilu"]))
    elif kind == "apply_box":
        case.update(op="box", **edges(20, 56), fill=rng.choice([0, 1]), kind="ilu")
    elif kind == "apply_mesh":
        case.update(op="mesh", **edges(100, 390, 2), fill=0, kind="ilu")
    elif kind == "apply_sweeps":
        case.update(op="seven", **edges(40, 124), fill=0, kind="ic", mode="sweeps",
                    val=rng.choice(["f64", "f32", "bf16"]))
    elif kind == "refactor":
        if rng.random() < 0.5:
            return {"path": "refactor", "op": "box", **edges(20, 48), "order": "rows",
                    "fill": rng.choice([0, 1]), "kind": "ilu", "val": "f64"}
        return {"path": "refactor", "op": "seven", **edges(24, 72), "order": "rows",
                "fill": 0, "kind": rng.choice(["ic", "ilu"]), "val": "f64"}
    elif kind == "fgmres":
        return {"path": "fgmres", "op": "seven", **edges(32, 90), "order": "rows",
                "fill": 0, "kind": "ilu", "val": "f64"}
    elif kind == "adjoint":
        return {"path": "adjoint", "op": "five", **edges(48, 128, 2), "order": "rows",
                "fill": 0, "kind": "ic", "val": "f64"}
    return case


# ------------------------------------------------------------------ operators


def _grid(case):
    return case["nx"], case["ny"], case["nz"]


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed, stream):
    g = torch.Generator(device=_device())
    g.manual_seed(int(seed) * 1009 + stream)
    return g


def _lognormal(n, seed, stream, sigma):
    z = torch.randn(n, generator=_generator(seed, stream), device=_device(), dtype=torch.float64)
    return torch.exp(sigma * z)


def _vector(n, seed, stream):
    return 2.0 * torch.rand(n, generator=_generator(seed, stream), device=_device(),
                            dtype=torch.float64) - 1.0


def _offsets(op):
    if op == "box":
        return [(x, y, z) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]
    return [(0, 0, -1), (0, -1, 0), (-1, 0, 0), (0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)]


def _neighbours(grid, offsets):
    """Per cell and offset: the neighbour's index and whether it is inside."""
    nx, ny, nz = grid
    dev = _device()
    c = torch.arange(nx * ny * nz, device=dev)
    x, y, z = c % nx, (c // nx) % ny, c // (nx * ny)
    nb, ok = [], []
    for dx, dy, dz in offsets:
        ok.append((x + dx >= 0) & (x + dx < nx) & (y + dy >= 0) & (y + dy < ny) &
                  (z + dz >= 0) & (z + dz < nz))
        nb.append(c + dx + nx * (dy + ny * dz))
    return torch.stack(nb, 1), torch.stack(ok, 1)


def _weight(op, d):
    dx, dy, dz = d
    if op == "box":  # strong coupling along z
        r2 = dx * dx + dy * dy + dz * dz
        return (dx * dx + dy * dy + 100.0 * dz * dz) / (r2 * r2)
    return 1.0


def _grid_operator(case, seed):
    """Diffusion with lognormal cell coefficients, harmonic means on the
    edges and Dirichlet walls; an ILU case adds upwind convection along x."""
    op, grid = case["op"], _grid(case)
    offs = [d for d in _offsets(op) if d[2] == 0 or grid[2] > 1 or op == "box"]
    nb, ok = _neighbours(grid, offs)
    n = nb.shape[0]
    kappa = _lognormal(n, seed, 1, 1.0)
    cols, vals = torch.where(ok, nb, n), torch.zeros(nb.shape, dtype=torch.float64,
                                                     device=nb.device)
    centre, diag = offs.index((0, 0, 0)), torch.zeros(n, dtype=torch.float64, device=nb.device)
    wind = 0.5 if case.get("kind") == "ilu" else 0.0
    for t, d in enumerate(offs):
        if t == centre:
            continue
        other = kappa[nb[:, t].clamp(0, n - 1)]
        edge = torch.where(ok[:, t], 2.0 * kappa * other / (kappa + other), kappa)
        edge = edge * _weight(op, d) + wind * float(d == (-1, 0, 0))
        vals[:, t] = torch.where(ok[:, t], -edge, 0.0)
        diag += edge
    vals[:, centre] = diag
    return cols, vals


def _mesh_operator(case, seed):
    """Stiffness of a triangulated sheet: a quadrilateral net cut along
    random diagonals, three per cent of the nodes left out."""
    nx, ny, _ = _grid(case)
    n0 = nx * ny
    dev = _device()
    u = torch.rand(2, n0, generator=_generator(7, 2), device=dev)  # one mesh per size
    keep, flip = u[0] > 0.03, u[1] > 0.5
    node = torch.cumsum(keep, 0) - 1
    c = torch.arange(n0, device=dev)
    x, y = c % nx, c // nx
    right, up = x + 1 < nx, y + 1 < ny
    pairs = [torch.stack((c, c + 1), 1)[right], torch.stack((c, c + nx), 1)[up],
             torch.stack((c, c + nx + 1), 1)[right & up & flip],
             torch.stack((c + 1, c + nx), 1)[right & up & ~flip]]
    e = torch.cat(pairs)
    e = e[keep[e[:, 0]] & keep[e[:, 1]]]
    n = int(keep.sum())
    i, j = node[e[:, 0]], node[e[:, 1]]
    w = _lognormal(i.numel(), seed, 3, 0.5)
    d = torch.arange(n, device=dev)
    rows, cs, vs = torch.cat((i, j, d)), torch.cat((j, i, d)), torch.cat((-w, -1.1 * w, 0.0 * d))
    order = torch.argsort(rows * n + cs)
    rows, cs, vs = rows[order], cs[order], vs[order]
    start = torch.searchsorted(rows, torch.arange(n + 1, device=dev))
    width = int((start[1:] - start[:-1]).max())
    slot = torch.arange(rows.numel(), device=dev) - start[rows]
    cols = torch.full((n, width), n, dtype=torch.int64, device=dev)
    vals = torch.zeros((n, width), dtype=torch.float64, device=dev)
    cols[rows, slot], vals[rows, slot] = cs, vs
    vals = torch.where(cols == d[:, None], 1e-2 - vals.sum(1)[:, None], vals)
    return cols, vals


def _reorder(cols, vals, grid):
    """Cells by diagonal planes x + y + z, the order a bandwidth-reducing
    renumbering gives on a grid."""
    nx, ny, _ = grid
    n = cols.shape[0]
    c = torch.arange(n, device=cols.device)
    plane = c % nx + (c // nx) % ny + c // (nx * ny)
    new_to_old = torch.argsort(plane * n + c)
    old_to_new = torch.empty(n + 1, dtype=torch.int64, device=cols.device)
    old_to_new[new_to_old] = c
    old_to_new[n] = n
    cols, vals = old_to_new[cols[new_to_old]], vals[new_to_old]
    cols, by = torch.sort(cols, 1)
    return cols, torch.gather(vals, 1, by)


def _operator(case, seed):
    """(columns, values), one padded row per row; padding has column n."""
    if case["op"] == "mesh":
        return _mesh_operator(case, seed)
    cols, vals = _grid_operator(case, seed)
    if case["order"] == "planes":
        cols, vals = _reorder(cols, vals, _grid(case))
    return cols, vals


def _csr(cols, vals):
    n = cols.shape[0]
    real = cols < n
    ai = np.zeros(n + 1, np.int32)
    ai[1:] = torch.cumsum(real.sum(1), 0).to(torch.int32).cpu().numpy()
    return la.CSR(n, ai, cols[real].to(torch.int32).cpu().numpy(), vals[real].cpu().numpy())


def _scattered(case, seed):
    """Row, column and value of each entry: row lengths lognormal with mean
    16, columns anywhere, the diagonal always there."""
    n, dev = case["rows"], _device()
    z = torch.randn(n, generator=_generator(seed, 4), device=dev, dtype=torch.float64)
    length = torch.exp(np.log(16.0) - 0.5 + z).round().clamp(1, 20000).to(torch.int64)
    rows = torch.repeat_interleave(torch.arange(n, device=dev), length - 1)
    cs = torch.randint(0, n, (rows.numel(),), generator=_generator(seed, 5), device=dev)
    d = torch.arange(n, device=dev)
    key = torch.unique(torch.cat((rows * n + cs, d * n + d)))
    rows, cs = key // n, key % n
    return rows, cs, _vector(rows.numel(), seed, 6)


# --------------------------------------------------- the measured calls


def _matrix(case, seed):
    if case["op"] != "scattered":
        return _csr(*_operator(case, seed))
    rows, cs, vs = _scattered(case, seed)
    n = case["rows"]
    ai = torch.searchsorted(rows, torch.arange(n + 1, device=rows.device)).to(torch.int32)
    return la.CSR(n, ai.cpu().numpy(), cs.to(torch.int32).cpu().numpy(), vs.cpu().numpy())


def _vec_dtype(case):
    return torch.float64 if case["val"] == "f64" else torch.float32


def _factor(A, case):
    if case["kind"] == "ilu":
        return la.Preconditioner(la.iluk(A, case["fill"]), "ilu")
    R, ok = la.icc(la.split_triangle(A, upper=True), case["fill"])
    if not ok:
        raise RuntimeError("IC factorisation failed")
    return la.Preconditioner(R, "ic")


def prepare(case, seed):
    path, dt = case["path"], _vec_dtype(case)
    A = _matrix(case, seed)
    x = _vector(A.n, seed, 10)
    state = {"case": case, "x": x.to(dt), "y": torch.empty(A.n, dtype=dt, device=x.device)}
    if path == "spmv":
        dA = la.DeviceMatrix(A)
        dA.add_dtype(_DTYPE[case["val"]])
        if case["form"] != "transpose":
            dA.preprocess(la.SPMV_AUTO)
        state.update(A=dA, b=_vector(A.n, seed, 11).to(dt))
    elif path == "apply":
        P = _factor(A, case)
        P.add_dtype(_DTYPE[case["val"]])
        if case["mode"] == "sweeps":
            P.set_sweeps(3)
        state.update(P=P)
    elif path == "refactor":
        make = la.Preconditioner.ilu_gpu if case["kind"] == "ilu" else la.Preconditioner.ic_gpu
        state.update(P=make(A, case["fill"]), v=torch.from_numpy(A.av).to(x.device))
    elif path == "fgmres":
        state.update(A=la.DeviceMatrix(A), P=_factor(A, case))
    else:
        from linearalgebra_amd.autograd import SparseSystem
        state.update(S=SparseSystem(A, "ic", case["fill"], rel_tol=_ADJOINT_TOL),
                     v=torch.from_numpy(A.av).to(x.device).requires_grad_(),
                     b=x.clone().requires_grad_(), target=_vector(A.n, seed, 12))
    return state


def run(state):
    case, x, y = state["case"], state["x"], state["y"]
    path, val = case["path"], _DTYPE[case["val"]]
    if path == "spmv":
        if case["form"] == "plain":
            return state["A"].spmv(x, y, val=val)
        if case["form"] == "residual":
            return state["A"].spmv(x, y, alpha=-1.0, beta=1.0, z=state["b"], val=val)
        return state["A"].spmv_transpose(x, y, val=val)
    if path == "apply":
        mode = la.TRSV_JACOBI if case["mode"] == "sweeps" else la.TRSV_SYNCFREE
        return state["P"].apply(x, y, mode=mode, val=val)
    if path == "refactor":
        state["P"].refactor(state["v"])
        return state["P"].apply(x, y)
    if path == "fgmres":
        y.zero_()
        la.fgmres(state["A"], state["P"], x, y, rel_tol=1e-30, max_iters=_FGMRES_STEPS,
                  restart=_FGMRES_STEPS, trsv_mode=la.TRSV_SYNCFREE)
        return y
    from linearalgebra_amd.autograd import sparse_solve
    sol = sparse_solve(state["v"], state["b"], state["S"])
    misfit = 0.5 * ((sol - state["target"]) ** 2).sum()
    gv, gb = torch.autograd.grad(misfit, (state["v"], state["b"]))
    return sol.detach(), gv, gb


# ------------------------------------------------------------------ costs


def _counts(case):
    """Rows, entries of A and entries of the factor."""
    if case["op"] == "scattered":
        return case["rows"], 16 * case["rows"], 0
    nx, ny, nz = _grid(case)
    if case["op"] == "mesh":
        n = int(0.97 * nx * ny)
        return n, int(6.8 * n), int(6.8 * n)
    offs = _offsets(case["op"])

    def entries(ds):
        return sum(max(0, nx - abs(x)) * max(0, ny - abs(y)) * max(0, nz - abs(z))
                   for x, y, z in ds)
    fill = _fill_offsets(case["op"]) if case.get("fill") else offs
    return nx * ny * nz, entries(offs), entries(fill)


def work(case):
    n, nnz, fnnz = _counts(case)
    sv, sx = _BYTES[case["val"]], 8 if case["val"] == "f64" else 4
    spmv = nnz * (sv + 4) + 4 * n + 2 * n * sx
    apply = fnnz * (sv + 4) + 8 * n + 2 * n * sx
    path = case["path"]
    if path == "spmv":
        return {"bytes": spmv + n * sx * (case["form"] == "residual"), "flops": 2 * nnz}
    if path == "apply":
        return {"bytes": apply, "flops": (6 if case["mode"] == "sweeps" else 2) * fnnz}
    # an entry of the factor is updated once per elimination that reaches it
    update = 2 * fnnz * max(1, fnnz // n // 4)
    if path == "refactor":
        return {"bytes": 8 * nnz + 12 * fnnz + apply, "flops": update + 2 * fnnz}
    if path == "fgmres":
        k = _FGMRES_STEPS
        return {"bytes": k * (spmv + apply) + n * sx * k * (k + 1),
                "flops": k * 2 * (nnz + fnnz) + 4 * n * k * (k + 1)}
    steps = 2 * 2 * max(_grid(case))  # about two iterations per cell of an edge, two solves
    return {"bytes": steps * (2 * spmv + apply + 8 * n * sx) + 24 * nnz + 12 * fnnz,
            "flops": steps * (4 * nnz + 2 * fnnz + 12 * n) + update}


# ------------------------------------------------------------------ 64 bits


def _fill_offsets(op):
    """Level-1 fill of a grid stencil: itself and lower + upper offsets."""
    offs = _offsets(op)
    low = [d for d in offs if d[::-1] < (0, 0, 0)]
    high = [d for d in offs if d[::-1] > (0, 0, 0)]
    more = {tuple(p + q for p, q in zip(a, b)) for a in low for b in high}
    return sorted(set(offs) | more, key=lambda d: d[::-1])


def _with_fill(case, cols, vals):
    """The rows widened by their level-1 fill (zero values): an entry a + b
    exists where both the cell at a and the one at a + b are inside."""
    if not case["fill"]:
        return cols, vals
    grid, n = _grid(case), cols.shape[0]
    offs, fill = _offsets(case["op"]), _fill_offsets(case["op"])
    nb, inside = _neighbours(grid, fill)
    _, ok = _neighbours(grid, offs)
    there = torch.zeros_like(inside)
    wide = torch.zeros(nb.shape, dtype=torch.float64, device=nb.device)
    for t, d in enumerate(offs):
        there[:, fill.index(d)] = ok[:, t]
        wide[:, fill.index(d)] = vals[:, t]
    for t, a in enumerate(offs):
        if a[::-1] < (0, 0, 0):
            for b in offs:
                if b[::-1] > (0, 0, 0):
                    f = fill.index(tuple(p + q for p, q in zip(a, b)))
                    there[:, f] |= ok[:, t] & inside[:, f]
    return torch.where(there, nb, n), wide


class _Exact:
    """ILU on a given pattern and its solves, level by level, in float64. An
    IC factor's M = R^T R is the same matrix as L U on a symmetric operator."""

    def __init__(self, cols, vals):
        n, w = cols.shape
        self.n = n
        row = torch.arange(n, device=cols.device)[:, None]
        self.low, self.up = cols < row, (cols > row) & (cols < n)
        self.cols, self.f = cols, vals.clone()
        self.diag_at = (cols == row).to(torch.int64).argmax(1)
        self.down, self.back = self._levels(self.low), self._levels(self.up)

    def _levels(self, part):
        n = self.n
        level = torch.zeros(n + 1, dtype=torch.int64, device=self.cols.device)
        while True:
            new = torch.where(part, level[self.cols] + 1, 0).amax(1)
            if torch.equal(new, level[:n]):
                break
            level[:n] = new
        order = torch.argsort(level[:n], stable=True)
        return torch.split(order, torch.bincount(level[:n]).tolist())

    def factor(self):
        cols, f, n, w = self.cols, self.f, self.n, self.cols.shape[1]
        inv = torch.zeros(n + 1, dtype=f.dtype, device=f.device)
        lower_most = int(self.low.sum(1).max())
        padded = torch.cat((torch.where(self.up, cols, -1),
                            torch.full((1, w), -1, device=cols.device)))
        for rows in self.down:
            c, v, low = cols[rows], f[rows], self.low[rows]
            for t in range(lower_most):
                if rows is self.down[0]:
                    break
                k = torch.where(low[:, t], c[:, t], n)
                ratio = v[:, t] * inv[k]
                v[:, t] = torch.where(low[:, t], ratio, v[:, t])
                fk = f[k.clamp(max=n - 1)]
                hit = c[:, :, None] == padded[k][:, None, :]
                upd = (hit * fk[:, None, :]).sum(2)
                v -= torch.where(low[:, t], ratio, 0.0)[:, None] * upd
            f[rows] = v
            inv[rows] = 1.0 / v.gather(1, self.diag_at[rows][:, None])[:, 0]
        self.inv = inv[:n]
        return self

    def _sweep(self, levels, part, b, scale):
        x = torch.zeros(self.n + 1, dtype=b.dtype, device=b.device)
        for rows in levels:
            s = (torch.where(part[rows], self.f[rows], 0.0) * x[self.cols[rows]]).sum(1)
            x[rows] = (b[rows] - s) * (scale[rows] if scale is not None else 1.0)
        return x[:self.n]

    def solve(self, b):
        return self._sweep(self.back, self.up, self._sweep(self.down, self.low, b, None), self.inv)

    def sweeps(self, b, k):
        """k Jacobi sweeps on each triangle from its scaled right-hand side."""
        def product(part, x):
            return (torch.where(part, self.f, 0.0) * torch.cat((x, x[:1]))[self.cols]).sum(1)
        y = b
        for _ in range(k):
            y = b - product(self.low, y)
        x = y * self.inv
        for _ in range(k):
            x = (y - product(self.up, x)) * self.inv
        return x


def _exact_fgmres(cols, vals, M, b, steps):
    def product(x):
        return (vals * torch.cat((x, torch.zeros_like(x[:1])))[cols]).sum(1)
    beta = torch.linalg.vector_norm(b)
    V, Z, H = [b / beta], [], torch.zeros(steps + 1, steps, dtype=b.dtype, device=b.device)
    for j in range(steps):
        Z.append(M.solve(V[j]))
        w = product(Z[j])
        B = torch.stack(V)
        for _ in range(2):
            h = B @ w
            w = w - h @ B
            H[:j + 1, j] += h
        H[j + 1, j] = torch.linalg.vector_norm(w)
        V.append(w / H[j + 1, j])
    rhs = torch.zeros(steps + 1, dtype=b.dtype, device=b.device)
    rhs[0] = beta
    y = torch.linalg.lstsq(H.cpu(), rhs.cpu()[:, None]).solution[:, 0].to(b.device)
    return y @ torch.stack(Z)


def _exact_cg(cols, vals, b):
    """Conjugate gradients restarted on the true residual until it stalls."""
    def product(x):
        return (vals * torch.cat((x, torch.zeros_like(x[:1])))[cols]).sum(1)
    n = cols.shape[0]
    row = torch.arange(n, device=cols.device)[:, None]
    inv = 1.0 / torch.where(cols == row, vals, 0.0).sum(1)
    x = torch.zeros_like(b)
    for _ in range(3):
        r = b - product(x)
        d, p, rz, first = torch.zeros_like(b), None, None, None
        for it in range(40 * int(n ** 0.5)):
            z = inv * r
            new = r @ z
            p = z if p is None else z + (new / rz) * p
            rz = new
            q = product(p)
            a = rz / (p @ q)
            d, r = d + a * p, r - a * q
            if it % 50 == 0:
                size = float(r @ r)
                first = size if first is None else first
                if size < 1e-26 * first or size == 0.0:
                    break
        x = x + d
    return x


def exact(case, seed):
    path = case["path"]
    if path == "spmv":
        if case["op"] == "scattered":
            rows, cs, vs = _scattered(case, seed)
            n = case["rows"]
        else:
            cols, vals = _operator(case, seed)
            n, real = cols.shape[0], cols < cols.shape[0]
            rows = torch.arange(n, device=cols.device)[:, None].expand_as(cols)[real]
            cs, vs = cols[real], vals[real]
        x = _vector(n, seed, 10).to(_vec_dtype(case)).double()
        if case["form"] == "transpose":
            rows, cs = cs, rows
        y = torch.zeros(n, dtype=torch.float64, device=x.device).index_add(0, rows, vs * x[cs])
        if case["form"] == "residual":
            y = _vector(n, seed, 11).to(_vec_dtype(case)).double() - y
        return y
    cols, vals = _operator(case, seed)
    n = cols.shape[0]
    b = _vector(n, seed, 10).to(_vec_dtype(case)).double()
    if path == "adjoint":
        x = _exact_cg(cols, vals, b)
        lam = _exact_cg(cols, vals, x - _vector(n, seed, 12))
        real = cols < n
        rows = torch.arange(n, device=cols.device)[:, None].expand_as(cols)[real]
        return x, -lam[rows] * x[cols[real]], lam
    M = _Exact(*_with_fill(case, cols, vals)).factor()
    if path == "fgmres":
        return _exact_fgmres(cols, vals, M, b, _FGMRES_STEPS)
    return M.sweeps(b, 3) if case.get("mode") == "sweeps" else M.solve(b)
