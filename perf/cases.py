"""Performance cases of the Krylov library: what its users have it do.

A case names a path through the public interface and the size of its system.
All matrices are seeded synthetic systems on structured grids of any extent
(7-point scalar diffusion and convection-diffusion with random face
coefficients, 27-point block systems, hexahedral meshes): the shapes of the
repository's benchmark and tests, with coefficients that differ everywhere.

Vectors and matrix handles are device-resident, as in a program that solves
more than once; ``host_solve`` is monolis's own calling convention on host
arrays.  Results are returned as torch views of the device buffers.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from monolis_amd import _lib, api
from monolis_amd.matrix import Matrix

METHODS = {"cg": 1, "gropcg": 2, "pipecg": 3, "bicgstab": 5}
TOL = 1e-8


def listed():
    return [
        # the product itself: an application's own eigensolver, smoother or time stepper
        {"name": "matvec_block27_100", "path": "matvec", "system": "block27", "nx": 100, "ny": 100, "nz": 100,
         "b": 3, "dtype": "f64"},
        # a small scalar solve: latency of an iteration, the inner problem of many coupled codes
        {"name": "cg_diffusion_32", "path": "solve", "system": "diffusion7", "nx": 32, "ny": 32, "nz": 32,
         "b": 1, "method": "cg", "mode": "f64"},
        # structural mechanics at 3.0 M unknowns
        {"name": "cg_block27_100", "path": "solve", "system": "block27", "nx": 100, "ny": 100, "nz": 100,
         "b": 3, "method": "cg", "mode": "f64"},
        # the same kind of system, uneven extents, FP32 corrections refined in FP64
        {"name": "refined_block27_72", "path": "solve", "system": "block27", "nx": 72, "ny": 81, "nz": 63,
         "b": 3, "method": "cg", "mode": "refined"},
        # transport: a nonsymmetric scalar system
        {"name": "bicgstab_convdiff_128", "path": "solve", "system": "convdiff7", "nx": 128, "ny": 128, "nz": 128,
         "b": 1, "method": "bicgstab", "mode": "f64"},
        # many load cases on one operator
        {"name": "multi_diffusion_96_rhs64", "path": "multi", "nx": 96, "ny": 96, "nz": 96, "rhs": 64},
        # many independent systems of uneven size, launch configuration tuned once
        {"name": "batch_512", "path": "batch", "count": 512, "lo": 10, "hi": 40, "tuned": True},
        # frequency response: complex symmetric system, COCG
        {"name": "cocg_block27_56", "path": "cocg", "nx": 56, "ny": 56, "nz": 56, "b": 3},
        # a differentiable solve: new values, forward solve, adjoint solve and dL/dA
        {"name": "grad_convdiff_64", "path": "grad", "system": "convdiff7", "nx": 64, "ny": 64, "nz": 64, "b": 1},
        # finite elements: pattern, element matrices and boundary conditions of a hexahedral mesh
        {"name": "assembly_hex_64", "path": "assembly", "nx": 64, "ny": 64, "nz": 64, "b": 3},
        # monolis_solve_R on host arrays: what a monolis application calls
        {"name": "host_cg_block27_40", "path": "host_solve", "system": "block27", "nx": 40, "ny": 40, "nz": 40, "b": 3},
        # coupled fields: nodes with 1, 2, 3 or 6 unknowns
        {"name": "vblock_cg_44", "path": "vblock", "nx": 44, "ny": 44, "nz": 44},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def box(lo, hi):
        e = log_int(lo, hi)
        ext = [min(hi, max(lo, int(round(e * rng.uniform(0.75, 1.3))))) for _ in range(3)]
        return {"nx": ext[0], "ny": ext[1], "nz": ext[2]}

    path = rng.choice(["matvec", "solve", "solve", "solve", "multi", "batch", "cocg", "grad", "assembly",
                       "host_solve", "vblock"])
    if path == "matvec":
        b = rng.choice([1, 2, 3, 3, 4, 6])
        return {"path": path, "system": "block27" if b > 1 else rng.choice(["block27", "diffusion7"]),
                **box(6, 100 if b <= 3 else 60), "b": b, "dtype": rng.choice(["f64", "f64", "f32"])}
    if path == "solve":
        system = rng.choice(["diffusion7", "block27", "convdiff7"])
        b = 1 if system != "block27" else rng.choice([2, 3, 3, 4])
        method = "bicgstab" if system == "convdiff7" else rng.choice(["cg", "cg", "cg", "gropcg", "pipecg", "bicgstab"])
        mode = rng.choice(["f64", "f64", "refined"]) if method in ("cg", "bicgstab") else "f64"
        return {"path": path, "system": system, **box(5, 128 if b == 1 else 90 if b <= 3 else 56), "b": b,
                "method": method, "mode": mode}
    if path == "multi":
        return {"path": path, **box(12, 96), "rhs": log_int(2, 64)}
    if path == "batch":
        lo = log_int(4, 20)
        return {"path": path, "count": log_int(8, 512), "lo": lo, "hi": min(40, lo + log_int(2, 24)),
                "tuned": rng.choice([True, False])}
    if path == "cocg":
        b = rng.choice([1, 3, 3, 2])
        return {"path": path, **box(6, 60), "b": b}
    if path == "grad":
        system = rng.choice(["convdiff7", "block27"])
        return {"path": path, "system": system, **box(6, 72 if system == "convdiff7" else 44),
                "b": 1 if system == "convdiff7" else 3}
    if path == "assembly":
        return {"path": path, **box(4, 64), "b": rng.choice([1, 2, 3, 3])}
    if path == "host_solve":
        system = rng.choice(["block27", "diffusion7"])
        return {"path": path, "system": system, **box(4, 44 if system == "block27" else 64),
                "b": 3 if system == "block27" else 1}
    return {"path": path, **box(5, 48)}


# ---------------------------------------------------------------------------
# Synthetic systems (torch, on the GPU; functions of their arguments alone)
# ---------------------------------------------------------------------------
DEV = "cuda"
_OFF = {
    7: [(-1, 0, 0), (0, -1, 0), (0, 0, -1), (0, 0, 0), (0, 0, 1), (0, 1, 0), (1, 0, 0)],
    27: [(dz, dy, dx) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1)],
}


@functools.lru_cache(maxsize=40)
def _pattern(nx, ny, nz, points):
    """Block CSR of a stencil on an nx x ny x nz grid (x fastest): row lengths and 0-based
    columns, rows in order, columns ascending."""
    n = nx * ny * nz
    ids = torch.arange(n, device=DEV)
    z, y, x = ids // (nx * ny), ids // nx % ny, ids % nx
    valid, cols = [], []
    for dz, dy, dx in _OFF[points]:
        valid.append((z + dz >= 0) & (z + dz < nz) & (y + dy >= 0) & (y + dy < ny) & (x + dx >= 0) & (x + dx < nx))
        cols.append(ids + (dz * ny + dy) * nx + dx)
    valid, cols = torch.stack(valid, 1), torch.stack(cols, 1)
    return valid.sum(1), cols[valid].to(torch.int32)


def _hash01(r, c, seed):
    """Uniform numbers in [0, 1) that depend on the unordered pair (r, c) and the seed."""
    salt = (seed + 1) * 1609587929392839161 % (1 << 62)
    h = torch.minimum(r, c) * -7046029254386353131 + torch.maximum(r, c) * -4417276706812531889 + salt
    h = (h ^ (h >> 31)) * -4658895280553007687
    h = (h ^ (h >> 29)) * -7723592293110705685
    h = h ^ (h >> 32)
    return (h & ((1 << 53) - 1)).to(torch.float64) * 2.0 ** -53


def _row_sums(v, lengths):
    return torch.segment_reduce(v, "sum", lengths=lengths, axis=0, unsafe=True)


def _blocks(lengths, cols, b, seed, peclet=0.0, shift=1.0):
    """Values (nz, b, b) of a symmetric diagonally dominant block system: off-diagonal entries in
    (-1, 0]; the diagonal is its row's absolute sum + `shift`.  With b = 1 and shift 0 a 7-point
    diffusion operator with face coefficients in [0.5, 2) and Dirichlet walls, `peclet` adding
    central-difference convection along x (nonsymmetric)."""
    n = lengths.numel()
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), lengths)
    cl = cols.long()
    k = torch.arange(b, device=DEV)
    u = _hash01((rows * b)[:, None, None] + k[:, None], (cl * b)[:, None, None] + k, seed)
    if shift:
        A = -u
    else:
        A = -0.5 * torch.exp(u * math.log(4.0))
    del u
    diag = (rows == cl).nonzero().reshape(-1)
    A[diag[:, None], k, k] = 0.0
    s = _row_sums(A.abs().sum(2), lengths)
    d = s + shift if shift else s + (7 - lengths)[:, None]
    A[diag[:, None], k, k] = d
    if peclet:
        A[rows - cl == 1] -= 0.5 * peclet
        A[cl - rows == 1] += 0.5 * peclet
    return A


def _product(lengths, cols, A, x):
    """Rows of A times x: x (n, b) or (n, k) for scalar systems with k columns."""
    xg = x[cols.long()]
    t = (A * xg[:, None, :]).sum(2) if A.shape[1] > 1 else A[:, 0] * xg
    return _row_sums(t, lengths)


def _transpose_product(lengths, cols, A, x):
    """A^T x of a scalar system with a symmetric pattern: the entry (j, i) of every (i, j)."""
    n = lengths.numel()
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), lengths)
    order = torch.argsort(cols.long() * n + rows)
    return _product(lengths, cols, A[order].transpose(1, 2), x)


def _uniform(shape, seed, dtype=torch.float64):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    if dtype == torch.complex128:
        return torch.complex(*(2.0 * torch.rand((2,) + tuple(shape), generator=g, device=DEV, dtype=torch.float64) - 1.0))
    return (2.0 * torch.rand(shape, generator=g, device=DEV, dtype=torch.float64) - 1.0).to(dtype)


def _system(case, seed):
    """(lengths, cols, A) of a fixed-block case."""
    ext = (case["nx"], case["ny"], case["nz"])
    if case["system"] == "block27":
        lengths, cols = _pattern(*ext, 27)
        return lengths, cols, _blocks(lengths, cols, case["b"], seed)
    lengths, cols = _pattern(*ext, 7)
    return lengths, cols, _blocks(lengths, cols, 1, seed, 0.5 if case["system"] == "convdiff7" else 0.0, 0.0)


def _offsets(lengths):
    index = torch.zeros(lengths.numel() + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(lengths, 0, out=index[1:])
    return index


def _host_matrix(lengths, cols, A, b):
    n = lengths.numel()
    return Matrix(n, n, b, _offsets(lengths).to(torch.int32).cpu().numpy(), (cols + 1).cpu().numpy(),
                  A.reshape(-1).cpu().numpy())


# ---------------------------------------------------------------------------
# Device buffers of the library as torch tensors (torch is imported first, so both use one runtime)
# ---------------------------------------------------------------------------
class _Shared:
    def __init__(self, buf, count, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (buf.ptr, False), "version": 2}


_KIND = {torch.float64: (np.float64, "<f8"), torch.float32: (np.float32, "<f4"),
         torch.complex128: (np.complex128, "<c16"), torch.int32: (np.int32, "<i4")}


def _buffer(count, dtype=torch.float64):
    """(DeviceBuffer, torch view of its memory)"""
    kind, typestr = _KIND[dtype]
    buf = api.DeviceBuffer(count, kind)
    return buf, torch.as_tensor(_Shared(buf, count, typestr), device=DEV)


def _filled(t):
    buf, view = _buffer(t.numel(), t.dtype)
    view.copy_(t.reshape(-1))
    return buf


def _prm(method=1, max_iter=5000):
    prm = api.Prm().quiet()
    prm.Iarray[api.MONOLIS_PRM_I_METHOD] = method
    prm.Iarray[api.MONOLIS_PRM_I_MAX_ITER] = max_iter
    prm.Rarray[api.MONOLIS_PRM_R_TOL] = TOL
    return prm


# ---------------------------------------------------------------------------
# The cases' inputs
# ---------------------------------------------------------------------------
def prepare(case, seed):
    state = _PREPARE[case["path"]](case, seed)
    torch.cuda.synchronize()
    return state


def _prepare_matvec(case, seed):
    lengths, cols, A = _system(case, seed)
    dtype = torch.float32 if case["dtype"] == "f32" else torch.float64
    n = lengths.numel() * case["b"]
    x = _filled(_uniform((n,), seed + 1000, dtype))
    y, out = _buffer(n, dtype)
    dm = api.DeviceMatrix(_host_matrix(lengths, cols, A, case["b"]))
    torch.cuda.synchronize()
    return {"case": case, "dm": dm, "x": x, "y": y, "out": out}


def _prepare_solve(case, seed):
    lengths, cols, A = _system(case, seed)
    b = case["b"]
    rhs = _filled(_product(lengths, cols, A, _uniform((lengths.numel(), b), seed + 1000)))
    x, out = _buffer(lengths.numel() * b)
    dm = api.DeviceMatrix(_host_matrix(lengths, cols, A, b))
    torch.cuda.synchronize()
    return {"case": case, "dm": dm, "rhs": rhs, "x": x, "out": out, "method": METHODS[case["method"]]}


def _prepare_multi(case, seed):
    lengths, cols, A = _system({**case, "system": "diffusion7"}, seed)
    n, k = lengths.numel(), case["rhs"]
    X = _uniform((n, k), seed + 1000)
    rhs, view = _buffer(n * k)
    view = view.reshape(n, k)
    for j in range(0, k, 8):
        view[:, j:j + 8] = _product(lengths, cols, A, X[:, j:j + 8])
    x, out = _buffer(n * k)
    dm = api.DeviceMatrix(_host_matrix(lengths, cols, A, 1))
    torch.cuda.synchronize()
    return {"case": case, "dm": dm, "rhs": rhs, "x": x, "out": out}


def _batch_system(case, seed):
    count, lo, hi = case["count"], case["lo"], case["hi"]
    edges = [lo + (k * 7919 % count) * (hi - lo + 1) // count for k in range(count)]  # every size, in mixed order
    lengths, cols, start = [], [], [0]
    for e in edges:
        le, co = _pattern(e, e, e, 7)
        lengths.append(le)
        cols.append(co + start[-1])
        start.append(start[-1] + e ** 3)
    lengths, cols = torch.cat(lengths), torch.cat(cols)
    return lengths, cols, _blocks(lengths, cols, 1, seed, 0.0, 0.0), np.array(start, np.int64)


def _prepare_batch(case, seed):
    lengths, cols, A, start = _batch_system(case, seed)
    n = lengths.numel()
    rhs = _filled(_product(lengths, cols, A, _uniform((n, 1), seed + 1000)))
    x, out = _buffer(n)
    batch = api.DeviceBatch(_host_matrix(lengths, cols, A, 1), start)
    torch.cuda.synchronize()
    if case["tuned"]:
        batch.autotune(rhs, x, _prm(), reps=1)
    return {"case": case, "batch": batch, "rhs": rhs, "x": x, "out": out}


def _complex_system(case, seed):
    """K + 0.5 i D with D the diagonal blocks of K."""
    lengths, cols, K = _system({**case, "system": "block27"}, seed)
    rows = torch.repeat_interleave(torch.arange(lengths.numel(), device=DEV), lengths)
    return lengths, cols, torch.complex(K, 0.5 * K * (rows == cols.long())[:, None, None])


def _prepare_cocg(case, seed):
    lengths, cols, A = _complex_system(case, seed)
    n, b = lengths.numel(), case["b"]
    X = _uniform((n, b), seed + 1000, torch.complex128)
    # segment sums take real numbers
    Ax = torch.complex(_product(lengths, cols, A.real, X.real) - _product(lengths, cols, A.imag, X.imag),
                       _product(lengths, cols, A.real, X.imag) + _product(lengths, cols, A.imag, X.real))
    rhs = _filled(Ax)
    x, out = _buffer(n * b, torch.complex128)
    dm = api.DeviceMatrixC(_host_matrix(lengths, cols, A, b))
    torch.cuda.synchronize()
    return {"case": case, "dm": dm, "rhs": rhs, "x": x, "out": out}


def _prepare_grad(case, seed):
    lengths, cols, A = _system(case, seed)
    n, b = lengths.numel(), case["b"]
    X, Lam = _uniform((n, b), seed + 1000), _uniform((n, b), seed + 2000)
    sym = case["system"] == "block27"
    rhs = _filled(_product(lengths, cols, A, X))
    g = _filled((_product if sym else _transpose_product)(lengths, cols, A, Lam))
    values = _filled(A)
    # the handle was made with the values of an earlier step
    dm = api.DeviceMatrix(_host_matrix(lengths, cols, A * 1.25, b))
    (x, xo), (lam, lo), (dA, do) = _buffer(n * b), _buffer(n * b), _buffer(A.numel())
    torch.cuda.synchronize()
    return {"case": case, "dm": dm, "values": values, "rhs": rhs, "g": g, "x": x, "lam": lam, "dA": dA,
            "out": {"x": xo, "lam": lo, "dA": do}, "method": 1 if sym else 5, "sym": sym}


def _mesh(case):
    """Hexahedra of an nx x ny x nz element box: node ids of each element, in monolis's corner order."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    ids = torch.arange(nx * ny * nz, device=DEV)
    x, y, z = ids % nx, ids // nx % ny, ids // (nx * ny)
    corner = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
    return torch.stack([((z + dz) * (ny + 1) + y + dy) * (nx + 1) + x + dx for dx, dy, dz in corner], 1)


def _assembly_inputs(case, seed):
    """Element matrices (symmetric, positive diagonal), right-hand side, and the conditions on the face z = 0."""
    elems, b = _mesh(case), case["b"]
    m = 8 * b
    Ke = _uniform((elems.shape[0], m, m), seed + 1000)
    Ke = Ke + Ke.transpose(1, 2) + 2.0 * m * torch.eye(m, device=DEV, dtype=torch.float64)
    n_node = (case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1)
    rhs = _uniform((n_node * b,), seed + 2000)
    face = (case["nx"] + 1) * (case["ny"] + 1)
    nodes = torch.arange(face, device=DEV).repeat_interleave(b)
    dofs = torch.arange(b, device=DEV).repeat(face)
    return elems, Ke, rhs, nodes, dofs, _uniform((face * b,), seed + 3000)


def _prepare_assembly(case, seed):
    elems, Ke, rhs, nodes, dofs, vals = _assembly_inputs(case, seed)
    n_node, b = rhs.numel() // case["b"], case["b"]
    nz = (3 * case["nx"] + 1) * (3 * case["ny"] + 1) * (3 * case["nz"] + 1)
    f, fo = _buffer(rhs.numel())
    (A, Ao), (index, io), (item, to) = (_buffer(nz * b * b), _buffer(n_node + 1, torch.int32), _buffer(nz, torch.int32))
    state = {"case": case, "n_node": n_node, "n_elem": elems.shape[0], "nz": nz,
             "elems": _filled(elems.to(torch.int32)), "Ke": _filled(Ke), "load": _filled(rhs), "rhs": f, "A": A,
             "index": index, "item": item, "nodes": _filled(nodes.to(torch.int32)),
             "dofs": _filled(dofs.to(torch.int32)), "vals": _filled(vals),
             "out": {"A": Ao, "rhs": fo, "index": io, "item": to}}
    torch.cuda.synchronize()
    return state


def _prepare_host_solve(case, seed):
    lengths, cols, A = _system(case, seed)
    b = case["b"]
    rhs = _product(lengths, cols, A, _uniform((lengths.numel(), b), seed + 1000)).reshape(-1).cpu().numpy()
    return {"case": case, "mat": _host_matrix(lengths, cols, A, b).ensure_dof_index(), "rhs": rhs,
            "x": np.zeros(lengths.numel() * b)}


def _vblock_system(case, seed):
    """7-point block pattern with 1, 2, 3 or 6 unknowns a node: the scalar entries (r, c) in
    monolis's block-by-block order and their values, and the block arrays."""
    lengths, cols = _pattern(case["nx"], case["ny"], case["nz"], 7)
    n, cl = lengths.numel(), cols.long()
    ids = torch.arange(n, device=DEV)
    dof = torch.tensor([1, 2, 3, 3, 6, 3, 2, 6], device=DEV)[(ids * 2654435761 >> 7) % 8]
    first = _offsets(dof)
    rows = torch.repeat_interleave(ids, lengths)
    index2 = _offsets(dof[rows] * dof[cl])
    blk = torch.repeat_interleave(torch.arange(cl.numel(), device=DEV), dof[rows] * dof[cl])
    local = torch.arange(blk.numel(), device=DEV) - index2[blk]
    nc = dof[cl[blk]]
    r, c = first[rows[blk]] + local // nc, first[cl[blk]] + local % nc
    A = -_hash01(r, c, seed)
    A[r == c] = 0.0
    order = torch.argsort(r, stable=True)
    per_row = torch.bincount(r, minlength=int(first[-1]))
    A[r == c] = _row_sums(A[order].abs(), per_row) + 0.05
    return lengths, cols, dof, first, index2, r, c, A, order, per_row


def _prepare_vblock(case, seed):
    lengths, cols, dof, first, index2, r, c, A, order, per_row = _vblock_system(case, seed)
    m = int(first[-1])
    X = _uniform((m,), seed + 1000)
    rhs = _filled(_row_sums((A * X[c])[order], per_row))
    x, out = _buffer(m)
    i32 = lambda t: t.to(torch.int32).cpu().numpy()  # noqa: E731
    n = lengths.numel()
    dm = api.DeviceMatrix(Matrix(n, n, -1, i32(_offsets(lengths)), i32(cols + 1), A.cpu().numpy(), i32(dof), i32(first),
                                 i32(index2)))
    torch.cuda.synchronize()
    return {"case": case, "dm": dm, "rhs": rhs, "x": x, "out": out, "method": 1}


_PREPARE = {"matvec": _prepare_matvec, "solve": _prepare_solve, "multi": _prepare_multi, "batch": _prepare_batch,
            "cocg": _prepare_cocg, "grad": _prepare_grad, "assembly": _prepare_assembly,
            "host_solve": _prepare_host_solve, "vblock": _prepare_vblock}


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    return _RUN[state["case"]["path"]](state)


def _run_matvec(s):
    s["dm"].matvec(s["x"], s["y"])
    return s["out"]


def _run_solve(s):
    if s["case"].get("mode") == "refined":
        s["dm"].solve_refined(s["rhs"], s["x"], _prm(s["method"]))
    else:
        s["dm"].solve(s["rhs"], s["x"], _prm(s["method"]))
    return s["out"]


def _run_multi(s):
    s["dm"].solve_multi(s["rhs"], s["x"], s["case"]["rhs"], _prm())
    return s["out"]


def _run_batch(s):
    s["batch"].solve(s["rhs"], s["x"], _prm())
    return s["out"]


def _run_cocg(s):
    s["dm"].solve(s["rhs"], s["x"], _prm(13))
    return s["out"]


def _run_grad(s):
    dm = s["dm"]
    dm.set_values(s["values"])
    dm.solve(s["rhs"], s["x"], _prm(s["method"]))
    dm.adjoint(s["x"], s["g"], s["lam"], s["dA"], _prm(s["method"]), symmetric=s["sym"])
    return s["out"]


def _run_assembly(s):
    L, h = _lib.load(), ctypes.c_void_p()
    p = {k: ctypes.c_void_p(s[k].ptr) for k in ("elems", "Ke", "load", "rhs", "A", "index", "item", "nodes", "dofs", "vals")}
    _lib.check(L.monolis_hip_memcpy(p["rhs"], p["load"], s["rhs"].nbytes), "memcpy")
    _lib.check(L.monolis_hip_matrix_create_by_simple_mesh(ctypes.byref(h), s["n_node"], 8, s["case"]["b"], s["n_elem"],
                                                          p["elems"]), "create_by_simple_mesh")
    try:
        _lib.check(L.monolis_hip_matrix_add_elements_R(h, s["n_elem"], 8, p["elems"], p["Ke"]), "add_elements")
        _lib.check(L.monolis_hip_set_Dirichlet_bc_R(h, p["rhs"], s["nodes"].count, p["nodes"], p["dofs"], p["vals"]),
                   "set_Dirichlet_bc")
        info = (ctypes.c_longlong * 8)()
        _lib.check(L.monolis_hip_matrix_info(h, info), "info")
        if info[2] != s["nz"]:
            raise RuntimeError("unexpected pattern")
        _lib.check(L.monolis_hip_matrix_get_pattern(h, p["index"], p["item"]), "get_pattern")
        _lib.check(L.monolis_hip_matrix_get_values_R(h, p["A"]), "get_values")
    finally:
        L.monolis_hip_matrix_destroy(h)
    return s["out"]


def _run_host_solve(s):
    api.monolis_solve_R(api.Monolis(s["mat"], _prm()), s["rhs"], s["x"])
    return s["x"]


_RUN = {"matvec": _run_matvec, "solve": _run_solve, "multi": _run_multi, "batch": _run_batch, "cocg": _run_cocg,
        "grad": _run_grad, "assembly": _run_assembly, "host_solve": _run_host_solve, "vblock": _run_solve}


# ---------------------------------------------------------------------------
# Bytes and operations one pass needs
# ---------------------------------------------------------------------------
def _nnz(ext, points):
    nx, ny, nz = ext
    if points == 27:
        return (3 * nx - 2) * (3 * ny - 2) * (3 * nz - 2)
    n = nx * ny * nz
    return 7 * n - 2 * (n // nx + n // ny + n // nz)


def _iterations(system, ext, method):
    """Iterations to TOL (measured; they follow the mesh for the scalar operators)."""
    e = (ext[0] * ext[1] * ext[2]) ** (1 / 3)
    if system == "block27":
        it = min(55.0, 8.0 + 1.6 * e)
    elif system == "vblock":
        it = min(130.0, 10.0 + 3.5 * e)
    else:
        it = 12.0 + 3.6 * e
    return 0.65 * it if method == "bicgstab" else it


def _solve_work(system, ext, b, method, size, k=1):
    """Per iteration: the matrix once (twice in BiCGSTAB) with 4-byte columns, its block-diagonal
    factors and the recurrence's vectors (11 in CG, 20 in BiCGSTAB), k right-hand sides."""
    points = 27 if system == "block27" else 7
    n, nnz = ext[0] * ext[1] * ext[2], _nnz(ext, points)
    it = _iterations(system, ext, method)
    products, vectors = (2, 20) if method == "bicgstab" else (1, 11)
    nbytes = it * (products * (nnz * (b * b * size + 4) + n * b * b * size) + vectors * n * b * size * k)
    flops = it * (products * 2 * nnz * b * b * k + vectors * 2 * n * b * k) * (4 if size == 16 else 1)
    return {"bytes": nbytes, "flops": flops}


def work(case):
    path = case["path"]
    if path == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        edges = case["hi"] - case["lo"] + 1
        for e in range(case["lo"], case["hi"] + 1):
            w = _solve_work("diffusion7", (e, e, e), 1, "cg", 8)
            total = {q: total[q] + w[q] * case["count"] / edges for q in total}
        return total
    ext = (case["nx"], case["ny"], case["nz"])
    n = ext[0] * ext[1] * ext[2]
    if path == "matvec":
        b, size = case["b"], 4 if case["dtype"] == "f32" else 8
        nnz = _nnz(ext, 27 if case["system"] == "block27" else 7)
        return {"bytes": nnz * (b * b * size + 4) + (n + 1) * 4 + 2 * n * b * size, "flops": 2 * nnz * b * b}
    if path == "solve":
        return _solve_work(case["system"], ext, case["b"], case["method"], 4 if case["mode"] == "refined" else 8)
    if path == "multi":
        return _solve_work("diffusion7", ext, 1, "cg", 8, case["rhs"])
    if path == "cocg":
        w = _solve_work("block27", ext, case["b"], "cg", 16)
        return {q: 0.4 * v for q, v in w.items()}  # the damping shortens the iteration
    if path == "grad":
        w = _solve_work(case["system"], ext, case["b"], "cg" if case["system"] == "block27" else "bicgstab", 8)
        return {q: 2 * v for q, v in w.items()}
    if path == "assembly":
        b = case["b"]
        nz = (3 * ext[0] + 1) * (3 * ext[1] + 1) * (3 * ext[2] + 1)
        return {"bytes": n * (64 * b * b * 8 + 32) + nz * (b * b * 8 + 4), "flops": n * 64 * b * b}
    if path == "host_solve":
        return _solve_work(case["system"], ext, case["b"], "cg", 8)
    # vblock: 3.25 unknowns a node on average, 10.5 x 10.5 / 3.25 scalar entries a block
    points, nodes = _nnz(ext, 7), n
    it = _iterations("vblock", ext, "cg")
    return {"bytes": it * (points * 10.6 * 12 + nodes * (13.5 * 8 + 11 * 3.25 * 8)),
            "flops": it * (points * 21 + nodes * 72)}


# ---------------------------------------------------------------------------
# Results: 64-bit values and how far another correct implementation may be from them
# ---------------------------------------------------------------------------
def tolerance(case):
    path = case["path"]
    if path == "matvec":  # sums of up to 162 products in another order
        return {"rel": 1e-6, "max": 1e-5} if case["dtype"] == "f32" else {"rel": 2e-15, "max": 2e-14}
    if path == "assembly":  # sums of at most 8 entries
        return {"rel": 2e-15, "max": 2e-14}
    # solves to a relative residual of 1e-8: an iteration more or less moves the result by the
    # residual times the condition of the system (measured against the exact solutions: 1e-7 for
    # block27, 7e-9 for its damped complex form, 3.3e-7 for vblock, 1.2e-7, 9e-7 and 1.6e-6 for
    # the scalar operators on 32, 96 and 128 nodes per axis); here four times that
    if path == "cocg":
        return {"rel": 4e-8}
    if path == "vblock":
        return {"rel": 1.3e-6}
    if case.get("system") == "block27":
        return {"rel": 4e-7}
    edge = case["hi"] if path == "batch" else max(case["nx"], case["ny"], case["nz"])
    return {"rel": 4e-8 + 4.5e-10 * edge * edge}


def exact(case, seed):
    path = case["path"]
    if path == "matvec":
        lengths, cols, A = _system(case, seed)
        dtype = torch.float32 if case["dtype"] == "f32" else torch.float64
        x = _uniform((lengths.numel() * case["b"],), seed + 1000, dtype).double()
        return _product(lengths, cols, A, x.reshape(-1, case["b"])).reshape(-1)
    if path == "batch":
        return _uniform((sum(_batch_rows(case)),), seed + 1000)
    n = case["nx"] * case["ny"] * case["nz"]
    if path in ("solve", "host_solve"):
        return _uniform((n, case["b"]), seed + 1000).reshape(-1)
    if path == "multi":
        return _uniform((n, case["rhs"]), seed + 1000).reshape(-1)
    if path == "cocg":
        return _uniform((n, case["b"]), seed + 1000, torch.complex128).reshape(-1)
    if path == "vblock":
        return _uniform((int(_vblock_system(case, seed)[3][-1]),), seed + 1000)
    if path == "grad":
        lengths, cols, _ = _system(case, seed)
        X, Lam = _uniform((n, case["b"]), seed + 1000), _uniform((n, case["b"]), seed + 2000)
        rows = torch.repeat_interleave(torch.arange(n, device=DEV), lengths)
        return {"x": X.reshape(-1), "lam": Lam.reshape(-1),
                "dA": -(Lam[rows][:, :, None] * X[cols.long()][:, None, :]).reshape(-1)}
    return _exact_assembly(case, seed)


def _batch_rows(case):
    count, lo, hi = case["count"], case["lo"], case["hi"]
    return [(lo + (k * 7919 % count) * (hi - lo + 1) // count) ** 3 for k in range(count)]


def _exact_assembly(case, seed):
    elems, Ke, rhs, nodes, dofs, vals = _assembly_inputs(case, seed)
    b, n_node = case["b"], rhs.numel() // case["b"]
    lengths, cols = _pattern(case["nx"] + 1, case["ny"] + 1, case["nz"] + 1, 27)
    index, cl = _offsets(lengths), cols.long()
    rows = torch.repeat_interleave(torch.arange(n_node, device=DEV), lengths)
    key = rows * n_node + cl
    A = torch.zeros((cl.numel(), b, b), device=DEV, dtype=torch.float64)
    for a in range(8):
        for c in range(8):
            pos = torch.searchsorted(key, elems[:, a] * n_node + elems[:, c])
            A.index_add_(0, pos, Ke[:, a * b:(a + 1) * b, c * b:(c + 1) * b].contiguous())
    v = torch.zeros(n_node * b, device=DEV, dtype=torch.float64)
    fixed = torch.zeros(n_node * b, device=DEV, dtype=torch.bool)
    v[nodes * b + dofs] = vals
    fixed[nodes * b + dofs] = True
    v, fixed = v.reshape(-1, b), fixed.reshape(-1, b)
    f = rhs.reshape(-1, b) - _product(lengths, cols, A, v)
    f = torch.where(fixed, v, f)
    A = A * (~fixed[rows])[:, :, None] * (~fixed[cl])[:, None, :]
    diag = (rows == cl).nonzero().reshape(-1)
    k = torch.arange(b, device=DEV)
    A[diag[:, None], k, k] = torch.where(fixed, torch.ones_like(v), A[diag[:, None], k, k])
    return {"A": A.reshape(-1), "rhs": f.reshape(-1), "index": None, "item": None}
