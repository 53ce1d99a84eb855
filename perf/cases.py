"""The work that programs have this library do on one GPU, as measurable cases.

Every case calls the public C interface (through the `gooseberry_amd` module) on data that is
resident on the GPU, as a program that keeps its matrices and vectors there does. The inputs are
made with torch from the case and the seed alone, and `exact` computes each result in plain torch
in 64 bits.

Kinds of case and the ranges that `draw` spreads over:

  spmv      y = A x in FP64 or FP32 on grid Laplacians and random symmetric diagonally dominant
            matrices, a thousand to four million rows
  spmm      C = A B for 2 to 32 right-hand sides
  cg        one FP64 conjugate-gradient solve to a relative residual of 1e-8 or 1e-10
  mixed     one mixed-precision solve (FP32 inner, FP64 refined) to 1e-10
  batch     independent solves of uneven sizes advanced together
  spgemm    a sparse product C = A B kept on the GPU, and its first use, y = C x
  pagerank  PageRank of a directed, weighted graph, column normalisation included
  parse     CSR text that lies in device memory into CSR arrays in device memory
"""
import ctypes
import math
import random

import torch

import gooseberry_amd as gb

DEV = "cuda"
VALUE_BITS = 20  # off-diagonals are multiples of 2^-20: their sums are exact in any order


def listed():
    return [
        # one product of the drop-in program's example system: a launch and little else
        {"name": "spmv_2d_256", "kind": "spmv", "matrix": "lap", "nx": 256, "ny": 256, "nz": 1,
         "dtype": "f64"},
        # the headline product: a 3D stencil that no cache holds
        {"name": "spmv_3d_160", "kind": "spmv", "matrix": "lap", "nx": 160, "ny": 160, "nz": 160,
         "dtype": "f64"},
        # the inner product of a served mixed-precision request: random columns, about 29 a row
        {"name": "spmv_f32_sdd", "kind": "spmv", "matrix": "sdd", "n": 300007, "law": "uniform",
         "dmin": 3, "dmax": 27, "dtype": "f32", "xtile": 0},
        # a block of right-hand sides through one matrix
        {"name": "spmm_3d_8", "kind": "spmm", "matrix": "lap", "nx": 101, "ny": 100, "nz": 99,
         "cols": 8},
        # the example system's solve: several hundred short iterations
        {"name": "cg_2d_256", "kind": "cg", "nx": 256, "ny": 256, "nz": 1, "tol": 1e-8},
        # the headline solve
        {"name": "cg_3d_160", "kind": "cg", "nx": 160, "ny": 160, "nz": 160, "tol": 1e-10},
        # irregular rows: Zipf degrees, mixed precision, the plan that suits scattered columns
        {"name": "mixed_zipf", "kind": "mixed", "n": 400000, "law": "zipf", "dmin": 2,
         "dmax": 4096, "xtile": 8192},
        # many uneven systems at once, as a batch program or a solve server holds them
        {"name": "batch_48", "kind": "batch", "systems": 48, "sizes": 3, "nmin": 1000,
         "nmax": 200000, "precision": "mixed_jacobi"},
        # squaring a stencil: short rows
        {"name": "spgemm_3d_90", "kind": "spgemm", "matrix": "lap", "nx": 90, "ny": 91, "nz": 89},
        # a product of random matrices: several hundred products to a row
        {"name": "spgemm_sdd", "kind": "spgemm", "matrix": "sdd", "n": 60000, "law": "uniform",
         "dmin": 3, "dmax": 27},
        # PageRank of a graph with Zipf degrees, a hundred iterations at most
        {"name": "pagerank_zipf", "kind": "pagerank", "n": 300000, "law": "zipf", "dmin": 2,
         "dmax": 4096, "niter": 100, "xtile": 8192},
        # a matrix file's text, six digits a value
        {"name": "parse_6", "kind": "parse", "rows": 500000, "dmin": 3, "dmax": 27, "digits": 6},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, nmin, nmax):
    """An uneven 2D or 3D grid of about nmin to nmax points."""
    n = _log(rng, nmin, nmax)
    if rng.random() < 0.5:
        nx = max(2, int(n ** 0.5 * rng.uniform(0.7, 1.4)))
        return {"nx": nx, "ny": max(2, n // nx), "nz": 1}
    nx = max(2, int(n ** (1 / 3) * rng.uniform(0.8, 1.25)))
    ny = max(2, int(n ** (1 / 3) * rng.uniform(0.8, 1.25)))
    return {"nx": nx, "ny": ny, "nz": max(2, n // (nx * ny))}


def draw(rng):
    kind = rng.choice(["spmv", "spmv", "spmm", "cg", "mixed", "batch", "spgemm", "spgemm",
                       "pagerank", "parse"])
    c = {"kind": kind}
    if kind == "spmv":
        c["dtype"] = rng.choice(["f64", "f32"])
        if rng.random() < 0.5:
            c["matrix"] = "lap"
            c.update(_grid(rng, 1000, 4000000))
        else:
            c.update({"matrix": "sdd", "n": _log(rng, 2000, 1048576), "law": "uniform",
                      "dmin": 3, "dmax": 27, "xtile": 0})
    elif kind == "spmm":
        c["cols"] = rng.choice([2, 3, 4, 5, 7, 8, 11, 16, 32])
        top = 8000000 // c["cols"]
        if rng.random() < 0.5:
            c["matrix"] = "lap"
            c.update(_grid(rng, 1000, top))
        else:
            c.update({"matrix": "sdd", "n": _log(rng, 2000, top // 4), "law": "uniform",
                      "dmin": 3, "dmax": 27})
    elif kind == "cg":
        c["tol"] = rng.choice([1e-8, 1e-10])
        c.update(_grid(rng, 1000, 300000 if rng.random() < 0.5 else 1000000))
    elif kind == "mixed":
        if rng.random() < 0.5:
            c.update({"n": _log(rng, 20000, 400000), "law": "zipf", "dmin": 2, "dmax": 4096,
                      "xtile": rng.choice([0, 8192])})
        else:
            c.update({"n": _log(rng, 4096, 1048576), "law": "uniform", "dmin": 3, "dmax": 27,
                      "xtile": 0})
    elif kind == "batch":
        c.update({"systems": _log(rng, 4, 48), "sizes": rng.randrange(1000), "nmin": 1000,
                  "nmax": _log(rng, 20000, 200000),
                  "precision": rng.choice(["fp64", "mixed", "mixed_jacobi"])})
    elif kind == "spgemm":
        if rng.random() < 0.4:
            c["matrix"] = "lap"
            c.update(_grid(rng, 2000, 700000))
        else:
            dmax = rng.choice([5, 9, 16, 27, 40])
            c.update({"matrix": "sdd", "n": _log(rng, 2000, 40000000 // dmax ** 2),
                      "law": "uniform", "dmin": 3, "dmax": dmax})
    elif kind == "pagerank":
        c.update({"n": _log(rng, 10000, 300000), "law": rng.choice(["zipf", "uniform"]),
                  "dmin": 2, "niter": rng.choice([20, 50, 100])})
        c["dmax"] = 4096 if c["law"] == "zipf" else 40
        c["xtile"] = rng.choice([0, 8192])
    else:
        c.update({"rows": _log(rng, 1000, 500000), "dmin": rng.choice([1, 3, 20]),
                  "digits": rng.choice([1, 6, 15])})
        c["dmax"] = c["dmin"] + rng.choice([4, 20, 24])
    return c


# ------------------------------------------------------------------ inputs

def _gen(seed, what):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 64 + what)
    return g


def _uniform(seed, n, what=0):
    return torch.rand(n, dtype=torch.float64, device=DEV, generator=_gen(seed, what)) * 2 - 1


def _laplacian(nx, ny, nz):
    """(rowptr, col, val) of the 5- or 7-point Dirichlet Laplacian, columns ascending."""
    n = nx * ny * nz
    i = torch.arange(n, device=DEV)
    x, y, z = i % nx, (i // nx) % ny, i // (nx * ny)
    here = torch.ones_like(x, dtype=torch.bool)
    cols, have, vals = [i], [here], [4.0 if nz == 1 else 6.0]
    for pos, size, step in ((x, nx, 1), (y, ny, nx), (z, nz, nx * ny)):
        if size == 1:
            continue
        cols = [i - step] + cols + [i + step]
        have = [pos > 0] + have + [pos < size - 1]
        vals = [-1.0] + vals + [-1.0]
    have = torch.stack(have, 1)
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(have.sum(1), 0, out=ptr[1:])
    col = torch.stack(cols, 1)[have]
    val = torch.tensor(vals, dtype=torch.float64, device=DEV).expand(n, len(vals))[have]
    return ptr, col, val


def _degrees(n, law, dmin, dmax, g):
    u = torch.rand(n, dtype=torch.float64, device=DEV, generator=g)
    if law == "uniform":
        return dmin + (u * (dmax - dmin + 1)).long().clamp(max=dmax - dmin)
    k = torch.arange(1, 1 << 16, dtype=torch.float64, device=DEV)  # Zipf(1.5), clipped
    cdf = torch.cumsum(k ** -1.5, 0)
    return (torch.searchsorted(cdf / cdf[-1], u) + 1).clamp(dmin, dmax)


def _csr(n, row, col, val):
    order = torch.sort(row * n + col, stable=True).indices
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(torch.bincount(row, minlength=n), 0, out=ptr[1:])
    return ptr, col[order], val[order]


def _edges(n, law, dmin, dmax, seed, spare):
    """Directed edges: each row draws its degree less `spare`, uniform heads other than itself,
    and weights that are multiples of 2^-20 in (0, 1]."""
    g = _gen(seed, 1)
    deg = _degrees(n, law, dmin, dmax, g) - spare
    row = torch.repeat_interleave(torch.arange(n, device=DEV), deg)
    col = torch.randint(0, n - 1, (row.numel(),), device=DEV, generator=g)
    col = col + (col >= row)
    w = torch.randint(1, (1 << VALUE_BITS) + 1, (row.numel(),), device=DEV, generator=g)
    return row, col, w.double() / (1 << VALUE_BITS)


def _sdd(n, law, dmin, dmax, seed):
    """A random symmetric, strictly diagonally dominant matrix, columns ascending."""
    row, col, w = _edges(n, law, dmin, dmax, seed, 1)
    row, col, w = torch.cat([row, col]), torch.cat([col, row]), torch.cat([w, w])
    diag = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, row, w) * 1.01
    diag = torch.where(diag > 0, diag, torch.ones_like(diag))
    own = torch.arange(n, device=DEV)
    return _csr(n, torch.cat([row, own]), torch.cat([col, own]), torch.cat([-w, diag]))


def _graph(case, seed):
    return _csr(case["n"], *_edges(case["n"], case["law"], case["dmin"], case["dmax"], seed, 0))


def _matrix(case, seed):
    if case.get("matrix", "sdd" if "n" in case else "lap") == "lap":
        return _laplacian(case["nx"], case["ny"], case["nz"])
    return _sdd(case["n"], case["law"], case["dmin"], case["dmax"], seed)


def _sizes(case):
    """The grids of a batch: 2D and 3D in turn, sizes log-uniform."""
    rng = random.Random(case["sizes"])
    got = []
    for k in range(case["systems"]):
        n = math.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"])))
        if k % 2 == 0:
            m = max(2, int(round(n ** 0.5)))
            got.append((m, m, 1))
        else:
            m = max(2, int(round(n ** (1 / 3))))
            got.append((m, m, m))
    return got


def _text(case, seed):
    """CSR text (1-based columns) and the arrays that it says. The row lengths go by the case, so
    that the outputs have one shape; columns and values go by the seed."""
    g = _gen(seed, 2)
    n, digits = case["rows"], case["digits"]
    deg = _degrees(n, "uniform", case["dmin"], case["dmax"], _gen(n, 3))
    row = torch.repeat_interleave(torch.arange(n, device=DEV), deg)
    nnz = row.numel()
    col = torch.randint(0, n, (nnz,), device=DEV, generator=g)
    col[0], col[-1] = 0, n - 1
    neg = torch.randint(0, 2, (nnz,), device=DEV, generator=g).bool()
    m = torch.randint(1, 10 ** digits, (nnz,), device=DEV, generator=g)
    frac = digits > 1
    val = m.double() / (10.0 ** digits if frac else 1.0)
    val = torch.where(neg, -val, val)
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(deg, 0, out=ptr[1:])
    wide = len(str(n))
    chars = torch.zeros((nnz, 1 + wide + 2 + (2 if frac else 0) + digits), dtype=torch.uint8,
                        device=DEV)
    chars[:, 0] = 32
    chars[ptr[:-1], 0] = 10
    chars[0, 0] = 0
    for k in range(wide):  # leading zeros are left out
        p = 10 ** (wide - 1 - k)
        chars[:, 1 + k] = torch.where(col + 1 >= p, ((col + 1) // p) % 10 + 48, 0).to(torch.uint8)
    at = 1 + wide
    chars[:, at] = 32
    chars[:, at + 1] = torch.where(neg, 45, 0).to(torch.uint8)
    at += 2
    if frac:
        chars[:, at], chars[:, at + 1] = 48, 46
        at += 2
    for k in range(digits):
        chars[:, at + k] = ((m // 10 ** (digits - 1 - k)) % 10 + 48).to(torch.uint8)
    text = torch.cat([chars[chars != 0], torch.tensor([10], dtype=torch.uint8, device=DEV)])
    return text, ptr, col, val


# ----------------------------------------------------------- library objects

class Vec:
    """A torch tensor where the library takes a device vector."""

    def __init__(self, t):
        self.t, self.ptr, self.n = t, t.data_ptr(), t.numel()


class DeviceBlock:
    """Device memory that the library handed over, as a tensor; given back when unused."""

    def __init__(self, ptr, n, kind):
        self.ptr = ptr
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": kind, "data": (ptr, False),
                                         "version": 2}

    def __del__(self):
        gb.lib().gooseberry_device_free(self.ptr)


def _resident(n, csr, xtile=0):
    ptr, col, val = csr[0], csr[1].to(torch.int32), csr[2]
    torch.cuda.synchronize()  # the library reads them on its own stream
    M = gb.Matrix.from_device64(n, n, ptr.data_ptr(), col.data_ptr(), val.data_ptr(),
                                plan={"xtile": xtile} if xtile else None)
    gb.synchronize()
    return M


def _order(case):
    if case["kind"] == "parse":
        return case["rows"]
    return case["n"] if "n" in case else case["nx"] * case["ny"] * case["nz"]


PRECISION = {"fp64": gb.PRECISION_FP64, "mixed": gb.PRECISION_MIXED,
             "mixed_jacobi": gb.PRECISION_MIXED_JACOBI}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "parse":
        return {"case": case, "text": _text(case, seed)[0]}
    if kind == "batch":
        grids = _sizes(case)
        ns = [a * b * c for a, b, c in grids]
        total = sum(ns)
        b, x = _uniform(seed, total), torch.zeros(total, dtype=torch.float64, device=DEV)
        systems, at = [], 0
        for g, n in zip(grids, ns):
            systems.append((_resident(n, _laplacian(*g)), Vec(b[at:at + n]), Vec(x[at:at + n])))
            at += n
        return {"case": case, "x": x, "b": b, "systems": systems,
                "batch": gb.Batch(case["systems"])}
    n = _order(case)
    if kind == "pagerank":
        M = _resident(n, _graph(case, seed), case["xtile"])
        return {"case": case, "M": M, "out": Vec(torch.zeros(n, dtype=torch.float64, device=DEV))}
    M = _resident(n, _matrix(case, seed), case.get("xtile", 0))
    st = {"case": case, "M": M}
    if kind == "spgemm":
        st["B"] = M if case["matrix"] == "lap" else _resident(n, _matrix(case, seed + (1 << 24)))
    k = case.get("cols", 1)
    x = _uniform(seed, n * k)
    y = torch.zeros(n * k, dtype=torch.float64, device=DEV)
    if case.get("dtype") == "f32":
        x, y = x.float(), y.float()
    st["x"], st["y"] = Vec(x), Vec(y)
    return st


def run(st):
    case, kind = st["case"], st["case"]["kind"]
    L = gb.lib()
    if kind == "spmv":
        if case["dtype"] == "f64":
            st["M"].spmv_device(st["x"], st["y"])
        else:
            gb.check(L.gooseberry_matrix_spmv_f32(st["M"].h, st["x"].ptr, st["y"].ptr), "spmv_f32")
        return st["y"].t
    if kind == "spmm":
        gb.check(L.gooseberry_matrix_spmm(st["M"].h, case["cols"], st["x"].ptr, st["y"].ptr),
                 "spmm")
        return st["y"].t.view(-1, case["cols"])
    if kind == "cg":
        st["M"].cgd_device(st["x"], st["y"], case["tol"])
        return st["y"].t
    if kind == "mixed":
        info = gb.CgdInfo()
        gb.check(L.gooseberry_matrix_cgd_mixed(st["M"].h, st["x"].ptr, st["y"].ptr, 1e-10,
                                               gb.TOL_RELATIVE, 0, ctypes.byref(info)), "mixed")
        return st["y"].t
    if kind == "batch":
        B, p = st["batch"], PRECISION[case["precision"]]
        slots = [B.add(M, b, x, 1e-10, precision=p) for M, b, x in st["systems"]]
        B.solve()
        for s in slots:
            B.remove(s)
        return st["x"]
    if kind == "spgemm":
        C = st["M"].spmultsp(st["B"])
        C.spmv_device(st["x"], st["y"])
        nnz = C.nnz
        C.free()
        return {"nnz": nnz, "y": st["y"].t}
    if kind == "pagerank":
        st["M"].pagerank_device(st["out"], damping=0.85, niter=case["niter"])
        return st["out"].t
    nr, nc = ctypes.c_uint32(), ctypes.c_uint32()
    p = [ctypes.c_void_p() for _ in range(3)]
    text = st["text"]
    gb.check(L.gooseberry_parse_csr_device(text.data_ptr(), text.numel(), ctypes.byref(nr),
                                           ctypes.byref(nc), *[ctypes.byref(q) for q in p]),
             "parse")
    last = ctypes.c_uint32()
    gb.check(L.gooseberry_memcpy_dtoh(ctypes.byref(last), p[0].value + 4 * nr.value, 4), "dtoh")
    nnz = last.value
    return {"rows": nr.value, "cols": nc.value,
            "ptr": torch.as_tensor(DeviceBlock(p[0].value, nr.value + 1, "<i4"), device=DEV),
            "col": torch.as_tensor(DeviceBlock(p[1].value, nnz, "<i4"), device=DEV),
            "val": torch.as_tensor(DeviceBlock(p[2].value, nnz, "<f8"), device=DEV)}


# -------------------------------------------------------- work and tolerance

def _mean_degree(law, dmin, dmax):
    if law == "uniform":
        return (dmin + dmax) / 2
    w = [k ** -1.5 for k in range(1, 1 << 16)]
    return sum(p * min(max(k, dmin), dmax) for k, p in enumerate(w, 1)) / sum(w)


def _entries(case):
    if "n" in case:
        d = _mean_degree(case["law"], case["dmin"], case["dmax"])
        return case["n"] * (d if case["kind"] == "pagerank" else 2 * (d - 1) + 1)
    return _grid_entries(case["nx"], case["ny"], case["nz"])


def _grid_entries(nx, ny, nz):
    n = nx * ny * nz
    return n + 2 * sum(n - n // s for s in (nx, ny, nz))


def _grid_iterations(nx, ny, nz, tol):
    """About the iterations that CG takes on this grid from a random right-hand side."""
    per = 0.17 if nz > 1 else 0.115
    return max(4.0, per * max(nx, ny, nz) * -math.log(tol) * (1.0 if nz > 1 else 2.0) / 2)


def _solve_bytes(n, nnz, iterations, value=8):
    # an iteration reads the matrix and the three vectors r, p and x, and writes them and A p
    return iterations * ((4 + value) * nnz + 4 * (n + 1) + 8 * value * n)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        b = f = 0.0
        for g in _sizes(case):
            n, nnz, it = g[0] * g[1] * g[2], _grid_entries(*g), _grid_iterations(*g, 1e-10)
            b += _solve_bytes(n, nnz, it, 8 if case["precision"] == "fp64" else 4)
            f += it * (2 * nnz + 10 * n)
        return {"bytes": b, "flops": f}
    if kind == "parse":
        entries = case["rows"] * (case["dmin"] + case["dmax"]) / 2
        text = entries * (len(str(case["rows"])) + case["digits"]
                          + (4.5 if case["digits"] > 1 else 2.5))
        return {"bytes": text + 12 * entries + 4 * case["rows"], "flops": entries}
    n, nnz = _order(case), _entries(case)
    if kind == "spmv":
        v = 8 if case["dtype"] == "f64" else 4
        return {"bytes": (4 + v) * nnz + 4 * (n + 1) + 2 * v * n, "flops": 2 * nnz}
    if kind == "spmm":
        k = case["cols"]
        return {"bytes": 12 * nnz + 4 * (n + 1) + 16 * n * k, "flops": 2 * nnz * k}
    if kind == "cg":
        it = _grid_iterations(case["nx"], case["ny"], case["nz"], case["tol"])
        return {"bytes": _solve_bytes(n, nnz, it), "flops": it * (2 * nnz + 10 * n)}
    if kind == "mixed":  # about these many FP32 iterations, and 9 FP64 refreshes
        it = 170 if case["law"] == "zipf" else 50
        return {"bytes": _solve_bytes(n, nnz, it, 4) + _solve_bytes(n, nnz, 9),
                "flops": (it + 9) * (2 * nnz + 10 * n)}
    if kind == "pagerank":
        it = case["niter"]
        return {"bytes": (it + 2) * (12 * nnz + 4 * (n + 1) + 16 * n), "flops": it * 2 * nnz}
    if case["matrix"] == "lap":
        products, out = nnz * nnz / n, n * (25 if case["nz"] > 1 else 13)
    else:
        products = out = nnz * nnz / n
    return {"bytes": 24 * nnz + 12 * 2 * out + 16 * n, "flops": 2 * products + 2 * out}


def tolerance(case):
    """About four times the error against 64-bit results that the cases show (and for solves, the
    distance that two stops at the same relative residual can have in x)."""
    kind = case["kind"]
    if kind == "parse":
        return "exact"
    if kind == "spmv" and case["dtype"] == "f32":
        return {"rel": 5e-7, "max": 1e-5}
    if kind in ("spmv", "spmm", "spgemm"):
        return {"rel": 1.5e-15, "max": 5e-14}
    if kind == "pagerank":
        return {"rel": 1e-14, "max": 4e-13}
    if kind == "mixed":
        return {"rel": 5e-10, "max": 2e-8}
    return {"rel": 60 * case.get("tol", 1e-10), "max": 2400 * case.get("tol", 1e-10)}


# ------------------------------------------------------------------- exact

def _apply(csr):
    """x -> A x in torch, in 64 bits."""
    ptr, col, val = csr
    n = ptr.numel() - 1
    row = torch.repeat_interleave(torch.arange(n, device=DEV), ptr[1:] - ptr[:-1])

    def mul(x):
        return torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, row, val * x[col])

    diag = torch.zeros(n, dtype=torch.float64, device=DEV)
    on = row == col
    diag.index_add_(0, row[on], val[on])
    return mul, diag


def _solve(csr, b, rel=1e-14, most=6000):
    """Conjugate gradients with a diagonal preconditioner, far past the tolerance of the cases."""
    mul, diag = _apply(csr)
    x, r = torch.zeros_like(b), b.clone()
    z = r / diag
    p, rz = z.clone(), torch.dot(r, z)
    stop = rel * float(torch.linalg.vector_norm(b))
    for k in range(most):
        q = mul(p)
        a = rz / torch.dot(p, q)
        x += a * p
        r -= a * q
        if k % 16 == 15 and float(torch.linalg.vector_norm(r)) <= stop:
            break
        z = r / diag
        new = torch.dot(r, z)
        p = z + (new / rz) * p
        rz = new
    return x


def _stack(parts):
    """The block-diagonal matrix of several."""
    ptrs, cols, vals, rows, ents = [torch.zeros(1, dtype=torch.int64, device=DEV)], [], [], 0, 0
    for ptr, col, val in parts:
        ptrs.append(ptr[1:] + ents)
        cols.append(col + rows)
        vals.append(val)
        rows += ptr.numel() - 1
        ents += val.numel()
    return torch.cat(ptrs), torch.cat(cols), torch.cat(vals)


def _pagerank(case, seed):
    """The reference program's iteration (src/gooseberry_bin.c:2622-2737) without empty rows:
    each weight over its column's sum, then rank' = d A rank + (1 - d) / n from 1 / n, and the
    vector before the last iterate."""
    n, d = case["n"], 0.85
    ptr, col, val = _graph(case, seed)
    sums = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, col, val)
    mul, _ = _apply((ptr, col, val / sums[col]))
    rank = torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEV)
    out = rank
    for _ in range(case["niter"]):
        rank, out = out, mul(out) * d + (1 - d) / n
    return rank


def exact(case, seed):
    kind = case["kind"]
    if kind == "parse":
        _, ptr, col, val = _text(case, seed)
        return {"rows": case["rows"], "cols": case["rows"], "ptr": None, "col": None, "val": val}
    if kind == "batch":
        parts = [_laplacian(*g) for g in _sizes(case)]
        csr = _stack(parts)
        return _solve(csr, _uniform(seed, csr[0].numel() - 1))
    n = _order(case)
    if kind == "pagerank":
        return _pagerank(case, seed)
    csr = _matrix(case, seed)
    k = case.get("cols", 1)
    x = _uniform(seed, n * k)
    if kind in ("cg", "mixed"):
        return _solve(csr, x)
    if kind == "spmv" and case["dtype"] == "f32":
        x = x.float().double()
        csr = (csr[0], csr[1], csr[2].float().double())
    mul, _ = _apply(csr)
    if kind == "spmm":
        return torch.stack([mul(x[j * n:(j + 1) * n]) for j in range(k)], 1)
    if kind == "spgemm":
        first = mul if case["matrix"] == "lap" else _apply(_matrix(case, seed + (1 << 24)))[0]
        return {"nnz": None, "y": mul(first(x))}
    return mul(x)
