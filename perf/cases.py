"""Timed workloads of the library: single products, Jacobi-PCG, Jacobi-GMRES,
the adjoint, batches of systems and the assembly of a matrix from unordered
entries, each through the C ABI (include/cel_gpu.h) or the Python front end.

Vectors live in HBM, as a program keeps them that solves with the same
matrix many times; the smallest solve takes host arrays, as a Fortran caller
does.  Right-hand sides are b = A x_true with x_true ~ U[0,1) from the seed,
so the exact solution is known.
"""
import ctypes as C
import math

import numpy as np
import torch

import cel_v3_amd as cel

FORMATS = {"csr": cel.FMT_CSR, "jad": cel.FMT_JAD, "dia": cel.FMT_DIA}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one product on the smallest block a program meets: latency
        {"name": "spmv_32", "kind": "spmv", "problem": "poisson", "nx": 32, "ny": 32, "nz": 32,
         "fmt": "csr", "f32": False, "accumulate": False},
        # y += A x on an unstructured mesh matrix, rows of uneven length, odd size
        {"name": "spmv_mesh_1m", "kind": "spmv", "problem": "mesh", "n": 1000003, "deg": 6,
         "fmt": "csr", "f32": False, "accumulate": True},
        # the reference's own size and settings (x0 = 1, absolute tolerance), host arrays
        {"name": "pcg_32_host", "kind": "pcg", "problem": "poisson", "nx": 32, "ny": 32, "nz": 32,
         "fmt": "csr", "mixed": False, "host": True, "x0": "one"},
        # an odd box with variable coefficients in the reference's other block format
        {"name": "pcg_61x47x73_jad", "kind": "pcg", "problem": "diffusion", "nx": 61, "ny": 47,
         "nz": 73, "fmt": "jad", "mixed": False, "host": False, "x0": "one"},
        # variable coefficients in diagonal storage, an ordinary block
        {"name": "pcg_128_dia", "kind": "pcg", "problem": "diffusion", "nx": 128, "ny": 128,
         "nz": 128, "fmt": "dia", "mixed": False, "host": False, "x0": "zero"},
        # mixed precision on an unstructured mesh
        {"name": "pcg_mesh_600k_mixed", "kind": "pcg", "problem": "mesh", "n": 600011, "deg": 5,
         "fmt": "csr", "mixed": True, "host": False, "x0": "zero"},
        # the library's headline: mixed precision on the 256^3 Poisson block, CSR
        {"name": "pcg_256_mixed", "kind": "pcg", "problem": "poisson", "nx": 256, "ny": 256,
         "nz": 256, "fmt": "csr", "mixed": True, "host": False, "x0": "zero"},
        # plain FP64 on a large block with variable coefficients, CSR
        {"name": "pcg_200_fp64", "kind": "pcg", "problem": "diffusion", "nx": 200, "ny": 200,
         "nz": 200, "fmt": "csr", "mixed": False, "host": False, "x0": "zero"},
        # the backward pass: adjoint solve, dL/dA on the pattern, dL/dkappa
        {"name": "adjoint_128", "kind": "adjoint", "problem": "diffusion", "nx": 128, "ny": 128,
         "nz": 128, "fmt": "csr"},
        # the element solver's method and settings
        {"name": "gmres_48", "kind": "gmres", "problem": "poisson", "nx": 48, "ny": 48, "nz": 48,
         "fmt": "dia"},
        # 64 systems of uneven size and one block of 16 right-hand sides, together
        {"name": "batch_64_and_128x16", "kind": "batch", "systems": 64, "lo": 24, "hi": 96,
         "edge": 128, "rhs": 16},
        # a matrix from unordered entries: order, row offsets, build, diagonal form, product
        {"name": "assemble_128", "kind": "assemble", "problem": "diffusion", "nx": 128, "ny": 128,
         "nz": 128, "fmt": "dia"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    """A box of about e^3 cells, e log-uniform, edges uneven and often odd."""
    e = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return {"nx": max(4, int(e * rng.uniform(0.75, 1.33))), "ny": max(4, int(e * rng.uniform(0.75, 1.33))),
            "nz": max(4, int(e * rng.uniform(0.75, 1.33)))}


def _one(rng):
    kind = rng.choice(["spmv", "spmv", "pcg", "pcg", "pcg", "pcg", "adjoint", "gmres", "batch", "assemble"])
    if kind == "batch":
        lo = rng.randint(8, 40)
        return {"kind": kind, "systems": rng.randint(2, 64), "lo": lo, "hi": lo + rng.randint(4, 50),
                "edge": rng.choice([0, rng.randint(16, 100)]), "rhs": rng.choice([2, 3, 4, 8, 11, 16])}
    if kind in ("adjoint", "gmres"):
        c = {"kind": kind, "problem": "diffusion" if kind == "adjoint" else "poisson"}
        c.update(_box(rng, 12, 110 if kind == "adjoint" else 52))
        c["fmt"] = rng.choice(["csr", "dia"])
        return c
    c = {"kind": kind, "problem": rng.choice(["poisson", "diffusion", "mesh"])}
    if c["problem"] == "mesh":
        c.update(n=_log_int(rng, 3000, 2000000), deg=rng.randint(3, 8))
        c["fmt"] = rng.choice(["csr", "csr", "jad"])
    else:
        c.update(_box(rng, 14, 200 if kind != "assemble" else 128))
        c["fmt"] = rng.choice(["csr", "csr", "jad", "dia"])
    if kind == "spmv":
        c.update(f32=rng.random() < 0.4, accumulate=rng.random() < 0.3)
    elif kind == "pcg":
        c.update(mixed=rng.random() < 0.5, host=rng.random() < 0.2, x0=rng.choice(["zero", "one"]))
    return c


def draw(rng):
    most = max(max(w["bytes"], w["flops"] / 50) for w in map(work, listed()))
    while True:
        c = _one(rng)
        w = work(c)
        if max(w["bytes"], w["flops"] / 50) <= 0.9 * most:
            return c


# ---------------------------------------------------------------- what a pass cannot do without
def _size(case):
    if case["problem"] == "mesh":
        # every row keeps 0.85 deg edges on average, each stored twice, and its diagonal
        return case["n"], int(case["n"] * (1 + 1.7 * case["deg"]))
    x, y, z = case["nx"], case["ny"], case["nz"]
    return x * y * z, 7 * x * y * z - 2 * (x * y + y * z + x * z)


def _pcg_cost(n, nnz, iters, vb):
    """One PCG iteration reads the matrix once (values; a column index of 4 bytes
    each), reads and writes p, r and x and reads the Jacobi vector."""
    return iters * (nnz * (vb + 4.0) + 7.0 * vb * n), iters * (2.0 * nnz + 12.0 * n)


def _iters(case):
    """About the iterations to 1e-10 (measured: 3.2 per edge for a constant and 6 for
    a variable coefficient; a mesh of n rows has the width of a box of n cells)."""
    if case["problem"] == "mesh":
        return 1.5 * case["n"] ** (1.0 / 3.0)
    return (3.2 if case["problem"] == "poisson" else 6.0) * max(case["nx"], case["ny"], case["nz"])


def work(case):
    kind = case["kind"]
    if kind == "batch":
        mean = (case["lo"] + case["hi"]) / 2.0
        n, e = mean ** 3, float(case["edge"]) ** 3
        by, fl = _pcg_cost(n, 7 * n, 6.0 * mean, 8.0)
        by, fl = by * case["systems"], fl * case["systems"]
        it = 3.2 * case["edge"]
        return {"bytes": by + it * (84.0 * e + 56.0 * e * case["rhs"]),
                "flops": fl + it * 26.0 * e * case["rhs"]}
    n, nnz = _size(case)
    if kind == "spmv":
        vb = 4.0 if case["f32"] else 8.0
        return {"bytes": nnz * (vb + 4.0) + 4.0 * n + vb * n * (3 if case["accumulate"] else 2),
                "flops": 2.0 * nnz}
    if kind == "assemble":
        # entries in and out, the row offsets, the matrix once more for its product
        return {"bytes": 32.0 * nnz + 4.0 * n + 12.0 * nnz + 20.0 * n, "flops": 2.0 * nnz}
    if kind == "gmres":
        # outer iterations of the defective rotation grow with the square of the
        # edge (2474 at 128); four cycles each, of three products and a residual
        cycles = 4 * 0.15 * max(case["nx"], case["ny"], case["nz"]) ** 2
        return {"bytes": cycles * (4 * 12.0 * nnz + 40 * 8.0 * n), "flops": cycles * (8.0 * nnz + 60.0 * n)}
    by, fl = _pcg_cost(n, nnz, _iters(case), 4.0 if case.get("mixed") else 8.0)
    if kind == "adjoint":
        by, fl = by + 12.0 * nnz + 40.0 * n, fl + nnz + 40.0 * n
    return {"bytes": by, "flops": fl}


# ---------------------------------------------------------------- inputs
def _ok(rc):
    if rc not in (cel.OK, cel.NOT_CONVERGED):
        raise RuntimeError("%d: %s" % (rc, cel.lib().cel_gpu_last_error().decode()))


def _p(t):
    return C.c_void_p(t.data_ptr())


def _rand(gen, *shape):
    return torch.rand(*shape, generator=gen, dtype=torch.float64, device="cuda")


def _kappa(gen, n):
    """A lognormal coefficient field, log kappa ~ N(0, 1)."""
    return torch.exp(torch.randn(n, generator=gen, dtype=torch.float64, device="cuda"))


def _mesh(case, gen):
    """Symmetric positive definite matrix of an unstructured mesh in a banded numbering:
    a graph Laplacian with a small shift; edge weights are multiples of 1/1024, so
    the diagonal is exact.  Returns 0-based row-sorted (rows, cols, vals)."""
    n, deg = case["n"], case["deg"]
    band = max(8, int(n ** (2.0 / 3.0)))
    i = torch.arange(n, device="cuda").repeat_interleave(deg)
    j = i + 1 + (_rand(gen, n * deg) * band).long()
    keep = (j < n) & (_rand(gen, n * deg) < 0.85)
    key = torch.unique(i[keep] * n + j[keep])
    i, j = key // n, key % n
    w = torch.randint(512, 1537, (key.numel(),), generator=gen, device="cuda").double() / 1024.0
    d = torch.full((n,), 1.0 / 256.0, dtype=torch.float64, device="cuda")
    d.index_add_(0, i, w)
    d.index_add_(0, j, w)
    a = torch.arange(n, device="cuda")
    rows, cols, vals = torch.cat([i, j, a]), torch.cat([j, i, a]), torch.cat([-w, -w, d])
    order = torch.argsort(rows * n + cols)
    return rows[order], cols[order], vals[order]


def _grid(case, kappa):
    """0-based row-sorted entries of the 7-point matrix in float64: harmonic-mean face
    coefficients of kappa with kappa itself on boundary faces; kappa None: 6 and -1."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    idx = torch.arange(n, device="cuda").view(nz, ny, nx)
    k = None if kappa is None else kappa.view(nz, ny, nx)
    d = torch.zeros(nz, ny, nx, dtype=torch.float64, device="cuda")
    rows, cols, vals = [], [], []
    for axis, m in ((0, nz), (1, ny), (2, nx)):
        lo, hi = idx.narrow(axis, 0, m - 1), idx.narrow(axis, 1, m - 1)
        if k is None:
            f = torch.ones(lo.shape, dtype=torch.float64, device="cuda")
            edge = torch.ones_like(d.narrow(axis, 0, 1))
            first = last = edge
        else:
            a, b = k.narrow(axis, 0, m - 1), k.narrow(axis, 1, m - 1)
            f = 2.0 * a * b / (a + b)
            first, last = k.narrow(axis, 0, 1), k.narrow(axis, m - 1, 1)
        d.narrow(axis, 0, m - 1).add_(f)
        d.narrow(axis, 1, m - 1).add_(f)
        d.narrow(axis, 0, 1).add_(first)
        d.narrow(axis, m - 1, 1).add_(last)
        rows += [lo.reshape(-1), hi.reshape(-1)]
        cols += [hi.reshape(-1), lo.reshape(-1)]
        vals += [-f.reshape(-1), -f.reshape(-1)]
    a = idx.reshape(-1)
    rows, cols = torch.cat(rows + [a]), torch.cat(cols + [a])
    vals = torch.cat(vals + [d.reshape(-1)])
    order = torch.argsort(rows * n + cols)
    return rows[order], cols[order], vals[order]


def _matrix(case, gen):
    """The matrix handle (and kappa, where there is one), with its Jacobi vector and
    the storage form the program solves in."""
    h, kappa = C.c_void_p(), None
    if case["problem"] == "mesh":
        rows, cols, vals = _mesh(case, gen)
        n = case["n"]
        xadj = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
        xadj[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0).int()
        cols = cols.int()
        torch.cuda.synchronize()
        _ok(cel.lib().cel_gpu_mat_create_csr(C.byref(h), n, n, cols.numel(), _p(xadj), _p(cols), _p(vals),
                                             0, 0, 0, cel.MEM_DEVICE))
        _ok(cel.lib().cel_gpu_synchronize())
    elif case["problem"] == "diffusion":
        kappa = _kappa(gen, case["nx"] * case["ny"] * case["nz"])
        torch.cuda.synchronize()
        _ok(cel.lib().cel_gpu_mat_gen_diffusion7(C.byref(h), case["nx"], case["ny"], case["nz"], _p(kappa),
                                                 cel.MEM_DEVICE))
    else:
        _ok(cel.lib().cel_gpu_mat_gen_poisson7(C.byref(h), case["nx"], case["ny"], case["nz"]))
    m = cel.Matrix(h)
    m.set_jacobi()
    if case["fmt"] == "jad":
        m.to_jad()
    elif case["fmt"] == "dia":
        m.to_dia()
    return m, kappa


def _gen(seed):
    cel.init()
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _product(m, x):
    y = torch.zeros(m.n, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    _ok(cel.lib().cel_gpu_spmv(m.h, cel.FMT_CSR, _p(x), _p(y), 0, cel.MEM_DEVICE))
    return y


def _batch_boxes(case):
    """Edges spread evenly over [lo, hi], the three edges of a box unequal."""
    s, lo, hi = case["systems"], case["lo"], case["hi"]
    at = lambda k: lo + (hi - lo) * (k % s) // max(1, s - 1)  # noqa: E731
    return [{"problem": "diffusion", "fmt": "csr", "nx": at(k), "ny": at(k), "nz": at(k + s // 3)} for k in range(s)]


def prepare(case, seed):
    gen, kind = _gen(seed), case["kind"]
    if kind == "batch":
        st = {"kind": kind, "mats": [], "nrhs": []}
        xs, bs = [], []
        for box in _batch_boxes(case):
            m, _ = _matrix(box, gen)
            x = _rand(gen, m.n)
            st["mats"].append(m)
            st["nrhs"].append(1)
            bs.append(_product(m, x))
        if case["edge"]:
            e = case["edge"]
            m, _ = _matrix({"problem": "poisson", "fmt": "csr", "nx": e, "ny": e, "nz": e}, gen)
            st["mats"].append(m)
            st["nrhs"].append(case["rhs"])
            bs += [_product(m, _rand(gen, m.n)) for _ in range(case["rhs"])]
        st["b"] = torch.cat(bs)
        st["x"] = torch.zeros_like(st["b"])
        st["batch"] = cel.Batch(st["mats"], st["nrhs"])
        at, k = 0, len(st["mats"])
        st["bp"], st["xp"] = (C.c_void_p * k)(), (C.c_void_p * k)()
        for s, (m, r) in enumerate(zip(st["mats"], st["nrhs"])):
            st["bp"][s], st["xp"][s] = st["b"].data_ptr() + 8 * at, st["x"].data_ptr() + 8 * at
            at += m.n * r
        st["params"] = cel.params(tol=1e-9, tol_mode=cel.TOL_REL_B, iter_max=20000, x0_mode=cel.X0_ZERO,
                                  alpha_stop=0, memspace=cel.MEM_DEVICE)
        st["lane_stats"] = (cel.PcgStats * sum(st["nrhs"]))()
        return st
    if kind == "assemble":
        rows, cols, vals = _mesh(case, gen) if case["problem"] == "mesh" else _grid(
            case, None if case["problem"] == "poisson" else _kappa(gen, case["nx"] * case["ny"] * case["nz"]))
        n = _size(case)[0]
        order = torch.argsort(_rand(gen, rows.numel()))
        st = {"kind": kind, "n": n, "nnz": rows.numel(), "fmt": case["fmt"],
              "coo": (rows[order].int(), cols[order].int(), vals[order].contiguous()), "x": _rand(gen, n)}
        st["work"] = tuple(torch.empty_like(t) for t in st["coo"])
        st["xadj"] = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
        st["y"] = torch.zeros(n, dtype=torch.float64, device="cuda")
        return st
    m, kappa = _matrix(case, gen)
    st = {"kind": kind, "m": m, "fmt": FORMATS[case["fmt"]]}
    x = _rand(gen, m.n)
    if kind == "spmv":
        st["f32"], st["accumulate"] = case["f32"], int(case["accumulate"])
        st["x"] = x.float() if case["f32"] else x
        st["y0"] = _rand(gen, m.n).to(st["x"].dtype)
        st["y"] = torch.zeros_like(st["x"])
        return st
    st["b"] = _product(m, x)
    st["x"] = torch.zeros_like(st["b"])
    if kind == "gmres":
        p = cel.GmresParams()
        cel.lib().cel_gpu_gmres_params_default(C.byref(p))
        p.memspace, p.format = cel.MEM_DEVICE, st["fmt"]
    elif kind == "adjoint":
        # x: the forward solution, b: dL/dx
        st.update(kappa=kappa, fwd=_rand(gen, m.n), box=(case["nx"], case["ny"], case["nz"]),
                  dLda=torch.zeros(m.nnz, dtype=torch.float64, device="cuda"), grad=torch.zeros_like(x))
        p = cel.params(tol=1e-12, tol_mode=cel.TOL_REL_B, iter_max=20000, x0_mode=cel.X0_ZERO, alpha_stop=0,
                       format=st["fmt"], memspace=cel.MEM_DEVICE)
    else:
        ref = case["host"] and case["x0"] == "one"  # the reference's absolute test
        p = cel.params(tol=1e-8 if ref else 1e-10, tol_mode=cel.TOL_ABS if ref else cel.TOL_REL_B, iter_max=20000,
                       x0_mode=cel.X0_ONE if case["x0"] == "one" else cel.X0_ZERO, alpha_stop=1 if ref else 0,
                       precision=cel.PREC_MIXED if case["mixed"] else cel.PREC_FP64, format=st["fmt"],
                       memspace=cel.MEM_HOST if case["host"] else cel.MEM_DEVICE)
        if case["host"]:
            st["b"], st["x"] = st["b"].cpu().numpy(), np.zeros(m.n)
    st["params"], st["stats"] = p, cel.PcgStats()
    return st


# ---------------------------------------------------------------- one pass
def run(st):
    L, kind = cel.lib(), st["kind"]
    if kind == "spmv":
        if st["accumulate"]:  # y starts from the caller's values each time
            _ok(L.cel_gpu_memcpy_d2d(_p(st["y"]), _p(st["y0"]),
                                     C.c_size_t(st["y"].numel() * st["y"].element_size())))
        f = L.cel_gpu_spmv_f32 if st["f32"] else L.cel_gpu_spmv
        _ok(f(st["m"].h, st["fmt"], _p(st["x"]), _p(st["y"]), st["accumulate"], cel.MEM_DEVICE))
        return st["y"]
    if kind == "pcg":
        if isinstance(st["b"], np.ndarray):
            _ok(L.cel_gpu_pcg_solve(st["m"].h, st["b"].ctypes.data_as(C.c_void_p), st["x"].ctypes.data_as(C.c_void_p),
                                    C.byref(st["params"]), C.byref(st["stats"]), None))
        else:
            _ok(L.cel_gpu_pcg_solve(st["m"].h, _p(st["b"]), _p(st["x"]), C.byref(st["params"]),
                                    C.byref(st["stats"]), None))
        return st["x"]
    if kind == "adjoint":
        _ok(L.cel_gpu_cg_adjoint(st["m"].h, _p(st["fwd"]), _p(st["b"]), _p(st["x"]), _p(st["dLda"]),
                                 C.byref(st["params"]), C.byref(st["stats"])))
        _ok(L.cel_gpu_diffusion7_kappa_grad(*st["box"], _p(st["kappa"]), _p(st["fwd"]), _p(st["x"]),
                                            _p(st["grad"]), cel.MEM_DEVICE))
        return {"dLdb": st["x"], "dLda": st["dLda"], "dLdkappa": st["grad"]}
    if kind == "gmres":
        _ok(L.cel_gpu_gmres_solve(st["m"].h, _p(st["b"]), _p(st["x"]), C.byref(st["params"]), C.byref(st["stats"])))
        return st["x"]
    if kind == "batch":
        total = cel.PcgStats()
        _ok(L.cel_gpu_batch_solve(st["batch"].h, st["bp"], st["xp"], C.byref(st["params"]), st["lane_stats"],
                                  C.byref(total)))
        return st["x"]
    # assemble: the entries are ordered in place, so they are copied first
    n, nnz = st["n"], st["nnz"]
    for dst, src in zip(st["work"], st["coo"]):
        _ok(L.cel_gpu_memcpy_d2d(_p(dst), _p(src), C.c_size_t(src.numel() * src.element_size())))
    rows, cols, vals = st["work"]
    _ok(L.cel_gpu_coo_sort(n, n, nnz, _p(rows), _p(cols), _p(vals), 0, 0, 0, cel.SORT_ROW_COL, cel.MEM_DEVICE))
    _ok(L.cel_gpu_coo_row_offsets(n, nnz, _p(rows), 0, 0, _p(st["xadj"]), cel.MEM_DEVICE))
    h = C.c_void_p()
    _ok(L.cel_gpu_mat_create_csr(C.byref(h), n, n, nnz, _p(st["xadj"]), _p(cols), _p(vals), 0, 0, 0, cel.MEM_DEVICE))
    _ok(L.cel_gpu_mat_set_jacobi(h, 0))
    if st["fmt"] == "dia":
        _ok(L.cel_gpu_mat_to_dia(h))
    elif st["fmt"] == "jad":
        _ok(L.cel_gpu_mat_to_jad(h, cel.JAD_SPARSKIT))
    _ok(L.cel_gpu_spmv(h, FORMATS[st["fmt"]], _p(st["x"]), _p(st["y"]), 0, cel.MEM_DEVICE))
    _ok(L.cel_gpu_mat_destroy(h))
    return {"rows": rows, "cols": cols, "vals": vals, "xadj": st["xadj"], "y": st["y"]}


# ---------------------------------------------------------------- in 64 bits, without the library
def exact(case, seed):
    gen, kind = _gen(seed), case["kind"]
    if kind == "batch":
        xs = []
        for box in _batch_boxes(case):
            n = box["nx"] * box["ny"] * box["nz"]
            _kappa(gen, n)
            xs.append(_rand(gen, n))
        xs += [_rand(gen, case["edge"] ** 3) for _ in range(case["rhs"] if case["edge"] else 0)]
        return torch.cat(xs)
    n = _size(case)[0]
    # the generator is read in prepare's order: the matrix, then the vectors
    mesh = _mesh(case, gen) if case["problem"] == "mesh" else None
    kappa = _kappa(gen, n) if case["problem"] == "diffusion" else None
    if kind in ("pcg", "gmres"):
        return _rand(gen, n)  # b = A x
    rows, cols, vals = mesh if mesh is not None else _grid(case, kappa)
    if kind == "assemble":
        _rand(gen, rows.numel())
        x = _rand(gen, n)
        xadj = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
        xadj[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0).int()
        y = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, rows, vals * x[cols])
        return {"rows": rows.int(), "cols": cols.int(), "vals": vals, "xadj": xadj, "y": y}
    x = _rand(gen, n)
    if kind == "spmv":
        dt = torch.float32 if case["f32"] else torch.float64
        x, y = x.to(dt).double(), _rand(gen, n).to(dt).double()
        if not case["accumulate"]:
            y = torch.zeros_like(y)
        return y.index_add_(0, rows, vals * x[cols])
    # adjoint: lambda = x; dL/da_ij = -lambda_i x_j; dL/dkappa through the face coefficients
    lam, fwd = x, _rand(gen, n)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    k, u, v = (t.view(nz, ny, nx) for t in (kappa, fwd, lam))
    g = torch.zeros_like(k)
    for axis, m in ((0, nz), (1, ny), (2, nx)):
        lo = lambda t: t.narrow(axis, 0, m - 1)  # noqa: E731
        hi = lambda t: t.narrow(axis, 1, m - 1)  # noqa: E731
        df = -(lo(v) - hi(v)) * (lo(u) - hi(u))
        s = (lo(k) + hi(k)) ** 2
        lo(g).add_(df * 2.0 * hi(k) ** 2 / s)
        hi(g).add_(df * 2.0 * lo(k) ** 2 / s)
        for at in (0, m - 1):
            g.narrow(axis, at, 1).sub_(v.narrow(axis, at, 1) * u.narrow(axis, at, 1))
    return {"dLdb": lam, "dLda": -lam[rows] * fwd[cols], "dLdkappa": g.reshape(-1)}
