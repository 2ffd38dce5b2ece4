"""Which path a solve takes: the tests of the paths that sizes, bands, forms and
values choose compare bits between them, and would pass as well if a path were
never taken.  Here the library says which kernels the last solve of a handle
ran on."""
import ctypes as C

import numpy as np
import pytest

from helpers import stencil27
from test_gpu_derived import kappa_of
from test_gpu_gmres_window import banded as gmres_banded
from test_gpu_wide import BASE, banded
from test_gpu_window import mesh

pytestmark = pytest.mark.gpu

BOX = (97, 93, 91)  # 820,911 rows


def path(gpu, M):
    s = C.create_string_buffer(96)
    assert gpu.lib().cel_gpu_internal_path(M.h, s, 96) == 0
    return s.value.decode()


def solve(gpu, M, fmt="CSR", prec="FP64", iter_max=40, **kw):
    M.pcg(np.ones(M.n), fmt=getattr(gpu, "FMT_" + fmt), precision=getattr(gpu, "PREC_" + prec), tol=1e-300,
          tol_mode=gpu.TOL_REL_B, alpha_stop=0, x0_mode=gpu.X0_ZERO, iter_max=iter_max, **kw)
    return path(gpu, M)


def box(gpu, shape, kind="random"):
    rng = np.random.default_rng(31)
    if kind == "poisson":
        M = gpu.Matrix.poisson7(*shape)
    elif kind == "random":
        M = gpu.Matrix.diffusion7(*shape, np.exp(rng.normal(0.0, 0.5, int(np.prod(shape)))))
    else:
        M = gpu.Matrix.diffusion7(*shape, kappa_of(kind, rng))
    M.set_jacobi()
    return M


@pytest.mark.parametrize("kind", ["poisson", "two_materials", "layers", "random"])
def test_derived_forms(gpu, kind):
    M = box(gpu, BOX, kind)
    classes = kind in ("poisson", "two_materials")
    form = "classes wide" if classes else "dia wide keep"
    assert solve(gpu, M, iter_max=8) == "csr keep"
    assert solve(gpu, M, prec="MIXED", iter_max=8) == "csr step keep"
    assert solve(gpu, M, "COO") == "csr keep"
    assert solve(gpu, M) == solve(gpu, M, prec="MIXED") == form
    assert solve(gpu, M, iter_max=8) == form  # the form that is there
    M.to_dia()
    assert solve(gpu, M, "DIA") == form
    assert solve(gpu, M, "DIA", "MIXED") == (form if classes else "dia step keep")  # line at 850,000 rows
    M.scale_diagonal()
    M.set_jacobi(row_scaled=True)
    # scaled rows: a few more forms, or diagonals that are not symmetric
    scaled = {"poisson": "classes wide", "layers": "dia keep", "random": "dia keep"}
    if kind in scaled:
        assert solve(gpu, M) == solve(gpu, M, prec="MIXED") == scaled[kind]
    M.set_jacobi()
    assert solve(gpu, M, iter_max=8) in ("csr keep",)  # dropped with the Jacobi vector


def test_blocks_without_a_derived_form(gpu):
    A = stencil27(94, 93, 92)
    M = gpu.Matrix.from_csr(A.indptr, A.indices, A.data, index_base=0)
    M.set_jacobi()
    assert solve(gpu, M).split()[0] == "csr-long" and "window" not in path(gpu, M)
    assert solve(gpu, box(gpu, (92, 93, 93), "poisson")) == "csr keep"  # 795,708 rows


@pytest.mark.parametrize("values", ["constant", "symmetric", "general"])
@pytest.mark.parametrize("n,offsets", [(BASE - 1, (-8101, -89, -1, 0, 1, 89, 8101)),
                                       (BASE + 255, (-8100, -90, -1, 0, 1, 2, 90, 8100)),
                                       (BASE + 129, (-500000, -1, 0, 1, 500000))])
def test_wide_walks(gpu, n, offsets, values):
    M = gpu.Matrix.from_csr(*banded(n, offsets, values, np.random.default_rng(1)), index_base=0)
    M.set_jacobi()
    form = {"constant": "classes wide", "symmetric": "dia wide keep", "general": "dia keep"}[values]
    assert solve(gpu, M) == solve(gpu, M, prec="MIXED") == form
    M.to_dia()
    assert solve(gpu, M, "DIA") == form
    # below 850,000 rows mixed solves iterate with two kernels instead, but for
    # rows that average more than 7.5 entries
    two_kernels = values != "constant" and len(offsets) < 8
    assert solve(gpu, M, "DIA", "MIXED") == ("dia step keep" if two_kernels else form)


@pytest.mark.parametrize("n,band,window", [(119999, 900, False), (120000, 900, True), (120001, 3582, True),
                                           (130817, 3583, False)])
def test_windows(gpu, n, band, window):
    for far in (False, True):
        M = gpu.Matrix.from_csr(*mesh(n, band, far, np.random.default_rng(7)), index_base=0)
        M.set_jacobi()
        for fmt in ("CSR", "COO"):
            assert solve(gpu, M, fmt, iter_max=33) == "csr-long window keep" if window and not far else "csr-long keep"
        assert solve(gpu, M, prec="MIXED", iter_max=33) == "csr-long keep"


@pytest.mark.parametrize("edge,fp64,mixed", [
    (32, "step direct", "step direct"), (41, "step direct", "step direct"), (42, "step", "step direct"),
    (49, "step", "step direct"), (50, "step", "step"), (66, "step", "step"), (67, "", "step"),
    (106, "", "step"), (107, "", ""),
])
def test_steps(gpu, edge, fp64, mixed):
    M = box(gpu, (edge, edge, edge))
    for prec, form in (("FP64", fp64), ("MIXED", mixed)):
        words = ["csr"] + form.split() + ["keep"]
        assert solve(gpu, M, prec=prec, iter_max=6) == " ".join(words)
        assert solve(gpu, M, prec=prec, iter_max=6, profile=1) == "csr keep"
    if edge in (32, 66):
        M.to_dia()
        M.to_jad()
        for fmt in ("DIA", "JAD"):
            for prec in ("FP64", "MIXED"):
                assert solve(gpu, M, fmt, prec, iter_max=6) == fmt.lower() + " step keep"


@pytest.mark.parametrize("shape,csr,dia,jad", [((71, 67, 69), 1, 1, 1), ((136, 135, 137), 0, 1, 0),
                                               ((144, 143, 145), 0, 0, 0)])
def test_matrices_kept_in_the_cache(gpu, shape, csr, dia, jad):
    M = box(gpu, shape)
    M.to_dia()
    M.to_jad()
    for fmt, keep in (("CSR", csr), ("DIA", dia), ("JAD", jad)):
        assert solve(gpu, M, fmt, iter_max=6) == fmt.lower() + " keep" * keep


@pytest.mark.parametrize("shape,prec,walk,classes", [((187, 186, 188), "FP64", 1, 0), ((219, 218, 220), "FP64", 2, 1),
                                                     ((237, 236, 238), "MIXED", 1, 0)])
def test_vectors_read_once(gpu, shape, prec, walk, classes):
    M = box(gpu, shape, "poisson")
    assert solve(gpu, M, "COO", prec, iter_max=33) == "csr" + (f" stream{walk}" if walk else "")
    assert solve(gpu, M, "CSR", prec, iter_max=33) == "classes wide" + (f" stream{classes}" if classes else "")


@pytest.mark.parametrize("scaled", [False, True])
def test_batch_forms(gpu, scaled):
    rng = np.random.default_rng(43)
    shapes = ((9, 8, 7), (31, 29, 33), (28, 27, 27), (400, 50, 1), (1, 1, 20001), (27, 27, 27), (47, 47, 47))
    mats = [gpu.Matrix.diffusion7(*s, np.exp(rng.normal(0.0, 0.3, int(np.prod(s))))) for s in shapes]
    mats.append(gpu.Matrix.poisson7(*BOX))
    for m in mats:
        m.set_jacobi()
        if scaled:
            m.scale_diagonal()
            m.set_jacobi(row_scaled=True)
    bs = [rng.normal(size=m.n) for m in mats]
    batch = gpu.Batch(mats)

    def forms(**kw):
        batch.solve(bs, tol_mode=gpu.TOL_REL_B, x0_mode=gpu.X0_ZERO, alpha_stop=0, **kw)
        kind, arrays = ((C.c_int * len(mats))() for _ in range(2))
        assert gpu.lib().cel_gpu_internal_batch_forms(batch.h, kind, arrays) == 0
        return list(kind), [a for k, a in zip(kind, arrays) if k == 2]

    # few iterations, or a solve that stops after a few: none
    assert forms(tol=1e-300, iter_max=31) == ([0] * 8, [])
    assert forms(tol=0.9, iter_max=1000) == ([0] * 8, [])
    full = ([0, 2, 2, 2, 2, 0, 2, 1], [7, 7, 5, 3, 7] if scaled else [4, 4, 3, 2, 4])
    assert forms(tol=1e-300, iter_max=40) == full
    assert forms(tol=0.9, iter_max=8) == full  # those that are there


def test_gmres_columns(gpu):
    M = box(gpu, (48, 48, 48))
    M.to_dia()
    M.to_jad()
    W = gpu.Matrix.from_csr(*gmres_banded(6143, (-2050, -1025, -1, 0, 1, 1025, 2050), np.random.default_rng(2)),
                            index_base=0)
    W.set_jacobi()
    W.to_dia()
    L = box(gpu, (85, 85, 85), "poisson")
    L.to_dia()
    for m, fmt, form in ((M, "CSR", "gmres step"), (M, "DIA", "gmres step window"), (M, "JAD", "gmres"),
                         (W, "DIA", "gmres step"), (L, "DIA", "gmres")):
        m.gmres(np.ones(m.n), fmt=getattr(gpu, "FMT_" + fmt), iter_max=0)
        assert path(gpu, m) == form
