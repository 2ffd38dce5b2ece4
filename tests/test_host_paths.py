"""Decisions of the library's host code, without a GPU: the library runs in a
child process over a stand-in for the HIP runtime (hoststub/hip_stub.cpp),
where device memory has a budget and a kernel launch is a line of a log.
No result is computed here; what is looked at is which calls succeed, which
kernels they launch, and on how many blocks."""
import json
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
STUB = os.path.join(HERE, "hoststub", "hip_stub.cpp")

PRELUDE = """
import ctypes as C, json, sys
import numpy as np
sys.path.insert(0, %r)
import cel_v3_amd as cel
S = C.CDLL(None)
S.stub_log.restype = C.c_char_p
S.stub_budget.argtypes = [C.c_size_t]
S.stub_used.restype = S.stub_peak.restype = C.c_size_t
cel.init(0)

def box(nx, ny, nz):
    '''7-point block, 0-based CSR arrays'''
    n = nx * ny * nz
    i = np.arange(n)
    x, y, z = i %% nx, i // nx %% ny, i // (nx * ny)
    cols = np.stack([i - nx * ny, i - nx, i - 1, i, i + 1, i + nx, i + nx * ny], 1)
    on = np.stack([z > 0, y > 0, x > 0, i >= 0, x < nx - 1, y < ny - 1, z < nz - 1], 1)
    xadj = np.concatenate([[0], np.cumsum(on.sum(1))])
    vals = np.where(np.arange(7) == 3, 6.0, -1.0) * np.ones((n, 1))
    return xadj, cols[on], vals[on]

def matrix(*shape):
    M = cel.Matrix.from_csr(*box(*shape), index_base=0)
    M.set_jacobi()
    return M

def launches(name=None):
    '''(kernel, blocks) since the log was cleared'''
    out = [tuple(l.rsplit(" ", 1)) for l in S.stub_log().decode().splitlines() if " " in l]
    return [(k, int(g)) for k, g in out if name is None or k.split("<")[0] == name]
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    import cel_v3_amd as cel

    if not os.path.exists(cel.LIB_PATH) or shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include/hip"):
        pytest.skip("needs libcel_gpu.so, g++ and the HIP headers")
    so = tmp_path_factory.mktemp("hoststub") / "libamdhip64.so.7"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-Wl,-soname,libamdhip64.so.7", STUB, "-o", str(so)], check=True)

    def run(body):
        """The JSON value that `body` assigns to `out`."""
        code = PRELUDE % ROOT + body + "\nprint('OUT' + json.dumps(out))\n"
        env = dict(os.environ, LD_PRELOAD=str(so))
        r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-2000:]
        return json.loads(r.stdout.split("OUT", 1)[1])

    return run


def test_kept_blocks_go_back_when_a_callers_allocation_fails(stub):
    out = stub("""
M = matrix(64, 64, 64)
held = S.stub_used()
del M
kept = S.stub_used()
S.stub_budget(kept + 1000)
a = cel.DeviceArray(kept // 16)       # half of what is kept
out = {"held": held, "kept": kept, "used": S.stub_used(), "got": kept // 16 * 8}
""")
    assert out["kept"] > 0.9 * out["held"]  # destroyed, and not with the driver
    assert out["used"] == out["got"]


@pytest.mark.parametrize("more", [0, 1])
def test_an_allocation_that_cannot_be_had_is_still_refused(stub, more):
    out = stub(f"""
S.stub_budget(1 << 20)
p = C.c_void_p(1)
out = [cel.lib().cel_gpu_malloc(C.byref(p), C.c_size_t((1 << 20) + {more})), p.value]
""")
    assert (out[0] == 0 and out[1]) if not more else out == [-8, None]


# A block of 820,911 rows: its derived diagonal storage takes 47 MB in FP64, 24 MB
# in FP32; a solve on the CSR arrays needs 42 MB in FP64 (r, p, v, b, x in
# pieces of 2 MB), 57 MB mixed (r, p, v, e, b, x and the FP32 values).
@pytest.mark.parametrize("prec,spare", [("FP64", 44), ("FP64", 60), ("MIXED", 57)])
def test_a_solve_has_its_memory_before_a_derived_form_has(stub, prec, spare):
    out = stub(f"""
S.stub_classes_fit(0)
M = matrix(97, 93, 91)
S.stub_budget(S.stub_used() + {spare} * 1000000)
S.stub_log_clear()
r = M.pcg(np.ones(M.n), precision=cel.PREC_{prec}, iter_max=40)
out = [k for k, _ in launches("k_pcg_spmv")]
S.stub_budget(1 << 34)
S.stub_log_clear()
N = matrix(97, 93, 91)
N.pcg(np.ones(N.n), precision=cel.PREC_{prec}, iter_max=40)
out = [out, [k for k, _ in launches("k_pcg_spmv")]]
""")
    vt = "double" if prec == "FP64" else "float"
    assert len(out[0]) >= 40 and {k.split(",")[0] + k.split(",")[1] for k in out[0]} == {f"k_pcg_spmv<{vt} 1"}  # CSR
    assert {k.split(",")[0] + k.split(",")[1] for k in out[1]} == {f"k_pcg_spmv<{vt} 4"}  # diagonals, with memory


def test_derived_forms_go_back_when_memory_is_short(stub):
    out = stub("""
S.stub_classes_fit(0)
M = matrix(97, 93, 91)
kw = dict(iter_max=40)
M.pcg(np.ones(M.n), fmt=cel.FMT_COO, **kw)
plain = S.stub_used()                      # matrix and workspace
M.pcg(np.ones(M.n), **kw)
form = S.stub_used() - plain
S.stub_budget(S.stub_used() + 1000000)
a = cel.DeviceArray(5000000)               # 40 MB, which only the form can give
short = S.stub_used()
S.stub_log_clear()
M.pcg(np.ones(M.n), **kw)                  # on the CSR arrays
csr = sorted({k for k, _ in launches("k_pcg_spmv")})
a.free()
S.stub_budget(1 << 34)
B = cel.Batch([M, matrix(31, 30, 29)])     # a batch's forms likewise
B.solve([np.ones(m.n) for m in B.mats], iter_max=40)
S.stub_budget(S.stub_used())
p = C.c_void_p()
rc = cel.lib().cel_gpu_malloc(C.byref(p), C.c_size_t(3000000))
out = {"form": form, "short": short - plain - 40000000, "csr": csr, "rc": rc}
""")
    assert out["form"] > 45e6
    assert out["short"] <= 2e6
    assert len(out["csr"]) == 1 and out["csr"][0].startswith("k_pcg_spmv<double, 1")
    assert out["rc"] == 0


def test_solve_grids_do_not_depend_on_occupancy(stub):
    out = stub("""
M = matrix(80, 80, 80)
M.to_dia()
out = []
for per_cu in (8, 5, 1):
    S.stub_occupancy(per_cu)
    S.stub_log_clear()
    for prec in (cel.PREC_FP64, cel.PREC_MIXED):
        for fmt in (cel.FMT_CSR, cel.FMT_COO, cel.FMT_DIA):
            M.pcg(np.ones(M.n), fmt=fmt, precision=prec, iter_max=3)
    out.append([l for l in launches() if l[0].startswith(("k_residual", "k_pcg"))])
""")
    assert out[0] == out[1] == out[2]
    # the residual: 6 blocks per CU; 2,000 tiles of 256 rows
    assert {g for k, g in out[0] if k.startswith("k_residual<")} == {1536}


def test_one_wait_serves_all_kept_blocks(stub):
    out = stub("""
M = matrix(4, 5, 6)
x = np.ones(M.n)
out = []
for _ in range(3):                      # two device buffers a call, kept from the one before
    before = S.stub_waits()
    M.spmv(x)
    out.append(S.stub_waits() - before)
""")
    # the end of the call, and one before the first kept block is used again
    assert out == [1, 2, 2]


@pytest.mark.parametrize("longest,deep", [(8, False), (24, False), (25, True), (3000, True)])
def test_matrices_with_a_few_long_rows(stub, longest, deep):
    out = stub(f"""
n = 30011
count = np.full(n, 5)
count[n // 2] = {longest}
cols = np.concatenate([np.sort((i + np.arange(c) - c // 2) % n) for i, c in enumerate(count)])
xadj = np.concatenate([[0], np.cumsum(count)])
M = cel.Matrix.from_csr(xadj, cols, np.ones(cols.size), index_base=0)
M.set_jacobi()
out = []
for prec in (cel.PREC_FP64, cel.PREC_MIXED):
    S.stub_log_clear()
    M.pcg(np.ones(n), precision=prec, iter_max=3)
    out.append(sorted({{k for k, _ in launches() if k.startswith(("k_pcg_spmv", "k_pcg_step"))}}))
""")
    for vt, got in zip(("double", "float"), out):
        assert got == [f"k_pcg_spmv<{vt}, 1, false, false, true, 8>" if deep else f"k_pcg_step<{vt}, 1, true>"]


def test_a_block_without_row_classes_is_not_scanned_whole(stub):
    out = stub("""
out = []
for fit in (0, 1):
    S.stub_classes_fit(fit)
    M = matrix(97, 93, 91)
    S.stub_log_clear()
    M.pcg(np.ones(M.n), iter_max=40)
    out.append([g for _, g in launches("k_class_scan")])
""")
    assert out[0] == [5]          # 1,025 rows, spread over the block
    assert out[1] == [5, 3207]    # then all 820,911


def test_a_batch_that_stops_early_builds_no_forms(stub):
    out = stub("""
B = cel.Batch([matrix(30, 31, 32), matrix(45, 46, 47), matrix(97, 93, 91)])
S.stub_log_clear()
B.solve([np.ones(m.n) for m in B.mats], iter_max=1000)   # (every lane is found stopped at the first look)
out = [k for k, _ in launches() if "scan" in k or "fill<" in k]
""")
    assert out == []


@pytest.mark.parametrize("prec", ["FP64", "MIXED"])
@pytest.mark.parametrize("every", [1, 3, 4, 16, 17])
def test_graph_solves_replay_a_graph(stub, every, prec):
    out = stub(f"""
M = matrix(12, 13, 14)
S.stub_log_clear()
M.pcg(np.ones(M.n), iter_max=99, use_graph=1, check_every={every}, precision=cel.PREC_{prec})
log = S.stub_log().decode().splitlines()
at = log.index("capture")
end = log.index("graph")
out = [sum("k_pcg_step" in l for l in log[at:end]), log.count("graph"),
       sum("k_pcg_step" in l for l in log[:at] + log[end:])]
""")
    steps = every if every % 2 == 0 else 2 * every   # an even chunk of the two-kernel form
    slots = 100 * (3 if prec == "MIXED" else 1)
    assert out == [steps, slots // steps, slots % steps]


@pytest.mark.parametrize("shape,symmetric", [((94, 93, 92), False), ((97, 96, 95), True), ((106, 105, 106), True)])
def test_mixed_solves_in_the_callers_diagonal_storage(stub, shape, symmetric):
    out = stub(f"""
M = matrix(*{shape})
M.to_dia()
S.stub_classes_fit(0)
S.stub_log_clear()
r = M.pcg(np.ones(M.n), fmt=cel.FMT_DIA, precision=cel.PREC_MIXED, iter_max=40)
ks = {{k.split("<")[0] for k, _ in launches()}}
out = ["k_dia_symmetric" in ks, "k_pcg_step" in ks, "k_pcg_spmv" in ks, r["spmv_bytes"] / M.n]
""")
    # checked, two kernels, the wide walk, bytes a row (4 of 7 arrays, or all and the product's own)
    assert out[:3] == [symmetric, not symmetric, symmetric]
    assert out[3] == 25.0 if symmetric else out[3] >= 37.0
