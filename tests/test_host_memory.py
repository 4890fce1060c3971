"""Device memory of the library's host code, without a GPU: libminife_hip.so on a
stand-in HIP runtime (hip_stub.cpp) whose kernels do nothing.  Each case runs in a
process of its own, so that no other test sees the stand-in."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = r"""
import ctypes, os, sys, threading, time
import numpy as np
os.environ["MINIFE_SYSTEM_HIP_RUNTIME"] = "1"
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_used.restype = ctypes.c_size_t
for f in ("mallocs", "frees", "hazards", "foreign_waits", "capture_breaks"):
    getattr(stub, "stub_" + f).restype = ctypes.c_long
stub.stub_capacity.argtypes = [ctypes.c_size_t]
stub.stub_host_fail.argtypes = [ctypes.c_long]
import minife_amd as m
L = m.lib()
MB = 1 << 20
def vec(mb, ctx):
    return m.Vector(mb * MB // 8, ctx)
"""


@pytest.fixture(scope="session")
def stub_lib(tmp_path_factory):
    if not os.path.exists(os.path.join(ROOT, "minife_amd", "libminife_hip.so")):
        pytest.skip("libminife_hip.so is not built")
    out = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(ROOT, "tests", "hip_stub.cpp"), "-o", out],
                   check=True)
    return out


def run(stub_lib, body):
    r = subprocess.run([sys.executable, "-c", PRELUDE + body, stub_lib], cwd=ROOT, text=True,
                       capture_output=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


def test_memory_is_kept_on_one_context(stub_lib):
    """A vector's memory serves the next one of its size on the same context."""
    run(stub_lib, """
ctx = m.Context(0)
vec(4, ctx).close()
n = stub.stub_mallocs()
for _ in range(5):
    v = vec(4, ctx); v.fill(1.0); v.close()
assert stub.stub_mallocs() == n and stub.stub_frees() == 0
""")


def test_memory_used_on_another_context_is_not_handed_out(stub_lib):
    """A vector or matrix that another context's stream may still work on does
    not become the next one's: its memory goes back to the driver, which waits
    for the device."""
    run(stub_lib, """
c1, c2 = m.Context(0), m.Context(0)
y = vec(4, c1)
x = vec(4, c2)
L.mfe_waxpby(c1.h, ctypes.c_double(1.0), x.h, ctypes.c_double(0.0), x.h, y.h)  # x's owner is c2
x.close()
z = vec(4, c2)
assert stub.stub_hazards() == 0
mesh = m.simple_mesh_description([0, 20, 0, 20, 0, 20])
A = m.CSRMatrix(c2)
m.generate_matrix_structure(mesh, A)
c2.synchronize()
xa, ya = m.Vector(A.nrows, c1), m.Vector(A.nrows, c1)
assert L.mfe_matvec(c1.h, A.h, xa.h, ya.h) == 0
assert m.generate_matrix_structure(mesh, A) == 0   # A's memory is replaced under c1's product
assert stub.stub_hazards() == 0
assert L.mfe_matvec(c1.h, A.h, xa.h, ya.h) == 0
A.close()
B = m.CSRMatrix(c2)
m.generate_matrix_structure(mesh, B)
assert stub.stub_hazards() == 0
""")


def test_every_call_notes_a_foreign_context(stub_lib):
    """Each entry point that takes handles: what was used on another context
    than its own is given back when it is destroyed, not kept."""
    run(stub_lib, """
c1, c2 = m.Context(0), m.Context(0)
box = (ctypes.c_int * 6)(0, 6, 0, 5, 0, 4)
n, ne, K = 7 * 6 * 5, 6 * 5 * 4, 4
host = np.zeros(n * 27 * 16)
hp = host.ctypes.data_as(ctypes.c_void_p)
i4 = [ctypes.byref(ctypes.c_int()) for _ in range(4)]
d4 = [ctypes.byref(ctypes.c_double()) for _ in range(4)]
i64 = (ctypes.c_int64 * 8)()
D = ctypes.c_double

def matrix(ctx):
    A = m.CSRMatrix(ctx)
    assert L.mfe_generate_matrix_structure(ctx.h, box, box, A.h) == 0
    m.make_local_matrix(A)
    return A

V = lambda k: (lambda ctx: m.Vector(k, ctx))
ro, cols = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32)
P = lambda a: a.ctypes.data_as(ctypes.c_void_p)
bc = np.zeros(1, np.int32)
# name -> (makers of the handles, call with the context and the handles)
calls = {
  "mfe_csr_upload": ([matrix], lambda c, A: L.mfe_csr_upload(c, A, n, n, None, P(ro), P(cols), hp)),
  "mfe_csr_download": ([matrix], lambda c, A: L.mfe_csr_download(c, A, None, None, None, hp)),
  "mfe_vec_upload": ([V(n)], lambda c, v: L.mfe_vec_upload(c, v, hp, n)),
  "mfe_vec_download": ([V(n)], lambda c, v: L.mfe_vec_download(c, v, hp, n)),
  "mfe_vec_fill": ([V(n)], lambda c, v: L.mfe_vec_fill(c, v, D(1.0))),
  "mfe_element_gradient": ([V(n), V(n), V(ne)], lambda c, *h: L.mfe_element_gradient(c, box, *h)),
  "mfe_generate_matrix_structure":
      ([matrix], lambda c, A: L.mfe_generate_matrix_structure(c, box, box, A)),
  "mfe_perform_element_loop": ([matrix, V(n), V(ne)],
                               lambda c, *h: L.mfe_perform_element_loop(c, box, box, *h)),
  "mfe_assemble_FE_data": ([matrix, V(n), V(ne)],
                           lambda c, *h: L.mfe_assemble_FE_data(c, box, box, *h)),
  "mfe_assemble_FE_data_ex": ([matrix, V(n), V(ne)],
                              lambda c, *h: L.mfe_assemble_FE_data_ex(c, box, box, *h, D(1.0))),
  "mfe_impose_dirichlet": ([matrix, V(n)],
                           lambda c, A, b: L.mfe_impose_dirichlet(c, D(0.0), A, b, 7, 6, 5, P(bc), 1)),
  "mfe_spmv_plan": ([matrix], lambda c, A: L.mfe_spmv_plan(c, A, 0, i64)),
  "mfe_matvec": ([matrix, V(n), V(n)], lambda c, *h: L.mfe_matvec(c, *h)),
  "mfe_matvec_and_dot": ([matrix, V(n), V(n)], lambda c, *h: L.mfe_matvec_and_dot(c, *h, d4[0])),
  "mfe_matvec_and_dot_noalloc": ([matrix, V(n), V(n)],
                                 lambda c, *h: L.mfe_matvec_and_dot_noalloc(c, *h, hp) * 0),
  "mfe_dot": ([V(n), V(n)], lambda c, *h: L.mfe_dot(c, *h, d4[0])),
  "mfe_dot_replay": ([V(n), V(n)], lambda c, *h: L.mfe_dot_replay(c, *h, d4[0])),
  "mfe_waxpby": ([V(n), V(n), V(n)],
                 lambda c, x, y, w: L.mfe_waxpby(c, D(1.0), x, D(1.0), y, w)),
  "mfe_cg_solve": ([matrix, V(n), V(n)],
                   lambda c, *h: L.mfe_cg_solve(c, *h, 2, D(0.0), 0, i4[0], d4[0], None, None)),
  "mfe_cg_solve_mixed": ([matrix, V(n), V(n)],
                         lambda c, *h: L.mfe_cg_solve_mixed(c, *h, 1, 1, D(.1), D(.1), i4[0], i4[1],
                                                            d4[0], None)),
  "mfe_cg_solve_mixed_ex": ([matrix, V(n), V(n)],
                            lambda c, *h: L.mfe_cg_solve_mixed_ex(c, *h, 1, 1, D(.1), D(.1), 0, i4[0],
                                                                  i4[1], d4[0], None)),
  "mfe_matvec_fp32": ([matrix, V(n), V(n)], lambda c, *h: L.mfe_matvec_fp32(c, *h)),
  "mfe_time_matvec": ([matrix, V(n), V(n)], lambda c, *h: L.mfe_time_matvec(c, *h, 1, 1, d4[0])),
  "mfe_verify_solution": ([V(n)], lambda c, x: L.mfe_verify_solution(c, box, x, D(9.0), 0, d4[0])),
  "mfe_verify_solution_ex": ([V(n)],
                             lambda c, x: L.mfe_verify_solution_ex(c, box, x, D(9.0), 0, 1, d4[0])),
  "mfe_spmm": ([matrix, V(n * K), V(n * K)], lambda c, *h: L.mfe_spmm(c, *h, K, 0)),
  "mfe_spmm_tune": ([matrix], lambda c, A: L.mfe_spmm_tune(c, A, K, i4[0], None, i4[1])),
  "mfe_spmm_select": ([matrix], lambda c, A: L.mfe_spmm_select(c, A, K, 0)),
  "mfe_cg_solve_multi": ([matrix, V(n * K), V(n * K)],
                         lambda c, *h: L.mfe_cg_solve_multi(c, *h, K, 2, D(.1), None, None, d4[0])),
}
# take no vector or matrix, or do not touch its memory
exempt = {x for x in m.EXPORTS if x.startswith(("mfe_ctx_", "mfe_timer_", "mfe_batch_"))} | {
    "mfe_last_error", "mfe_device_info", "mfe_trim_memory", "mfe_csr_create", "mfe_csr_destroy", "mfe_csr_shape",
    "mfe_vec_create", "mfe_vec_destroy", "mfe_vec_size", "mfe_vec_wrap", "mfe_make_local_matrix",
    "mfe_soln", "mfe_spmm_tile_info"}
assert set(calls) | exempt == set(m.EXPORTS), set(calls) ^ (set(m.EXPORTS) - exempt)
for name, (make, call) in calls.items():
    for foreign in (False, True):
        hs = [f(c2) for f in make]
        c2.synchronize()
        if name == "mfe_matvec_and_dot_noalloc":
            assert L.mfe_spmv_plan(c2.h, hs[0].h, 0, None) == 0
        st = call((c1 if foreign else c2).h, *[h.h for h in hs])
        assert st == 0, (name, st, L.mfe_last_error(c1.h), L.mfe_last_error(c2.h))
        c1.synchronize()
        for h in hs:
            before = stub.stub_frees()
            h.close()
            gone = stub.stub_frees() - before
            assert (gone > 0) == foreign, (name, type(h).__name__, foreign, gone)
""")


@pytest.mark.parametrize("why", ["cap", "failure"])
def test_giving_kept_memory_back_leaves_other_streams_alone(stub_lib, why):
    """Memory that one context kept goes when another context's thread frees more
    than the device keeps, or runs out of memory -- without a wait for the first
    one's stream, which its own thread may be capturing."""
    run(stub_lib, f"why = {why!r}" + """
stub.stub_capacity(256 * MB)      # 32 MB may be kept
c1, c2 = m.Context(0), m.Context(0)
kept = [vec(8, c2) for _ in range(3)]
for v in kept: v.close()
assert stub.stub_frees() == 0
stub.stub_thread_stream(0)
stub.stub_begin_capture(1)        # c2's stream
if why == "cap":
    vs = [vec(8, c1) for _ in range(2)]
    for v in vs: v.close()
    assert stub.stub_frees() == 1
else:
    v = vec(240, c1)
    assert stub.stub_frees() == 3
    v.close()
stub.stub_end_capture(1)
assert stub.stub_capture_breaks() == 0 and stub.stub_foreign_waits() == 0
""")


WORKSPACES = {
    "cg_solve": "m.cg_solve(A, b, x, max_iter=2)",
    "cg_solve_mixed": "m.cg_solve_mixed(A, b, x, max_outer=1, max_inner=2)",
    "matvec_fp32": "m.matvec_fp32(A, b, x)",
    "matvec_and_dot": "m.matvec_and_dot(A, b, x)",
    "dot": "m.dot(b, x)",
    "spmm": "m.spmm(A, X, X2, 16)",
    "cg_solve_multi": "m.cg_solve_multi(A, X, X2, 16, max_iter=2)",
    "batch": "m.Batch([(40, 40, 40), (30, 30, 30)], ctx)",
}


@pytest.mark.parametrize("what", sorted(WORKSPACES))
def test_workspaces_get_the_kept_memory(stub_lib, what):
    """Calls whose own allocations fit the device only once the memory kept for
    matrices and vectors has gone back."""
    run(stub_lib, f"what, call = {what!r}, {WORKSPACES[what]!r}" + """
ctx = m.Context(0)
_, A, b = m.build_problem(40, ctx=ctx)
x = m.Vector(A.nrows, ctx)
X, X2 = m.Vector(16 * A.nrows, ctx), m.Vector(16 * A.nrows, ctx)
m.matvec(A, b, x)                     # A's plan
m.spmm(A, X, X2, 16, tile=0)
other = m.Context(0)                  # leaves its memory: half of it is another context's
stub.stub_capacity(1 << 40)
for c in (ctx, other):
    kept = [m.Vector(8 * MB // 8, c) for _ in range(40)]
    for v in kept: v.close()
frees = stub.stub_frees()
stub.stub_capacity(stub.stub_used())  # nothing is left but what is kept
eval(call)
assert stub.stub_frees() > frees
""")


def test_trim_memory(stub_lib):
    """The kept memory of every context goes back when asked for, and only that."""
    run(stub_lib, """
c1, c2 = m.Context(0), m.Context(0)
a = vec(4, c1)
vec(6, c1).close()
vec(8, c2).close()
used = stub.stub_used()
assert c1.trim_memory() == 14 * MB and stub.stub_used() == used - 14 * MB
assert c1.trim_memory() == 0 and stub.stub_used() == used - 14 * MB
a.fill(1.0)
""")


@pytest.mark.parametrize("nth", [1, 2])
def test_solve_after_a_failed_workspace(stub_lib, nth):
    """A solve whose pinned words could not be allocated reports it, and the next
    one allocates them."""
    run(stub_lib, f"nth = {nth}" + """
ctx = m.Context(0)
_, A, b = m.build_problem(6, ctx=ctx)
x = m.Vector(A.nrows, ctx)
m.matvec(A, b, x)
stub.stub_host_fail(nth)
try:
    m.cg_solve(A, b, x, max_iter=2)
    assert False
except m.MfeError as e:
    assert e.status == m.MFE_OOM
m.cg_solve(A, b, x, max_iter=2)
""")


def test_mixed_solve_after_a_failed_workspace(stub_lib):
    """The mixed solve's inner vectors could not grow for a larger system: that
    solve reports it, and the next one of the first size allocates its own."""
    run(stub_lib, """
ctx = m.Context(0)
def problem(n):
    _, A, b = m.build_problem(n, ctx=ctx)
    return A, b, m.Vector(A.nrows, ctx)
small, large = problem(6), problem(40)
m.cg_solve_mixed(*small, max_outer=1, max_inner=2, outer_tol=-1.0)
m.cg_solve(*large, max_iter=2)
m.matvec_fp32(*large)            # all that the large system needs but the inner vectors
ctx.trim_memory()
stub.stub_capacity(stub.stub_used() + 4096)
try:
    m.cg_solve_mixed(*large, max_outer=1, max_inner=2)
    assert False
except m.MfeError as e:
    assert e.status == m.MFE_OOM
stub.stub_capacity(1 << 30)
m.cg_solve_mixed(*small, max_outer=1, max_inner=2, outer_tol=-1.0)
""")


def test_allocating_among_many_kept_blocks(stub_lib):
    """A thousand allocations that find no block of their size take about as long
    beside 50,000 kept blocks as beside none (a look at every block takes more than
    a hundred times as long)."""
    run(stub_lib, """
ctx = m.Context(0)
h = ctypes.c_void_p()
def create(doubles):
    L.mfe_vec_create(ctx.h, doubles, ctypes.byref(h))
    return ctypes.c_void_p(h.value)
def seconds():
    best = 1e9
    for _ in range(5):
        t = time.perf_counter()
        for _ in range(1000): create(512)   # (never destroyed: nothing to find)
        best = min(best, time.perf_counter() - t)
    return best
stub.stub_capacity(1 << 40)
few = seconds()
for v in [create(8) for _ in range(50000)]: L.mfe_vec_destroy(v)
many = seconds()
print(many, few)
assert many < 5 * few, (many, few)
""")


def test_allocation_waits_for_memory_that_is_being_given_back(stub_lib):
    """An allocation that the device has no room for while another thread is still
    giving kept memory back succeeds once that is done."""
    run(stub_lib, """
stub.stub_capacity(512 * MB)
c1, c2 = m.Context(0), m.Context(0)
vec(60, c2).close()
stub.stub_capacity(stub.stub_used() + MB)
stub.stub_free_delay(500)
t = threading.Thread(target=c2.trim_memory)
t.start()
time.sleep(0.1)
v = vec(40, c1)
t.join()
""")
