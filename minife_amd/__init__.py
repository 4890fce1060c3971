"""minife_amd -- miniFE's assemble-and-solve path on MI355X (gfx950).

Python mirror of the reference ref/ operator surface over the C-ABI of
``libminife_hip.so`` (include/minife_hip.h).  Names, argument meaning and error
behaviour follow the reference:

  simple_mesh_description(global_box, local_box)   simple_mesh_description.hpp:38-244
  generate_matrix_structure(mesh, A)                generate_matrix_structure.hpp:47-149
  assemble_FE_data(mesh, A, b, params)              assemble_FE_data.hpp:38-73
  perform_element_loop(mesh, box, A, b, params)     perform_element_loop.hpp:40-104
  impose_dirichlet(value, A, b, gnx, gny, gnz, bc)  SparseMatrix_functions.hpp:431-480
  make_local_matrix(A)                              make_local_matrix.hpp:42-442
  cg_solve(A, b, x, max_iter, tol)                  cg_solve.hpp:69-229
  matvec / matvec_and_dot / dot / waxpby            SparseMatrix_functions.hpp:491-578,
                                                    Vector_functions.hpp:127-226
  verify_solution(mesh, x, tol, whole)              verify_solution.hpp:55-174

Matrices and vectors live in HBM (device handles); ``to_host`` copies out.
The HIP library is required: importing works without it, but the first call
raises if ``libminife_hip.so`` is missing or no GPU is visible.
"""
from __future__ import annotations

import atexit
import ctypes
import os
import sys
import weakref
from dataclasses import dataclass, field

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libminife_hip.so")

MFE_OK, MFE_BREAKDOWN, MFE_NOT_LOCAL, MFE_OOM, MFE_HIP_ERROR, MFE_BAD_ARG, MFE_UNSUPPORTED = range(7)
STATUS_NAMES = ["OK", "BREAKDOWN", "NOT_LOCAL", "OOM", "HIP_ERROR", "BAD_ARG", "UNSUPPORTED"]
CG_REPLAY, CG_TOL_RELATIVE, CG_EAGER = 0x1, 0x2, 0x4
SPMV_AUTO, SPMV_CSR, SPMV_SELL = 0, 1, 2
SPMV_KERNELS = ["csr-stream", "sell64", "csr-rowwise", "sell64-staged-x", "box", "box-sym",
                "box-sym-packed"]
# packed forms of the symmetric box layout's upper values (slots 0..13 =
# stencil slots 13..26): name -> (field bits of the cube's slots, of its
# analytically zero slots PACK_NEAR; 0: read at full width)
PACK_FORMS = {1: "all16", 2: "cube16+near32", 3: "cube16", 4: "all12", 5: "cube12+near24",
              6: "all10", 7: "cube10+near22"}
PACK_NEAR = (1, 3, 9)
PACK_WIDTHS = {"all16": (16, 16), "cube16+near32": (16, 32), "cube16": (16, 0),
               "all12": (12, 12), "cube12+near24": (12, 24), "all10": (10, 10),
               "cube10+near22": (10, 22)}


def pack_bnd_words(form: str) -> int:
    """32-bit words per (block, plane) of the packed boundary stream: 282
    fields, the 32 of lower slots 10 and 12 wide, the others narrow, and one
    word of padding (forms that give every entry a field: not "cube16")."""
    narrow, near = PACK_WIDTHS[form]
    return (250 * narrow + 32 * near + 31) // 32 + 1


def pack_row_layout(form: str):
    """(32-bit words per row, slots read at full width) of a packed form: the
    14 fields follow each other from bit 0 of the row's first word."""
    narrow, near = PACK_WIDTHS[form]
    bits = narrow * (14 - len(PACK_NEAR)) + near * len(PACK_NEAR)
    return (bits + 31) // 32, (len(PACK_NEAR) if near == 0 else 0)


T_WAXPY, T_DOT, T_MATVEC, T_MATVECDOT, T_TOTAL = range(5)

# Every extern "C" symbol declared in include/minife_hip.h.
EXPORTS = [
    "mfe_ctx_create", "mfe_ctx_destroy", "mfe_last_error", "mfe_ctx_synchronize", "mfe_trim_memory",
    "mfe_device_info", "mfe_timer_start", "mfe_timer_stop",
    "mfe_csr_create", "mfe_csr_destroy", "mfe_csr_shape", "mfe_csr_upload", "mfe_csr_download",
    "mfe_vec_create", "mfe_vec_destroy", "mfe_vec_size", "mfe_vec_upload", "mfe_vec_download",
    "mfe_vec_fill", "mfe_vec_wrap", "mfe_element_gradient",
    "mfe_generate_matrix_structure", "mfe_perform_element_loop", "mfe_assemble_FE_data",
    "mfe_assemble_FE_data_ex", "mfe_verify_solution_ex",
    "mfe_impose_dirichlet", "mfe_make_local_matrix", "mfe_spmv_plan",
    "mfe_matvec", "mfe_matvec_and_dot", "mfe_matvec_and_dot_noalloc", "mfe_dot", "mfe_dot_replay", "mfe_waxpby",
    "mfe_cg_solve", "mfe_cg_solve_mixed", "mfe_cg_solve_mixed_ex", "mfe_matvec_fp32", "mfe_time_matvec", "mfe_soln",
    "mfe_verify_solution", "mfe_batch_create", "mfe_batch_destroy", "mfe_batch_info",
    "mfe_batch_solve", "mfe_batch_download", "mfe_batch_timing", "mfe_spmm", "mfe_spmm_tune", "mfe_spmm_select", "mfe_spmm_tile_info",
    "mfe_cg_solve_multi",
]


class MfeError(RuntimeError):
    def __init__(self, status: int, msg: str):
        name = STATUS_NAMES[status] if 0 <= status < len(STATUS_NAMES) else str(status)
        super().__init__(f"{name}: {msg}")
        self.status = status


_lib = None
_vp = ctypes.c_void_p
_i64 = ctypes.c_int64
_int6 = ctypes.c_int * 6


def _share_torch_hip_runtime() -> None:
    """Keep one HIP runtime per process.  PyTorch wheels bundle their own
    libamdhip64/libhsa-runtime64 and load them by file name, so a process that
    loaded the system runtime first ends up with two HSA runtimes and torch
    then finds no GPU.  Loading torch's copy first (without importing torch)
    makes this library bind to it through the shared soname, so tensors and
    library vectors live in one runtime whatever the import order.
    MINIFE_SYSTEM_HIP_RUNTIME=1 keeps the system runtime (processes that
    never use torch)."""
    if os.environ.get("MINIFE_SYSTEM_HIP_RUNTIME") == "1":
        return
    import importlib.util
    try:
        spec = importlib.util.find_spec("torch")
    except (ImportError, ValueError):
        return
    if spec is None or not spec.submodule_search_locations:
        return
    for loc in spec.submodule_search_locations:
        path = os.path.join(loc, "lib", "libamdhip64.so")
        if os.path.exists(path):
            ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
            return


# Live handles: contexts, and what lives in a context (matrices, vectors,
# batches).  At interpreter exit every one still open is closed, dependents
# first, while the HIP runtime is up: none of the captured graphs, streams,
# events or pinned buffers is left to the runtime's own exit-time teardown,
# whose order against them is unspecified.
_live_contexts: "weakref.WeakSet" = weakref.WeakSet()
_live_dependents: "weakref.WeakSet" = weakref.WeakSet()
_shut_down = False


def _close_all_at_exit() -> None:
    global _shut_down
    for group in (_live_dependents, _live_contexts):
        for obj in list(group):
            try:
                obj.close()
            except Exception:
                pass
    _shut_down = True


def _release(obj, _finalizing=sys.is_finalizing) -> None:
    """Destructor body: free the handle unless the interpreter is shutting
    down (the exit hook has closed every live handle by then)."""
    if _shut_down or _finalizing():
        return
    try:
        obj.close()
    except Exception:
        pass


def lib() -> ctypes.CDLL:
    """Load libminife_hip.so (raises if it has not been built)."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(f"{LIB_PATH} is missing: build it with `python -m minife_amd.build`")
    _share_torch_hip_runtime()
    L = ctypes.CDLL(LIB_PATH)
    atexit.register(_close_all_at_exit)
    sig = {
        "mfe_ctx_create": ([ctypes.c_int, ctypes.POINTER(_vp)], ctypes.c_int),
        "mfe_ctx_destroy": ([_vp], None),
        "mfe_last_error": ([_vp], ctypes.c_char_p),
        "mfe_ctx_synchronize": ([_vp], ctypes.c_int),
        "mfe_trim_memory": ([_vp, ctypes.POINTER(_i64)], ctypes.c_int),
        "mfe_device_info": ([_vp, ctypes.c_char_p, ctypes.c_int, ctypes.POINTER(ctypes.c_int),
                             ctypes.POINTER(_i64)], ctypes.c_int),
        "mfe_timer_start": ([_vp], ctypes.c_int),
        "mfe_timer_stop": ([_vp, ctypes.POINTER(ctypes.c_double)], ctypes.c_int),
        "mfe_csr_create": ([_vp, ctypes.POINTER(_vp)], ctypes.c_int),
        "mfe_csr_destroy": ([_vp], None),
        "mfe_csr_shape": ([_vp, ctypes.POINTER(_i64), ctypes.POINTER(_i64)], ctypes.c_int),
        "mfe_csr_upload": ([_vp, _vp, _i64, _i64, _vp, _vp, _vp, _vp], ctypes.c_int),
        "mfe_csr_download": ([_vp, _vp, _vp, _vp, _vp, _vp], ctypes.c_int),
        "mfe_vec_create": ([_vp, _i64, ctypes.POINTER(_vp)], ctypes.c_int),
        "mfe_vec_destroy": ([_vp], None),
        "mfe_vec_size": ([_vp], _i64),
        "mfe_vec_upload": ([_vp, _vp, _vp, _i64], ctypes.c_int),
        "mfe_vec_download": ([_vp, _vp, _vp, _i64], ctypes.c_int),
        "mfe_vec_fill": ([_vp, _vp, ctypes.c_double], ctypes.c_int),
        "mfe_vec_wrap": ([_vp, _vp, _i64, ctypes.POINTER(_vp)], ctypes.c_int),
        "mfe_element_gradient": ([_vp, _int6, _vp, _vp, _vp], ctypes.c_int),
        "mfe_generate_matrix_structure": ([_vp, _int6, _int6, _vp], ctypes.c_int),
        "mfe_perform_element_loop": ([_vp, _int6, _int6, _vp, _vp, _vp], ctypes.c_int),
        "mfe_assemble_FE_data": ([_vp, _int6, _int6, _vp, _vp, _vp], ctypes.c_int),
        "mfe_assemble_FE_data_ex": ([_vp, _int6, _int6, _vp, _vp, _vp, ctypes.c_double],
                                    ctypes.c_int),
        "mfe_impose_dirichlet": ([_vp, ctypes.c_double, _vp, _vp, ctypes.c_int, ctypes.c_int,
                                  ctypes.c_int, _vp, _i64], ctypes.c_int),
        "mfe_make_local_matrix": ([_vp, _vp], ctypes.c_int),
        "mfe_spmv_plan": ([_vp, _vp, ctypes.c_int, _vp], ctypes.c_int),
        "mfe_matvec": ([_vp, _vp, _vp, _vp], ctypes.c_int),
        "mfe_matvec_and_dot": ([_vp, _vp, _vp, _vp, ctypes.POINTER(ctypes.c_double)], ctypes.c_int),
        "mfe_matvec_and_dot_noalloc": ([_vp, _vp, _vp, _vp, _vp], ctypes.c_int),
        "mfe_dot": ([_vp, _vp, _vp, ctypes.POINTER(ctypes.c_double)], ctypes.c_int),
        "mfe_dot_replay": ([_vp, _vp, _vp, ctypes.POINTER(ctypes.c_double)], ctypes.c_int),
        "mfe_waxpby": ([_vp, ctypes.c_double, _vp, ctypes.c_double, _vp, _vp], ctypes.c_int),
        "mfe_cg_solve": ([_vp, _vp, _vp, _vp, ctypes.c_int, ctypes.c_double, ctypes.c_uint,
                          ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_double), _vp, _vp],
                         ctypes.c_int),
        "mfe_cg_solve_mixed": ([_vp, _vp, _vp, _vp, ctypes.c_int, ctypes.c_int, ctypes.c_double,
                                ctypes.c_double, ctypes.POINTER(ctypes.c_int),
                                ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_double),
                                _vp], ctypes.c_int),
        "mfe_cg_solve_mixed_ex": ([_vp, _vp, _vp, _vp, ctypes.c_int, ctypes.c_int, ctypes.c_double,
                                   ctypes.c_double, ctypes.c_uint, ctypes.POINTER(ctypes.c_int),
                                   ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_double),
                                   _vp], ctypes.c_int),
        "mfe_matvec_fp32": ([_vp, _vp, _vp, _vp], ctypes.c_int),
        "mfe_time_matvec": ([_vp, _vp, _vp, _vp, ctypes.c_int, ctypes.c_int,
                             ctypes.POINTER(ctypes.c_double)], ctypes.c_int),
        "mfe_soln": ([ctypes.c_double] * 3 + [ctypes.c_int, ctypes.c_int], ctypes.c_double),
        "mfe_spmm": ([_vp, _vp, _vp, _vp, ctypes.c_int, ctypes.c_int], ctypes.c_int),
        "mfe_spmm_tune": ([_vp, _vp, ctypes.c_int, ctypes.POINTER(ctypes.c_int), _vp,
                           ctypes.POINTER(ctypes.c_int)], ctypes.c_int),
        "mfe_spmm_select": ([_vp, _vp, ctypes.c_int, ctypes.c_int], ctypes.c_int),
        "mfe_spmm_tile_info": ([ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.c_int),
                                ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_int),
                                ctypes.POINTER(ctypes.c_int)],
                               ctypes.c_int),
        "mfe_cg_solve_multi": ([_vp, _vp, _vp, _vp, ctypes.c_int, ctypes.c_int, ctypes.c_double,
                                _vp, _vp, ctypes.POINTER(ctypes.c_double)], ctypes.c_int),
        "mfe_batch_create": ([_vp, ctypes.c_int, _vp, ctypes.POINTER(_vp)], ctypes.c_int),
        "mfe_batch_destroy": ([_vp], None),
        "mfe_batch_info": ([_vp, ctypes.c_int, _vp], ctypes.c_int),
        "mfe_batch_solve": ([_vp, _vp, ctypes.c_int, ctypes.c_double, _vp, _vp,
                             ctypes.POINTER(ctypes.c_double)], ctypes.c_int),
        "mfe_batch_download": ([_vp, _vp, ctypes.c_int, _vp, _vp, _vp, _vp, _vp], ctypes.c_int),
        "mfe_batch_timing": ([_vp, _vp, _vp], ctypes.c_int),
        "mfe_verify_solution": ([_vp, _int6, _vp, ctypes.c_double, ctypes.c_int,
                                 ctypes.POINTER(ctypes.c_double)], ctypes.c_int),
        "mfe_verify_solution_ex": ([_vp, _int6, _vp, ctypes.c_double, ctypes.c_int, ctypes.c_int,
                                    ctypes.POINTER(ctypes.c_double)], ctypes.c_int),
    }
    for name, (args, res) in sig.items():
        f = getattr(L, name)
        f.argtypes = args
        f.restype = res
    _lib = L
    return L


def _ptr(a: np.ndarray | None):
    return None if a is None else a.ctypes.data_as(_vp)


class Context:
    """One device and one HIP stream (mfe_ctx)."""

    def __init__(self, device: int = 0):
        h = _vp()
        st = lib().mfe_ctx_create(int(device), ctypes.byref(h))
        if st != MFE_OK:
            raise MfeError(st, f"mfe_ctx_create(device={device}) failed (no GPU visible?)")
        self.h = h
        _live_contexts.add(self)
        self.device = device

    def check(self, st: int, what: str = ""):
        if st != MFE_OK:
            raise MfeError(st, f"{what}: {lib().mfe_last_error(self.h).decode(errors='replace')}")

    def synchronize(self):
        self.check(lib().mfe_ctx_synchronize(self.h), "synchronize")

    def trim_memory(self) -> int:
        """Gives the device memory kept for later matrices and vectors back to the
        driver (torch's allocator then finds it); returns the bytes."""
        n = _i64(0)
        self.check(lib().mfe_trim_memory(self.h, ctypes.byref(n)), "trim_memory")
        return n.value

    def device_info(self) -> dict:
        buf = ctypes.create_string_buffer(256)
        cu = ctypes.c_int(0)
        hbm = _i64(0)
        self.check(lib().mfe_device_info(self.h, buf, 256, ctypes.byref(cu), ctypes.byref(hbm)),
                   "device_info")
        return dict(name=buf.value.decode(), cu_count=cu.value, hbm_bytes=hbm.value)

    def timer_start(self):
        self.check(lib().mfe_timer_start(self.h), "timer_start")

    def timer_stop(self) -> float:
        ms = ctypes.c_double(0)
        self.check(lib().mfe_timer_stop(self.h, ctypes.byref(ms)), "timer_stop")
        return ms.value

    def close(self):
        """Destroy the context after what lives in it (their destroy calls
        synchronize on this context's stream)."""
        if getattr(self, "h", None):
            for obj in list(_live_dependents):
                if getattr(obj, "ctx", None) is self:
                    obj.close()
            lib().mfe_ctx_destroy(self.h)
            self.h = None

    def __del__(self):
        _release(self)


_default_ctx: Context | None = None


def default_context() -> Context:
    global _default_ctx
    if _default_ctx is None:
        _default_ctx = Context(int(os.environ.get("MFE_DEVICE", "0")))
    return _default_ctx


class CSRMatrix:
    """Device CSR with the fields of CSRMatrix.hpp:40-129 (int32 ordinals, float64)."""

    def __init__(self, ctx: Context | None = None):
        self.ctx = ctx or default_context()
        h = _vp()
        self.ctx.check(lib().mfe_csr_create(self.ctx.h, ctypes.byref(h)), "csr_create")
        self.h = h
        _live_dependents.add(self)

    @property
    def shape(self):
        n, z = _i64(), _i64()
        lib().mfe_csr_shape(self.h, ctypes.byref(n), ctypes.byref(z))
        return n.value, z.value

    @property
    def nrows(self) -> int:
        return self.shape[0]

    def num_nonzeros(self) -> int:
        return self.shape[1]

    @classmethod
    def from_host(cls, row_offsets, cols, vals, rows=None, ctx: Context | None = None):
        A = cls(ctx)
        ro = np.ascontiguousarray(row_offsets, dtype=np.int32)
        c = np.ascontiguousarray(cols, dtype=np.int32)
        v = np.ascontiguousarray(vals, dtype=np.float64)
        r = None if rows is None else np.ascontiguousarray(rows, dtype=np.int32)
        A.ctx.check(lib().mfe_csr_upload(A.ctx.h, A.h, ro.shape[0] - 1, c.shape[0], _ptr(r),
                                         _ptr(ro), _ptr(c), _ptr(v)), "csr_upload")
        return A

    def to_host(self, rows=True, row_offsets=True, cols=True, vals=True) -> dict:
        n, nnz = self.shape
        out = {}
        if rows:
            out["rows"] = np.empty(n, np.int32)
        if row_offsets:
            out["row_offsets"] = np.empty(n + 1, np.int32)
        if cols:
            out["cols"] = np.empty(nnz, np.int32)
        if vals:
            out["vals"] = np.empty(nnz, np.float64)
        self.ctx.check(lib().mfe_csr_download(self.ctx.h, self.h, _ptr(out.get("rows")),
                                              _ptr(out.get("row_offsets")), _ptr(out.get("cols")),
                                              _ptr(out.get("vals"))), "csr_download")
        return out

    def close(self):
        if getattr(self, "h", None):
            lib().mfe_csr_destroy(self.h)
            self.h = None

    def __del__(self):
        _release(self)


class Vector:
    """Device vector of float64 (Vector.hpp:36-61); zero-filled on creation."""

    def __init__(self, n: int, ctx: Context | None = None):
        self.ctx = ctx or default_context()
        h = _vp()
        self.ctx.check(lib().mfe_vec_create(self.ctx.h, int(n), ctypes.byref(h)), "vec_create")
        self.h = h
        _live_dependents.add(self)
        self.n = int(n)

    @classmethod
    def wrap(cls, device_ptr: int, n: int, ctx: Context | None = None, owner=None):
        """A view over caller-owned device memory (e.g. a torch tensor's
        data_ptr()); `owner` is kept alive with the view."""
        v = cls.__new__(cls)
        v.ctx = ctx or default_context()
        h = _vp()
        v.ctx.check(lib().mfe_vec_wrap(v.ctx.h, _vp(int(device_ptr)), int(n), ctypes.byref(h)),
                    "vec_wrap")
        v.h = h
        v.n = int(n)
        v._owner = owner
        _live_dependents.add(v)
        return v

    @classmethod
    def from_numpy(cls, a, ctx: Context | None = None):
        a = np.ascontiguousarray(a, dtype=np.float64)
        v = cls(a.shape[0], ctx)
        v.ctx.check(lib().mfe_vec_upload(v.ctx.h, v.h, _ptr(a), a.shape[0]), "vec_upload")
        return v

    def to_numpy(self) -> np.ndarray:
        out = np.empty(self.n, np.float64)
        self.ctx.check(lib().mfe_vec_download(self.ctx.h, self.h, _ptr(out), self.n), "vec_download")
        return out

    def fill(self, value: float):
        self.ctx.check(lib().mfe_vec_fill(self.ctx.h, self.h, float(value)), "vec_fill")

    def close(self):
        if getattr(self, "h", None):
            lib().mfe_vec_destroy(self.h)
            self.h = None

    def __del__(self):
        _release(self)


def _box6(box) -> "ctypes.Array":
    b = np.asarray(box, dtype=np.int64).reshape(-1)
    if b.shape[0] != 6:
        raise ValueError("a Box is 6 ints {x0,x1,y0,y1,z0,z1}")
    return _int6(*[int(v) for v in b])


@dataclass
class Parameters:
    """Runtime parameters of ref/utils/Parameters.hpp:40-90 used on this path."""
    nx: int = 10
    ny: int = -1
    nz: int = -1
    verify_solution: int = 0
    name: str = ""
    # not in the reference (its problem is fixed): the element source Q and
    # the face held at u = 1 (1: x = 1 as the reference, 0: x = 0)
    source: float = 1.0
    hot_face: int = 1
    extra: dict = field(default_factory=dict)

    def __post_init__(self):
        if self.ny < 0:
            self.ny = self.nx
        if self.nz < 0:
            self.nz = self.ny


class simple_mesh_description:
    """simple_mesh_description.hpp:38-244 for one rank: boxes and BC row sets.

    bc_rows_0: nodes on the faces x=0, y=0, z=0, y=1, z=1 (prescribed 0);
    bc_rows_1: nodes on the face x=1 (prescribed 1).  Sorted int32 arrays
    (the reference's std::set); one rank so node id == row.  hot_face=0 swaps
    the roles of x=0 and x=1 (u = 1 on x = 0).
    """

    def __init__(self, global_box, local_box=None, hot_face: int = 1):
        self.hot_face = int(hot_face)
        self.global_box = np.asarray(global_box, dtype=np.int64).reshape(6)
        self.local_box = self.global_box.copy() if local_box is None else \
            np.asarray(local_box, dtype=np.int64).reshape(6)
        gb = self.global_box
        if gb[0] != 0 or gb[2] != 0 or gb[4] != 0 or min(gb[1], gb[3], gb[5]) < 1:
            raise ValueError("global box must be {0,nx,0,ny,0,nz} with nx,ny,nz >= 1")
        if not np.array_equal(self.local_box, self.global_box):
            raise NotImplementedError("one rank: local box must equal the global box")
        gx, gy, gz = int(gb[1]) + 1, int(gb[3]) + 1, int(gb[5]) + 1
        hot, cold = (gx - 1, 0) if self.hot_face else (0, gx - 1)
        # u = 0: the first and last z planes whole, of every other plane its
        # first and last lines and the cold column, in ascending id
        line = np.zeros((gy, gx), bool)
        line[0] = line[-1] = True
        line[:, cold] = True
        edge = np.flatnonzero(line).astype(np.int32)
        plane = gx * gy
        inner = np.arange(1, gz - 1, dtype=np.int32)[:, None] * np.int32(plane) + edge
        first = np.arange(plane, dtype=np.int32)
        self.bc_rows_0 = np.concatenate([first, inner.reshape(-1), first + np.int32((gz - 1) * plane)])
        self.bc_rows_1 = np.arange(hot, plane * gz, gx, dtype=np.int32)

    @property
    def nodes(self):
        gb = self.global_box
        return int(gb[1]) + 1, int(gb[3]) + 1, int(gb[5]) + 1


def generate_matrix_structure(mesh: simple_mesh_description, A: CSRMatrix) -> int:
    """Returns 0 on success, 1 on allocation failure (generate_matrix_structure.hpp:140-148)."""
    st = lib().mfe_generate_matrix_structure(A.ctx.h, _box6(mesh.global_box),
                                             _box6(mesh.local_box), A.h)
    if st == MFE_OOM:
        return 1
    A.ctx.check(st, "generate_matrix_structure")
    return 0


def perform_element_loop(mesh, elem_box, A: CSRMatrix, b: Vector, params=None, kappa=None):
    st = lib().mfe_perform_element_loop(A.ctx.h, _box6(mesh.global_box), _box6(elem_box), A.h,
                                        b.h, kappa.h if kappa is not None else None)
    A.ctx.check(st, "perform_element_loop")


def assemble_FE_data(mesh, A: CSRMatrix, b: Vector, params=None, kappa=None, source=None):
    """assemble_FE_data.hpp:38-73; source (or params.source) is the element
    source Q, 1.0 as the reference."""
    if source is None:
        source = params.source if params is not None else 1.0
    st = lib().mfe_assemble_FE_data_ex(A.ctx.h, _box6(mesh.global_box), _box6(mesh.local_box),
                                       A.h, b.h, kappa.h if kappa is not None else None,
                                       float(source))
    A.ctx.check(st, "assemble_FE_data")


def impose_dirichlet(prescribed_value: float, A: CSRMatrix, b: Vector, global_nx: int,
                     global_ny: int, global_nz: int, bc_rows) -> None:
    bc = np.ascontiguousarray(bc_rows, dtype=np.int32)
    if bc.size > 1 and not bool(np.all(bc[1:] > bc[:-1])):
        bc = np.unique(bc)  # std::set semantics: sorted, each row once
    st = lib().mfe_impose_dirichlet(A.ctx.h, float(prescribed_value), A.h, b.h, int(global_nx),
                                    int(global_ny), int(global_nz), _ptr(bc), bc.shape[0])
    A.ctx.check(st, "impose_dirichlet")


def make_local_matrix(A: CSRMatrix) -> None:
    A.ctx.check(lib().mfe_make_local_matrix(A.ctx.h, A.h), "make_local_matrix")


def spmv_plan(A: CSRMatrix, fmt: int = SPMV_AUTO) -> dict:
    """Choose A's SpMV storage and build it now.  SPMV_AUTO: the box layout
    when A holds a box's stencil structure (values per 16 x 16-node block,
    plane and stencil slot; the SpMV marches along z with x planes in LDS;
    "box-sym" when A is symmetric bit for bit: each row stores its 14 upper
    slots and takes the others from its neighbours; "box-sym-packed" when,
    for a set of those slots, every value is also kept exactly as an offset
    of 10 to 32 bits from a base, times a power of two, per (block, plane,
    slot) -- then 'pack' names the form of the FP64 values and 'pack_fp32'
    that of the FP32 copy once it exists (PACK_FORMS, PACK_WIDTHS)),
    else a SELL-64 copy when every row has at most 27 entries, with x staged
    in LDS per 256-row tile when every tile's distinct columns form at most
    128 runs; SPMV_SELL: SELL-64 without the staging; SPMV_CSR: CSR kernels
    only."""
    info = (ctypes.c_int64 * 8)()
    A.ctx.check(lib().mfe_spmv_plan(A.ctx.h, A.h, int(fmt), info), "spmv_plan")
    kernel = SPMV_KERNELS[info[0]]
    if kernel in ("box", "box-sym", "box-sym-packed"):
        d = dict(kernel=kernel, stored=int(info[1]), workgroups=int(info[2]),
                 longest_row=27, planes_per_chunk=int(info[4]),
                 blocks_x=int(info[5]), blocks_y=int(info[6]), z_chunks=int(info[7]))
        if kernel == "box-sym-packed":
            d["pack"] = PACK_FORMS[int(info[3]) & 0xFF]
            d["pack_fp32"] = PACK_FORMS.get((int(info[3]) >> 8) & 0xFF)
            d["wpack"] = PACK_FORMS.get((int(info[3]) >> 16) & 0xFF)
        return d
    return dict(kernel=kernel, stored=int(info[1]), slices=int(info[2]),
                longest_row=int(info[3]), runs=int(info[4]), max_distinct=int(info[5]),
                explicit_entries=int(info[6]), base_slices=int(info[7]))


def matvec(A: CSRMatrix, x: Vector, y: Vector) -> None:
    A.ctx.check(lib().mfe_matvec(A.ctx.h, A.h, x.h, y.h), "matvec")


def matvec_and_dot(A: CSRMatrix, x: Vector, y: Vector) -> float:
    r = ctypes.c_double(0)
    A.ctx.check(lib().mfe_matvec_and_dot(A.ctx.h, A.h, x.h, y.h, ctypes.byref(r)), "matvec_and_dot")
    return r.value


def dot(x: Vector, y: Vector, replay: bool = False) -> float:
    r = ctypes.c_double(0)
    f = lib().mfe_dot_replay if replay else lib().mfe_dot
    x.ctx.check(f(x.ctx.h, x.h, y.h, ctypes.byref(r)), "dot")
    return r.value


def waxpby(alpha: float, x: Vector, beta: float, y: Vector, w: Vector) -> None:
    x.ctx.check(lib().mfe_waxpby(x.ctx.h, float(alpha), x.h, float(beta), y.h, w.h), "waxpby")


@dataclass
class CGResult:
    num_iters: int
    normr: float
    status: int
    times: np.ndarray
    history: np.ndarray | None  # [k, 4] = rtrans, p_ap_dot, alpha, beta

    @property
    def breakdown(self) -> bool:
        return self.status == MFE_BREAKDOWN


def cg_solve(A: CSRMatrix, b: Vector, x: Vector, max_iter: int = 200,
             tolerance: float = float(np.finfo(np.float64).eps), *, replay: bool = False,
             relative: bool = False, eager: bool = False, history: bool = False) -> CGResult:
    """cg_solve.hpp:69-229.  Breakdown is reported in the result (status), as
    the reference returns early rather than failing."""
    flags = (CG_REPLAY if replay else 0) | (CG_TOL_RELATIVE if relative else 0) | \
        (CG_EAGER if eager else 0)
    ni = ctypes.c_int(0)
    nr = ctypes.c_double(0)
    times = np.zeros(5, np.float64)
    hist = np.zeros((max(int(max_iter), 1) + 1, 4), np.float64) if history else None
    st = lib().mfe_cg_solve(A.ctx.h, A.h, b.h, x.h, int(max_iter), float(tolerance), flags,
                            ctypes.byref(ni), ctypes.byref(nr), _ptr(times), _ptr(hist))
    if st not in (MFE_OK, MFE_BREAKDOWN):
        A.ctx.check(st, "cg_solve")
    if hist is not None:
        hist = hist[: ni.value + (1 if st == MFE_BREAKDOWN else 0)]
    return CGResult(ni.value, nr.value, st, times, hist)


@dataclass
class MixedResult:
    outer_iters: int
    inner_iters: int
    rel_residual: float
    status: int
    seconds: float

    @property
    def converged(self) -> bool:
        return self.status == MFE_OK


MIXED_KEEP_DIRECTION = 0x1


def cg_solve_mixed(A: CSRMatrix, b: Vector, x: Vector, *, max_outer: int = 200,
                   max_inner: int = 20000, inner_tol: float | None = None,
                   outer_tol: float = 1e-10, keep_direction: bool = False) -> MixedResult:
    """Mixed-precision iterative refinement around cg_solve (FP32 inner CG on an
    FP32 copy of A, FP64 residual/update/norms on the GPU).  inner_tol is the
    residual reduction per refinement (default 1e-5 restarting, 0.1 keeping
    the direction).  keep_direction: the inner CG continues across
    refinements with its residual replaced by the FP64 one (reliable updates)
    instead of restarting; it needs frequent replacements (0.1)."""
    if inner_tol is None:
        inner_tol = 0.1 if keep_direction else 1e-5
    oi, ii = ctypes.c_int(0), ctypes.c_int(0)
    rel = ctypes.c_double(0)
    times = np.zeros(5, np.float64)
    st = lib().mfe_cg_solve_mixed_ex(A.ctx.h, A.h, b.h, x.h, int(max_outer), int(max_inner),
                                     float(inner_tol), float(outer_tol),
                                     MIXED_KEEP_DIRECTION if keep_direction else 0,
                                     ctypes.byref(oi), ctypes.byref(ii), ctypes.byref(rel),
                                     _ptr(times))
    if st not in (MFE_OK, MFE_BREAKDOWN, MFE_UNSUPPORTED):
        A.ctx.check(st, "cg_solve_mixed")
    return MixedResult(oi.value, ii.value, rel.value, st, float(times[T_TOTAL]))


def matvec_fp32(A: CSRMatrix, x: Vector, y: Vector) -> None:
    """y = A x as the mixed solve's FP32 inner SpMV (result widened to FP64)."""
    A.ctx.check(lib().mfe_matvec_fp32(A.ctx.h, A.h, x.h, y.h), "matvec_fp32")


def time_matvec(A: CSRMatrix, x: Vector, y: Vector, variant: int = 1, reps: int = 20) -> float:
    """Mean SpMV kernel time in ms over `reps` back-to-back launches (HIP events
    on the context's stream); variant 1 is the kernel inside the fast cg_solve,
    variant 2 the FP32 kernel inside cg_solve_mixed, 3 and 4 the same two on
    the CSR kernels whatever A's plan, 6 variant 1 on plain SELL-64 where the
    plan stages x, 13 variant 1 on the packed boundary stream whatever the size."""
    ms = ctypes.c_double(0)
    A.ctx.check(lib().mfe_time_matvec(A.ctx.h, A.h, x.h, y.h, int(variant), int(reps),
                                      ctypes.byref(ms)), "time_matvec")
    return ms.value


def element_gradient(mesh: simple_mesh_description, lam: Vector, utilde: Vector,
                     grad: Vector) -> None:
    """grad[e] = -lambda_e^T K_e(1) utilde_e (the adjoint element gradient)."""
    lam.ctx.check(lib().mfe_element_gradient(lam.ctx.h, _box6(mesh.global_box), lam.h, utilde.h,
                                             grad.h), "element_gradient")


def spmm(A: CSRMatrix, X: Vector, Y: Vector, nrhs: int, tile: int = -1) -> None:
    """Y = A X for row-major n x nrhs block vectors (nrhs 4, 8 or 16); tile -1
    uses the autotuned tile."""
    A.ctx.check(lib().mfe_spmm(A.ctx.h, A.h, X.h, Y.h, int(nrhs), int(tile)), "spmm")


def spmm_tune(A: CSRMatrix, nrhs: int) -> dict:
    """Run the SpMM autotuner on A: {'tile': chosen id, 'ms': [...], 'tiles': [...]};
    ms is +inf for a tile that cannot run on A (a staged tile whose plan does
    not fit)."""
    tiles = spmm_tiles(nrhs)
    ms = np.zeros(max(len(tiles), 1), np.float64)  # one entry per candidate tile
    tile, nt = ctypes.c_int(0), ctypes.c_int(0)
    A.ctx.check(lib().mfe_spmm_tune(A.ctx.h, A.h, int(nrhs), ctypes.byref(tile), _ptr(ms),
                                    ctypes.byref(nt)), "spmm_tune")
    return {"tile": tile.value, "ms": ms[:nt.value].tolist(), "tiles": tiles}


def spmm_select(A: CSRMatrix, nrhs: int, tile: int) -> None:
    """Pin `tile` as A's SpMM tile for nrhs (used by spmm(tile=-1) and
    cg_solve_multi) without timing."""
    A.ctx.check(lib().mfe_spmm_select(A.ctx.h, A.h, int(nrhs), int(tile)), "spmm_select")


def spmm_tiles(nrhs: int) -> list:
    """Shapes of the SpMM candidate tiles for nrhs (index = tile id)."""
    tiles = []
    i = 0
    while True:
        c, u, r, st = (ctypes.c_int(0) for _ in range(4))
        if lib().mfe_spmm_tile_info(int(nrhs), i, ctypes.byref(c), ctypes.byref(u),
                                    ctypes.byref(r), ctypes.byref(st)) != 0:
            return tiles
        kind = ("csr", "staged", "sell", "sell-lines", "box")[st.value]
        tiles.append({"cols_per_lane": c.value, "unroll": u.value, "rows_per_block": r.value,
                      "kind": kind, "staged": kind == "staged"})
        i += 1


@dataclass
class MultiResult:
    iters: np.ndarray
    rel_residual: np.ndarray
    seconds: float


def cg_solve_multi(A: CSRMatrix, B: Vector, X: Vector, nrhs: int, max_iter: int = 5000,
                   rel_tol: float = 1e-10) -> MultiResult:
    """nrhs simultaneous CG solves sharing one SpMM per iteration (row-major
    n x nrhs B and X)."""
    it = np.zeros(nrhs, np.int32)
    rel = np.zeros(nrhs, np.float64)
    sec = ctypes.c_double(0)
    A.ctx.check(lib().mfe_cg_solve_multi(A.ctx.h, A.h, B.h, X.h, int(nrhs), int(max_iter),
                                         float(rel_tol), _ptr(it), _ptr(rel), ctypes.byref(sec)),
                "cg_solve_multi")
    return MultiResult(it, rel, sec.value)


class Batch:
    """Many independent box problems (dims: (nprob, 3) elements per side),
    assembled and solved by FP64 CG together, every launch over all that are not done."""

    def __init__(self, dims, ctx: Context | None = None):
        self.ctx = ctx or default_context()
        d = np.ascontiguousarray(np.asarray(dims, dtype=np.int32).reshape(-1, 3))
        self.dims = d
        self.nprob = d.shape[0]
        h = _vp()
        self.ctx.check(lib().mfe_batch_create(self.ctx.h, int(self.nprob), _ptr(d), ctypes.byref(h)),
                       "batch_create")
        self.h = h
        _live_dependents.add(self)

    def info(self, p: int = -1) -> dict:
        a = np.zeros(6, np.int64)
        self.ctx.check(lib().mfe_batch_info(self.h, int(p), _ptr(a)), "batch_info")
        if p < 0:
            keys = ["problems", "workgroups", "rows", "stored", "nnz"]
        else:
            keys = ["rows", "nnz", "elements", "workgroups", "first_workgroup", "stored"]
        return {k: int(v) for k, v in zip(keys, a)}

    def solve(self, max_iter: int = 5000, rel_tol: float = 1e-10) -> dict:
        iters = np.zeros(self.nprob, np.int32)
        rel = np.zeros(self.nprob, np.float64)
        sec = ctypes.c_double(0)
        st = lib().mfe_batch_solve(self.ctx.h, self.h, int(max_iter), float(rel_tol), _ptr(iters),
                                   _ptr(rel), ctypes.byref(sec))
        if st not in (MFE_OK, MFE_BREAKDOWN):
            self.ctx.check(st, "batch_solve")
        per = np.zeros(self.nprob, np.float64)
        ph = np.zeros((self.nprob, 6), np.float64)
        lib().mfe_batch_timing(self.h, _ptr(per), _ptr(ph))
        return dict(iters=iters, rel_residual=rel, seconds=sec.value, status=st,
                    problem_seconds=per, phase_seconds=ph)

    # phase_seconds' columns: the problem's first workgroup in its own kernels, then the rest
    PHASES = ("elements", "rows", "xp_update", "spmv", "r_update", "outside_first_workgroup")

    def download(self, p: int, matrix: bool = True) -> dict:
        inf = self.info(p)
        n, nnz = inf["rows"], inf["nnz"]
        b = np.empty(n, np.float64)
        x = np.empty(n, np.float64)
        ro = np.empty(n + 1, np.int32) if matrix else None
        cols = np.empty(nnz, np.int32) if matrix else None
        vals = np.empty(nnz, np.float64) if matrix else None
        self.ctx.check(lib().mfe_batch_download(self.ctx.h, self.h, int(p), _ptr(ro), _ptr(cols),
                                                _ptr(vals), _ptr(b), _ptr(x)), "batch_download")
        return dict(row_offsets=ro, cols=cols, vals=vals, b=b, x=x)

    def close(self):
        if getattr(self, "h", None):
            lib().mfe_batch_destroy(self.h)
            self.h = None

    def __del__(self):
        _release(self)


def soln(x: float, y: float, z: float, max_p: int = 300, max_q: int = 300) -> float:
    return lib().mfe_soln(float(x), float(y), float(z), int(max_p), int(max_q))


def verify_solution(mesh: simple_mesh_description, x: Vector, tolerance: float = 0.06,
                    verify_whole_domain: bool = False):
    """Returns (rc, max_abs_err); rc = 0 when within tolerance."""
    e = ctypes.c_double(0)
    rc = lib().mfe_verify_solution_ex(x.ctx.h, _box6(mesh.global_box), x.h, float(tolerance),
                                      int(bool(verify_whole_domain)),
                                      int(getattr(mesh, "hot_face", 1)), ctypes.byref(e))
    if rc not in (0, 1):
        x.ctx.check(rc, "verify_solution")
    return rc, e.value


def build_problem(nx: int, ny: int | None = None, nz: int | None = None, ctx: Context | None = None,
                  kappa: Vector | None = None, source: float = 1.0, hot_face: int = 1):
    """Structure -> assembly -> Dirichlet (u=0 faces, then u=1 face) -> make_local_matrix,
    the order of driver.hpp:159-230.  Returns (mesh, A, b)."""
    ny = nx if ny is None else ny
    nz = ny if nz is None else nz
    mesh = simple_mesh_description([0, nx, 0, ny, 0, nz], hot_face=hot_face)
    A = CSRMatrix(ctx)
    if generate_matrix_structure(mesh, A) != 0:
        raise MfeError(MFE_OOM, "generate_matrix_structure ran out of device memory")
    b = Vector(A.nrows, A.ctx)
    assemble_FE_data(mesh, A, b, kappa=kappa, source=source)
    impose_dirichlet(0.0, A, b, nx + 1, ny + 1, nz + 1, mesh.bc_rows_0)
    impose_dirichlet(1.0, A, b, nx + 1, ny + 1, nz + 1, mesh.bc_rows_1)
    make_local_matrix(A)
    return mesh, A, b
