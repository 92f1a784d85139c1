"""ctypes binding of the C ABI in include/cubie_hip.h.

The shared library ``libcubie_hip.so`` is built in-tree by
:func:`build_runtime` (also run by ``__graft_entry__.build``). Loading it
always imports torch first, so that the HIP runtime torch ships and the one
this library links against are the same loaded copy (they share the
``libamdhip64.so.7`` soname); device buffers allocated through torch are then
valid for our launches. Missing or unloadable native code is an error: there
is no CPU fallback on the product path.
"""

from __future__ import annotations

import ctypes
import os
import subprocess
import threading
from typing import Optional

_HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(_HERE)
ROOT = os.path.dirname(PKG)
LIB_PATH = os.path.join(PKG, "csrc", "libcubie_hip.so")
RUNTIME_SRC = os.path.join(PKG, "csrc", "cubie_hip_runtime.cpp")
NOALLOC_SRC = os.path.join(PKG, "csrc", "cubie_noalloc.hip")
LAYOUT_SRC = os.path.join(PKG, "csrc", "cubie_layout.hip")
INCLUDE_DIR = os.path.join(ROOT, "include")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


class CubieNativeError(RuntimeError):
    pass


class SolveArgs(ctypes.Structure):
    """Mirror of ``cubie_solve_args`` (include/cubie_hip.h)."""

    _fields_ = [
        ("inits", ctypes.c_void_p),
        ("params", ctypes.c_void_p),
        ("driver_coeffs", ctypes.c_void_p),
        ("state_out", ctypes.c_void_p),
        ("observables_out", ctypes.c_void_p),
        ("state_summ_out", ctypes.c_void_p),
        ("obs_summ_out", ctypes.c_void_p),
        ("counters_out", ctypes.c_void_p),
        ("status_out", ctypes.c_void_p),
        ("rtol_per_run", ctypes.c_void_p),
        ("duration_per_run", ctypes.c_void_p),
        ("save_times", ctypes.c_void_p),
        ("work_counter", ctypes.c_void_p),
        ("work_tally", ctypes.c_void_p),
        ("checkpoints", ctypes.c_void_p),
        ("checkpoint_stride", ctypes.c_longlong),
        ("duration", ctypes.c_double),
        ("warmup", ctypes.c_double),
        ("t0", ctypes.c_double),
        ("save_stop", ctypes.c_double),
        ("summary_stop", ctypes.c_double),
        ("n_runs", ctypes.c_longlong),
        ("out_rows", ctypes.c_longlong),
        ("summary_rows", ctypes.c_longlong),
        ("chunk_runs", ctypes.c_int),
        ("reserved", ctypes.c_int),
    ]


class AdjointArgs(ctypes.Structure):
    """Mirror of ``cubie_adjoint_args`` (include/cubie_hip.h)."""
    _fields_ = [
        ("fwd", SolveArgs),
        ("checkpoints", ctypes.c_void_p),
        ("checkpoint_t", ctypes.c_void_p),
        ("tape_dt", ctypes.c_void_p),
        ("tape_flags", ctypes.c_void_p),
        ("tape_info", ctypes.c_void_p),
        ("replay", ctypes.c_void_p),
        ("replay_t", ctypes.c_void_p),
        ("replay_stages", ctypes.c_void_p),
        ("grad_state", ctypes.c_void_p),
        ("grad_state_summ", ctypes.c_void_p),
        ("grad_inits", ctypes.c_void_p),
        ("grad_params", ctypes.c_void_p),
        ("max_steps", ctypes.c_longlong),
        ("max_checkpoints", ctypes.c_longlong),
    ]


class Copy(ctypes.Structure):
    """Mirror of ``cubie_copy`` (include/cubie_hip.h)."""
    _fields_ = [("dst", ctypes.c_void_p), ("src", ctypes.c_void_p), ("bytes", ctypes.c_ulonglong)]


ABI_VERSION = 4


def build_runtime(force: bool = False) -> str:
    """Compile ``libcubie_hip.so`` (host code: hiprtc + module launch)."""
    if not force and os.path.exists(LIB_PATH) and os.path.getmtime(LIB_PATH) >= max(
            os.path.getmtime(RUNTIME_SRC), os.path.getmtime(NOALLOC_SRC),
            os.path.getmtime(LAYOUT_SRC),
            os.path.getmtime(os.path.join(INCLUDE_DIR, "cubie_hip.h"))):
        return LIB_PATH
    tmp = LIB_PATH + ".tmp"
    # host runtime (g++) plus the allocation-free entry point, whose scratch
    # array and clear kernel are device code (hipcc, gfx950)
    obj_rt = LIB_PATH + ".runtime.o"
    obj_na = LIB_PATH + ".noalloc.o"
    obj_ly = LIB_PATH + ".layout.o"
    hip_flags = ["-O3", "-std=c++17", "-c", "-fPIC", "--offload-arch=gfx950",
                 "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", f"-I{INCLUDE_DIR}"]
    steps = [
        ["g++", "-O2", "-std=c++17", "-c", "-fPIC", "-D__HIP_PLATFORM_AMD__",
         f"-I{ROCM}/include", f"-I{INCLUDE_DIR}", RUNTIME_SRC, "-o", obj_rt],
        [os.path.join(ROCM, "bin", "hipcc")] + hip_flags + [NOALLOC_SRC, "-o", obj_na],
        [os.path.join(ROCM, "bin", "hipcc")] + hip_flags + [LAYOUT_SRC, "-o", obj_ly],
        [os.path.join(ROCM, "bin", "hipcc"), "-shared", "-fPIC", obj_rt, obj_na, obj_ly, "-o", tmp,
         f"-L{ROCM}/lib", "-lhiprtc", "-lamdhip64", f"-Wl,-rpath,{ROCM}/lib"],
    ]
    try:
        for cmd in steps:
            res = subprocess.run(cmd, capture_output=True, text=True)
            if res.returncode != 0:
                raise CubieNativeError("building libcubie_hip.so failed:\n" + " ".join(cmd) +
                                       "\n" + res.stderr)
    finally:
        for o in (obj_rt, obj_na, obj_ly):
            if os.path.exists(o):
                os.remove(o)
    os.replace(tmp, LIB_PATH)
    return LIB_PATH


_lib: Optional[ctypes.CDLL] = None
_lock = threading.Lock()


def lib() -> ctypes.CDLL:
    global _lib
    with _lock:
        if _lib is not None:
            return _lib
        import torch  # noqa: F401  (share torch's HIP runtime, see module doc)
        if not os.path.exists(LIB_PATH):
            raise CubieNativeError(
                f"{LIB_PATH} is missing; build it with cubie_amd.runtime.native.build_runtime() "
                "or __graft_entry__.build()")
        L = ctypes.CDLL(LIB_PATH)
        L.cubie_hip_abi_version.restype = ctypes.c_int
        L.cubie_hip_last_error.argtypes = [ctypes.c_char_p, ctypes.c_size_t]
        L.cubie_hip_last_error.restype = ctypes.c_int
        L.cubie_hip_compile.argtypes = [ctypes.c_char_p, ctypes.c_char_p, ctypes.c_char_p,
                                        ctypes.POINTER(ctypes.c_void_p),
                                        ctypes.POINTER(ctypes.c_size_t),
                                        ctypes.c_char_p, ctypes.c_size_t]
        L.cubie_hip_compile.restype = ctypes.c_int
        L.cubie_hip_free_code.argtypes = [ctypes.c_void_p]
        L.cubie_hip_load.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_char_p,
                                     ctypes.POINTER(ctypes.c_void_p)]
        L.cubie_hip_load.restype = ctypes.c_int
        L.cubie_hip_unload.argtypes = [ctypes.c_void_p]
        L.cubie_hip_unload.restype = ctypes.c_int
        L.cubie_hip_kernel_info.argtypes = [ctypes.c_void_p] + [ctypes.POINTER(ctypes.c_int)] * 4
        L.cubie_hip_kernel_info.restype = ctypes.c_int
        L.cubie_hip_launch.argtypes = [ctypes.c_void_p, ctypes.POINTER(SolveArgs), ctypes.c_uint,
                                       ctypes.c_uint, ctypes.c_uint, ctypes.c_void_p]
        L.cubie_hip_launch.restype = ctypes.c_int
        L.cubie_hip_launch_timed.argtypes = [ctypes.c_void_p, ctypes.POINTER(SolveArgs),
                                             ctypes.c_uint, ctypes.c_uint, ctypes.c_uint,
                                             ctypes.c_void_p, ctypes.POINTER(ctypes.c_float)]
        L.cubie_hip_launch_timed.restype = ctypes.c_int
        L.cubie_hip_launch_adjoint.argtypes = [ctypes.c_void_p, ctypes.POINTER(AdjointArgs),
                                               ctypes.c_uint, ctypes.c_uint, ctypes.c_uint,
                                               ctypes.c_void_p]
        L.cubie_hip_launch_adjoint.restype = ctypes.c_int
        L.cubie_hip_launch_adjoint_timed.argtypes = [ctypes.c_void_p, ctypes.POINTER(AdjointArgs),
                                                     ctypes.c_uint, ctypes.c_uint, ctypes.c_uint,
                                                     ctypes.c_void_p, ctypes.POINTER(ctypes.c_float)]
        L.cubie_hip_launch_adjoint_timed.restype = ctypes.c_int
        L.cubie_hip_graph_create.argtypes = [ctypes.c_void_p, ctypes.POINTER(SolveArgs),
                                             ctypes.c_uint, ctypes.c_uint,
                                             ctypes.POINTER(Copy), ctypes.c_int,
                                             ctypes.POINTER(Copy), ctypes.c_int,
                                             ctypes.POINTER(ctypes.c_void_p)]
        L.cubie_hip_graph_create.restype = ctypes.c_int
        L.cubie_hip_graph_launch.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
        L.cubie_hip_graph_launch.restype = ctypes.c_int
        L.cubie_hip_graph_destroy.argtypes = [ctypes.c_void_p]
        L.cubie_hip_graph_destroy.restype = ctypes.c_int
        L.cubie_hip_runs_to_rows.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_longlong,
                                             ctypes.c_longlong, ctypes.c_int, ctypes.c_void_p]
        L.cubie_hip_runs_to_rows.restype = ctypes.c_int
        L.cubie_hip_morton_keys.argtypes = [
            ctypes.c_void_p, ctypes.c_longlong, ctypes.c_int, ctypes.c_int,
            ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_double),
            ctypes.POINTER(ctypes.c_double), ctypes.c_void_p, ctypes.c_void_p]
        L.cubie_hip_morton_keys.restype = ctypes.c_int
        if L.cubie_hip_abi_version() != ABI_VERSION:
            raise CubieNativeError("libcubie_hip.so ABI version mismatch; rebuild it")
        _lib = L
        return L


def last_error() -> str:
    buf = ctypes.create_string_buffer(8192)
    lib().cubie_hip_last_error(buf, len(buf))
    return buf.value.decode(errors="replace")


def check(rc: int, what: str) -> None:
    if rc != 0:
        raise CubieNativeError(f"{what} failed ({rc}): {last_error()}")


def runs_to_rows(src, dst, n_runs: int, inner: int, stream) -> None:
    """Enqueue the transpose of a run-major (n_runs, inner) device tensor
    into dst, an (inner, n_runs) device tensor of the same element size."""
    esize = src.element_size()
    if (src.numel() != n_runs * inner or dst.numel() != n_runs * inner
            or dst.element_size() != esize or not src.is_contiguous() or not dst.is_contiguous()):
        raise CubieNativeError("runs_to_rows: src and dst must be contiguous with "
                               "n_runs x inner elements of one size")
    check(lib().cubie_hip_runs_to_rows(ctypes.c_void_p(src.data_ptr()),
                                       ctypes.c_void_p(dst.data_ptr()), n_runs, inner, esize,
                                       ctypes.c_void_p(stream)), "cubie_hip_runs_to_rows")


def morton_keys(columns, keys, index, lo, span, bits: int, stream) -> None:
    """Enqueue the Morton keys (include/cubie_order.h) of the rows ``index``
    of a float64 (columns, n_runs) device tensor into an int64 one."""
    import torch
    n_cols, n_runs = len(index), int(columns.shape[1])
    if (columns.dtype != torch.float64 or keys.dtype != torch.int64 or keys.numel() != n_runs
            or not columns.is_contiguous() or not keys.is_contiguous()
            or columns.device != keys.device or max(index) >= columns.shape[0]):
        raise CubieNativeError("morton_keys: a contiguous float64 (columns, n_runs) matrix and "
                               "n_runs int64 keys on one device are needed")
    check(lib().cubie_hip_morton_keys(
        ctypes.c_void_p(columns.data_ptr()), n_runs, n_cols, bits, (ctypes.c_int * n_cols)(*index),
        (ctypes.c_double * n_cols)(*lo), (ctypes.c_double * n_cols)(*span),
        ctypes.c_void_p(keys.data_ptr()), ctypes.c_void_p(stream)), "cubie_hip_morton_keys")


def compile_source(source: str, options, name: str = "cubie_kernel.hip") -> bytes:
    L = lib()
    code = ctypes.c_void_p()
    size = ctypes.c_size_t()
    log = ctypes.create_string_buffer(1 << 16)
    rc = L.cubie_hip_compile(source.encode(), name.encode(), "\n".join(options).encode(),
                             ctypes.byref(code), ctypes.byref(size), log, len(log))
    if rc != 0:
        raise CubieNativeError("hiprtc compilation failed:\n" + last_error())
    try:
        return ctypes.string_at(code, size.value)
    finally:
        L.cubie_hip_free_code(code)


class Module:
    """A loaded code object with one resolved kernel."""

    def __init__(self, code: bytes, kernel_name: str):
        L = lib()
        self._code = code  # keep alive
        handle = ctypes.c_void_p()
        check(L.cubie_hip_load(code, len(code), kernel_name.encode(), ctypes.byref(handle)),
              "cubie_hip_load")
        self.handle = handle
        self.kernel_name = kernel_name

    def info(self):
        regs, lds, priv, maxt = (ctypes.c_int() for _ in range(4))
        check(lib().cubie_hip_kernel_info(self.handle, ctypes.byref(regs), ctypes.byref(lds),
                                          ctypes.byref(priv), ctypes.byref(maxt)), "kernel_info")
        return {"vgprs": regs.value, "lds_bytes": lds.value, "scratch_bytes": priv.value,
                "max_threads": maxt.value}

    def launch(self, args: SolveArgs, grid: int, block: int, stream: int = 0, lds: int = 0) -> None:
        check(lib().cubie_hip_launch(self.handle, ctypes.byref(args), grid, block, lds,
                                     ctypes.c_void_p(stream)), "cubie_hip_launch")

    def launch_timed(self, args: SolveArgs, grid: int, block: int, stream: int = 0, lds: int = 0) -> float:
        ms = ctypes.c_float()
        check(lib().cubie_hip_launch_timed(self.handle, ctypes.byref(args), grid, block, lds,
                                           ctypes.c_void_p(stream), ctypes.byref(ms)),
              "cubie_hip_launch_timed")
        return float(ms.value)

    def launch_adjoint(self, args: AdjointArgs, grid: int, block: int, stream: int = 0,
                       lds: int = 0, timed: bool = False):
        """Launch cubie_integrate_record / cubie_adjoint; returns the kernel
        time in ms when ``timed``."""
        if timed:
            ms = ctypes.c_float()
            check(lib().cubie_hip_launch_adjoint_timed(self.handle, ctypes.byref(args), grid, block,
                                                       lds, ctypes.c_void_p(stream),
                                                       ctypes.byref(ms)),
                  "cubie_hip_launch_adjoint_timed")
            return float(ms.value)
        check(lib().cubie_hip_launch_adjoint(self.handle, ctypes.byref(args), grid, block, lds,
                                             ctypes.c_void_p(stream)), "cubie_hip_launch_adjoint")
        return None

    def __del__(self):
        try:
            if getattr(self, "handle", None) is not None and _lib is not None:
                _lib.cubie_hip_unload(self.handle)
        except Exception:
            pass


class ChunkGraph:
    """One captured chunk sequence (copies before, the kernel, copies after)
    of ``Module``; replay with :meth:`launch`. Pointers are raw device or
    pinned-host addresses; the caller keeps those buffers alive."""

    def __init__(self, module: Module, args: SolveArgs, grid: int, block: int,
                 before=(), after=()):
        def copies(lst):
            arr = (Copy * max(len(lst), 1))()
            for i, (dst, src, nbytes) in enumerate(lst):
                arr[i].dst, arr[i].src, arr[i].bytes = dst, src, nbytes
            return arr
        b, a = copies(list(before)), copies(list(after))
        handle = ctypes.c_void_p()
        check(lib().cubie_hip_graph_create(module.handle, ctypes.byref(args), grid, block,
                                           b, len(before), a, len(after), ctypes.byref(handle)),
              "cubie_hip_graph_create")
        self.handle = handle
        self.module = module

    def launch(self, stream: int = 0) -> None:
        check(lib().cubie_hip_graph_launch(self.handle, ctypes.c_void_p(stream)),
              "cubie_hip_graph_launch")

    def __del__(self):
        try:
            if getattr(self, "handle", None) is not None and _lib is not None:
                _lib.cubie_hip_graph_destroy(self.handle)
        except Exception:
            pass
