"""ctypes binding of libapcost.so (see include/apcost.h for the contract).

There is no CPU fallback: if the library has not been built, or a launch fails,
a RuntimeError is raised.
"""

from __future__ import annotations

import ctypes
import os

import numpy as np

from ._build import LIB_PATH, TORCH_EXT_PATH

APC_ABI_VERSION = 3  # include/apcost.h: the interface this binding's structs and limits mirror
APC_MAX_RANK = 8
APC_MAX_MESH = 4
APC_MAX_DTYPES = 8
APC_TILE_MAX_COLS = 64
APC_TILE_MAX_ROWS = 64
APC_TILE_MAX_DUPS = 32
APC_PACKED_MAX_DUPS = 16
APC_SWEEP_MAX_WORKGROUPS = 224

EDGE_GRAD_RESCALE = 1
EDGE_NO_PRODUCER = 2


class ApcParams(ctypes.Structure):
    _fields_ = [
        ("mesh_ndim", ctypes.c_int32),
        ("mesh_size", ctypes.c_int32 * APC_MAX_MESH),
        ("bw", ctypes.c_double * APC_MAX_MESH),
        ("lat", ctypes.c_double * APC_MAX_MESH),
        ("base_latency", ctypes.c_double),
        ("a2a_scale", ctypes.c_double),
        ("hbm_bw", ctypes.c_double),
        ("rw_eff", ctypes.c_double),
        ("launch_floor", ctypes.c_double),
        ("compute_eff", ctypes.c_double),
        ("rescale", ctypes.c_double),
        ("gpu_flops", ctypes.c_double * APC_MAX_DTYPES),
        ("transition_scale", ctypes.c_int32),
        ("inv_bw", ctypes.c_double * APC_MAX_MESH),
        ("inv_mesh", ctypes.c_double * APC_MAX_MESH),
        ("inv_hbm_bw", ctypes.c_double),
        ("inv_rw_eff", ctypes.c_double),
        ("inv_compute_eff", ctypes.c_double),
        ("inv_gpu_flops", ctypes.c_double * APC_MAX_DTYPES),
    ]


class ApcTile(ctypes.Structure):
    _fields_ = [
        ("edge", ctypes.c_int32), ("row_begin", ctypes.c_int32), ("col_begin", ctypes.c_int32),
        ("counts", ctypes.c_int32),
        ("src_begin", ctypes.c_int32), ("n_src", ctypes.c_int32), ("tgt_begin", ctypes.c_int32),
        ("flags", ctypes.c_int32), ("strat_begin", ctypes.c_int32), ("tensor", ctypes.c_int32),
        ("entry_begin", ctypes.c_int64), ("pt_begin", ctypes.c_int64),
        ("dup_begin", ctypes.c_int32), ("dup_count", ctypes.c_int32),
    ]


class ApcRowMinima(ctypes.Structure):
    _fields_ = [
        ("edge_row_begin", ctypes.c_void_p), ("dup_row_begin", ctypes.c_void_p),
        ("row_min", ctypes.c_void_p), ("row_argmin", ctypes.c_void_p),
    ]


EXPORTS = (
    "apc_version",
    "apc_last_error",
    "apc_validate_tables_host",
    "apc_tensor_tables",
    "apc_spec_tables",
    "apc_compute_costs",
    "apc_input_tables",
    "apc_redistribute_tables",
    "apc_build_tables",
    "apc_redistribute_tables_row_min",
    "apc_build_tables_row_min",
    "apc_segmented_min",
    "apc_segmented_min_copies",
    "apc_strategy_bounds",
    "apc_greedy_strategies",
    "apc_edge_rows",
    "apc_report_inputs",
    "apc_copy_arrays",
    "apc_check_tables",
    "apc_edge_classes",
    "apc_pack_tiles",
    "apc_cost_objective",
    "apc_validate_row_minima_host",
    "apc_diffusion_sweeps",
    "apc_sweep_plan_host",
    "apc_diffusion_sweeps_resident",
    "apc_redistribute_tables_static",
    "apc_strategy_inputs",
    "apc_validate_packed_tiles_host",
    "apc_pack_tiles_host",
    "apc_edge_classes_host",
    "apc_count_tiles_host",
    "apc_fill_tiles_host",
    "apc_order_tiles_host",
    "apc_tile_records_host",
    "apc_validate_tiling_host",
    "apc_label_incidence_host",
    "apc_label_minima_host",
    "apc_round_labels_host",
    "apc_refine_labels_host",
    "apc_prune_masks_host",
    "apc_build_tables_packed",
    "apc_build_tables_packed_small",
    "apc_keep_next_launch",
    "apc_run_kept",
    "apc_calibrate_launch",
    "apc_calibrate_fill",
)

_lib = None


def library_path() -> str:
    return LIB_PATH


def lib() -> ctypes.CDLL:
    """Loads the built library; raises if it is missing (build it with
    ``python -m autoparallel_amd._build`` or ``__graft_entry__.build()``)."""
    global _lib
    if _lib is None:
        # torch ships its own HIP runtime; it must be in the process before this library
        # is mapped so that both resolve to the same runtime (streams and device pointers
        # are shared between them).
        import torch  # noqa: F401

        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: the HIP library has not been built "
                "(run `python -m autoparallel_amd._build`). There is no CPU fallback."
            )
        l = ctypes.CDLL(LIB_PATH, mode=ctypes.RTLD_GLOBAL)
        for name in EXPORTS:
            if not hasattr(l, name):
                raise RuntimeError(f"{LIB_PATH} does not export {name}")
        l.apc_last_error.restype = ctypes.c_char_p
        l.apc_version.restype = ctypes.c_int
        if int(l.apc_version()) != APC_ABI_VERSION:
            raise RuntimeError(f"{LIB_PATH} implements interface version {int(l.apc_version())}, this binding "
                               f"mirrors version {APC_ABI_VERSION} of include/apcost.h: rebuild the library")
        for name in EXPORTS:
            if name != "apc_last_error":
                getattr(l, name).restype = ctypes.c_int
        _lib = l
    return _lib


_runners = None
_ops = None


def torch_ops():
    """The ``apcost`` operator namespace of the torch layer (csrc/apcost_torch.cpp): operators
    over torch tensors on the HIP device, bound to the same library.  Raises if it has not
    been built."""
    global _ops
    if _ops is None:
        import torch

        lib()  # the C-ABI library first: the extension resolves its symbols against it
        if not os.path.exists(TORCH_EXT_PATH):
            raise RuntimeError(
                f"{TORCH_EXT_PATH} is missing: the torch layer has not been built "
                "(run `python -m autoparallel_amd._build`). There is no CPU fallback."
            )
        torch.ops.load_library(TORCH_EXT_PATH)
        _ops = torch.ops.apcost
        if int(_ops.abi_version()) != APC_ABI_VERSION or int(_ops.library_abi_version()) != APC_ABI_VERSION:
            raise RuntimeError(f"the torch layer was compiled against interface version {int(_ops.abi_version())} and "
                               f"sees a library of version {int(_ops.library_abi_version())}; this binding mirrors "
                               f"version {APC_ABI_VERSION}: rebuild both")
    return _ops


def bound_runners():
    """(run, run_on): ``BoundLaunch.run`` / ``run_on`` as functions of the object's ``handle()`` (``run_on``: and of a stream's
    handle and torch's number of it, ``stream_id``), 0 when the launch is enqueued (else ``bound_error()``).  The caller keeps the object."""
    global _runners
    if _runners is None:
        torch_ops()
        ext = ctypes.CDLL(TORCH_EXT_PATH)  # (the library that is loaded already)
        run, run_on = ext.apcost_run_bound, ext.apcost_run_bound_on
        run.argtypes, run_on.argtypes = (ctypes.c_void_p,), (ctypes.c_void_p, ctypes.c_int64, ctypes.c_int64)
        ext.apcost_run_error.restype = ctypes.c_char_p
        _runners = run, run_on, ext.apcost_run_error
    return _runners[:2]


def bound_error() -> RuntimeError:
    """Why the last launch of this thread through ``bound_runners`` failed."""
    return RuntimeError(_runners[2]().decode(errors="replace"))


def params_tensor(c_params: "ApcParams"):
    """``struct apc_params`` as the CPU uint8 tensor the operators take."""
    import torch

    return torch.frombuffer(bytearray(bytes(c_params)), dtype=torch.uint8)


def check(rc: int, what: str) -> None:
    if rc != 0:
        msg = lib().apc_last_error().decode("utf-8", "replace")
        raise RuntimeError(f"{what} failed ({rc}): {msg}")


_AT = (ctypes.c_char * 0).from_buffer  # (an object at the buffer's address, which holds the buffer: 0.2 us; ``a.ctypes.data`` 1.1)


def argument(a):
    """A host entry point's argument: what is one already, a contiguous numpy array as its address, ``None`` as NULL, an
    integer as int64, a float as double, a ctypes structure by reference."""
    if type(a) is np.ndarray:
        flags = a.flags
        if not flags.c_contiguous:
            raise ValueError("host entry points take contiguous arrays")
        return _AT(a) if flags.writeable else ctypes.c_void_p(a.ctypes.data)
    if a is None:
        return ctypes.c_void_p(None)
    if isinstance(a, ctypes.c_void_p):
        return a
    if isinstance(a, int):
        return ctypes.c_int64(a)
    if isinstance(a, float):
        return ctypes.c_double(a)
    if isinstance(a, ctypes.Structure):
        return ctypes.byref(a)
    raise TypeError(f"host entry points take contiguous arrays and plain numbers: {type(a).__name__}")


def host_call(name: str, *args) -> None:
    """Calls a host entry point of the library; raises RuntimeError with its message on an error."""
    check(getattr(lib(), name)(*[argument(a) for a in args]), name)


def host_counts(name: str, *args) -> tuple:
    """A host entry point whose last two arguments are ``int64_t *`` results: returns them."""
    first, second = ctypes.c_int64(), ctypes.c_int64()
    check(getattr(lib(), name)(*[argument(a) for a in args], ctypes.byref(first), ctypes.byref(second)), name)
    return first.value, second.value


def vp(ptr) -> ctypes.c_void_p:
    """int / None -> void*"""
    return ctypes.c_void_p(ptr if ptr else None)
