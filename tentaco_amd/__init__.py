"""Python host mirror of the tentaco C ABI (include/tentaco.h).

The product is ``libtentaco.so`` (HIP for gfx950, built in-tree by
``tentaco_amd/Makefile``); this module only binds it with ctypes, so callers in
Python see the same operator interface as C/C++ callers of the reference's
``gpu_kernels.cuh``: ``mttkrp`` / ``ttv`` take a CSF tensor and factor
matrices (host arrays) and return the output, ``DeviceCsf`` is the
device-resident handle for repeated calls. There is no CPU fallback: if the
library is missing or no gfx950 device is present, calls raise.
"""

from __future__ import annotations

import ctypes
import os
from ctypes import POINTER, c_double, c_float, c_int, c_int32, c_int64, c_size_t, c_uint64, c_void_p
from dataclasses import dataclass, field
from typing import List, Optional, Sequence

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libtentaco.so")

VARIANT_AUTO = -1
VARIANT_DEFAULT = -2
NUM_FEATURES = 24
TUNED_NONE, TUNED_SWEEP, TUNED_SELECTOR, TUNED_SET, TUNED_SELECTOR_TIMED = 0, 1, 2, 3, 4

OK, EINVAL, EHIP, ENOMEM, EUNSUPPORTED, ENOGPU = 0, 1, 2, 3, 4, 5


class TentacoError(RuntimeError):
    """A tentaco entry point returned a nonzero status."""

    def __init__(self, code: int, msg: str):
        super().__init__(f"tentaco error {code}: {msg}")
        self.code = code


class TacoTensor(ctypes.Structure):
    """ctypes mirror of ``taco_tensor_t`` (include/taco_tensor_t.h, 64 bytes)."""

    _fields_ = [
        ("order", c_int32),
        ("dimensions", POINTER(c_int32)),
        ("csize", c_int32),
        ("mode_ordering", POINTER(c_int32)),
        ("mode_types", POINTER(c_int)),
        ("indices", POINTER(POINTER(POINTER(c_int32)))),
        ("vals", POINTER(c_float)),
        ("vals_size", c_int32),
    ]


class SynthParams(ctypes.Structure):
    """ctypes mirror of ``tentaco_synth_params``."""

    _fields_ = [
        ("order", c_int),
        ("dims", c_int32 * 5),
        ("nnz", c_int64),
        ("slice_s", c_double),
        ("fanout_s", c_double),
        ("mid_mu", c_double),
        ("mid_sigma", c_double),
        ("leaf_mu", c_double),
        ("leaf_sigma", c_double),
        ("leaf_cap", c_int32),
        ("seed", c_uint64),
    ]


_lib = None


def lib() -> ctypes.CDLL:
    """Load libtentaco.so once; raise if it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise TentacoError(ENOGPU, f"{LIB_PATH} not built (run __graft_entry__.build())")
    L = ctypes.CDLL(LIB_PATH)
    P = POINTER(TacoTensor)
    sigs = {
        "tentaco_last_error": (ctypes.c_char_p, []),
        "tentaco_version": (c_int, []),
        "tentaco_device_check": (c_int, []),
        "tentaco_mttkrp3": (c_int, [P, P, P, P]),
        "tentaco_mttkrp4": (c_int, [P, P, P, P, P]),
        "tentaco_mttkrp5": (c_int, [P, P, P, P, P, P]),
        "tentaco_mttkrp": (c_int, [c_int, P, P, POINTER(P), c_int]),
        "tentaco_ttv": (c_int, [P, P, P]),
        "tentaco_ttv_n": (c_int, [c_int, P, P, P]),
        "get_gpu_timer_result": (c_float, []),
        "mttkrp_gpu_taco": (None, [P, P, P, P]),
        "ttv_csf_gpu_taco": (None, [P, P, P]),
        "tentaco_num_variants": (c_int, []),
        "tentaco_variant_name": (ctypes.c_char_p, [c_int]),
        "tentaco_variant_params": (c_int, [c_int, POINTER(c_int), POINTER(c_int), POINTER(c_int)]),
        "tentaco_default_variant": (c_int, []),
        "tentaco_variant_fits": (c_int, [c_int, c_int, c_int]),
        "tentaco_csf_resolve_variant": (c_int, [c_void_p, c_int, c_int, POINTER(c_int)]),
        "tentaco_csf_upload": (c_int, [P, c_int, POINTER(c_void_p)]),
        "tentaco_csf_free": (c_int, [c_void_p]),
        "tentaco_csf_info": (c_int, [c_void_p, POINTER(c_int), POINTER(c_int64), POINTER(c_int32)]),
        "tentaco_csf_reserve": (c_int, [c_void_p, c_int, c_int]),
        "tentaco_csf_reserve_rows": (c_int, [c_void_p, c_int, c_int, c_int32]),
        "tentaco_csf_reserve_level": (c_int, [c_void_p, c_int]),
        "tentaco_mttkrp_dev_noalloc": (c_int, [c_void_p, c_int, POINTER(c_void_p), c_void_p, c_int32, c_int,
                                               c_void_p]),
        "tentaco_legacy_variant": (c_int, [ctypes.c_char_p, c_int, c_int, POINTER(c_int)]),
        "tentaco_mttkrp_dev": (c_int, [c_void_p, c_int, POINTER(c_void_p), c_void_p, c_int32, c_int, c_void_p]),
        "tentaco_ttv_dev": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p]),
        "tentaco_csf_set_ttv_bands": (c_int, [c_void_p, c_int]),
        "tentaco_csf_ttv_layout": (c_int, [c_void_p, POINTER(c_int), POINTER(ctypes.c_int64)]),
        "tentaco_mttkrp_dev_repeat": (c_int, [c_void_p, c_int, POINTER(c_void_p), c_void_p, c_int32, c_int,
                                              c_void_p, c_int]),
        "tentaco_mttkrp_level_dev": (c_int, [c_void_p, c_int, c_int, POINTER(c_void_p), c_void_p, c_int32,
                                             c_void_p]),
        "tentaco_csf_autotune": (c_int, [c_void_p, c_int, POINTER(c_void_p), c_void_p, c_int32, c_int,
                                         c_void_p, POINTER(c_int), POINTER(c_float)]),
        "tentaco_csf_set_tuned": (c_int, [c_void_p, c_int, c_int]),
        "tentaco_csf_sweep": (c_int, [c_void_p, c_int, POINTER(c_void_p), c_void_p, c_int32, c_int,
                                      c_float, c_void_p, POINTER(c_float)]),
        "tentaco_csf_tuned": (c_int, [c_void_p, c_int, POINTER(c_int), POINTER(c_int)]),
        "tentaco_csf_features": (c_int, [c_void_p, c_int, POINTER(c_float)]),
        "tentaco_csf_set_selector": (c_int, [c_void_p, c_void_p, c_float]),
        "tentaco_csf_set_selector_fallback": (c_int, [c_void_p, c_int]),
        "tentaco_cpd_create": (c_int, [POINTER(c_void_p), POINTER(c_int), c_int, c_int, ctypes.c_uint64,
                                       POINTER(c_void_p)]),
        "tentaco_cpd_tune": (c_int, [c_void_p, c_int]),
        "tentaco_cpd_iterate": (c_int, [c_void_p, c_int, c_int, c_void_p, POINTER(ctypes.c_double)]),
        "tentaco_cpd_factor": (c_int, [c_void_p, c_int, c_int, POINTER(c_float), POINTER(c_float)]),
        "tentaco_cpd_set_factor": (c_int, [c_void_p, c_int, c_int, POINTER(c_float)]),
        "tentaco_cpd_free": (c_int, [c_void_p]),
        "tentaco_mlp_num_params": (c_int64, [c_int]),
        "tentaco_mlp_create": (c_int, [c_int, ctypes.c_uint64, POINTER(c_void_p)]),
        "tentaco_mlp_free": (c_int, [c_void_p]),
        "tentaco_mlp_set_scaling": (c_int, [c_void_p, POINTER(c_float), POINTER(c_float), c_float, c_float]),
        "tentaco_mlp_get_scaling": (c_int, [c_void_p, POINTER(c_float), POINTER(c_float), POINTER(c_float),
                                            POINTER(c_float)]),
        "tentaco_mlp_get_params": (c_int, [c_void_p, POINTER(c_float), c_int64]),
        "tentaco_mlp_set_params": (c_int, [c_void_p, POINTER(c_float), c_int64]),
        "tentaco_mlp_get_grads": (c_int, [c_void_p, POINTER(c_float), c_int64]),
        "tentaco_mlp_forward": (c_int, [c_void_p, c_void_p, c_int, c_void_p, c_void_p]),
        "tentaco_mlp_loss_grad": (c_int, [c_void_p, POINTER(c_float), POINTER(c_float), POINTER(c_float),
                                          c_int, POINTER(c_float)]),
        "tentaco_mlp_adam": (c_int, [c_void_p, c_float, c_float, c_float, c_float]),
        "tentaco_mlp_train": (c_int, [c_void_p, POINTER(c_float), POINTER(c_float), POINTER(c_float), c_int,
                                      c_int, c_int, c_float, ctypes.c_uint64, POINTER(c_float)]),
        "tentaco_mlp_select": (c_int, [c_void_p, c_int, c_int, POINTER(c_float), POINTER(c_int),
                                       POINTER(c_float), POINTER(c_float)]),
        "tentaco_select_variant": (c_int, [c_void_p, POINTER(c_float), c_int, c_int, POINTER(c_int)]),
        "tentaco_batch_create": (c_int, [POINTER(c_void_p), c_int, c_int, POINTER(c_void_p)]),
        "tentaco_batch_set_operands": (c_int, [c_void_p, POINTER(c_void_p), POINTER(c_void_p), POINTER(c_int32)]),
        "tentaco_batch_configure": (c_int, [c_void_p, c_int, c_int, c_int]),
        "tentaco_batch_configure_order": (c_int, [c_void_p, c_int, c_int, c_int, c_int, c_int]),
        "tentaco_batch_get_config": (c_int, [c_void_p, c_int, POINTER(c_int), POINTER(c_int), POINTER(c_int), POINTER(c_int)]),
        "tentaco_batch_run": (c_int, [c_void_p, c_void_p]),
        "tentaco_batch_capture": (c_int, [c_void_p, c_void_p]),
        "tentaco_batch_launch": (c_int, [c_void_p, c_void_p]),
        "tentaco_batch_items": (c_int, [c_void_p, POINTER(c_int32), POINTER(c_int32), POINTER(c_int32)]),
        "tentaco_batch_autotune": (c_int, [c_void_p, c_int, c_void_p, POINTER(c_int), POINTER(c_int), POINTER(c_int), POINTER(c_float)]),
        "tentaco_batch_free": (c_int, [c_void_p]),
        "tentaco_batch_set_schedule": (c_int, [c_void_p, c_int]),
        "tentaco_batch_get_schedule": (c_int, [c_void_p, POINTER(c_int)]),
        "tentaco_batch_set_output_mode": (c_int, [c_void_p, c_int]),
        "tentaco_batch_get_output_mode": (c_int, [c_void_p, POINTER(c_int)]),
        "tentaco_host_alloc": (c_int, [POINTER(c_void_p), c_size_t]),
        "tentaco_host_free": (c_int, [c_void_p]),
        "tentaco_stream_create": (c_int, [POINTER(c_void_p)]),
        "tentaco_stream_destroy": (c_int, [c_void_p]),
        "tentaco_stream_synchronize": (c_int, [c_void_p]),
        "tentaco_csf_upload_async": (c_int, [P, c_int, c_void_p, POINTER(c_void_p)]),
        "tentaco_mttkrp_host_async": (c_int, [c_void_p, c_int, POINTER(P), P, c_int, c_void_p]),
        "tentaco_dev_malloc": (c_int, [POINTER(c_void_p), c_size_t]),
        "tentaco_dev_free": (c_int, [c_void_p]),
        "tentaco_memcpy_h2d": (c_int, [c_void_p, c_void_p, c_size_t]),
        "tentaco_memcpy_d2h": (c_int, [c_void_p, c_void_p, c_size_t]),
        "tentaco_dev_synchronize": (c_int, []),
        "tentaco_timer_start": (c_int, [c_void_p]),
        "tentaco_flush_cache": (c_int, [c_void_p]),
        "tentaco_timer_stop": (c_int, [c_void_p, POINTER(c_float)]),
        "tentaco_ktimer_start": (c_int, []),
        "tentaco_ktimer_stop": (c_int, [POINTER(ctypes.c_double), POINTER(c_int), ctypes.c_char_p, c_int]),
        "tentaco_dev_copy": (c_int, [c_void_p, c_void_p, ctypes.c_size_t, c_void_p]),
        "tentaco_dev_gather": (c_int, [c_void_p, c_int64, c_int, c_int32, c_int, c_void_p, c_void_p,
                                       POINTER(ctypes.c_double)]),
        "tentaco_tns_read": (c_int, [ctypes.c_char_p, POINTER(c_int32), POINTER(c_int), POINTER(c_void_p),
                                     POINTER(c_int), POINTER(c_int)]),
        "tentaco_coo_to_csf": (c_int, [c_int, POINTER(c_int32), c_int64, POINTER(c_int32), POINTER(c_float), POINTER(c_void_p)]),
        "tentaco_synth_csf": (c_int, [POINTER(SynthParams), POINTER(c_void_p)]),
        "tentaco_host_csf_view": (P, [c_void_p]),
        "tentaco_csf_reorder": (c_int, [P, c_int, POINTER(c_int), POINTER(c_void_p)]),
        "tentaco_host_csf_nodes": (c_int64, [c_void_p, c_int]),
        "tentaco_host_csf_free": (c_int, [c_void_p]),
    }
    for name, (res, args) in sigs.items():
        fn = getattr(L, name)
        fn.restype = res
        fn.argtypes = args
    _lib = L
    return L


def _check(rc: int) -> None:
    if rc != OK:
        msg = lib().tentaco_last_error()
        raise TentacoError(rc, msg.decode() if msg else "")


def device_check() -> None:
    """Raise unless a gfx950 device is usable."""
    _check(lib().tentaco_device_check())


# ---------------------------------------------------------------------------
# host CSF
@dataclass
class Csf:
    """Host CSF tensor: level 0 is the root (pos[0] = [0, n0], crd[0]),
    levels 1..order-1 hold pos/crd, vals the nonzero values (int32/FP32)."""

    order: int
    dims: tuple
    pos: List[np.ndarray]
    crd: List[np.ndarray]
    vals: np.ndarray
    _owner: object = field(default=None, repr=False, compare=False)

    @property
    def nnz(self) -> int:
        return int(self.vals.shape[0])

    def nodes(self, m: int) -> int:
        return int(self.crd[m].shape[0])

    def as_taco(self):
        """taco_tensor_t view of this CSF (returns the struct and a keep-alive)."""
        dims = np.ascontiguousarray(self.dims, dtype=np.int32)
        keep = [dims]
        lvl = (POINTER(c_int32) * 2 * self.order)()
        ptrs = (POINTER(POINTER(c_int32)) * self.order)()
        for m in range(self.order):
            p = np.ascontiguousarray(self.pos[m], dtype=np.int32)
            c = np.ascontiguousarray(self.crd[m], dtype=np.int32)
            keep += [p, c]
            lvl[m][0] = p.ctypes.data_as(POINTER(c_int32))
            lvl[m][1] = c.ctypes.data_as(POINTER(c_int32))
            ptrs[m] = ctypes.cast(lvl[m], POINTER(POINTER(c_int32)))
        vals = np.ascontiguousarray(self.vals, dtype=np.float32)
        keep += [vals, lvl, ptrs]
        t = TacoTensor()
        t.order = self.order
        t.dimensions = dims.ctypes.data_as(POINTER(c_int32))
        t.csize = 4
        t.indices = ctypes.cast(ptrs, POINTER(POINTER(POINTER(c_int32))))
        t.vals = vals.ctypes.data_as(POINTER(c_float))
        t.vals_size = vals.shape[0]
        return t, keep

    @classmethod
    def from_coo(cls, dims: Sequence[int], coords: np.ndarray, vals: np.ndarray) -> "Csf":
        """Lexicographic COO -> CSF with duplicates summed (tentaco_coo_to_csf)."""
        dims = np.ascontiguousarray(dims, dtype=np.int32)
        coords = np.ascontiguousarray(coords, dtype=np.int32)
        vals = np.ascontiguousarray(vals, dtype=np.float32)
        order = dims.shape[0]
        nnz = vals.shape[0]
        assert coords.shape == (order, nnz)
        h = c_void_p()
        _check(
            lib().tentaco_coo_to_csf(
                order,
                dims.ctypes.data_as(POINTER(c_int32)),
                nnz,
                coords.ctypes.data_as(POINTER(c_int32)),
                vals.ctypes.data_as(POINTER(c_float)),
                ctypes.byref(h),
            )
        )
        return _wrap_host_csf(h)

    @classmethod
    def from_tns(cls, path: str, dims: Optional[Sequence[int]] = None,
                 mode_order: Optional[Sequence[int]] = None):
        """Read a FROSTT .tns file (tentaco_tns_read). Returns (csf, mode_order):
        CSF level l holds file mode mode_order[l]; by default the shortest mode
        comes first."""
        h = c_void_p()
        order = c_int()
        used = (c_int * 5)()
        d = None if dims is None else np.ascontiguousarray(dims, dtype=np.int32)
        mo = None if mode_order is None else (c_int * len(mode_order))(*mode_order)
        _check(lib().tentaco_tns_read(os.fsencode(path),
                                      None if d is None else d.ctypes.data_as(POINTER(c_int32)),
                                      mo, ctypes.byref(h), ctypes.byref(order), used))
        return _wrap_host_csf(h), [used[l] for l in range(order.value)]

    def reorder(self, mode_order: Sequence[int]) -> "Csf":
        """Same tensor with level m = mode mode_order[m] (tentaco_csf_reorder)."""
        t, keep = self.as_taco()
        mo = (c_int * self.order)(*[int(m) for m in mode_order])
        h = c_void_p()
        _check(lib().tentaco_csf_reorder(ctypes.byref(t), self.order, mo, ctypes.byref(h)))
        del keep
        return _wrap_host_csf(h)

    def mode_levels(self, m: int, policy: str = "natural") -> List[int]:
        """Level order of the mode-m CSF: m at the root, then the other modes
        in mode order ("natural"), by ascending dimension ("small_first", the
        splatt-like order, largest mode at the leaves) or by descending
        dimension ("large_first": the smallest mode, whose factor rows are
        gathered once per nonzero, at the leaves)."""
        rest = [k for k in range(self.order) if k != m]
        if policy == "small_first":
            rest.sort(key=lambda k: (self.dims[k], k))
        elif policy == "large_first":
            rest.sort(key=lambda k: (-self.dims[k], k))
        elif policy != "natural":
            raise ValueError(f"unknown mode order policy {policy!r}")
        return [m] + rest

    def mode_csfs(self, policy: str = "natural") -> List["Csf"]:
        """One CSF per mode, mode m at the root (levels as mode_levels)."""
        out = []
        for m in range(self.order):
            lv = self.mode_levels(m, policy)
            out.append(self if lv == list(range(self.order)) else self.reorder(lv))
        return out

    @classmethod
    def synth(cls, order: int, dims: Sequence[int], nnz: int, slice_s: float = 1.1,
              fanout_s: float = 1.3, mid_mu: float = 1.0, mid_sigma: float = 1.0,
              leaf_mu: float = 1.5, leaf_sigma: float = 1.0, leaf_cap: int = 10000,
              seed: int = 0) -> "Csf":
        """Synthetic Zipf / log-normal CSF (tentaco_synth_csf)."""
        p = SynthParams()
        p.order = order
        for m in range(5):
            p.dims[m] = int(dims[m]) if m < order else 0
        p.nnz = int(nnz)
        p.slice_s, p.fanout_s = slice_s, fanout_s
        p.mid_mu, p.mid_sigma = mid_mu, mid_sigma
        p.leaf_mu, p.leaf_sigma = leaf_mu, leaf_sigma
        p.leaf_cap = leaf_cap
        p.seed = seed
        h = c_void_p()
        _check(lib().tentaco_synth_csf(ctypes.byref(p), ctypes.byref(h)))
        return _wrap_host_csf(h)


class _HostCsfOwner:
    def __init__(self, h):
        self.h = h

    def __del__(self):
        try:
            if self.h:
                lib().tentaco_host_csf_free(self.h)
        except Exception:
            pass


def _wrap_host_csf(h: c_void_p) -> Csf:
    L = lib()
    owner = _HostCsfOwner(h)
    t = L.tentaco_host_csf_view(h).contents
    order = t.order
    dims = tuple(int(t.dimensions[m]) for m in range(order))
    nodes = [int(L.tentaco_host_csf_nodes(h, m)) for m in range(order)]
    pos, crd = [], []
    parents = 1
    for m in range(order):
        np_len = 2 if m == 0 else parents + 1
        pos.append(np.ctypeslib.as_array(t.indices[m][0], shape=(np_len,)))
        crd.append(np.ctypeslib.as_array(t.indices[m][1], shape=(max(nodes[m], 0),)) if nodes[m] > 0
                   else np.zeros(0, np.int32))
        parents = nodes[m]
    nnz = nodes[order - 1]
    vals = np.ctypeslib.as_array(t.vals, shape=(nnz,)) if nnz > 0 else np.zeros(0, np.float32)
    return Csf(order, dims, pos, crd, vals, _owner=owner)


def dense_taco(a: np.ndarray):
    """taco_tensor_t view of a dense row-major FP32 matrix or vector."""
    a = np.ascontiguousarray(a, dtype=np.float32)
    dims = np.ascontiguousarray(a.shape, dtype=np.int32)
    t = TacoTensor()
    t.order = a.ndim
    t.dimensions = dims.ctypes.data_as(POINTER(c_int32))
    t.csize = 4
    t.vals = a.ctypes.data_as(POINTER(c_float))
    t.vals_size = a.size
    return t, [a, dims]


# ---------------------------------------------------------------------------
# host-pointer entry points (layer 1)
def mttkrp(B: Csf, factors: Sequence[np.ndarray], variant: int = VARIANT_AUTO,
           out_rows: Optional[int] = None) -> np.ndarray:
    """A = MTTKRP(B, factors) on the GPU; factors[m-1] is the factor of level m
    (rows x R, FP32). Mirrors tentaco_mttkrp (gpu_kernels.cuh:5)."""
    assert len(factors) == B.order - 1
    R = int(factors[0].shape[1])
    rows = B.dims[0] if out_rows is None else out_rows
    A = np.empty((rows, R), dtype=np.float32)
    tA, kA = dense_taco(A)
    tB, kB = B.as_taco()
    fs = [dense_taco(f) for f in factors]
    arr = (POINTER(TacoTensor) * len(fs))(*[ctypes.pointer(t) for t, _ in fs])
    _check(lib().tentaco_mttkrp(B.order, ctypes.byref(tA), ctypes.byref(tB), arr, variant))
    del kA, kB
    return A


def ttv(B: Csf, c: np.ndarray) -> np.ndarray:
    """y = TTV(B, c) over the last mode (ttv_csf_gpu_taco, gpu_kernels.cuh:6)."""
    nf = B.nodes(B.order - 2)
    y = np.empty(nf, dtype=np.float32)
    tA, kA = dense_taco(y)
    tB, kB = B.as_taco()
    tc, kc = dense_taco(np.ascontiguousarray(c, dtype=np.float32))
    _check(lib().tentaco_ttv_n(B.order, ctypes.byref(tA), ctypes.byref(tB), ctypes.byref(tc)))
    del kA, kB, kc
    return y


def last_timer_ms() -> float:
    """get_gpu_timer_result(): hot-region ms of the last host-pointer call."""
    return float(lib().get_gpu_timer_result())


def legacy_variant(name: str, R: int, order: int = 3) -> int:
    """The variant the reference name `name` runs at rank R
    (tentaco_legacy_variant)."""
    v = c_int()
    _check(lib().tentaco_legacy_variant(name.encode(), R, order, ctypes.byref(v)))
    return v.value


def variants() -> List[str]:
    L = lib()
    return [L.tentaco_variant_name(v).decode() for v in range(L.tentaco_num_variants())]


def variant_params(v: int):
    fam, blk, grp = c_int(), c_int(), c_int()
    _check(lib().tentaco_variant_params(v, ctypes.byref(fam), ctypes.byref(blk), ctypes.byref(grp)))
    return fam.value, blk.value, grp.value


def default_variant() -> int:
    return int(lib().tentaco_default_variant())


def variant_fits(order: int, R: int, v: int) -> bool:
    """Whether variant v's tile fits the LDS limit at this order and rank."""
    return bool(lib().tentaco_variant_fits(order, R, v))


# ---------------------------------------------------------------------------
# device-resident API (layer 3)
class DeviceArray:
    """A device buffer owned by the library's HIP runtime."""

    def __init__(self, nbytes: int, dtype=np.float32, shape=None):
        self.ptr = c_void_p()
        self.nbytes = int(nbytes)
        self.dtype = np.dtype(dtype)
        self.shape = shape if shape is not None else (self.nbytes // self.dtype.itemsize,)
        _check(lib().tentaco_dev_malloc(ctypes.byref(self.ptr), max(self.nbytes, 4)))

    @classmethod
    def from_numpy(cls, a: np.ndarray) -> "DeviceArray":
        a = np.ascontiguousarray(a)
        d = cls(a.nbytes, a.dtype, a.shape)
        if a.nbytes:
            _check(lib().tentaco_memcpy_h2d(d.ptr, a.ctypes.data_as(c_void_p), a.nbytes))
        return d

    @classmethod
    def empty(cls, shape, dtype=np.float32) -> "DeviceArray":
        shape = tuple(int(s) for s in (shape if isinstance(shape, (tuple, list)) else (shape,)))
        n = int(np.prod(shape)) * np.dtype(dtype).itemsize
        return cls(n, dtype, shape)

    def upload(self, a: np.ndarray):
        """Copy a host array of the same byte size into this buffer."""
        a = np.ascontiguousarray(a, dtype=self.dtype)
        assert a.nbytes == self.nbytes
        if a.nbytes:
            _check(lib().tentaco_memcpy_h2d(self.ptr, a.ctypes.data_as(c_void_p), a.nbytes))

    def numpy(self) -> np.ndarray:
        out = np.empty(self.shape, dtype=self.dtype)
        if self.nbytes:
            _check(lib().tentaco_memcpy_d2h(out.ctypes.data_as(c_void_p), self.ptr, self.nbytes))
        return out

    def free(self):
        if self.ptr:
            lib().tentaco_dev_free(self.ptr)
            self.ptr = c_void_p()

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


class DeviceCsf:
    """Device-resident CSF handle (tentaco_csf_upload)."""

    def __init__(self, B: Csf):
        t, keep = B.as_taco()
        self.h = c_void_p()
        _check(lib().tentaco_csf_upload(ctypes.byref(t), B.order, ctypes.byref(self.h)))
        del keep
        self.order = B.order
        self.dims = B.dims
        self.nnz = B.nnz
        self.nodes = [B.nodes(m) for m in range(B.order)]

    def reserve(self, R: int, variant: int = VARIANT_AUTO, a_rows: Optional[int] = None):
        if a_rows is None:
            _check(lib().tentaco_csf_reserve(self.h, R, variant))
        else:
            _check(lib().tentaco_csf_reserve_rows(self.h, R, variant, a_rows))

    def mttkrp(self, factors: Sequence[DeviceArray], A: DeviceArray, R: int,
               variant: int = VARIANT_AUTO, stream=None, a_rows: Optional[int] = None):
        arr = (c_void_p * len(factors))(*[f.ptr for f in factors])
        rows = self.dims[0] if a_rows is None else a_rows
        _check(lib().tentaco_mttkrp_dev(self.h, R, arr, A.ptr, rows, variant, stream))

    def autotune(self, factors: Sequence[DeviceArray], A: DeviceArray, R: int, reps: int = 5,
                 stream=None, a_rows: Optional[int] = None):
        """Time every variant; the fastest becomes this handle's AUTO choice.
        Returns (best_variant, per-variant median ms, -1 where unsupported)."""
        arr = (c_void_p * len(factors))(*[f.ptr for f in factors])
        rows = self.dims[0] if a_rows is None else a_rows
        n = lib().tentaco_num_variants()
        times = (c_float * n)()
        best = c_int()
        _check(lib().tentaco_csf_autotune(self.h, R, arr, A.ptr, rows, reps, stream,
                                          ctypes.byref(best), times))
        return best.value, [float(t) for t in times]

    def reserve_level(self, level: int):
        """Build the structures mttkrp_level needs at `level` (the leaf
        level's transposed index)."""
        _check(lib().tentaco_csf_reserve_level(self.h, level))

    def resolve(self, R: int, variant: int = VARIANT_AUTO) -> int:
        """The variant a call with `variant` runs (recorded choice or the
        structural heuristic; no selector)."""
        v = c_int()
        _check(lib().tentaco_csf_resolve_variant(self.h, R, variant, ctypes.byref(v)))
        return v.value

    def set_tuned(self, R: int, variant: int):
        _check(lib().tentaco_csf_set_tuned(self.h, R, variant))

    def sweep(self, factors: Sequence[DeviceArray], A: DeviceArray, R: int, reps: int = 3,
              cut: float = 4.0, stream=None, a_rows: Optional[int] = None) -> List[float]:
        """Per-call ms of every variant (probe, then the median of `reps`
        repetitions within `cut` x the fastest probe); -1 where unsupported.
        Leaves the handle's recorded choices unchanged."""
        arr = (c_void_p * len(factors))(*[f.ptr for f in factors])
        rows = self.dims[0] if a_rows is None else a_rows
        n = lib().tentaco_num_variants()
        times = (c_float * n)()
        _check(lib().tentaco_csf_sweep(self.h, R, arr, A.ptr, rows, reps, cut, stream, times))
        return [float(t) for t in times]

    @classmethod
    def upload_async(cls, B: "Csf", stream: "Stream") -> "DeviceCsf":
        """Upload with the copies enqueued on `stream`; B must stay alive
        until the stream is synchronized."""
        self = cls.__new__(cls)
        t, keep = B.as_taco()
        self._keep_async = (B, t, keep)
        self.h = c_void_p()
        _check(lib().tentaco_csf_upload_async(ctypes.byref(t), B.order, stream.h, ctypes.byref(self.h)))
        self.order = B.order
        self.dims = B.dims
        self.nnz = B.nnz
        self.nodes = [B.nodes(m) for m in range(B.order)]
        return self

    def mttkrp_host_async(self, factors: Sequence[np.ndarray], A: np.ndarray, R: int,
                          stream: "Stream", variant: int = VARIANT_AUTO):
        """Host factors (levels 1..order-1) -> host A, enqueued on `stream`;
        keep the arrays alive and A unread until stream.synchronize()."""
        tf = [dense_taco(f) for f in factors]
        tA, kA = dense_taco(A)
        arr = (POINTER(TacoTensor) * len(tf))(*[ctypes.pointer(t) for t, _ in tf])
        self._keep_call = (tf, tA, kA, arr, factors, A)
        _check(lib().tentaco_mttkrp_host_async(self.h, R, arr, ctypes.byref(tA), variant, stream.h))

    def mttkrp_repeat(self, factors: Sequence[DeviceArray], A: DeviceArray, R: int, count: int,
                      variant: int = VARIANT_AUTO, stream=None, a_rows: Optional[int] = None):
        """`count` back-to-back MTTKRP calls issued from the library's loop."""
        arr = (c_void_p * len(factors))(*[f.ptr for f in factors])
        rows = self.dims[0] if a_rows is None else a_rows
        _check(lib().tentaco_mttkrp_dev_repeat(self.h, R, arr, A.ptr, rows, variant, stream, count))

    def mttkrp_level(self, level: int, factors: Sequence[Optional[DeviceArray]], A: DeviceArray,
                     R: int, stream=None, a_rows: Optional[int] = None):
        """MTTKRP for the mode at CSF level `level` on this CSF; factors[l]
        for every level l (the entry for `level` may be None)."""
        arr = (c_void_p * len(factors))(*[None if f is None else f.ptr for f in factors])
        rows = self.dims[level] if a_rows is None else a_rows
        _check(lib().tentaco_mttkrp_level_dev(self.h, level, R, arr, A.ptr, rows, stream))

    def tuned(self, R: int):
        """(variant, source) recorded for rank R; source is one of TUNED_*."""
        v, src = c_int(), c_int()
        _check(lib().tentaco_csf_tuned(self.h, R, ctypes.byref(v), ctypes.byref(src)))
        return v.value, src.value

    def features(self, R: int) -> np.ndarray:
        """The 24 selector features of this tensor at rank R."""
        f = np.zeros(NUM_FEATURES, np.float32)
        _check(lib().tentaco_csf_features(self.h, R, f.ctypes.data_as(POINTER(c_float))))
        return f

    def set_selector(self, selector: Optional["Selector"], min_margin: float = 0.03):
        """AUTO on an unrecorded rank uses the selector's pick, or the
        fallback (timing the top 4 predictions, set_selector_fallback) when
        the predicted margin is under min_margin."""
        self._selector = selector  # keep it alive while attached
        _check(lib().tentaco_csf_set_selector(self.h, selector.h if selector else None, min_margin))

    def set_selector_fallback(self, top_k: int):
        """k > 0 (4 by default): time the top k picks when the margin is
        small; 0: the full sweep."""
        _check(lib().tentaco_csf_set_selector_fallback(self.h, top_k))

    def ttv(self, c: DeviceArray, y: DeviceArray, stream=None):
        _check(lib().tentaco_ttv_dev(self.h, c.ptr, y.ptr, stream))

    def set_ttv_bands(self, bands: int):
        """TTV layout: 0 picks (banded when c exceeds one LDS window and the
        best window serves under 3/4 of the gathers), 1 one window, 2..8
        that many leaf-coordinate bands."""
        _check(lib().tentaco_csf_set_ttv_bands(self.h, bands))

    def ttv_layout(self):
        """(bands, device bytes of the banded copy): bands 0 before the
        first TTV, 1 for one window."""
        b = c_int(-1)
        n = ctypes.c_int64(-1)
        _check(lib().tentaco_csf_ttv_layout(self.h, ctypes.byref(b), ctypes.byref(n)))
        return b.value, n.value

    def close(self):
        if self.h:
            lib().tentaco_csf_free(self.h)
            self.h = c_void_p()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class Batch:
    """Batched persistent MTTKRP over many device-resident CSFs
    (tentaco_batch_*): one persistent launch for all tasks, optionally
    captured in a hipGraph."""

    def __init__(self, tasks: Sequence[DeviceCsf], R: int):
        self.tasks = list(tasks)
        self.R = R
        arr = (c_void_p * len(tasks))(*[t.h for t in tasks])
        self.h = c_void_p()
        _check(lib().tentaco_batch_create(arr, len(tasks), R, ctypes.byref(self.h)))
        self._keep = []

    def set_operands(self, factors: Sequence[Sequence[DeviceArray]], outs: Sequence[DeviceArray],
                     out_rows: Sequence[int]):
        n = len(self.tasks)
        fa = (c_void_p * (4 * n))()
        for t in range(n):
            for j, f in enumerate(factors[t]):
                fa[4 * t + j] = f.ptr
        oa = (c_void_p * n)(*[o.ptr for o in outs])
        rows = (c_int32 * n)(*[int(r) for r in out_rows])
        self._keep = [factors, outs]
        _check(lib().tentaco_batch_set_operands(self.h, fa, oa, rows))

    def configure(self, family: int, block: int, group: int):
        _check(lib().tentaco_batch_configure(self.h, family, block, group))

    def configure_order(self, order: int, family: int, block: int, group: int,
                        schedule: int = 0):
        """The tile and schedule of one tensor order's tasks only
        (tentaco_batch_configure_order)."""
        _check(lib().tentaco_batch_configure_order(self.h, order, family, block, group, schedule))

    def config(self, order: int):
        """(family, block, group, schedule) that an order group runs with."""
        f, b, g, sc = c_int(), c_int(), c_int(), c_int()
        _check(lib().tentaco_batch_get_config(self.h, order, ctypes.byref(f), ctypes.byref(b),
                                              ctypes.byref(g), ctypes.byref(sc)))
        return f.value, b.value, g.value, sc.value

    def run(self, stream=None):
        _check(lib().tentaco_batch_run(self.h, stream))

    def capture(self, stream=None):
        _check(lib().tentaco_batch_capture(self.h, stream))

    def launch(self, stream=None):
        _check(lib().tentaco_batch_launch(self.h, stream))

    def items(self):
        i, g, nb = c_int32(), c_int32(), c_int32()
        _check(lib().tentaco_batch_items(self.h, ctypes.byref(i), ctypes.byref(g), ctypes.byref(nb)))
        return i.value, g.value, nb.value

    OUTPUTS_WRITTEN, OUTPUTS_RETAINED = 0, 1

    def set_output_mode(self, mode: int):
        """OUTPUTS_WRITTEN: every run zeroes the rows of empty slices;
        OUTPUTS_RETAINED: they are zeroed once now and left alone by runs
        (the output buffers must not be written by anything else)."""
        _check(lib().tentaco_batch_set_output_mode(self.h, mode))

    @property
    def output_mode(self) -> int:
        m = c_int()
        _check(lib().tentaco_batch_get_output_mode(self.h, ctypes.byref(m)))
        return m.value

    def set_schedule(self, schedule: int):
        """0: device work counter (default); 1: static cyclic items."""
        _check(lib().tentaco_batch_set_schedule(self.h, schedule))

    @property
    def schedule(self) -> int:
        s = c_int()
        _check(lib().tentaco_batch_get_schedule(self.h, ctypes.byref(s)))
        return s.value

    def autotune(self, reps: int = 3, stream=None):
        """The joint sweep's best tile for all orders, then each order group's
        own tile (read with config(order)); returns (joint best tile,
        final ms)."""
        f, b, g, ms = c_int(), c_int(), c_int(), c_float()
        _check(lib().tentaco_batch_autotune(self.h, reps, stream, ctypes.byref(f), ctypes.byref(b),
                                            ctypes.byref(g), ctypes.byref(ms)))
        return (f.value, b.value, g.value), float(ms.value)

    def close(self):
        if self.h:
            lib().tentaco_batch_free(self.h)
            self.h = c_void_p()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def synchronize():
    _check(lib().tentaco_dev_synchronize())


def flush_cache(stream=None):
    """Read 512 MiB on the device so the next kernel starts cold."""
    _check(lib().tentaco_flush_cache(stream))


def timer_start(stream=None):
    _check(lib().tentaco_timer_start(stream))


def timer_stop(stream=None) -> float:
    ms = c_float()
    _check(lib().tentaco_timer_stop(stream, ctypes.byref(ms)))
    return float(ms.value)


def ktimer_start():
    """Start timing the main kernel of every following call (events on the
    launch stream around that kernel only)."""
    _check(lib().tentaco_ktimer_start())


def ktimer_stop():
    """Stop the kernel timer; returns (total_ms, launches, kernel_name)."""
    total = ctypes.c_double()
    n = c_int()
    name = ctypes.create_string_buffer(64)
    _check(lib().tentaco_ktimer_stop(ctypes.byref(total), ctypes.byref(n), name, 64))
    return float(total.value), int(n.value), name.value.decode()


def dev_copy(dst, src, nbytes=None, stream=None):
    """Device-to-device copy of DeviceArrays through the streaming copy kernel."""
    nbytes = min(dst.nbytes, src.nbytes) if nbytes is None else int(nbytes)
    _check(lib().tentaco_dev_copy(dst.ptr, src.ptr, nbytes, stream))


def dev_gather(table, rows: int, R: int, blocks: int, iters: int, out, stream=None) -> float:
    """Random row gathers from a rows x R table (tentaco_dev_gather); returns
    the bytes one launch gathers."""
    nb = ctypes.c_double()
    _check(lib().tentaco_dev_gather(table.ptr, rows, R, blocks, iters, out.ptr, stream,
                                    ctypes.byref(nb)))
    return nb.value


def _fp(a: np.ndarray):
    return a.ctypes.data_as(POINTER(c_float))


class Selector:
    """The learned variant selector (FP32 MLP 24 -> 64 -> 64 -> K on the
    device). Its forward, backward and Adam steps are the library's HIP
    kernels; this class only moves host arrays in and out."""

    def __init__(self, n_out: Optional[int] = None, seed: int = 0):
        self.n_out = int(n_out or lib().tentaco_num_variants())
        self.h = c_void_p()
        _check(lib().tentaco_mlp_create(self.n_out, seed, ctypes.byref(self.h)))
        self.n_params = int(lib().tentaco_mlp_num_params(self.n_out))

    def set_scaling(self, x_mean, x_std, y_mean: float, y_std: float):
        xm = np.ascontiguousarray(x_mean, np.float32)
        xs = np.ascontiguousarray(x_std, np.float32)
        _check(lib().tentaco_mlp_set_scaling(self.h, _fp(xm), _fp(xs), float(y_mean), float(y_std)))

    def scaling(self):
        xm = np.zeros(NUM_FEATURES, np.float32)
        xs = np.zeros(NUM_FEATURES, np.float32)
        ym, ys = c_float(), c_float()
        _check(lib().tentaco_mlp_get_scaling(self.h, _fp(xm), _fp(xs), ctypes.byref(ym), ctypes.byref(ys)))
        return xm, xs, float(ym.value), float(ys.value)

    def params(self) -> np.ndarray:
        p = np.zeros(self.n_params, np.float32)
        _check(lib().tentaco_mlp_get_params(self.h, _fp(p), self.n_params))
        return p

    def set_params(self, p):
        p = np.ascontiguousarray(p, np.float32)
        _check(lib().tentaco_mlp_set_params(self.h, _fp(p), int(p.size)))

    def grads(self) -> np.ndarray:
        g = np.zeros(self.n_params, np.float32)
        _check(lib().tentaco_mlp_get_grads(self.h, _fp(g), self.n_params))
        return g

    def forward(self, x) -> np.ndarray:
        """Predicted ln(ms) per output for rows of raw features (inference kernel)."""
        x = np.ascontiguousarray(np.atleast_2d(x), np.float32)
        n = x.shape[0]
        xd = DeviceArray.from_numpy(x)
        yd = DeviceArray.empty((n, self.n_out))
        _check(lib().tentaco_mlp_forward(self.h, xd.ptr, n, yd.ptr, None))
        return yd.numpy()

    def loss_grad(self, x, t, mask) -> float:
        x = np.ascontiguousarray(x, np.float32)
        t = np.ascontiguousarray(t, np.float32)
        m = np.ascontiguousarray(mask, np.float32)
        loss = c_float()
        _check(lib().tentaco_mlp_loss_grad(self.h, _fp(x), _fp(t), _fp(m), x.shape[0], ctypes.byref(loss)))
        return float(loss.value)

    def adam(self, lr=1e-3, beta1=0.9, beta2=0.999, eps=1e-8):
        _check(lib().tentaco_mlp_adam(self.h, lr, beta1, beta2, eps))

    def train(self, x, t, mask, epochs=300, batch=128, lr=3e-3, seed=0) -> float:
        x = np.ascontiguousarray(x, np.float32)
        t = np.ascontiguousarray(t, np.float32)
        m = np.ascontiguousarray(mask, np.float32)
        loss = c_float()
        _check(lib().tentaco_mlp_train(self.h, _fp(x), _fp(t), _fp(m), x.shape[0], epochs, batch, lr,
                                       seed, ctypes.byref(loss)))
        return float(loss.value)

    def select(self, order: int, R: int, features):
        """(variant, margin, predicted ms per variant) for one tensor."""
        f = np.ascontiguousarray(features, np.float32)
        v, margin = c_int(), c_float()
        pred = np.zeros(self.n_out, np.float32)
        _check(lib().tentaco_mlp_select(self.h, order, R, _fp(f), ctypes.byref(v), ctypes.byref(margin),
                                        _fp(pred)))
        return v.value, float(margin.value), pred

    def save(self, path: str, **meta):
        xm, xs, ym, ys = self.scaling()
        np.savez(path, params=self.params(), x_mean=xm, x_std=xs, y_mean=np.float32(ym),
                 y_std=np.float32(ys), n_out=np.int32(self.n_out),
                 variants=np.array(variants()), **meta)

    @classmethod
    def load(cls, path: str) -> "Selector":
        d = np.load(path, allow_pickle=False)
        if list(d["variants"]) != variants():
            raise TentacoError(EINVAL, f"{path}: trained for a different variant table")
        s = cls(int(d["n_out"]))
        s.set_params(d["params"])
        s.set_scaling(d["x_mean"], d["x_std"], float(d["y_mean"]), float(d["y_std"]))
        return s

    def close(self):
        if self.h:
            lib().tentaco_mlp_free(self.h)
            self.h = c_void_p()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class Cpd:
    """CP-ALS on the device for several tensors at once (tentaco_cpd_*).

    mode_handles[t][m] is tensor t's DeviceCsf with mode m at its root;
    level_modes[t][m] lists the tensor mode at each level of that CSF
    (default: m first, then the other modes in increasing order, as
    Csf.mode_csfs() builds them)."""

    def __init__(self, mode_handles: Sequence[Sequence["DeviceCsf"]], R: int, seed: int = 0,
                 level_modes=None):
        nt = len(mode_handles)
        hs = (c_void_p * (5 * nt))()
        lm = (c_int * (25 * nt))()
        self.orders = []
        self.dims = []
        for t, modes in enumerate(mode_handles):
            N = len(modes)
            self.orders.append(N)
            for m, H in enumerate(modes):
                hs[5 * t + m] = H.h
                levels = (level_modes[t][m] if level_modes is not None
                          else [m] + [k for k in range(N) if k != m])
                for l, md in enumerate(levels):
                    lm[(5 * t + m) * 5 + l] = md
            dims = [0] * N
            levels0 = level_modes[t][0] if level_modes is not None else list(range(N))
            for l, md in enumerate(levels0):
                dims[md] = modes[0].dims[l]
            self.dims.append(dims)
        self.R = R
        self._keep = [list(m) for m in mode_handles]
        self.h = c_void_p()
        _check(lib().tentaco_cpd_create(hs, lm, nt, R, seed, ctypes.byref(self.h)))

    def tune(self, reps: int = 3):
        _check(lib().tentaco_cpd_tune(self.h, reps))

    def iterate(self, sweeps: int = 1, use_graphs: bool = False, stream=None) -> np.ndarray:
        """Run ALS sweeps; returns each tensor's fit after the last one."""
        fits = (ctypes.c_double * len(self.orders))()
        _check(lib().tentaco_cpd_iterate(self.h, sweeps, int(use_graphs), stream, fits))
        return np.array(fits[:])

    def factor(self, t: int, m: int):
        a = np.empty((self.dims[t][m], self.R), np.float32)
        lam = np.empty(self.R, np.float32)
        _check(lib().tentaco_cpd_factor(self.h, t, m, _fp(a), _fp(lam)))
        return a, lam

    def set_factor(self, t: int, m: int, a):
        a = np.ascontiguousarray(a, np.float32)
        assert a.shape == (self.dims[t][m], self.R)
        _check(lib().tentaco_cpd_set_factor(self.h, t, m, _fp(a)))

    def close(self):
        if self.h:
            lib().tentaco_cpd_free(self.h)
            self.h = c_void_p()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class Stream:
    """A HIP stream at the default priority (tentaco_stream_create)."""

    def __init__(self):
        self.h = c_void_p()
        _check(lib().tentaco_stream_create(ctypes.byref(self.h)))

    def synchronize(self):
        _check(lib().tentaco_stream_synchronize(self.h))

    def close(self):
        if self.h:
            lib().tentaco_stream_destroy(self.h)
            self.h = c_void_p()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class _PinnedOwner:
    def __init__(self, ptr):
        self.ptr = ptr

    def __del__(self):
        try:
            lib().tentaco_host_free(self.ptr)
        except Exception:
            pass


class PinnedArray(np.ndarray):
    """numpy array over pinned host memory; views keep it (and the memory)
    alive through their base."""


def pinned_empty(shape, dtype=np.float32) -> np.ndarray:
    """A numpy array in pinned (page-locked) host memory (tentaco_host_alloc);
    the memory is freed when the array and its views are collected."""
    dtype = np.dtype(dtype)
    shape = tuple(np.atleast_1d(shape).tolist()) if not isinstance(shape, tuple) else shape
    n = int(np.prod(shape)) if shape else 1
    nbytes = max(n * dtype.itemsize, 4)
    ptr = c_void_p()
    _check(lib().tentaco_host_alloc(ctypes.byref(ptr), nbytes))
    buf = (ctypes.c_char * nbytes).from_address(ptr.value)
    arr = np.frombuffer(buf, dtype=dtype, count=n).reshape(shape).view(PinnedArray)
    arr._owner = _PinnedOwner(ptr)
    return arr


def pinned_copy(a: np.ndarray) -> np.ndarray:
    out = pinned_empty(a.shape, a.dtype)
    out[...] = a
    return out
