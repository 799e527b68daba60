"""ctypes binding of libfmdbzp.so (declared in include/fmdbzp.h).

The library is the only compute path: if it is not built, importing this
module raises, and every plan creation or search call goes through it.
"""
from __future__ import annotations

import ctypes
import os

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "_lib", "libfmdbzp.so")

ABI_VERSION = 1
FMDBZP_OK = 0

ELTYPE = {"cf32": 0, "cf64": 1, "i16": 2, "ci8": 3, "ci16": 4, "f32": 5, "f64": 6, "c2bit": 7}
FLAG_STORE_SURFACES = 0x1
FLAG_DEVICE_SIGNAL = 0x2
FLAG_DEVICE_OUTPUT = 0x4

KERNEL_CLASSES = ("code_fft", "signal_fft", "corr_tile", "column", "reduce", "finalize", "export")


class PlanDesc(ctypes.Structure):
    _fields_ = [
        ("abi_version", ctypes.c_int32),
        ("samples_per_code", ctypes.c_int32),
        ("num_blocks", ctypes.c_int32),
        ("block_size", ctypes.c_int32),
        ("fft_size", ctypes.c_int32),
        ("num_coh", ctypes.c_int32),
        ("num_data_bits", ctypes.c_int32),
        ("bit_edge_search_steps", ctypes.c_int32),
        ("num_noncoherent", ctypes.c_int32),
        ("num_secondary_rotations", ctypes.c_int32),
        ("num_doppler_bins", ctypes.c_int32),
        ("samples_per_code_eff", ctypes.c_int32),
        ("num_patterns", ctypes.c_int32),
        ("path", ctypes.c_int32),
        ("noise_estimator", ctypes.c_int32),
        ("samples_per_chip", ctypes.c_int32),
        ("precision", ctypes.c_int32),
        ("options", ctypes.c_int32),
        ("reserved", ctypes.c_int32 * 6),
        ("sampling_freq_hz", ctypes.c_double),
    ]


class PrnStats(ctypes.Structure):
    _fields_ = [
        ("peak_power", ctypes.c_float),
        ("peak_row", ctypes.c_int32),
        ("peak_col", ctypes.c_int32),
        ("noise_power", ctypes.c_float),
        ("code_left", ctypes.c_float),
        ("code_right", ctypes.c_float),
        ("dop_left", ctypes.c_float),
        ("dop_right", ctypes.c_float),
        ("noise_sum", ctypes.c_double),
        ("noise_cells", ctypes.c_int64),
    ]


class PrnResult(ctypes.Structure):
    _fields_ = [
        ("cn0_dbhz", ctypes.c_double),
        ("code_phase", ctypes.c_double),
        ("doppler_offset", ctypes.c_double),
        ("peak_to_noise", ctypes.c_float),
        ("reserved", ctypes.c_int32),
    ]


class Request(ctypes.Structure):
    _fields_ = [
        ("plan", ctypes.c_void_p),
        ("signal", ctypes.c_void_p),
        ("eltype", ctypes.c_int32),
        ("nprn", ctypes.c_int32),
        ("n_samples", ctypes.c_int64),
        ("interm_freq_hz", ctypes.c_double),
        ("prn_index", ctypes.c_void_p),
        ("flags", ctypes.c_uint32),
        ("reserved", ctypes.c_uint32),
        ("out_stats", ctypes.c_void_p),
        ("out_surfaces", ctypes.c_void_p),
    ]


class Emitter(ctypes.Structure):
    _fields_ = [
        ("chips", ctypes.c_void_p),
        ("code_length", ctypes.c_int32),
        ("boc", ctypes.c_int32),
        ("secondary", ctypes.c_void_p),
        ("secondary_length", ctypes.c_int32),
        ("secondary_phase", ctypes.c_int32),
        ("bits", ctypes.c_void_p),
        ("num_bits", ctypes.c_int32),
        ("bit_ms", ctypes.c_int32),
        ("bit_edge_ms", ctypes.c_int32),
        ("reserved", ctypes.c_int32),
        ("amplitude", ctypes.c_double),
        ("code_freq_hz", ctypes.c_double),
        ("code_phase_chips", ctypes.c_double),
        ("carrier_hz", ctypes.c_double),
        ("carrier_phase", ctypes.c_double),
    ]


class SceneDesc(ctypes.Structure):
    _fields_ = [
        ("n_samples", ctypes.c_int64),
        ("sampling_freq_hz", ctypes.c_double),
        ("complex_samples", ctypes.c_int32),
        ("out_eltype", ctypes.c_int32),
        ("noise_scale", ctypes.c_double),
        ("seed", ctypes.c_uint64),
        ("noise_stream", ctypes.c_uint32),
        ("reserved", ctypes.c_int32),
    ]


class SecondaryRequest(ctypes.Structure):
    _fields_ = [
        ("code", ctypes.c_void_p),
        ("secondary", ctypes.c_void_p),
        ("doppler_hz", ctypes.c_double),
        ("num_rotations", ctypes.c_int32),
        ("reserved", ctypes.c_int32),
    ]


EXPORTED_SYMBOLS = (
    "fmdbzp_plan_create",
    "fmdbzp_acquire",
    "fmdbzp_acquire_batch",
    "fmdbzp_prn_results",
    "fmdbzp_acquire_noalloc",
    "fmdbzp_plan_destroy",
    "fmdbzp_last_error",
    "fmdbzp_query",
    "fmdbzp_plan_set_timing",
    "fmdbzp_plan_graph_counts",
    "fmdbzp_plan_tuning",
    "fmdbzp_plan_column_kernel",
    "fmdbzp_plan_call_kernels",
    "fmdbzp_full_period_form",
    "fmdbzp_plan_kernel_times",
    "fmdbzp_synthesize",
    "fmdbzp_plan_set_surface_layout",
    "fmdbzp_secondary_phase",
)


def load_library(path: str = LIB_PATH) -> ctypes.CDLL:
    if not os.path.exists(path):
        raise ImportError(f"libfmdbzp.so is not built ({path}); run __graft_entry__.build() "
                          "or `make -C acquisition.jl_amd/csrc`")
    lib = ctypes.CDLL(path)
    P = ctypes.c_void_p
    lib.fmdbzp_plan_create.argtypes = [ctypes.POINTER(PlanDesc), ctypes.c_int32, P, ctypes.c_int32, P, P, P,
                                       ctypes.POINTER(ctypes.c_void_p)]
    lib.fmdbzp_plan_create.restype = ctypes.c_int
    lib.fmdbzp_acquire.argtypes = [P, P, ctypes.c_int32, ctypes.c_int64, ctypes.c_double, P, ctypes.c_int32,
                                   ctypes.c_uint32, P, P]
    lib.fmdbzp_acquire.restype = ctypes.c_int
    D, I = ctypes.c_double, ctypes.c_int32
    lib.fmdbzp_prn_results.argtypes = [P, I, I, I, I, D, D, D, D, D, I, P]
    lib.fmdbzp_prn_results.restype = ctypes.c_int
    lib.fmdbzp_acquire_batch.argtypes = [P, ctypes.c_int32]
    lib.fmdbzp_acquire_batch.restype = ctypes.c_int
    lib.fmdbzp_plan_destroy.argtypes = [P]
    lib.fmdbzp_plan_destroy.restype = ctypes.c_int
    lib.fmdbzp_last_error.argtypes = []
    lib.fmdbzp_last_error.restype = ctypes.c_char_p
    lib.fmdbzp_query.argtypes = [ctypes.c_char_p, ctypes.c_size_t]
    lib.fmdbzp_query.restype = ctypes.c_int
    lib.fmdbzp_plan_set_timing.argtypes = [P, ctypes.c_int32]
    lib.fmdbzp_plan_set_timing.restype = ctypes.c_int
    lib.fmdbzp_plan_kernel_times.argtypes = [P, P, P, ctypes.c_int32]
    lib.fmdbzp_plan_kernel_times.restype = ctypes.c_int
    lib.fmdbzp_secondary_phase.argtypes = [P, P, ctypes.c_int32, ctypes.c_int64, ctypes.c_double, ctypes.c_uint32,
                                           P, ctypes.c_int32, P]
    lib.fmdbzp_secondary_phase.restype = ctypes.c_int
    lib.fmdbzp_plan_set_surface_layout.argtypes = [P, ctypes.c_int32, P]
    lib.fmdbzp_plan_set_surface_layout.restype = ctypes.c_int
    lib.fmdbzp_synthesize.argtypes = [ctypes.POINTER(SceneDesc), P, ctypes.c_int32, P]
    lib.fmdbzp_synthesize.restype = ctypes.c_int
    lib.fmdbzp_acquire_noalloc.argtypes = [P, P, ctypes.c_int32, ctypes.c_int64, ctypes.c_double, P, ctypes.c_int32,
                                           P]
    lib.fmdbzp_acquire_noalloc.restype = ctypes.c_int
    if hasattr(lib, "fmdbzp_plan_graph_counts"):
        lib.fmdbzp_plan_graph_counts.argtypes = [P, P, P]
        lib.fmdbzp_plan_graph_counts.restype = ctypes.c_int
    if hasattr(lib, "fmdbzp_plan_tuning"):
        lib.fmdbzp_plan_tuning.argtypes = [P, ctypes.c_char_p, ctypes.c_size_t]
        lib.fmdbzp_plan_tuning.restype = ctypes.c_int
    if hasattr(lib, "fmdbzp_plan_column_kernel"):
        lib.fmdbzp_plan_column_kernel.argtypes = [P, ctypes.c_char_p, ctypes.c_size_t]
        lib.fmdbzp_plan_column_kernel.restype = ctypes.c_int
    lib.fmdbzp_full_period_form.argtypes = [I, I, I, I, I]
    lib.fmdbzp_full_period_form.restype = ctypes.c_int
    if hasattr(lib, "fmdbzp_plan_call_kernels"):
        lib.fmdbzp_plan_call_kernels.argtypes = [P, ctypes.c_int32, ctypes.c_int32, ctypes.c_uint32, ctypes.c_char_p,
                                                 ctypes.c_size_t]
        lib.fmdbzp_plan_call_kernels.restype = ctypes.c_int
    return lib


_lib = None


def lib() -> ctypes.CDLL:
    global _lib
    if _lib is None:
        _lib = load_library()
    return _lib


def prn_results(stats, n: int, spc: int, nb: int, bs: int, fs: float, fc: float, code_length: float, tcoh: float,
                spacing: float, interpolate: int, out_ptr: int):
    """`fmdbzp_prn_results` over a ctypes array of `PrnStats`."""
    _check(lib().fmdbzp_prn_results(stats, n, spc, nb, bs, fs, fc, code_length, tcoh, spacing, interpolate, out_ptr),
           "fmdbzp_prn_results")


def full_period_form(samples_per_code: int, num_blocks: int, num_coh: int, num_noncoherent: int, nprn: int) -> str:
    """Form of the full-period correlation of a statistics-only call: "radix",
    "axis31", or "" where the call runs on the tile (`fmdbzp_full_period_form`)."""
    rc = lib().fmdbzp_full_period_form(samples_per_code, num_blocks, num_coh, num_noncoherent, nprn)
    _check(min(rc, 0), "fmdbzp_full_period_form")
    return ("", "radix", "axis31")[rc]


def acquire_batch(reqs):
    """Submit a list of `Request`s as one batch."""
    arr = (Request * len(reqs))(*reqs)
    _check(lib().fmdbzp_acquire_batch(ctypes.cast(arr, ctypes.c_void_p), len(reqs)), "fmdbzp_acquire_batch")


class EngineError(RuntimeError):
    """A negative status from libfmdbzp (HIP error, OOM, no device, bad handle)."""


def _check(rc: int, what: str):
    if rc != FMDBZP_OK:
        msg = lib().fmdbzp_last_error().decode(errors="replace")
        raise EngineError(f"{what} failed (status {rc}): {msg}")


def query() -> str:
    buf = ctypes.create_string_buffer(512)
    rc = lib().fmdbzp_query(buf, len(buf))
    _check(rc, "fmdbzp_query")
    return buf.value.decode()


def make_desc(fields: dict) -> PlanDesc:
    d = PlanDesc()
    d.abi_version = ABI_VERSION
    for k, v in fields.items():
        setattr(d, k, v)
    return d


class NativePlan:
    """Owner of one `fmdbzp_plan*`."""

    def __init__(self, handle, desc: PlanDesc, nprn: int):
        self.handle = handle
        self.desc = desc
        self.nprn = nprn

    @classmethod
    def create(cls, plan) -> "NativePlan":
        from .plan import plan_code_samples, plan_desc_fields, plan_patterns

        desc = make_desc(plan_desc_fields(plan))
        codes = np.ascontiguousarray(plan_code_samples(plan), dtype=np.int8)
        nsets, pats, pset = plan_patterns(plan)
        pats = np.ascontiguousarray(pats, dtype=np.float32)
        pset = np.ascontiguousarray(pset, dtype=np.int32)
        shifts = np.ascontiguousarray(plan.code_drift_shifts, dtype=np.int32)
        h = ctypes.c_void_p()
        rc = lib().fmdbzp_plan_create(ctypes.byref(desc), len(plan.avail_prns), codes.ctypes.data, nsets,
                                      pats.ctypes.data, pset.ctypes.data, shifts.ctypes.data, ctypes.byref(h))
        _check(rc, "fmdbzp_plan_create")
        return cls(h, desc, len(plan.avail_prns))

    def acquire(self, signal_ptr: int, eltype: int, n_samples: int, if_hz: float, prn_index, flags: int,
                surfaces=None):
        idx = np.ascontiguousarray(prn_index, dtype=np.int32)
        stats = (PrnStats * len(idx))()
        surf_arg = None
        if surfaces is not None:
            arr = (ctypes.c_void_p * len(idx))(*[ctypes.c_void_p(int(s)) if s else None for s in surfaces])
            surf_arg = arr
        rc = lib().fmdbzp_acquire(self.handle, ctypes.c_void_p(signal_ptr), eltype, n_samples, float(if_hz),
                                  idx.ctypes.data, len(idx), flags, ctypes.cast(stats, ctypes.c_void_p),
                                  ctypes.cast(surf_arg, ctypes.c_void_p) if surf_arg is not None else None)
        _check(rc, "fmdbzp_acquire")
        return stats

    def acquire_noalloc(self, signal_ptr: int, eltype: int, n_samples: int, if_hz: float, prn_index):
        """`fmdbzp_acquire_noalloc`: the same search on device-resident samples
        with the library's static scratch instead of any allocation."""
        idx = np.ascontiguousarray(prn_index, dtype=np.int32)
        stats = (PrnStats * len(idx))()
        rc = lib().fmdbzp_acquire_noalloc(self.handle, ctypes.c_void_p(signal_ptr), eltype, n_samples, float(if_hz),
                                          idx.ctypes.data, len(idx), ctypes.cast(stats, ctypes.c_void_p))
        _check(rc, "fmdbzp_acquire_noalloc")
        return stats

    def request(self, signal_ptr: int, eltype: int, n_samples: int, if_hz: float, prn_index, flags: int,
                surfaces=None):
        """A filled `Request` plus the buffers it points to (kept alive by the caller)."""
        idx = np.ascontiguousarray(prn_index, dtype=np.int32)
        stats = (PrnStats * len(idx))()
        surf_arg = None
        if surfaces is not None:
            surf_arg = (ctypes.c_void_p * len(idx))(*[ctypes.c_void_p(int(x)) if x else None for x in surfaces])
        q = Request(self.handle, signal_ptr, eltype, len(idx), n_samples, float(if_hz), idx.ctypes.data, flags, 0,
                    ctypes.cast(stats, ctypes.c_void_p).value,
                    ctypes.cast(surf_arg, ctypes.c_void_p).value if surf_arg is not None else None)
        return q, (idx, stats, surf_arg)

    def secondary_phase(self, signal_ptr: int, eltype: int, n_samples: int, if_hz: float, flags: int, items):
        """items: (code int8 [spc], secondary int8 [L], doppler_hz) per detected PRN; returns the phases."""
        keep = []
        arr = (SecondaryRequest * len(items))()
        for i, (code, sec, dop) in enumerate(items):
            c = np.ascontiguousarray(code, dtype=np.int8)
            q = np.ascontiguousarray(sec, dtype=np.int8)
            keep += [c, q]
            arr[i] = SecondaryRequest(c.ctypes.data, q.ctypes.data, float(dop), len(q), 0)
        out = np.zeros(len(items), dtype=np.int32)
        _check(lib().fmdbzp_secondary_phase(self.handle, ctypes.c_void_p(signal_ptr), eltype, n_samples,
                                            float(if_hz), flags, ctypes.cast(arr, ctypes.c_void_p), len(items),
                                            out.ctypes.data), "fmdbzp_secondary_phase")
        return [int(v) for v in out]

    def set_surface_layout(self, nbins: int, chip_order=None):
        order = None if chip_order is None else np.ascontiguousarray(chip_order, dtype=np.int32)
        _check(lib().fmdbzp_plan_set_surface_layout(self.handle, int(nbins),
                                                    None if order is None else order.ctypes.data),
               "fmdbzp_plan_set_surface_layout")

    def set_timing(self, enable: bool):
        _check(lib().fmdbzp_plan_set_timing(self.handle, 1 if enable else 0), "fmdbzp_plan_set_timing")

    def tuning(self) -> str:
        """The autotuner's record for this plan ("" when it did not run)."""
        buf = ctypes.create_string_buffer(4096)
        _check(lib().fmdbzp_plan_tuning(self.handle, buf, len(buf)), "fmdbzp_plan_tuning")
        return buf.value.decode()

    def column_kernel(self) -> str:
        """Form of this plan's column stage on the tile."""
        buf = ctypes.create_string_buffer(128)
        _check(lib().fmdbzp_plan_column_kernel(self.handle, buf, len(buf)), "fmdbzp_plan_column_kernel")
        return buf.value.decode()

    def call_kernels(self, eltype: int, nreq: int, flags: int = 0) -> str:
        """Kernels that a call over `nreq` PRNs launches for the search: the
        full-period correlation, or block correlation and column kernel."""
        buf = ctypes.create_string_buffer(160)
        _check(lib().fmdbzp_plan_call_kernels(self.handle, eltype, int(nreq), flags, buf, len(buf)),
               "fmdbzp_plan_call_kernels")
        return buf.value.decode()

    def graph_counts(self):
        """(captures, replays) of a plan created with graphs=True."""
        c, r = ctypes.c_int64(), ctypes.c_int64()
        _check(lib().fmdbzp_plan_graph_counts(self.handle, ctypes.byref(c), ctypes.byref(r)),
               "fmdbzp_plan_graph_counts")
        return c.value, r.value

    def kernel_times(self) -> dict:
        n = len(KERNEL_CLASSES)
        ms = (ctypes.c_double * n)()
        cnt = (ctypes.c_int64 * n)()
        lib().fmdbzp_plan_kernel_times(self.handle, ctypes.cast(ms, ctypes.c_void_p),
                                       ctypes.cast(cnt, ctypes.c_void_p), n)
        return {name: (ms[i], cnt[i]) for i, name in enumerate(KERNEL_CLASSES)}

    def destroy(self):
        if self.handle:
            lib().fmdbzp_plan_destroy(self.handle)
            self.handle = None
