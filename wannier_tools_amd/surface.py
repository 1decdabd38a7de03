"""Host-side mirror of the reference's surface Green's function interface.

Thin ctypes front over ``libwtsurf.so`` (the HIP library, C ABI in
``include/wtsurf.h``).  The names and argument meanings follow the
reference's Fortran routines:

* ``SurfaceGF.ham_qlayer2qlayer``  -- src/ham_qlayer2qlayer.f90:1-102
* ``SurfaceGF.surfgreen_1985``     -- src/surfgreen.f90:7-137
* ``SurfaceGF.spectral_grid``      -- the (k, omega) loops and traces of
  surfstat (src/surfstat.f90:123-160) and SurfaceDOSkk
  (src/fermiarc.f90:206-248)
* ``SurfaceGF.set_spin_traces`` / ``spin_download`` -- the spin-resolved
  traces of surfstat (src/surfstat.f90:163-192) and SurfaceDOSkk
  (src/fermiarc.f90:250-328)
* ``SurfaceGF.kplane_autocorrelation`` -- the QPI jdos / jsdos sums of
  SurfaceDOSkk (src/fermiarc.f90:496-560)
* ``SurfaceGF.kpath_jdos`` -- the k-path jdos of surfstat_jdos
  (src/surfstat.f90:891-907)

There is no CPU fallback: constructing a ``SurfaceGF`` without the built
library, or without a HIP device, raises.
"""
from __future__ import annotations

import ctypes
import os
from typing import Optional, Sequence

import numpy as np

from .model import DECIMATION_ACCURACY, DECIMATION_ITERMAX, TBModel

LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libwtsurf.so")

FP64 = 0
FP32 = 1
MIXED = 2
_PRECISION = {"fp64": FP64, "fp32": FP32, "mixed": MIXED, FP64: FP64, FP32: FP32, MIXED: MIXED}

STATUS_SINGULAR = 1
STATUS_NOT_CONVERGED = 2

_dp = ctypes.POINTER(ctypes.c_double)
_ip = ctypes.POINTER(ctypes.c_int)
_fp = ctypes.POINTER(ctypes.c_float)

# Every symbol include/wtsurf.h declares: (name, restype, argtypes)
SIGNATURES = {
    "wtsurf_ctx_create": (ctypes.c_int, [ctypes.c_int, ctypes.POINTER(ctypes.c_void_p)]),
    "wtsurf_ctx_destroy": (None, [ctypes.c_void_p]),
    "wtsurf_last_error": (ctypes.c_char_p, [ctypes.c_void_p]),
    "wtsurf_set_model": (ctypes.c_int, [ctypes.c_void_p] + [ctypes.c_int] * 4 + [_ip, _dp]),
    "wtsurf_set_stop_rule": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, ctypes.c_double]),
    "wtsurf_set_orbitals": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, _ip, ctypes.c_int, _ip]),
    "wtsurf_ham_qlayer2qlayer": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, _dp, _dp, _dp]),
    "wtsurf_surfgreen_1985": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, ctypes.c_double,
                                             ctypes.c_double, _dp, _dp, _dp, _dp, _dp, _ip]),
    "wtsurf_surfgreen_1985_noalloc": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, ctypes.c_double,
                                                     ctypes.c_double] + [ctypes.c_void_p] * 6),
    "wtsurf_spectral_grid": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, _dp, ctypes.c_int, _dp,
                                            ctypes.c_double, ctypes.c_double, ctypes.c_int,
                                            _dp, _dp, _dp, _ip, _ip]),
    "wtsurf_spectral_batch": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, _dp, ctypes.c_int, _ip,
                                             _dp, _dp, ctypes.c_double, ctypes.c_int,
                                             _dp, _dp, _dp, _ip, _ip]),
    "wtsurf_grid_upload": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int, _dp, ctypes.c_int, _dp]),
    "wtsurf_grid_run_async": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_double, ctypes.c_double,
                                             ctypes.c_int]),
    "wtsurf_sync": (ctypes.c_int, [ctypes.c_void_p]),
    "wtsurf_grid_timing": (ctypes.c_int, [ctypes.c_void_p, _fp, _fp]),
    "wtsurf_grid_download": (ctypes.c_int, [ctypes.c_void_p, _dp, _dp, _dp, _ip, _ip]),
    "wtsurf_set_spin_traces": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int]),
    "wtsurf_set_schedule": (ctypes.c_int, [ctypes.c_void_p, ctypes.c_int]),
    "wtsurf_spin_download": (ctypes.c_int, [ctypes.c_void_p, _dp, _dp]),
    "wtsurf_kplane_autocorrelation": (ctypes.c_int, [ctypes.c_void_p] + [ctypes.c_int] * 5
                                      + [_dp, _dp]),
    "wtsurf_kpath_jdos": (ctypes.c_int, [ctypes.c_void_p] + [ctypes.c_int] * 3 + [_dp, _dp]),
    "wtsurf_kpath_jdos_energy_fastest": (ctypes.c_int, [ctypes.c_void_p] + [ctypes.c_int] * 3
                                         + [_dp, _dp]),
    "wtsurf_max_ndim": (ctypes.c_int, []),
}

# Spin-resolved trace modes (which orbitals GRR's spin sums run over)
SPIN_OFF = 0
SPIN_SURFSTAT = 1   # top orbital indices, as surfstat (src/surfstat.f90:178-191)
SPIN_ARC = 2        # bottom orbitals of the last layer, as SurfaceDOSkk (src/fermiarc.f90:298-327)
_SPIN = {"off": SPIN_OFF, "surfstat": SPIN_SURFSTAT, "arc": SPIN_ARC,
         SPIN_OFF: SPIN_OFF, SPIN_SURFSTAT: SPIN_SURFSTAT, SPIN_ARC: SPIN_ARC}

_lib: Optional[ctypes.CDLL] = None


def load_library(path: str = LIB_PATH) -> ctypes.CDLL:
    """Load libwtsurf.so and declare every C-ABI signature (no device calls)."""
    global _lib
    if _lib is not None and path == LIB_PATH:
        return _lib
    if not os.path.exists(path):
        raise RuntimeError(f"{path} is not built; run __graft_entry__.build() first")
    lib = ctypes.CDLL(path)
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    if path == LIB_PATH:
        _lib = lib
    return lib


def _dptr(a: np.ndarray):
    return a.ctypes.data_as(_dp)


def _iptr(a: np.ndarray):
    return a.ctypes.data_as(_ip)


class WtsurfError(RuntimeError):
    pass


class SurfaceGF:
    """One wtsurf context (device buffers + stream) on HIP device ``device``."""

    def __init__(self, device: int = 0):
        self.lib = load_library()
        h = ctypes.c_void_p()
        rc = self.lib.wtsurf_ctx_create(device, ctypes.byref(h))
        if rc != 0 or not h.value:
            raise WtsurfError(f"wtsurf_ctx_create(device={device}) failed ({rc}): no usable HIP device")
        self.ctx = h
        self.n = 0
        self.nw = 0
        self.np = 0
        self._grid = (0, 0)
        self._last_shape = None  # output shape of the last grid or batch run

    def close(self) -> None:
        if getattr(self, "ctx", None) is not None and self.ctx.value:
            self.lib.wtsurf_ctx_destroy(self.ctx)
            self.ctx = None

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.close()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def _check(self, rc: int, what: str) -> None:
        if rc != 0:
            msg = self.lib.wtsurf_last_error(self.ctx)
            raise WtsurfError(f"{what} failed ({rc}): {msg.decode() if msg else ''}")

    # ---- model state (module para in the reference) -----------------------
    def set_model_arrays(self, nw: int, np_: int, irvec: np.ndarray, hr: np.ndarray,
                         ijmax: int = 10) -> None:
        """irvec (nr, 3) ints and hr (nr, nw, nw) complex, already in the units
        and ndegen normalisation of HmnR_surfacecell."""
        irvec = np.ascontiguousarray(irvec, dtype=np.int32).reshape(-1, 3)
        hr = np.asarray(hr, dtype=np.complex128).reshape(-1, nw, nw)
        if hr.shape[0] != irvec.shape[0]:
            raise ValueError("irvec and hr disagree on the number of R vectors")
        hr_cm = np.ascontiguousarray(hr.transpose(0, 2, 1))  # column-major blocks
        self._check(self.lib.wtsurf_set_model(self.ctx, nw, np_, irvec.shape[0], ijmax,
                                              _iptr(irvec), _dptr(hr_cm.view(np.float64))),
                    "wtsurf_set_model")
        self.nw, self.np, self.n = nw, np_, nw * np_
        self._grid = (0, 0)  # the library drops the grid and the last run with the model
        self._last_shape = None

    def set_model(self, model: TBModel, np_: int, ijmax: int = 10) -> None:
        irvec, hr = model.surface_cell()
        self.set_model_arrays(model.num_wann, np_, irvec, hr, ijmax)

    def set_stop_rule(self, itermax: int = DECIMATION_ITERMAX,
                      accuracy: float = DECIMATION_ACCURACY) -> None:
        self._check(self.lib.wtsurf_set_stop_rule(self.ctx, int(itermax), float(accuracy)),
                    "wtsurf_set_stop_rule")

    def set_orbitals(self, top: Sequence[int], bot: Sequence[int]) -> None:
        """1-based TopOrbitals (1..Ndim) and BottomOrbitals (1..Num_wann)."""
        t = np.ascontiguousarray(top, dtype=np.int32)
        b = np.ascontiguousarray(bot, dtype=np.int32)
        self._check(self.lib.wtsurf_set_orbitals(self.ctx, t.size, _iptr(t), b.size, _iptr(b)),
                    "wtsurf_set_orbitals")

    # ---- per-call entry points ---------------------------------------------
    def ham_qlayer2qlayer(self, kpts) -> tuple[np.ndarray, np.ndarray]:
        """H00(k), H01(k) for kpts of shape (nk, 2) or (2,); returns arrays of
        shape (nk, N, N) (or (N, N) for a single k)."""
        k = np.ascontiguousarray(kpts, dtype=np.float64)
        single = k.ndim == 1
        k = k.reshape(-1, 2)
        nk, n = k.shape[0], self.n
        h00 = np.zeros((nk, n, n), dtype=np.complex128)
        h01 = np.zeros((nk, n, n), dtype=np.complex128)
        self._check(self.lib.wtsurf_ham_qlayer2qlayer(self.ctx, nk, _dptr(k), _dptr(h00.view(np.float64)),
                                                      _dptr(h01.view(np.float64))),
                    "wtsurf_ham_qlayer2qlayer")
        self._grid = (0, 0)  # the call replaces the device's k points and H00/H01
        self._last_shape = None
        h00 = h00.transpose(0, 2, 1)
        h01 = h01.transpose(0, 2, 1)
        return (h00[0], h01[0]) if single else (h00, h01)

    def surfgreen_1985(self, omega: float, h00: np.ndarray, h01: np.ndarray,
                       eta: float) -> tuple[np.ndarray, np.ndarray, np.ndarray, int]:
        """(GLL, GRR, GB, iterations) for one (omega, eta) instance."""
        h00 = np.asfortranarray(h00, dtype=np.complex128)
        h01 = np.asfortranarray(h01, dtype=np.complex128)
        n = h00.shape[0]
        if h00.shape != (n, n) or h01.shape != (n, n):
            raise ValueError("H00 and H01 must be square and of the same order")
        g = [np.zeros((n, n), dtype=np.complex128, order="F") for _ in range(3)]
        it = np.zeros(1, dtype=np.int32)
        self._check(self.lib.wtsurf_surfgreen_1985(
            self.ctx, n, float(omega), float(eta), h00.ctypes.data_as(_dp), h01.ctypes.data_as(_dp),
            g[0].ctypes.data_as(_dp), g[1].ctypes.data_as(_dp), g[2].ctypes.data_as(_dp), _iptr(it)),
            "wtsurf_surfgreen_1985")
        # the call works in buffers of its own: the grid and the last run stay
        return g[0], g[1], g[2], int(it[0])

    def surfgreen_1985_noalloc(self, n: int, omega: float, eta: float, d_h00: int, d_h01: int,
                               d_gll: int, d_grr: int, d_gb: int, d_iters: int = 0) -> None:
        """surfgreen_1985 on device buffers (integer device addresses of
        column-major n x n complex128 arrays; d_iters of one int32 or 0),
        allocating no device memory (n <= 80)."""
        self._check(self.lib.wtsurf_surfgreen_1985_noalloc(
            self.ctx, int(n), float(omega), float(eta), d_h00, d_h01, d_gll, d_grr, d_gb,
            d_iters or None), "wtsurf_surfgreen_1985_noalloc")

    def spectral_grid(self, kpts, omegas, eta: float, divisor: float = 1.0,
                      precision="fp64"):
        """dos_l, dos_r, dos_bulk (shape (nk, nomega)), iterations, status."""
        self.upload_grid(kpts, omegas)
        self.run_async(eta, divisor, precision)
        self.sync()
        return self.download()

    def spectral_batch(self, kpts, k_index, omegas, etas, divisor: float = 1.0,
                       precision="fp64"):
        """Per-instance (k_index[i] into kpts, omegas[i], etas[i]): dos_l, dos_r,
        dos_bulk, iterations, status, each of shape (ninst,)."""
        if precision not in _PRECISION:
            raise ValueError(f"unknown precision {precision!r}")
        k = np.ascontiguousarray(kpts, dtype=np.float64).reshape(-1, 2)
        ki = np.ascontiguousarray(k_index, dtype=np.int32).ravel()
        w = np.ascontiguousarray(omegas, dtype=np.float64).ravel()
        e = np.ascontiguousarray(etas, dtype=np.float64).ravel()
        if not (ki.size == w.size == e.size):
            raise ValueError("k_index, omegas and etas must have one entry per instance")
        out = [np.empty(ki.size) for _ in range(3)]
        it = np.empty(ki.size, dtype=np.int32)
        st = np.empty(ki.size, dtype=np.int32)
        self._check(self.lib.wtsurf_spectral_batch(self.ctx, k.shape[0], _dptr(k), ki.size, _iptr(ki),
                                                   _dptr(w), _dptr(e), float(divisor),
                                                   _PRECISION[precision], _dptr(out[0]),
                                                   _dptr(out[1]), _dptr(out[2]), _iptr(it),
                                                   _iptr(st)),
                    "wtsurf_spectral_batch")
        self._grid = (0, 0)
        self._last_shape = (ki.size,)
        return out[0], out[1], out[2], it, st

    def set_schedule(self, schedule="auto") -> None:
        """Decimation schedule (see include/wtsurf.h): "rounds", "persistent"
        (orders up to 80), "small" (FP64, orders up to 32) or "auto"."""
        code = {"rounds": 0, "persistent": 1, "small": 2, "auto": 3}.get(schedule, schedule)
        if code not in (0, 1, 2, 3):
            raise ValueError(f"unknown schedule {schedule!r}")
        self._check(self.lib.wtsurf_set_schedule(self.ctx, code), "wtsurf_set_schedule")

    def set_spin_traces(self, mode="surfstat") -> None:
        """Take spin-resolved traces in the runs that follow: "surfstat",
        "arc" or "off" (see include/wtsurf.h)."""
        if mode not in _SPIN:
            raise ValueError(f"unknown spin trace mode {mode!r}")
        self._check(self.lib.wtsurf_set_spin_traces(self.ctx, _SPIN[mode]),
                    "wtsurf_set_spin_traces")

    def spin_download(self):
        """(spin_l, spin_r) of the last run, each (3,) + that run's output
        shape: sx, sy, sz."""
        if self._last_shape is None:
            raise WtsurfError("no run to download spin traces from")
        shp = self._last_shape
        sl = np.zeros(shp + (3,), dtype=np.float64, order="F")
        sr = np.zeros_like(sl)
        self._check(self.lib.wtsurf_spin_download(self.ctx, _dptr(sl), _dptr(sr)),
                    "wtsurf_spin_download")
        return np.moveaxis(sl, -1, 0), np.moveaxis(sr, -1, 0)

    def kplane_autocorrelation(self, fields, m1: int, m2: int) -> np.ndarray:
        """QPI autocorrelation (see include/wtsurf.h): fields (nfield, nkx, nky)
        or (nkx, nky) indexed [f, ik1-1, ik2-1]; returns (nkx, nky) indexed
        [iq1-1, iq2-1]."""
        f = np.asarray(fields, dtype=np.float64)
        if f.ndim == 2:
            f = f[None]
        nfield, nkx, nky = f.shape
        if max(m1, m2) <= 2048 and m2 >= min(m1, 32):
            # the sum is the same with the axes exchanged, and so is its result:
            # no transposes (the library limits the length of its rows, and is
            # at its best with long ones: 1025 x 3 points 1.0 ms as rows of 2,
            # 0.1 as rows of 1024)
            buf = np.ascontiguousarray(f)
            out = np.empty((nkx, nky), dtype=np.float64)
            self._check(self.lib.wtsurf_kplane_autocorrelation(
                self.ctx, nky, nkx, int(m2), int(m1), nfield, _dptr(buf), _dptr(out)),
                "wtsurf_kplane_autocorrelation")
            return out
        buf = np.ascontiguousarray(f.transpose(0, 2, 1))
        out = np.zeros((nky, nkx), dtype=np.float64)
        self._check(self.lib.wtsurf_kplane_autocorrelation(self.ctx, nkx, nky, int(m1), int(m2),
                                                           nfield, _dptr(buf), _dptr(out)),
                    "wtsurf_kplane_autocorrelation")
        return out.T.copy()

    def kpath_jdos(self, fields) -> np.ndarray:
        """k-path joint density of states (see include/wtsurf.h): fields
        (nfield, nk, nomega) or (nk, nomega) indexed [f, ik-1, j-1]; returns the
        same shape."""
        f = np.asarray(fields, dtype=np.float64)
        single = f.ndim == 2
        if single:
            f = f[None]
        nfield, nk, nom = f.shape
        buf = np.ascontiguousarray(f)
        out = np.empty_like(buf)
        self._check(self.lib.wtsurf_kpath_jdos_energy_fastest(self.ctx, nk, nom, nfield, _dptr(buf),
                                                              _dptr(out)),
                    "wtsurf_kpath_jdos_energy_fastest")
        return out[0] if single else out

    # ---- resident split (inputs stay in device memory) -------------------
    def upload_grid(self, kpts, omegas) -> None:
        k = np.ascontiguousarray(kpts, dtype=np.float64).reshape(-1, 2)
        w = np.ascontiguousarray(omegas, dtype=np.float64).ravel()
        self._check(self.lib.wtsurf_grid_upload(self.ctx, k.shape[0], _dptr(k), w.size, _dptr(w)),
                    "wtsurf_grid_upload")
        self._grid = (k.shape[0], w.size)

    def run_async(self, eta: float, divisor: float = 1.0, precision="fp64") -> None:
        if precision not in _PRECISION:
            raise ValueError(f"unknown precision {precision!r}")
        self._check(self.lib.wtsurf_grid_run_async(self.ctx, float(eta), float(divisor),
                                                   _PRECISION[precision]),
                    "wtsurf_grid_run_async")
        self._last_shape = tuple(self._grid)

    def sync(self) -> None:
        self._check(self.lib.wtsurf_sync(self.ctx), "wtsurf_sync")

    def timing(self) -> tuple[float, float]:
        """Device ms of the Fourier and decimation stages of the last grid run
        or spectral_batch call."""
        a = ctypes.c_float()
        b = ctypes.c_float()
        self._check(self.lib.wtsurf_grid_timing(self.ctx, ctypes.byref(a), ctypes.byref(b)),
                    "wtsurf_grid_timing")
        return a.value, b.value

    def lib_download_raw(self, n: int = 1):
        """wtsurf_grid_download into buffers of n elements, whatever grid the
        host side believes is current (for checking the library's own state)."""
        outs = [np.zeros(n, dtype=np.float64) for _ in range(3)]
        ii = [np.zeros(n, dtype=np.int32) for _ in range(2)]
        self._check(self.lib.wtsurf_grid_download(self.ctx, *(o.ctypes.data_as(_dp) for o in outs),
                                                  *(i.ctypes.data_as(_ip) for i in ii)),
                    "wtsurf_grid_download")
        return outs, ii

    def download(self):
        nk, nw_ = self._grid
        if nk * nw_ == 0 or self._last_shape != (nk, nw_):
            raise WtsurfError("no completed grid run to download")
        outs = [np.zeros((nk, nw_), dtype=np.float64, order="F") for _ in range(3)]
        its = np.zeros((nk, nw_), dtype=np.int32, order="F")
        st = np.zeros((nk, nw_), dtype=np.int32, order="F")
        self._check(self.lib.wtsurf_grid_download(self.ctx, *(o.ctypes.data_as(_dp) for o in outs),
                                                  its.ctypes.data_as(_ip), st.ctypes.data_as(_ip)),
                    "wtsurf_grid_download")
        return outs[0], outs[1], outs[2], its, st


def max_ndim() -> int:
    return int(load_library().wtsurf_max_ndim())
