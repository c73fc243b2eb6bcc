"""Autotuning of the spreading / interpolation geometry.

No reference counterpart: the reference declares ``gpu_method``,
``gpu_binsize{x,y,z}`` and ``gpu_maxsubprobsize`` (src/jax_finufft/
options.py:66-79) but forwards no bin size to the GPU library, whose defaults
are fixed.  Here

- ``autotune(...)`` times the backend's candidate choices for one type-1 or
  type-2 transform on the caller's own device data (``jfa_autotune``), records
  the fastest under the workload's key, and returns it; every later transform
  of that workload that leaves the knobs at their defaults uses the record
  (the C-ABI entry points consult it too).  With ``JFA_TUNE_CACHE=<file>`` in
  the environment the records persist in that JSON file.
- ``tune_ragged(...)`` does the same for a ragged batch: it times ragged plans
  with candidate unit heights and piece sizes and returns the fastest plan.

Explicit knob settings in ``opts`` are never overridden; ``autotune`` refuses
them.
"""

import ctypes
import time

import torch

from . import _native, options
from .ragged import RaggedPlan

__all__ = ["autotune", "tune_ragged", "clear"]

_KNOBS = ("gpu_method", "gpu_binsizex", "gpu_binsizey", "gpu_binsizez", "gpu_maxsubprobsize")


def _lib():
    L = _native.lib()
    L.jfa_autotune.argtypes = [
        ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.c_int64), ctypes.c_int, ctypes.c_int,
        ctypes.c_double, ctypes.c_int, ctypes.POINTER(_native.JfaOpts), ctypes.c_int64,
        ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
        ctypes.POINTER(_native.JfaOpts), ctypes.POINTER(ctypes.c_double),
        ctypes.POINTER(ctypes.c_double)]
    L.jfa_autotune.restype = ctypes.c_int
    L.jfa_tuned_opts.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.c_int64),
                                 ctypes.c_int, ctypes.c_double, ctypes.c_int, ctypes.c_int64,
                                 ctypes.POINTER(_native.JfaOpts)]
    L.jfa_tuned_opts.restype = ctypes.c_int
    L.jfa_tune_clear.restype = None
    return L


def _base_opts(opts, nufft_type, device):
    o = options.unpack_opts(opts, nufft_type, True) or options.Opts()
    native = o.to_native_opts()
    jo = _native.JfaOpts()
    _native.lib().jfa_default_opts(ctypes.byref(jo))
    for k in ("modeord", "upsampfac", "gpu_kerevalmeth", "gpu_sort"):
        setattr(jo, k, native[k])
    # the option set of the transform entry points: explicit knobs only when
    # the caller changed them from the defaults
    if int(o.gpu_method) != 0:
        jo.gpu_method = int(o.gpu_method)
    for k in ("gpu_binsizex", "gpu_binsizey", "gpu_binsizez"):
        setattr(jo, k, native[k])
    jo.gpu_stream = torch.cuda.current_stream(device).cuda_stream
    return jo


def autotune(nufft_type, source, *points, n_modes=None, iflag=None, eps=1e-6, opts=None):
    """Tune one transform and record the choice.

    Type 1: ``source`` is (M,) or (T, M) strengths, ``n_modes`` the output
    shape.  Type 2: ``source`` is (*N) or (T, *N) modes.  ``points`` are the
    (M,) coordinate arrays.  Returns a dict of the chosen knobs plus
    ``best_ms`` and ``default_ms`` (setpts + execute, best of three runs).
    """
    if nufft_type not in (1, 2):
        raise ValueError("autotune covers types 1 and 2")
    ndim = len(points)
    if not 1 <= ndim <= 3:
        raise ValueError("Only 1-, 2-, and 3-dimensions are supported")
    _native._require_device(source, *points)
    single = source.dtype == torch.complex64
    M = int(points[0].numel())
    if nufft_type == 1:
        if n_modes is None or len(n_modes) != ndim:
            raise ValueError("type 1 needs n_modes of length ndim")
        T = source.numel() // max(M, 1) if M else (source.shape[0] if source.dim() == 2 else 1)
        modes = tuple(int(n) for n in n_modes)
        c = source.contiguous()
        fk = torch.empty((T, *modes), dtype=source.dtype, device=source.device)
        iflag = 1 if iflag is None else iflag
    else:
        modes = tuple(int(n) for n in source.shape[-ndim:])
        T = source.numel() // max(1, int(torch.tensor(modes).prod()))
        fk = source.contiguous()
        c = torch.empty((T, M), dtype=source.dtype, device=source.device)
        iflag = -1 if iflag is None else iflag
    jo = _base_opts(opts, nufft_type, source.device)
    if any(getattr(jo, k) for k in _KNOBS) or int(jo.gpu_maxsubprobsize):
        raise ValueError("autotune tunes gpu_method, bin sizes and gpu_maxsubprobsize: leave "
                         "them at their defaults")
    nm = (ctypes.c_int64 * 3)(*(list(modes[::-1]) + [1] * (3 - ndim)))
    pts = [p.contiguous() for p in points[::-1]] + [None] * (3 - ndim)
    P = ctypes.c_void_p
    chosen = _native.JfaOpts()
    best, default = ctypes.c_double(), ctypes.c_double()
    with torch.cuda.device(source.device):
        rc = _lib().jfa_autotune(
            nufft_type, ndim, nm, 1 if iflag >= 0 else -1, int(T), float(eps), int(not single),
            ctypes.byref(jo), M, *[P(p.data_ptr() if p is not None else None) for p in pts],
            P(c.data_ptr()), P(fk.data_ptr()), ctypes.byref(chosen), ctypes.byref(best),
            ctypes.byref(default))
    _native.check(rc, "autotune")
    out = {k: int(getattr(chosen, k)) for k in _KNOBS}
    out.update(best_ms=best.value, default_ms=default.value)
    return out


def tuned_opts(nufft_type, n_modes, ntransf, M, eps, double, upsampfac=2.0):
    """The recorded knobs for a workload (backend defaults where none), as a
    dict, or None when nothing is recorded."""
    jo = _native.JfaOpts()
    _native.lib().jfa_default_opts(ctypes.byref(jo))
    jo.upsampfac = float(upsampfac)
    ndim = len(n_modes)
    nm = (ctypes.c_int64 * 3)(*(list(n_modes[::-1]) + [1] * (3 - ndim)))
    if not _lib().jfa_tuned_opts(nufft_type, ndim, nm, int(ntransf), float(eps), int(double),
                                 int(M), ctypes.byref(jo)):
        return None
    return {k: int(getattr(jo, k)) for k in _KNOBS}


def clear():
    """Forget the in-memory records (the JSON file is left alone)."""
    _lib().jfa_tune_clear()


# unit height (rows, at most 33 - width where that is 25 or more) x piece size for ragged
# batches; (0, 0) is the default rule
RAGGED_CANDIDATES = [(0, 0), (16, 0), (32, 0), (0, 2048), (32, 2048), (32, 8192)]


def tune_ragged(output_shapes, sources, points_x, points_y, iflag=1, eps=1e-6, opts=None,
                graph=True, candidates=RAGGED_CANDIDATES, reps=3):
    """Time ragged plans over candidate (unit height, piece size) pairs on the
    caller's batch; returns ``(best_plan, report)`` with report = list of
    ((rows, pmax), ms) and the default's time first."""
    dtype = sources[0].dtype
    n_points = [int(x.numel()) for x in points_x]
    ntransf = [int(c.numel()) // max(m, 1) if m else (c.shape[0] if c.dim() == 2 else 1)
               for c, m in zip(sources, n_points)]
    dev = sources[0].device
    report, best = [], None
    for rows, pmax in candidates:
        plan = RaggedPlan(output_shapes, n_points, ntransf, iflag=iflag, eps=eps, dtype=dtype,
                          opts=opts, graph=graph, device=dev, rows=rows, pmax=pmax)
        plan.run(points_x, points_y, sources)  # first run (graph capture)
        torch.cuda.synchronize(dev)
        times = []
        for _ in range(reps):
            t0 = time.perf_counter()
            plan.run(points_x, points_y, sources)
            torch.cuda.synchronize(dev)
            times.append((time.perf_counter() - t0) * 1e3)
        ms = min(times)
        report.append(((rows, pmax), ms))
        if best is None or ms < best[1]:
            if best is not None:
                best[0].destroy()
            best = (plan, ms)
        else:
            plan.destroy()
    return best[0], report
