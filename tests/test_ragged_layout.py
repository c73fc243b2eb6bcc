"""Host-side tables of ragged batches (no device work): jfa_ragged_check_layout
builds the tables jfa_ragged_makeplan builds and checks every offset and range
against the buffer sizes the plan allocates.  Run over the benchmark's
64-problem batch, edge cases and many random batches, with the totals checked
against an independent recount here."""

import ctypes

import numpy as np
import pytest

from jax_finufft_amd import _native

I64P = ctypes.POINTER(ctypes.c_int64)


@pytest.fixture(scope="module")
def L():
    L = _native.lib()
    L.jfa_ragged_check_layout.argtypes = [ctypes.c_int, ctypes.c_int, I64P, I64P, I64P,
                                          ctypes.c_double, ctypes.c_int,
                                          ctypes.POINTER(_native.JfaOpts), I64P]
    L.jfa_ragged_check_layout.restype = ctypes.c_int
    L.jfa_fine_grid_size.argtypes = [ctypes.c_int64, ctypes.c_double, ctypes.c_int]
    L.jfa_fine_grid_size.restype = ctypes.c_int64
    return L


def _check(L, Ns, Ts, Ms, eps=1e-6, dbl=0, **opts):
    nmodes = np.array([[n0, n1] for n0, n1 in Ns], dtype=np.int64).ravel()
    ntr = np.asarray(Ts, dtype=np.int64)
    npts = np.asarray(Ms, dtype=np.int64)
    o = _native.JfaOpts()
    L.jfa_default_opts(ctypes.byref(o))
    for k, v in opts.items():
        setattr(o, k, v)
    info = np.zeros(8, dtype=np.int64)
    rc = L.jfa_ragged_check_layout(2, len(Ms), nmodes.ctypes.data_as(I64P),
                                   ntr.ctypes.data_as(I64P), npts.ctypes.data_as(I64P), eps,
                                   dbl, ctypes.byref(o), info.ctypes.data_as(I64P))
    return rc, info


def _fine(L, n, ns):
    return int(L.jfa_fine_grid_size(int(n), 2.0, int(ns)))


def test_benchmark_batch(L):
    # the bench's 64-problem batch: M log-uniform in [1e4, 2e6], N in {64..512}^2,
    # 1-8 transforms, default_rng(7)
    rng = np.random.default_rng(7)
    nprob = 64
    Ms = np.round(10 ** rng.uniform(4, np.log10(2e6), nprob)).astype(int)
    Ns = rng.choice([64, 128, 256, 512], nprob)
    Ts = rng.integers(1, 9, nprob)
    rc, info = _check(L, [(n, n) for n in Ns], Ts, Ms)
    assert rc == 0, _native.last_error()
    ns = 8  # eps 1e-6, single precision
    assert info[0] == Ms.sum()
    assert info[3] == Ts.sum()
    assert info[4] == sum(t * _fine(L, n, ns) ** 2 for n, t in zip(Ns, Ts))
    assert info[5] == sum(t * n * _fine(L, n, ns) for n, t in zip(Ns, Ts))


@pytest.mark.parametrize("case", [
    ([(32, 32)], [1], [0]),                    # one empty problem, smallest fine grid
    ([(32, 40)], [7], [123]),                  # odd transform count, unequal axes
    ([(64, 64)] * 9, [2] * 9, [5000] * 9),     # one fine-grid class
    ([(512, 512), (40, 300)], [8, 1], [2_000_000, 1]),
    ([(100, 33), (33, 100), (100, 33)], [3, 4, 5], [0, 70000, 9]),
])
def test_edge_batches(L, case):
    Ns, Ts, Ms = case
    rc, info = _check(L, Ns, Ts, Ms)
    assert rc == 0, _native.last_error()
    assert info[0] == sum(Ms) and info[3] == sum(Ts)


@pytest.mark.parametrize("case", [
    # many full pieces a unit and several transforms: one workgroup per piece
    # of every transform
    ([(64, 64)], [3], [2_000_000]),
    ([(64, 64)], [8], [2_000_000]),
    ([(128, 128), (33, 40)], [4, 1], [1_000_000, 0]),
    ([(64, 64), (100, 80)], [5, 2], [100_000, 60_000]),
])
@pytest.mark.parametrize("pmax", [0, 256])
def test_workgroups_cover_every_piece(L, case, pmax):
    Ns, Ts, Ms = case
    rc, info = _check(L, Ns, Ts, Ms, gpu_maxsubprobsize=pmax)
    assert rc == 0, _native.last_error()


@pytest.mark.parametrize("seed", range(12))
def test_random_batches(L, seed):
    rng = np.random.default_rng(100 + seed)
    nprob = int(rng.integers(1, 40))
    Ns = [(int(rng.integers(32, 600)), int(rng.integers(8, 600))) for _ in range(nprob)]
    Ts = rng.integers(1, 10, nprob)
    Ms = np.round(10 ** rng.uniform(0, 6, nprob)).astype(int)
    dbl = int(seed % 2)
    eps = [1e-3, 1e-6, 1e-9][seed % 3] if dbl else [1e-3, 1e-5, 1e-6][seed % 3]
    rows = [0, 16, 32][seed % 3]
    rc, info = _check(L, Ns, Ts, Ms, eps=eps, dbl=dbl, gpu_binsizey=rows,
                      gpu_maxsubprobsize=[0, 1024, 8192][seed % 3])
    assert rc == 0, _native.last_error()
    assert info[0] == Ms.sum() and info[3] == Ts.sum()


@pytest.mark.parametrize("eps", [1e-1, 1e-3, 1e-6])
def test_tuning_candidates_differ(L, eps):
    # dense problems, whose default units are the short ones
    from jax_finufft_amd.autotune import RAGGED_CANDIDATES

    units = []
    for rows, pmax in RAGGED_CANDIDATES:
        rc, info = _check(L, [(200, 300)], [2], [900_000], eps=eps, gpu_binsizey=rows,
                          gpu_maxsubprobsize=pmax)
        assert rc == 0, _native.last_error()
        units.append((int(info[2]), int(info[7])))
    assert len(set(units)) == len(units), units


def test_bad_arguments_are_rejected(L):
    rc, _ = _check(L, [(32, 32)], [0], [10])
    assert rc == 2 and "ntransf" in _native.last_error()
    # below the strip spreader's 64-column minimum
    rc, _ = _check(L, [(32, 32), (16, 64)], [1, 1], [10, 10])
    assert rc == 6 and "minimum" in _native.last_error()
