"""Pruned FFT passes (one kernel per axis) against the FP64 direct sums.

Mode counts are chosen so that the fine axes take every radix, one to four
stages, partial column tiles and both mode orders; the last shape has an axis
beyond the passes' 4096 points, which runs the rocFFT passes instead.
"""

import numpy as np
import pytest

import oracle
from gpu_helpers import cnormal, dev, host, rel_l2, uniform_points
from jax_finufft_amd import nufft1, nufft2
from jax_finufft_amd.options import Opts

pytestmark = pytest.mark.gpu

SHAPES = [(1, 9), (7, 20), (33, 50), (64, 81), (101, 128), (243, 16), (12, 405), (9, 500),
          (1024, 5), (6, 2048), (2050, 7), (16, 20, 12), (9, 25, 30), (13, 50, 8), (10, 8, 100)]


@pytest.mark.parametrize("prec,eps", [("f32", 1e-6), ("f64", 1e-11)])
@pytest.mark.parametrize("modeord", [0, 1])
@pytest.mark.parametrize("n_modes", SHAPES, ids=str)
def test_fft_axis_vs_direct_sum(n_modes, modeord, prec, eps):
    rng = np.random.default_rng(31)
    M = 300
    x = uniform_points(rng, len(n_modes), M, prec)
    c = np.stack([cnormal(rng, M, prec) for _ in range(2)])
    f = np.stack([cnormal(rng, n_modes, prec) for _ in range(2)])
    opts = Opts(modeord=modeord)
    xd = [dev(a) for a in x]
    got1 = host(nufft1(n_modes, dev(c), *xd, eps=eps, opts=opts))
    got2 = host(nufft2(dev(f), *xd, eps=eps, opts=opts))
    axes = tuple(range(len(n_modes)))
    for t in range(2):
        want1 = oracle.type1(x, c[t], n_modes, 1)
        centred = f[t]
        if modeord:
            want1 = np.fft.ifftshift(want1, axes=axes)
            centred = np.fft.fftshift(centred, axes=axes)
        assert rel_l2(got1[t], want1) <= eps
        assert rel_l2(got2[t], oracle.type2(centred, x, -1)) <= eps
