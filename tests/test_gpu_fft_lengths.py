"""Fine axes below 4096 cells that the one-kernel passes refuse (2000 and 3000 in fp32,
3000 and 3600 in fp64, among others) run through rocFFT, as do their plans' other axes:
against the FP64 direct sums."""

import numpy as np
import pytest

import oracle
from gpu_helpers import cnormal, dev, host, rel_l2, uniform_points
from jax_finufft_amd import nufft1, nufft2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,eps", [("f32", 1e-6), ("f64", 1e-11)])
@pytest.mark.parametrize("n_modes", [(1000, 9), (12, 1500), (1800, 7), (5, 6, 1000)], ids=str)
def test_lengths_between_vs_direct_sum(n_modes, prec, eps):
    rng = np.random.default_rng(32)
    M = 300
    x = uniform_points(rng, len(n_modes), M, prec)
    c, f = cnormal(rng, M, prec), cnormal(rng, n_modes, prec)
    xd = [dev(a) for a in x]
    assert rel_l2(host(nufft1(n_modes, dev(c), *xd, eps=eps)), oracle.type1(x, c, n_modes, 1)) <= eps
    assert rel_l2(host(nufft2(dev(f), *xd, eps=eps)), oracle.type2(f, x, -1)) <= eps
