"""Type-3 deconvolution factors from the fp32 plans' series, over the whole range of
target frequencies: ends of the range, flat axes, both upsampling factors, against the
FP64 direct sum.  Bars as for the other type-3 tests: eps, and twice eps at 1.25."""

import numpy as np
import pytest

import oracle
from gpu_helpers import cnormal, dev, host, rel_l2
from jax_finufft_amd import nufft3
from jax_finufft_amd.options import Opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("upsampfac,eps", [(2.0, 1e-2), (2.0, 1e-4), (2.0, 1e-5), (1.25, 1e-3),
                                           (1.25, 1e-4)])
@pytest.mark.parametrize("flat", [0, 1])
@pytest.mark.parametrize("ndim", [1, 2, 3])
def test_factors_over_the_range(ndim, flat, upsampfac, eps):
    if ndim == 3 and not flat and upsampfac != 2.0:
        pytest.skip("targets in the corners of three axes: their small psi_hat at 1.25 amplifies "
                    "fp32 rounding past eps, with the quadrature's factors as well")
    rng = np.random.default_rng(71)
    M, N = 600, 300
    x = [rng.uniform(-3.0, 3.0, M).astype(np.float32) for _ in range(ndim)]
    s = [rng.uniform(-9.0, 9.0, N).astype(np.float32) for _ in range(ndim)]
    for a in s:  # half of the targets at the ends of the range
        a[: N // 2] = np.float32(9.0) * rng.choice([-1, 1], N // 2)
    if flat:
        s[-1][:] = np.float32(4.5)
    c = cnormal(rng, M, "f32")
    opts = Opts(gpu_upsampfac=upsampfac)
    got = host(nufft3(dev(c), *[dev(a) for a in x], *[dev(a) for a in s], eps=eps, opts=opts))
    bar = eps if upsampfac == 2.0 else 2 * eps
    assert rel_l2(got, oracle.type3(c, x, s, -1)) <= bar
