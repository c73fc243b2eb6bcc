"""FFT passes of more threads than one launch may have: 5600 transforms whose y pass has
one column a workgroup, 4.4e9 threads in all.  The last and the first transforms against
single calls."""

import numpy as np
import pytest
import torch

from gpu_helpers import cnormal, dev, host, rel_l2, uniform_points
from jax_finufft_amd import _native, nufft2

pytestmark = pytest.mark.gpu


def test_passes_beyond_one_launch():
    if torch.cuda.mem_get_info()[0] < (80 << 30):
        pytest.skip("needs 80 GB of device memory")
    rng = np.random.default_rng(91)
    T, modes, eps = 5600, (2048, 30, 1), 1e-1
    x = [dev(a) for a in uniform_points(rng, 3, 50, "f32")]
    f = torch.zeros((T,) + modes, dtype=torch.complex64, device="cuda")
    some = [0, 1, T - 2, T - 1]
    for t in some:
        f[t] = dev(cnormal(rng, modes, "f32"))
    got = nufft2(f, *x, eps=eps)
    for t in some:
        assert rel_l2(host(got[t]), host(nufft2(f[t], *x, eps=eps))) <= 1e-6, t
    assert not got[2:T - 2].any()
    del got, f
    _native.lib().jfa_cache_clear()  # the plan holds 54 GB
    torch.cuda.empty_cache()
