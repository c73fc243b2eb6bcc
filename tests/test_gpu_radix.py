"""The point sort at the sizes where its launches change: one workgroup (2, 4,
8 or 16 keys per thread), narrow tiles, wide tiles, and one to three passes.
The checks are those of test_gpu_setpts (bijection, order, stability, bin starts).
"""

import pytest

from jax_finufft_amd import Plan
from test_gpu_setpts import _pts, check_sort

pytestmark = pytest.mark.gpu

# (type, modes, options): 3- and 11-bit bins, a strip grid (18 key bits), a 3D
# interpolation grid of 23-bit bins
GRIDS = {
    "keyed_1d": (2, (3000,), dict(gpu_method=2)),
    "keyed_2d": (2, (700, 600), dict(gpu_method=2)),
    "strip_2d": (1, (300, 500), {}),
    "gathered_3d": (2, (96, 80, 100), dict(gpu_method=2, gpu_binsizex=2, gpu_binsizey=1,
                                           gpu_binsizez=1)),
}
SIZES = [11, 2048, 2049, 4097, 8193, 16384, 16385, (1 << 21) - 1, (1 << 21) + 3]


@pytest.mark.parametrize("M", SIZES)
@pytest.mark.parametrize("grid", list(GRIDS))
@pytest.mark.parametrize("dist", ["uniform", "clustered"])
def test_sort_at_size_edges(grid, dist, M):
    import torch

    typ, modes, opts = GRIDS[grid]
    plan = Plan(typ, modes, eps=1e-5, dtype=torch.complex64, device="cuda", **opts)
    # a larger call first: the sort then runs in buffers sized for more points
    big = _pts(M + 5000, len(modes), dist, 3, torch.float32)
    plan.setpts(*big)
    pts = _pts(M, len(modes), dist, 18, torch.float32)
    plan.setpts(*pts)
    check_sort(plan, pts)
    plan.destroy()
