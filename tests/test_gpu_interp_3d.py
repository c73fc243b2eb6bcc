"""3D interpolation from LDS tiles (loaded by slabs in 16-byte values, or by rows
where grid, bins or the caller's pointer do not allow it; a lane or two per point),
against the plain gather on the same grid.

Both sum the same terms f kx ky kz: in units u of rounding, a term's three weights
are off by a few u each of their peak and its three products by 3, sums of random
terms by no more than that again: 96 u in the rel-l2 norm bounds the difference."""

import numpy as np
import pytest
import torch

from gpu_helpers import CDT, NPR, clustered_points, cnormal, dev, host, rel_l2, uniform_points
from jax_finufft_amd._native import Plan

pytestmark = pytest.mark.gpu


def _interp(grid, x, f, eps, prec, method, **opts):
    M = len(x[0])
    plan = Plan(2, grid, iflag=1, ntransf=1, eps=eps, dtype=CDT[prec], gpu_method=method,
                gpu_spreadinterponly=True, **opts)
    plan.setpts(*[dev(a) for a in x])
    out = torch.empty((1, M), dtype=CDT[prec], device="cuda")
    plan.execute(out, f)
    torch.cuda.synchronize()
    plan.destroy()
    return host(out)


@pytest.mark.parametrize("prec,eps", [("f32", e) for e in (1e-1, 1e-2, 1e-3, 1e-4, 1e-5, 1e-6)] +
                         [("f64", e) for e in (1e-4, 1e-7, 1e-9, 1e-11, 1e-14)])
@pytest.mark.parametrize("grid,bins", [((40, 36, 44), (0, 0, 0)), ((35, 34, 33), (0, 0, 0)),
                                       ((40, 36, 44), (5, 4, 6)), ((36, 48, 40), (12, 6, 4))],
                         ids=str)
def test_tiles_match_gather(prec, eps, grid, bins):
    rng = np.random.default_rng(63)
    bar = 96 * (np.finfo(np.float32).eps if prec == "f32" else np.finfo(np.float64).eps) / 2
    opts = dict(gpu_binsizex=bins[0], gpu_binsizey=bins[1], gpu_binsizez=bins[2])
    # the grid on a 16-byte boundary and 8 (16 for doubles) bytes past one
    values = dev(cnormal(rng, (1 + int(np.prod(grid)),), prec))
    aligned = values[:-1].clone().reshape((1,) + grid)
    # points of one bin: about the half and the whole of a workgroup's lanes
    for M, gen in ((1, uniform_points), (20000, clustered_points), (127, None), (129, None),
                   (257, None), (385, None), (1500, None)):
        if gen:
            x = gen(rng, 3, M, prec)
        else:
            x = [rng.uniform(0.0, 0.05, M).astype(NPR[prec]) for _ in range(3)]
        for f in (aligned, values[1:].reshape((1,) + grid)):
            a = _interp(grid, x, f, eps, prec, 2, **opts)
            b = _interp(grid, x, f, eps, prec, 1)
            assert rel_l2(a, b) <= bar, (M,)
