"""The strip spreader's tiles at every kernel width: both precisions, both kernel
evaluations, one and several waves a piece, short last batches, points at every
column and row of a strip, against the plain scatter on the same grid.

Both add the same terms c kx ky.  In units u of rounding, a term's two weights are
off by a few u each of their peak (Horner of at most 19 coefficients) and its two
products by 2, sums of random terms by no more than that again: 64 u in the
rel-l2 norm bounds the difference."""

import numpy as np
import pytest
import torch

from gpu_helpers import CDT, clustered_points, cnormal, dev, host, rel_l2, uniform_points
from jax_finufft_amd._native import Plan

pytestmark = pytest.mark.gpu

WIDTHS = [("f32", e) for e in (1e-1, 1e-2, 1e-3, 1e-4, 1e-5, 1e-6)] + \
         [("f64", e) for e in (1e-1, 1e-4, 1e-6, 1e-7, 1e-8, 1e-9, 1e-11, 1e-13, 1e-15)]


def _spread(grid, x, c, eps, prec, method, kerevalmeth, pmax=0):
    plan = Plan(1, grid, iflag=1, ntransf=1, eps=eps, dtype=CDT[prec], gpu_method=method,
                gpu_kerevalmeth=kerevalmeth, gpu_spreadinterponly=True, gpu_maxsubprobsize=pmax)
    plan.setpts(*[dev(a) for a in x])
    out = torch.empty((1,) + tuple(grid), dtype=CDT[prec], device="cuda")
    plan.execute(dev(c), out)
    torch.cuda.synchronize()
    plan.destroy()
    return host(out)


# fewer columns than a strip: one strip that wraps onto itself, or a second of few
@pytest.mark.parametrize("columns", [32, 33, 48, 49, 50, 53, 57, 58, 60, 61, 63])
@pytest.mark.parametrize("prec,eps", [("f32", 1e-2), ("f32", 1e-4), ("f32", 1e-6),
                                      ("f64", 1e-7), ("f64", 1e-11), ("f64", 1e-15)])
def test_narrow_grids_match_scatter(prec, eps, columns):
    rng = np.random.default_rng(58)
    bar = 64 * (np.finfo(np.float32).eps if prec == "f32" else np.finfo(np.float64).eps) / 2
    for grid, M in (((32, columns), 33), ((75, columns), 9001), ((33, 34, columns), 2500)):
        x = uniform_points(rng, len(grid), M, prec)
        c = cnormal(rng, M, prec)
        a = _spread(grid, x, c, eps, prec, 0, 1)
        b = _spread(grid, x, c, eps, prec, 1, 1)
        assert rel_l2(a, b) <= bar, (grid, M)


@pytest.mark.parametrize("prec,eps", WIDTHS)
@pytest.mark.parametrize("kerevalmeth", [0, 1])
def test_tiles_match_scatter(prec, eps, kerevalmeth):
    rng = np.random.default_rng(57)
    bar = 64 * (np.finfo(np.float32).eps if prec == "f32" else np.finfo(np.float64).eps) / 2
    for grid, M, pmax in (((64, 67), 1, 0), ((45, 131), 65, 0), ((97, 200), 6001, 0),
                          ((97, 200), 6001, 130), ((33, 34, 71), 700, 0)):
        for gen in (uniform_points, clustered_points):
            x = gen(rng, len(grid), M, prec)
            c = cnormal(rng, M, prec)
            a = _spread(grid, x, c, eps, prec, 3, kerevalmeth, pmax)
            b = _spread(grid, x, c, eps, prec, 1, kerevalmeth)
            assert rel_l2(a, b) <= bar, (grid, M, pmax)
