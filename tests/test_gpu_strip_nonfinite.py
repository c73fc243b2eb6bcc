"""Infinite, NaN and nearly overflowing strengths, and NaN coordinates, in spread-only
calls: they reach the cells of their points' taps and no others, as with the plain
scatter, and the cells that only the other points reach hold what those give (a nearly
overflowing strength leaves finite values at its smallest weights, whose rounding, of
the largest weight, is all there is of them)."""

import numpy as np
import pytest
import torch

from gpu_helpers import CDT, NPC, cnormal, dev, host, rel_l2, uniform_points
from jax_finufft_amd._native import Plan

pytestmark = pytest.mark.gpu


def _spread(grid, x, c, eps, prec, method, rows=0):
    plan = Plan(1, grid, iflag=1, ntransf=1, eps=eps, dtype=CDT[prec], gpu_method=method,
                gpu_spreadinterponly=True, gpu_binsizey=rows)
    plan.setpts(*[dev(a) for a in x])
    out = torch.empty((1,) + tuple(grid), dtype=CDT[prec], device="cuda")
    plan.execute(dev(c), out)
    torch.cuda.synchronize()
    plan.destroy()
    return host(out)


# a narrow grid, several strips, many points a unit (four waves a piece), tall units, 3D
@pytest.mark.parametrize("grid,M,rows", [((80, 48), 300, 0), ((150, 300), 900, 0),
                                         ((40, 130), 9000, 0), ((150, 300), 900, 25),
                                         ((36, 34, 70), 500, 0)], ids=str)
@pytest.mark.parametrize("prec,eps", [("f32", 1e-2), ("f32", 1e-6), ("f64", 1e-6), ("f64", 1e-10)])
def test_reach_of_nonfinite_points(prec, eps, grid, M, rows):
    rng = np.random.default_rng(97)
    x = uniform_points(rng, len(grid), M, prec)
    c = cnormal(rng, M, prec)
    big = 3e38 if prec == "f32" else 1.7e308
    special = np.zeros(M, NPC[prec])
    for k, v in enumerate((complex(np.inf, 0), complex(0, -np.inf), complex(np.nan, 1),
                           complex(1, np.nan), complex(big, -big))):
        c[k * (M // 7) + 3] = v
        special[k * (M // 7) + 3] = 1
    x[0][5] = np.nan
    x[-1][M - 2] = np.nan
    a = _spread(grid, x, c, eps, prec, 3 if rows else 0, rows)
    b = _spread(grid, x, c, eps, prec, 1)
    reached = _spread(grid, x, special, eps, prec, 1) != 0  # (NaN, too)
    for u, v in ((a.real, b.real), (a.imag, b.imag)):
        assert np.array_equal(np.isfinite(u), np.isfinite(v))
        bar = 64 * np.finfo(u.dtype).eps / 2
        assert rel_l2(u[~reached], v[~reached]) <= bar
