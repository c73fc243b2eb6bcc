"""Tall units of the strip spreader (up to 33 - w rows, in 16-column frames; of widths above
8 up to 128 rows, over which the accumulators roll): asked for through gpu_binsizey on
grids of whole and part units, against the plain scatter on the same grid, and chosen by the
density of a ragged batch and of a plan.

The bound is that of test_gpu_strip_tiles: both add the same terms."""

import numpy as np
import pytest
import torch

from gpu_helpers import CDT, clustered_points, cnormal, dev, host, rel_l2, uniform_points
from jax_finufft_amd import RaggedPlan, nufft1
from jax_finufft_amd._native import Plan

pytestmark = pytest.mark.gpu

BAR = {"f32": 64 * np.finfo(np.float32).eps / 2, "f64": 64 * np.finfo(np.float64).eps / 2}


def _spread(grid, x, c, eps, prec, method, rows=0):
    plan = Plan(1, grid, iflag=1, ntransf=1, eps=eps, dtype=CDT[prec], gpu_method=method,
                gpu_spreadinterponly=True, gpu_binsizey=rows)
    plan.setpts(*[dev(a) for a in x])
    out = torch.empty((1,) + tuple(grid), dtype=CDT[prec], device="cuda")
    plan.execute(dev(c), out)
    torch.cuda.synchronize()
    plan.destroy()
    return host(out)


@pytest.mark.parametrize("prec,eps", [("f32", e) for e in (1e-1, 1e-2, 1e-3, 1e-4, 1e-5, 1e-6)] +
                         [("f64", e) for e in (1e-1, 1e-4, 1e-6, 1e-7, 1e-8, 1e-9, 1e-11, 1e-12, 1e-14)])
@pytest.mark.parametrize("rows", [10, 17, 40, 100])
def test_unit_heights_match_scatter(prec, eps, rows):
    rng = np.random.default_rng(59)
    for grid, M in (((64, 67), 1), ((45, 131), 65), ((97, 200), 2500), ((33, 34, 71), 700)):
        for gen in (uniform_points, clustered_points):
            x = gen(rng, len(grid), M, prec)
            c = cnormal(rng, M, prec)
            a = _spread(grid, x, c, eps, prec, 3, rows)
            b = _spread(grid, x, c, eps, prec, 1)
            assert rel_l2(a, b) <= BAR[prec], (grid, M)


@pytest.mark.parametrize("prec,eps", [("f32", 1e-4), ("f32", 1e-6), ("f64", 1e-6), ("f64", 1e-14)])
def test_sparse_grids_match_scatter(prec, eps):
    # a few to some tens of points a short unit of many
    rng = np.random.default_rng(60)
    for grid, M in (((2000, 1500), 60_000), ((96, 100, 110), 6_000),
                    ((4100, 4050), 300_000)):
        x = uniform_points(rng, len(grid), M, prec)
        c = cnormal(rng, M, prec)
        assert rel_l2(_spread(grid, x, c, eps, prec, 0), _spread(grid, x, c, eps, prec, 1)) <= \
            BAR[prec], grid


@pytest.mark.parametrize("prec,eps", [("f32", 1e-5), ("f64", 1e-6), ("f64", 1e-10)])
@pytest.mark.parametrize("rows", [0, 60])
def test_sparse_ragged_batch_matches_single_calls(prec, eps, rows):
    rng = np.random.default_rng(61)
    nprob = 24
    shapes = [(128, 128) if i % 3 else (70, 150) for i in range(nprob)]
    ms = [int(m) for m in rng.integers(300, 3000, nprob)]
    ts = [1 + i % 3 for i in range(nprob)]
    pts = [uniform_points(rng, 2, m, prec) for m in ms]
    xs, ys = [dev(p[0]) for p in pts], [dev(p[1]) for p in pts]
    cs = [dev(cnormal(rng, (t, m), prec)) for t, m in zip(ts, ms)]
    plan = RaggedPlan(shapes, ms, ts, eps=eps, dtype=CDT[prec], graph=False, rows=rows)
    got = plan.run(xs, ys, cs)
    for s, x, y, c, f in zip(shapes, xs, ys, cs, got):
        one = nufft1(s, c, x, y, eps=eps)
        assert rel_l2(host(f).ravel(), host(one).ravel()) < (2e-6 if prec == "f32" else 1e-13)
