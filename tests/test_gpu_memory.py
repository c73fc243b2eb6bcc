"""What the strip spreader does when its keys, records and tiles are many: a bound on
narrow grids, fewer transforms at a time and then LDS tiles where the device has no room.
Memory is filled by a tensor of the test; what is left is many times what the kernels
that run need."""

import contextlib
import gc

import numpy as np
import pytest
import torch

from gpu_helpers import cnormal, dev, host, rel_l2, uniform_points
from jax_finufft_amd import _native
from jax_finufft_amd._native import Plan

pytestmark = pytest.mark.gpu

TILES, STRIPS = 2, 3
GIB = 1 << 30


def _method(plan):
    return plan.setpts_info()["method"]


@contextlib.contextmanager
def _memory_left(nbytes):
    # what earlier tests left behind goes first, or it would be freed meanwhile
    gc.collect()
    _native.lib().jfa_cache_clear()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # (the driver may hold more than it reports as free, so the last of it is found by
    # asking for it)
    chunk = 64 << 20
    filler = []
    if (free := torch.cuda.mem_get_info()[0] - nbytes) > 0:
        filler.append(torch.empty(free, dtype=torch.uint8, device="cuda"))
    last = []
    with contextlib.suppress(torch.cuda.OutOfMemoryError):
        while len(last) < 16 * nbytes // chunk:
            last.append(torch.empty(chunk, dtype=torch.uint8, device="cuda"))
    filler += last[nbytes // chunk:]
    del last
    torch.cuda.empty_cache()
    try:
        yield
    finally:
        torch.cuda.synchronize()
        del filler
        torch.cuda.empty_cache()


def _run(plan, x, c, shape):
    out = torch.empty(shape, dtype=torch.complex64, device="cuda")
    plan.setpts(*x)
    plan.execute(c, out)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("modes", [(40, 16), (300, 31), (20, 24, 18)], ids=str)
def test_auto_takes_strips_on_narrow_grids(modes):
    # (what test_gpu_strip_tiles compares there, and cannot ask for by method 3)
    x = [torch.rand(5000, device="cuda") for _ in modes]
    plan = Plan(1, modes, iflag=1, eps=1e-5, dtype=torch.complex64)
    plan.setpts(*x)
    assert _method(plan) == STRIPS
    plan.destroy()


def test_narrow_grid_memory_is_bounded():
    # 24^3 modes, 48^3 cells, width 8: eight slice points of 64 bytes per point
    plan = Plan(1, (24, 24, 24), iflag=1, eps=1e-6, dtype=torch.complex64)
    small, large = 1_000_000, 17_000_000
    x = [torch.rand(large, device="cuda") for _ in range(3)]
    plan.setpts(*[a[:small] for a in x])
    assert _method(plan) == STRIPS
    free, _ = torch.cuda.mem_get_info()
    plan.setpts(*x)
    torch.cuda.synchronize()
    assert _method(plan) == TILES
    assert free - torch.cuda.mem_get_info()[0] < 2 * GIB
    plan.setpts(*[a[:small] for a in x])
    assert _method(plan) == STRIPS
    plan.destroy()


def test_no_room_for_strips_spreads_by_tiles():
    rng = np.random.default_rng(81)
    M, modes = 6_000_000, (64, 64, 64)
    x = [dev(a) for a in uniform_points(rng, 3, M, "f32")]
    c = dev(cnormal(rng, M, "f32"))
    ref = Plan(1, modes, iflag=1, eps=1e-6, dtype=torch.complex64)
    want = host(_run(ref, x, c, modes))
    assert _method(ref) == STRIPS
    ref.destroy()
    # 3 GB for strips, 0.4 GB for tiles
    plan = Plan(1, modes, iflag=1, eps=1e-6, dtype=torch.complex64)
    with _memory_left(2 * GIB):
        got = host(_run(plan, x, c, modes))
        assert _method(plan) == TILES
    assert rel_l2(got, want) <= 2e-6
    # fewer points take strips again
    plan.setpts(*[a[:100_000] for a in x])
    assert _method(plan) == STRIPS
    plan.destroy()


def test_no_room_for_every_transform_spreads_fewer_at_a_time():
    rng = np.random.default_rng(82)
    M, modes, T = 1_000_000, (1024, 1024), 24
    x = [dev(a) for a in uniform_points(rng, 2, M, "f32")]
    c = dev(cnormal(rng, (T, M), "f32"))
    want = torch.empty((T,) + modes, dtype=torch.complex64, device="cuda")
    got = torch.empty_like(want)
    ref = Plan(1, modes, iflag=1, ntransf=T, eps=1e-6, dtype=torch.complex64)
    ref.setpts(*x)
    ref.execute(c, want)
    torch.cuda.synchronize()
    ref.destroy()
    # tiles and records of 24 transforms: about 3 GB; the FFT's buffer 0.4 GB
    plan = Plan(1, modes, iflag=1, ntransf=T, eps=1e-6, dtype=torch.complex64)
    with _memory_left(2 * GIB):
        for _ in range(2):
            plan.setpts(*x)
            plan.execute(c, got)
            torch.cuda.synchronize()
        assert _method(plan) == STRIPS
    assert torch.equal(got, want)
    plan.destroy()
