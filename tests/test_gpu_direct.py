"""Items over many tiles (listed per job and matched by the tiles instead of
being binned) and the checkpoint column spacing, where they can go wrong: a
list that runs over (the rest is binned), several jobs with lists of their own
beside jobs without, tiles with listed items only, checkpoints spaced wider
than a tile, the persistent kernel.  All against the oracle, bit for bit in
winner and depth."""
import math

import numpy as np
import pytest

from minirender_amd import scenes
from minirender_amd.scenes import Draw, FrameSpec, Material
from oracle import oracle_py
from tests.parity import assert_parity, fuzz_frame, stack_frame

pytestmark = pytest.mark.gpu
KINDS = ("rgb8", "depth", "winner")


def soup(n, seed, w, h, lo=0.2, hi=1.5):
    tris = scenes.random_triangles(n, seed, lo=lo, hi=hi, center_lo=(-1, -1, -3), center_hi=(1, 1, -1))
    return FrameSpec(w, h, scenes.projection_frustum(math.radians(60), w / h, 0.5, 50.0),
                     draws=[Draw(tris, Material(shininess=30.0))], light=(0.3, 0.5, 1.0))


def check(ctx, frame, what):
    assert_parity(ctx.render(frame, KINDS), oracle_py.render(frame, KINDS), what)


@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("n,w,h", [(1, 127, 129), (64, 333, 251), (900, 640, 360)])
def test_large_triangles(gpu_ctx, tile, n, w, h):
    """From one triangle to overdraw that fills the checkpoint buffer at the
    tile's column spacing (900 layers of a 640 x 360 frame)."""
    gpu_ctx.set_tile(tile, tile)
    try:
        check(gpu_ctx, soup(n, 40 + n, w, h), f"soup {n} t{tile}")
    finally:
        gpu_ctx.set_tile(16, 16)


def test_list_runs_over(gpu_ctx):
    """More large items than a job's list holds (4096): the rest is binned."""
    gpu_ctx.set_tile(8, 8)
    try:
        check(gpu_ctx, stack_frame(4600, 72, 56, seed=9), "list overflow")
    finally:
        gpu_ctx.set_tile(16, 16)


@pytest.mark.parametrize("persistent", [False, True])
def test_jobs_with_and_without_lists(gpu_ctx, persistent):
    """Jobs of large triangles, of small ones only, and empty ones in one
    batch: each tile meets its own job's list."""
    empty = FrameSpec(50, 40, scenes.projection_frustum(1.0, 1.25, 0.1, 10))
    frames = [soup(200, 1, 321, 203), scenes.config_sphere(160, 120), empty, fuzz_frame(5, 201, 99),
              soup(30, 2, 65, 63), fuzz_frame(8, 640, 480), soup(3, 3, 640, 16)]
    gpu_ctx.set_persistent(persistent)
    try:
        out = gpu_ctx.render_batch(frames, KINDS)
    finally:
        gpu_ctx.set_persistent(False)
    for i, (g, f) in enumerate(zip(out, frames)):
        assert_parity(g, oracle_py.render(f, KINDS), f"job {i}")


def test_bin_list_too_small(gpu_ctx):
    """Pairs of listed items that do not fit behind the bin list: the batch is
    run again with a larger list."""
    import minirender_amd as mra
    frame = soup(900, 77, 1920, 1080, lo=0.5, hi=2.0)
    with mra.Context(0) as ctx:
        ctx.set_bin_factor(1.0)
        g = ctx.render(frame, KINDS)
        assert ctx.stats().retries >= 1
    assert_parity(g, oracle_py.render(frame, KINDS), "bin list too small")
