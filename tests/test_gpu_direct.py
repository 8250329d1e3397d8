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


def flat_frame(w, h, tris):
    """Triangles given in pixel coordinates (x right, y up) under an
    orthographic projection, at depths of their own."""
    n = len(tris)
    rng = np.random.default_rng(n)
    pos = np.empty((n, 3, 3), np.float32)
    pos[:, :, :2] = tris
    pos[:, :, 2] = rng.uniform(-0.9, 0.9, n).astype(np.float32)[:, None]
    nrm = np.tile(np.array([[0, 0, 1]], np.float32), (3 * n, 1))
    idx = np.arange(3 * n, dtype=np.int32).reshape(-1, 3)
    return FrameSpec(w, h, scenes.projection_ortho(0, w, 0, h, -1, 1),
                     draws=[Draw(scenes.Mesh(pos.reshape(-1, 3), nrm, idx), Material())], lighting=False)


@pytest.mark.parametrize("persistent", [False, True])
@pytest.mark.parametrize("small_first", [False, True])
def test_both_ends_of_the_bin_list_meet(persistent, small_first):
    """Two jobs whose listed pairs (48,960 of 6 triangles over a 1920 x 1080
    frame) and binned pairs (up to 45,000 of 3,000 triangles that leave a
    200 x 150 frame, 3 x 5 tiles each) both fit the 65,536 entries of the bin
    list alone, but not together: nothing may be drawn from the list before
    the batch has run again with a longer one."""
    import minirender_amd as mra
    rng = np.random.default_rng(5)
    large = flat_frame(1920, 1080, np.array([[-10, -10], [4000, -10], [-10, 2300]], np.float32)[None] +
                       rng.uniform(0, 5, (6, 1, 2)).astype(np.float32))
    off = flat_frame(200, 150, np.array([[170, 55], [900, 90], [170, 130]], np.float32)[None] +
                     rng.uniform(0, 4, (3000, 1, 2)).astype(np.float32))
    frames = [off, large] if small_first else [large, off]
    with mra.Context(0) as ctx:
        ctx.set_tile(16, 16)
        ctx.set_bin_factor(1.0)
        ctx.set_persistent(persistent)
        out = ctx.render_batch(frames, KINDS)
        assert ctx.stats().retries >= 1
    for i, (g, f) in enumerate(zip(out, frames)):
        assert_parity(g, oracle_py.render(f, KINDS), f"job {i}")


@pytest.mark.parametrize("tile,n,w,h,persistent", [
    (16, 1300, 1040, 16, False), (16, 1300, 1040, 31, False), (16, 1300, 1033, 64, False), (16, 1300, 1040, 128, False),
    (16, 1300, 1040, 31, True), (16, 1300, 1033, 64, True), (8, 1300, 1026, 8, False), (32, 2000, 1057, 70, False)])
def test_bands_of_listed_items(gpu_ctx, tile, n, w, h, persistent):
    """Few tiles (8, 4, 2 and 1 row bands each) and more large triangles than
    one round of the raster: tiles with binned entries, with listed ones only
    and with both, frames that end inside a band."""
    tris = scenes.random_triangles(600, 13, lo=0.02, hi=0.02, center_lo=(-30, -2, -3), center_hi=(30, 2, -1))
    big = scenes.random_triangles(n, 12, lo=0.5, hi=8.0, center_lo=(-20, -0.2, -3), center_hi=(8, 0.2, -1))
    f = FrameSpec(w, h, scenes.projection_frustum(math.radians(5), w / h, 0.5, 50.0),
                  draws=[Draw(big, Material()), Draw(tris, Material())], light=(0.3, 0.5, 1.0))
    gpu_ctx.set_tile(tile, tile)
    gpu_ctx.set_persistent(persistent)
    try:
        check(gpu_ctx, f, f"bands {w} x {h} t{tile}")
    finally:
        gpu_ctx.set_persistent(False)
        gpu_ctx.set_tile(16, 16)


@pytest.mark.parametrize("frag", [256, 1000])
def test_split_tiles_share_listed_items(gpu_ctx, frag):
    """Tiles split by their binned entries, with listed ones beside them: a
    list that runs over, in parts of both kinds."""
    tris = scenes.random_triangles(14000, 14, lo=0.3, hi=3.0, center_lo=(-8, -0.3, -3), center_hi=(8, 0.3, -1))
    f = FrameSpec(1100, 40, scenes.projection_frustum(math.radians(10), 27.5, 0.5, 50.0),
                  draws=[Draw(tris, Material(shininess=5.0))], light=(0.3, 0.5, 1.0))
    gpu_ctx.set_frag_size(frag)
    try:
        check(gpu_ctx, f, f"split {frag}")
    finally:
        gpu_ctx.set_frag_size(1024)
