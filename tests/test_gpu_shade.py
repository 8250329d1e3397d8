"""Shading blocks of frames whose tiles are mostly empty: tiles smaller than,
equal to and larger than a block (16 pixels), ragged right and lower edges,
every output, against the oracle."""
import pytest

from minirender_amd import scenes
from minirender_amd.scenes import Draw, FrameSpec, Material
from oracle import oracle_py
from tests.parity import assert_parity

pytestmark = pytest.mark.gpu
ALL = ("rgb8", "depth", "winner", "rgb", "normals", "points")


@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("w,h", [(1040, 48), (1041, 33), (1055, 17)])
def test_empty_tiles(gpu_ctx, tile, w, h):
    f = FrameSpec(w, h, scenes.projection_frustum(1.0, w / h, 0.1, 10.0),
                  draws=[Draw(scenes.create_cube(0.4), Material(), scenes.translate(x, 0, -3))
                         for x in (-20.0, -3.0, 0.0, 9.0)])
    f.save_normals = True
    gpu_ctx.set_tile(tile, tile)
    try:
        got = gpu_ctx.render_batch([f, f], ALL)
        assert gpu_ctx.stats().launches > 2
        ref = oracle_py.render(f, ALL)
        for i in range(2):
            assert_parity(got[i], ref, f"{w}x{h} tile {tile} job {i}")
    finally:
        gpu_ctx.set_tile(16, 16)
