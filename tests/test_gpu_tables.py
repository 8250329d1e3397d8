"""Batch tables on both sides of what a kernel argument holds, and of one and
several workgroups of the kernel that fetches larger ones: frames of many
draws, small (k_front + k_small) and general, against the oracle."""
import numpy as np
import pytest

from minirender_amd import scenes
from minirender_amd.scenes import Draw, FrameSpec, Material
from tests.parity import assert_parity
from oracle import oracle_py

pytestmark = pytest.mark.gpu
KINDS = ("rgb8", "depth", "winner")


def frame(ndraws, w, h):
    rng = np.random.default_rng(ndraws)
    cube = scenes.create_cube(0.3)
    draws = [Draw(cube, Material(), scenes.translate(*rng.uniform((-1.5, -1.0, -4), (1.5, 1.0, -2))))
             for _ in range(ndraws)]
    return FrameSpec(w, h, scenes.projection_frustum(1.0, w / h, 0.1, 10.0), draws=draws)


@pytest.mark.parametrize("ndraws", [1, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 33, 300])
@pytest.mark.parametrize("w,h", [(97, 61), (1040, 20)])
def test_many_draws(gpu_ctx, ndraws, w, h):
    f = frame(ndraws, w, h)
    got = gpu_ctx.render(f, KINDS)
    ref = oracle_py.render(f, KINDS)
    assert_parity(got, ref, f"{ndraws} draws")
