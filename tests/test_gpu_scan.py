"""Tile counts at the edges of the scan's workgroups (256 tiles, or 2048 of
more than 16384), with tiles split over several work items and in row bands,
and jobs that share a workgroup, against the oracle."""
import pytest

from oracle import oracle_py
from tests.parity import assert_parity, fuzz_frame

pytestmark = pytest.mark.gpu
KINDS = ("rgb8", "depth", "winner")


@pytest.mark.parametrize("w,h", [(2048, 8), (2056, 8), (1032, 511), (1024, 1024), (1032, 1024),
                                 (1040, 1090)])
@pytest.mark.parametrize("frag", [64, 1024])
def test_tile_counts(gpu_ctx, w, h, frag):
    f = fuzz_frame(1200 + w % 7 + h, w, h)
    gpu_ctx.set_tile(8, 8)
    gpu_ctx.set_frag_size(frag)
    try:
        assert_parity(gpu_ctx.render(f, KINDS), oracle_py.render(f, KINDS), f"{w}x{h}")
        assert gpu_ctx.stats().launches > 2
    finally:
        gpu_ctx.set_frag_size(1024)
        gpu_ctx.set_tile(16, 16)


def test_jobs_share_workgroups(gpu_ctx):
    frames = [fuzz_frame(1300 + i, (1030, 77, 500, 333, 1200)[i % 5], (640, 70, 410, 8, 120)[i % 5])
              for i in range(10)]
    gpu_ctx.set_tile(8, 8)
    try:
        for i, (g, f) in enumerate(zip(gpu_ctx.render_batch(frames, KINDS), frames)):
            assert_parity(g, oracle_py.render(f, KINDS), f"job {i}")
    finally:
        gpu_ctx.set_tile(16, 16)
