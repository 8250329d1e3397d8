"""Outputs in host memory (chunks through pinned staging) against the same
outputs in device memory, byte for byte: outputs that end at, before and
after a chunk's edge, more chunks than the ring holds, several jobs in one
chunk, pinned outputs between pageable ones, and a batch that runs again."""
import ctypes as C

import numpy as np
import pytest
import torch

import minirender_amd as mra
from minirender_amd import scenes
from minirender_amd._capi import mr_outputs
from minirender_amd.scenes import Draw, FrameSpec, Material
from tests.parity import fuzz_frame

pytestmark = pytest.mark.gpu
SHAPE = {"rgb8": (3, torch.uint8), "depth": (1, torch.float32), "winner": (1, torch.int32),
         "rgb": (3, torch.float32), "normals": (3, torch.float32), "points": (3, torch.float32)}


def buffers(f, kinds, **kw):
    return {k: torch.zeros(f.height * f.width * SHAPE[k][0], dtype=SHAPE[k][1], **kw) for k in kinds}


def render(ctx, frames, bufs, on_device):
    """One batch into the buffers (per frame, by kind)."""
    built = [ctx.frame(f) for f in frames]
    outs = (mr_outputs * len(frames))()
    for o, b, dev in zip(outs, bufs, on_device):
        for k, t in b.items():
            setattr(o, k, C.c_void_p(t.data_ptr()))
        o.on_device = int(dev)
    arr = (type(built[0][0]) * len(frames))(*[b[0] for b in built])
    assert ctx.lib.mr_render_batch(ctx.h, arr, len(frames), outs) == 0


def check(ctx, frames, kinds, host=None):
    ref = [buffers(f, k, device="cuda") for f, k in zip(frames, kinds)]
    torch.cuda.synchronize()
    render(ctx, frames, ref, [True] * len(frames))
    host = host or [buffers(f, k) for f, k in zip(frames, kinds)]
    render(ctx, frames, host, [False] * len(frames))
    for i, (r, h) in enumerate(zip(ref, host)):
        for k in r:
            a, b = r[k].cpu().numpy(), h[k].numpy()
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), (i, k)


@pytest.mark.parametrize("w,h,kinds", [
    (1, 1, ("rgb8",)),
    (512, 512, ("depth",)),                      # one chunk exactly
    (512, 512, ("depth", "winner")),
    (699, 500, ("rgb8", "depth")),               # rgb8: 76 bytes less than a chunk
    (700, 500, ("rgb8", "depth", "winner")),     # and 1424 more
    (900, 620, tuple(SHAPE)),                    # more than the ring
])
def test_host_outputs(gpu_ctx, w, h, kinds):
    f = fuzz_frame(31, w, h)
    f.save_normals = "normals" in kinds
    check(gpu_ctx, [f], [kinds])


def test_host_batch(gpu_ctx):
    frames = [fuzz_frame(40 + i, 40 + 97 * (i % 5), 30 + 61 * (i % 4)) for i in range(24)]
    kinds = [("rgb8", "depth"), ("winner",), ("depth", "points", "rgb8"), ()]
    check(gpu_ctx, frames, [kinds[i % 4] for i in range(len(frames))])


def test_pinned_between(gpu_ctx):
    frames = [fuzz_frame(70 + i, 300, 10 + 5 * i) for i in range(6)]
    kinds = [("rgb8", "depth", "winner")] * 6
    host = [buffers(f, k) for f, k in zip(frames, kinds)]
    for i, h in enumerate(host):
        pin = ("depth",) if i < 3 else ("rgb8", "winner") if i < 5 else kinds[0]
        for k in pin:
            h[k] = torch.empty(h[k].shape, dtype=h[k].dtype, pin_memory=True)
    check(gpu_ctx, frames, kinds, host)


def test_host_after_rerun():
    # about ten 16 x 16 tiles per triangle where the bin list starts with three
    tris = scenes.random_triangles(60000, 9, lo=0.05, hi=0.08, center_lo=(-1, -1, -2.2),
                                   center_hi=(1, 1, -2))
    f = FrameSpec(1920, 1080, scenes.projection_frustum(1.0, 1920 / 1080, 0.5, 50.0),
                  draws=[Draw(tris, Material())])
    with mra.Context() as a, mra.Context() as b:
        host = [buffers(f, ("rgb8", "depth"))]
        render(a, [f], host, [False])
        assert a.stats().retries >= 1
        ref = [buffers(f, ("rgb8", "depth"), device="cuda")]
        torch.cuda.synchronize()
        render(b, [f], ref, [True])
        for k in ref[0]:
            assert np.array_equal(ref[0][k].cpu().numpy().view(np.uint8),
                                  host[0][k].numpy().view(np.uint8)), k
