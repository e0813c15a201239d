"""Results on their way to the caller's arrays: by the runtime's copy up to 1
MB, through the pinned slots in one part up to 1.5 MB, in parts above.  The sizes
are the edges of those, part sizes that do not divide the result, and enough
parts to reuse every slot; each must bring every byte to its place."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 16 bytes a pixel; the byte image is a quarter of that
SIZES = [(1, 1), (256, 256), (257, 256), (512, 256), (513, 256), (1, 131_073), (1023, 511), (1920, 1080), (2050, 2051)]


@pytest.mark.parametrize("w,h", SIZES)
def test_read_back(ct, gpu_ctx, w, h):
    rng = np.random.default_rng(w)
    gpu_ctx.resize(w, h)
    acc = rng.uniform(0.0, 4.0, (h, w, 4)).astype(np.float32)
    gpu_ctx.write_accum(acc, 3)
    for _ in range(2):  # a context's first large result goes by the runtime's copy
        got, samples = gpu_ctx.read_accum()
        assert samples == 3 and np.array_equal(got.view(np.uint32), acc.view(np.uint32))
    # a pixel's colour does not depend on where it is: the image of a repeated
    # row of 64 pixels is that row's image, read in one piece
    n, row = w * h, rng.uniform(0.0, 4.0, (64, 4)).astype(np.float32)
    order = np.arange(n) * 37 % 64
    gpu_ctx.write_accum(row[order].reshape(h, w, 4), 3)
    image, bytes8 = gpu_ctx.read_image(), gpu_ctx.read_image_rgba8()
    gpu_ctx.resize(64, 1)
    gpu_ctx.write_accum(row.reshape(1, 64, 4), 3)
    assert np.array_equal(image.reshape(n, 4).view(np.uint32), gpu_ctx.read_image().reshape(64, 4)[order].view(np.uint32))
    assert np.array_equal(bytes8.reshape(n, 4), gpu_ctx.read_image_rgba8().reshape(64, 4)[order])
    gpu_ctx.reset()


@pytest.mark.parametrize("n", [262_144, 262_145, 524_289, 2_200_001])
def test_host_hits(ct, gpu_ctx, c1, n):
    """The hits of n rays, 4 bytes each and 1 byte a shadow flag (offsets in
    the device arrays that are not multiples of 16), are those of the same
    rays in small calls."""
    from conftest import ray_set
    scene, arrays, _ = c1
    gpu_ctx.upload(scene)
    opts, _, _ = scene.frame_opts()
    m = 50_001
    o, d = ray_set(scene, arrays, m, seed=5)
    tmax = np.random.default_rng(5).uniform(0.0, 60.0, m).astype(np.float32)
    order = np.arange(n) * 101 % m
    t, p = gpu_ctx.trace_rays(o, d, opts)
    occ = gpu_ctx.trace_shadow_rays(o, d, tmax, opts)
    t2, p2 = gpu_ctx.trace_rays(o[order], d[order], opts)
    assert np.array_equal(t2.view(np.uint32), t[order].view(np.uint32)) and np.array_equal(p2, p[order])
    assert np.array_equal(gpu_ctx.trace_shadow_rays(o[order], d[order], tmax[order], opts), occ[order])


@pytest.mark.parametrize("w,h", [(64, 64), (1920, 1080)])
def test_first_image_of_a_context(ct, gpu_ctx, w, h):
    acc = np.random.default_rng(3).uniform(0.0, 4.0, (h, w, 4)).astype(np.float32)
    ctx = ct.Context(0)
    ctx.resize(w, h)
    ctx.write_accum(acc, 2)
    first, second, bytes8 = ctx.read_image(), ctx.read_image(), ctx.read_image_rgba8()
    ctx.close()
    gpu_ctx.resize(w, h)
    gpu_ctx.write_accum(acc, 2)
    ref = gpu_ctx.read_image()
    assert np.array_equal(first.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(second.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(bytes8, gpu_ctx.read_image_rgba8())
    gpu_ctx.reset()


@pytest.mark.parametrize("w,h", [(384, 256), (385, 256), (448, 256), (449, 256)])
def test_read_back_up_to_four_parts(ct, gpu_ctx, w, h):
    """One part up to 1.5 MB, then three and a bit, and four."""
    test_read_back(ct, gpu_ctx, w, h)


def test_host_hits_in_two_parts(ct, gpu_ctx, c1):
    """Host rays go to the device 4,194,304 at a time: a second part of one ray."""
    test_host_hits(ct, gpu_ctx, c1, (1 << 22) + 1)
