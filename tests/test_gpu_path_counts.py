"""Frames at the path counts where the frame loop changes: whole paths in one
launch with eight lanes each (up to 40,960 paths on 256 CUs) or two (up to
131,072), the queue pipeline above.  These frames ask for statistics, so they
take the pipeline at every count (test_gpu_whole_paths.py holds the whole paths
against them).  Each must equal the FP32 oracle bit for
bit, ray counts included, on the trees whose traversal is exact; on the
compact and the wide tree 99.9% of the pixels must equal the exact frame (t is
equal there, ids on exact ties of t may differ)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# width, height, samples per pixel
SIZES = [(1, 1, 1), (7, 3, 5), (160, 256, 1), (331, 125, 1), (256, 256, 2), (401, 329, 1)]


@pytest.mark.parametrize("tree", ["quad", "binary", "compact", "wide"])
@pytest.mark.parametrize("config", [1, 2])
def test_frames_at_path_counts(ct, orc, gpu_ctx, config, tree):
    from conftest import get_scene
    scene, _, osc = get_scene(ct, orc, config)
    gpu_ctx.upload(scene)
    opts, _, _ = scene.frame_opts()
    opts.max_depth = 5
    for w, h, spp in SIZES:
        cam = scene.camera(w, h)
        opts.spp = spp
        opts.accel = ct.ACCEL_BVH2 if tree == "binary" else ct.ACCEL_BVH4
        opts.traversal = {"compact": ct.TRAV_COMPACT, "wide": ct.TRAV_FAST}.get(tree, ct.TRAV_EXACT)
        gpu_ctx.resize(w, h)
        st = gpu_ctx.trace_frame(cam, opts)
        acc = gpu_ctx.read_accum()[0].view(np.uint32)
        if tree in ("quad", "binary"):
            ref, ost = osc.render(cam, opts, w, h, 0, spp, threads=16)
            assert np.array_equal(acc, ref.view(np.uint32)), (w, h, spp)
            assert (st.primary_rays, st.extension_rays, st.shadow_rays) == (
                ost["primary_rays"], ost["extension_rays"], ost["shadow_rays"])
        else:
            opts.traversal = ct.TRAV_EXACT
            gpu_ctx.resize(w, h)
            gpu_ctx.trace_frame(cam, opts)
            same = np.all(acc == gpu_ctx.read_accum()[0].view(np.uint32), axis=-1)
            assert same.mean() >= 0.999, (w, h, spp, same.mean())
