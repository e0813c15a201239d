"""Frames without statistics of up to 131,072 paths run as whole paths in one
launch (eight lanes each up to 40,960 on 256 CUs, two above); with statistics
through the queue pipeline, whose stages are timed.  Both must give the same
bits and ray counts, on every tree, and the FP32 oracle's on the exact ones."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_path_counts import SIZES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tree", ["quad", "binary", "compact", "wide"])
@pytest.mark.parametrize("config,depth,rr", [(1, 5, -1), (2, 5, -1), (2, 9, 3)])
def test_whole_paths(ct, orc, gpu_ctx, config, depth, rr, tree):
    from conftest import get_scene
    scene, _, osc = get_scene(ct, orc, config)
    gpu_ctx.upload(scene)
    opts, _, _ = scene.frame_opts()
    opts.max_depth, opts.rr_start = depth, rr
    opts.accel = ct.ACCEL_BVH2 if tree == "binary" else ct.ACCEL_BVH4
    opts.traversal = {"compact": ct.TRAV_COMPACT, "wide": ct.TRAV_FAST}.get(tree, ct.TRAV_EXACT)
    for w, h, spp in SIZES:
        cam = scene.camera(w, h)
        opts.spp = spp
        gpu_ctx.resize(w, h)
        gpu_ctx.trace_frame(cam, opts, stats=False)
        whole = gpu_ctx.read_accum()[0].view(np.uint32)
        gpu_ctx.resize(w, h)
        st = gpu_ctx.trace_frame(cam, opts)
        assert np.array_equal(whole, gpu_ctx.read_accum()[0].view(np.uint32)), (w, h, spp)
        _, bst = gpu_ctx.render_batch([(cam, w, h, spp, 0)], opts)
        assert (bst.primary_rays, bst.extension_rays, bst.shadow_rays) == (
            st.primary_rays, st.extension_rays, st.shadow_rays)
        assert st.extend_launches > 0 and st.extend_ms > 0.0 and st.shade_ms > 0.0
        if tree in ("quad", "binary"):
            ref, _ = osc.render(cam, opts, w, h, 0, spp, threads=16)
            assert np.array_equal(whole, ref.view(np.uint32)), (w, h, spp)
