"""Wide-tree queries whose rays run parallel to an axis or a plane of axes:
the header promises the exact tree's distances for them too."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import ray_set

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("zero", [(0,), (1,), (2,), (0, 1), (0, 2), (1, 2)])
@pytest.mark.parametrize("sign", [0.0, -0.0])
def test_wide_tree_rays_parallel_to_axes(ct, orc, gpu_ctx, c1, zero, sign):
    """Half of the rays have the components `zero` at +0 or -0 (1 / d is +inf
    or -inf), some all three, or NaN (which hit
    nothing).  As for other rays, a few of
    the exact tree's ulp-level culls (1 in 100,000) may be found here."""
    scene, arrays, osc = c1
    gpu_ctx.upload_build(scene, wide=True)
    opts, _, _ = scene.frame_opts()
    opts.accel, opts.traversal = ct.ACCEL_BVH4, ct.TRAV_FAST
    n = 1 << 17
    o, d = ray_set(scene, arrays, n, seed=80 + sum(zero))
    d[::2, list(zero)] = sign
    d[::4096] = 0.0
    d[1::4096] = np.nan
    tmax = np.random.default_rng(3).uniform(0.0, 60.0, n).astype(np.float32)
    t, p = gpu_ctx.trace_rays(o, d, opts)
    t_ref, p_ref = osc.trace(o, d, 1, 32, opts.triangle_epsilon, threads=16)
    assert np.mean(p_ref[::2] >= 0) > 0.1  # the parallel rays hit something
    assert np.sum(_bits(t) != _bits(t_ref)) <= n // 100_000
    assert np.sum((p >= 0) != (p_ref >= 0)) <= n // 100_000
    occ = gpu_ctx.trace_shadow_rays(o, d, tmax, opts)
    assert np.sum(occ != osc.trace_shadow(o, d, tmax, 1, 32, opts.triangle_epsilon, threads=16)) <= n // 100_000
