"""Ray-level queries at the ray counts where the traversal changes how it
shares rays out: four lanes a ray while a launch has at most 16 rays for each
wave of the full grid (131,072 on 256 CUs), one lane a ray above, and four
lanes again for the last rays of a launch.  Both must give the oracle's bits,
also for rays on box planes, for stacks deep in the spill region and for a
binary tree's empty leaves."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import ArrayView, ray_set
from test_gpu_stack import chain_rays, chain_scene
from test_gpu_traversal_edges import _edge_rays

pytestmark = pytest.mark.gpu

COUNTS = (1, 3, 63, 1001, 32_769, 131_072, 131_073, 300_001)


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


def _same(gpu_ctx, osc, o, d, tmax, opts, accel):
    t, p = gpu_ctx.trace_rays(o, d, opts)
    t_ref, p_ref = osc.trace(o, d, accel, 32, opts.triangle_epsilon, threads=16)
    assert np.array_equal(_bits(t), _bits(t_ref))
    assert np.array_equal(p, p_ref)
    occ = gpu_ctx.trace_shadow_rays(o, d, tmax, opts)
    assert np.array_equal(occ, osc.trace_shadow(o, d, tmax, accel, 32, opts.triangle_epsilon, threads=16))


@pytest.mark.parametrize("tree", ["quad", "compact", "binary"])
def test_ray_counts(ct, orc, gpu_ctx, c1, tree):
    scene, arrays, osc = c1
    gpu_ctx.upload(scene)
    opts, _, _ = scene.frame_opts()
    opts.accel = ct.ACCEL_BVH2 if tree == "binary" else ct.ACCEL_BVH4
    opts.traversal = ct.TRAV_COMPACT if tree == "compact" else ct.TRAV_EXACT
    accel = 0 if tree == "binary" else 1
    o, d = _edge_rays(arrays, max(COUNTS), 7)
    tmax = np.random.default_rng(8).uniform(0.0, 60.0, len(o)).astype(np.float32)
    for n in COUNTS:
        if tree == "compact":  # ids may differ on exact ties of t
            t, p = gpu_ctx.trace_rays(o[:n], d[:n], opts)
            t_ref, p_ref = osc.trace(o[:n], d[:n], accel, 32, opts.triangle_epsilon, threads=16)
            assert np.array_equal(_bits(t), _bits(t_ref)), n
            assert np.array_equal(p >= 0, p_ref >= 0), n
        else:
            _same(gpu_ctx, osc, o[:n], d[:n], tmax[:n], opts, accel)


@pytest.mark.parametrize("n", [5, 140_001])
def test_deep_stacks(ct, orc, gpu_ctx, n):
    """127 stack entries, 111 of them spilled, with both ways of sharing rays."""
    arrays = chain_scene(ct, 42, seed=3)
    gpu_ctx.upload_view(ArrayView(ct, arrays).view)
    osc = orc.Scene(arrays, build=False)
    osc.set_trees(arrays["bvh"], arrays["mbvh"], arrays["prim_indices"])
    o, d = chain_rays(n, 4)
    _same(gpu_ctx, osc, o, d, np.full(n, 40.0, np.float32), ct.default_opts(), 1)


@pytest.mark.parametrize("axis", [1, 2])
def test_wide_tree_axis_parallel(ct, orc, gpu_ctx, c1, axis):
    """Rays without a y or z component have infinite slab terms in the wide
    tree and take its general node test (which leaves that axis out, so a
    superset of the exact boxes is entered); the others take the hardware
    minimum and maximum.  Both find the oracle's distances, but for the few
    rays of the exact tree's ulp-level culls (1 in 100,000, as for the rays of
    test_fast_traversal_closest_hit)."""
    scene, arrays, osc = c1
    gpu_ctx.upload_build(scene, wide=True)
    opts, _, _ = scene.frame_opts()
    opts.accel, opts.traversal = ct.ACCEL_BVH4, ct.TRAV_FAST
    n = 1 << 18
    o, d = ray_set(scene, arrays, n, seed=60 + axis)
    d[::2, axis] = 0.0
    tmax = np.random.default_rng(axis).uniform(0.0, 60.0, n).astype(np.float32)
    t, p = gpu_ctx.trace_rays(o, d, opts)
    t_ref, p_ref = osc.trace(o, d, 1, 32, opts.triangle_epsilon, threads=16)
    assert np.sum(_bits(t) != _bits(t_ref)) <= n // 100_000
    assert np.sum((p >= 0) != (p_ref >= 0)) <= n // 100_000
    occ = gpu_ctx.trace_shadow_rays(o, d, tmax, opts)
    assert np.sum(occ != osc.trace_shadow(o, d, tmax, 1, 32, opts.triangle_epsilon, threads=16)) <= n // 100_000


def _binary_tree(nodes):
    """nodes: (left_first, count) in export order, every box around the scene."""
    b = np.zeros((len(nodes), 8), np.float32)
    b[:, 0:3], b[:, 4:7] = -20.0, 20.0
    i = b.view(np.int32)
    for k, (first, count) in enumerate(nodes):
        i[k, 3], i[k, 7] = first, count
    return b.view(np.uint8).ravel()


@pytest.mark.parametrize("tree", ["empty_leaf_left", "empty_leaf_right", "leaf_root", "empty_root", "infinite_box"])
def test_odd_binary_trees(ct, orc, gpu_ctx, tree):
    arrays = chain_scene(ct, 3, seed=6)
    n = len(arrays["prim_indices"])
    # an interior root has its children at 2 and 3, node 1 is padding
    arrays["bvh"] = _binary_tree({
        "empty_leaf_left": [(2, -1), (0, 0), (0, 0), (0, n)],
        "empty_leaf_right": [(2, -1), (0, 0), (0, n), (3, 0)],
        "leaf_root": [(0, n)],
        "empty_root": [(0, 0)],
        "infinite_box": [(2, -1), (0, 0), (4, -1), (0, 2), (2, 2), (4, n - 4)],
    }[tree])
    if tree == "infinite_box":  # of an interior node: 0 * inf for the axis-parallel rays
        arrays["bvh"].view(np.float32).reshape(-1, 8)[2, [0, 5]] = -np.inf, np.inf
    arrays["mbvh"] = np.zeros(0, np.uint8)
    gpu_ctx.upload_view(ArrayView(ct, arrays).view)
    osc = orc.Scene(arrays, build=False)
    osc.set_trees(arrays["bvh"], arrays["mbvh"], arrays["prim_indices"])
    opts = ct.default_opts()
    opts.accel = ct.ACCEL_BVH2
    o, d = chain_rays(1000, 9)
    d[::5] = [1.0, 0.0, 0.0]
    _same(gpu_ctx, osc, o, d, np.full(1000, 40.0, np.float32), opts, 0)


@pytest.mark.parametrize("n", [5, 140_001])
@pytest.mark.parametrize("levels", [14, 15, 16, 17, 40, 127])
def test_deep_binary_stacks(ct, orc, gpu_ctx, levels, n):
    """Every box around the scene, so each level leaves its right leaf on the
    stack under the left child: up to the LDS part's 16 entries and past it, up
    to 127 and the entry kept in a register, which is the bound."""
    _binary_chain(ct, orc, gpu_ctx, levels, n)


@pytest.mark.parametrize("n", [5, 140_001])
def test_binary_stack_bound(ct, orc, gpu_ctx, n):
    with pytest.raises(ct.CTError) as e:
        _binary_chain(ct, orc, gpu_ctx, 128, n)
    assert e.value.code == ct.CT_ERR_STACK_OVERFLOW


def _binary_chain(ct, orc, gpu_ctx, levels, n):
    arrays = chain_scene(ct, 64, seed=8)
    assert len(arrays["prim_indices"]) > levels
    nodes = [(2, -1), (0, 0)]
    for k in range(levels):
        left = (4 + 2 * k, -1) if k + 1 < levels else (levels, len(arrays["prim_indices"]) - levels)
        nodes += [left, (k, 1)]
    arrays["bvh"] = _binary_tree(nodes)
    arrays["mbvh"] = np.zeros(0, np.uint8)
    gpu_ctx.upload_view(ArrayView(ct, arrays).view)
    osc = orc.Scene(arrays, build=False)
    osc.set_trees(arrays["bvh"], arrays["mbvh"], arrays["prim_indices"])
    opts = ct.default_opts()
    opts.accel = ct.ACCEL_BVH2
    o, d = chain_rays(n, 4)
    _same(gpu_ctx, osc, o, d, np.full(n, 40.0, np.float32), opts, 0)


@pytest.mark.parametrize("n", [2, 4095, 4096, 4097])
def test_hits_in_one_copy(ct, orc, gpu_ctx, c1, n):
    """Up to 4,096 host rays' distances and ids come in one copy."""
    scene, arrays, osc = c1
    gpu_ctx.upload(scene)
    opts, _, _ = scene.frame_opts()
    o, d = ray_set(scene, arrays, n, 21)
    _same(gpu_ctx, osc, o, d, np.full(n, 20.0, np.float32), opts, int(opts.accel == ct.ACCEL_BVH4))
