"""What the library asks of the HIP runtime, counted on the CPU: the library runs
in a process of its own over a stand-in for the runtime (hip_calls/standin.cpp:
device memory is host memory, kernels do nothing)."""
from __future__ import annotations

import ctypes as C
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

HERE = Path(__file__).resolve().parent
MB = 1 << 20
CASES = {}


def case(f):
    CASES[f.__name__] = f
    return f


@pytest.fixture(scope="module")
def standin(tmp_path_factory):
    so = tmp_path_factory.mktemp("hip") / "standin.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", str(so), str(HERE / "hip_calls" / "standin.cpp")], check=True)
    return so


class Hip:
    """The stand-in's records."""

    def __init__(self, so):
        self.lib = C.CDLL(so, mode=C.RTLD_GLOBAL)
        for f in ("standin_used", "standin_peak", "standin_copied"):
            getattr(self.lib, f).restype = C.c_size_t

    def calls(self, name):
        return self.lib.standin_calls(name.encode())

    def fail(self, name, times):
        self.lib.standin_fail(name.encode(), times)

    def capacity(self, n):
        self.lib.standin_capacity(C.c_size_t(n))

    def used(self):
        return self.lib.standin_used()

    def peak(self):
        """The largest use since the last call."""
        p = self.lib.standin_peak(0)
        self.lib.standin_peak(1)
        return p

    def copied(self, a):
        """Bytes the runtime has copied to the array since the last call."""
        return self.lib.standin_copied(C.c_void_p(a.ctypes.data), C.c_size_t(a.nbytes))

    def pinned(self, shape, dtype=np.float32):
        n = int(np.prod(shape)) * np.dtype(dtype).itemsize
        p = C.c_void_p()
        assert self.lib.hipHostMalloc(C.byref(p), C.c_size_t(n), 0) == 0
        return np.frombuffer((C.c_char * n).from_address(p.value), dtype).reshape(shape)


@case
def refused_allocation(hip, ct):
    """An allocation the runtime refuses is reported by the call that asked for
    it, and not again by the next call's launch."""
    scene = ct.HostScene.generate(ct.SCENE_C1, 7)
    ctx = ct.Context(0, mem_budget=1 << 40)
    ctx.upload(scene)
    hip.capacity(hip.used() + 512 * MB)
    try:
        ctx.resize(8192, 8192)
        raise AssertionError("1 GiB fitted")
    except ct.CTError as e:
        assert e.code == ct.CT_ERR_OUT_OF_MEMORY
    ctx.resize(64, 64)
    ctx.trace_frame(scene.camera(64, 64), scene.frame_opts()[0], stats=False)


@case
def failures_reported_once(hip, ct):
    """So it is with other calls that fail: in a frame's first buffers, and where
    a launch shape is looked for (a fixed one is taken then)."""
    scene = ct.HostScene.generate(ct.SCENE_C1, 7)
    frame = scene.camera(64, 64), scene.frame_opts()[0]
    hip.fail("hipOccupancyMaxActiveBlocksPerMultiprocessor", 1)
    ctx = ct.Context(0)
    ctx.upload(scene)
    ctx.resize(64, 64)
    hip.fail("hipMemsetAsync", 1)
    try:
        ctx.trace_frame(*frame, stats=False)
        raise AssertionError("the path buffers were not cleared")
    except ct.CTError as e:
        assert e.code == ct.CT_ERR_DEVICE
    ctx.trace_frame(*frame, stats=False)


def _textured(ct, n, side):
    """A view of n separate triangles with one float texture of side^2 texels."""
    from conftest import ArrayView
    rng = np.random.default_rng(5)
    v = rng.uniform(-8, 8, (n, 1, 3)) + rng.uniform(-0.5, 0.5, (n, 3, 3))
    cn = np.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    none = np.zeros(0, np.uint8)
    arrays = dict(vertices=v.reshape(-1, 3), normals=np.repeat(cn, 3, axis=0), center_normals=cn,
                  texcoords=rng.uniform(0, 1, (3 * n, 2)), indices=np.arange(3 * n).reshape(-1, 3),
                  material_idx=np.zeros(n), light_indices=np.zeros(0), prim_indices=np.arange(n), bvh=none, mbvh=none,
                  sky_enabled=0, sky=(0.0, 0.0, 0.0))
    return ArrayView(ct, arrays, textures=[rng.uniform(0, 1, (side, side, 4))], mats=[ct.Material()])


@case
def build_beside_textures(hip, ct):
    """upload_build needs the finished scene's memory for its textures, and not
    that of the arrays its kernels read as well: 124 bytes a triangle here."""
    n = 5_000
    scene = _textured(ct, n, 1024)
    budget = 1 << 40
    for _ in range(2):
        ctx = ct.Context(0, mem_budget=budget)
        before = hip.used()
        ctx.upload_build(scene.view)
        budget = hip.used() - before + 16 * n
        ctx.close()


@case
def no_copies_on_the_null_stream(hip, ct):
    """The null stream takes a hardware queue for the rest of the process, and
    a later context's two lanes then share one."""
    scene = ct.HostScene.generate(ct.SCENE_C1, 7)
    ctx = ct.Context(0)
    ctx.upload_build(scene, wide=True)
    ctx.read_trees()
    ctx.upload(scene)
    ctx.resize(64, 64)
    ctx.trace_frame(scene.camera(64, 64), scene.frame_opts()[0])
    ctx.read_image()
    assert hip.calls("hipMemcpyAsync") > 0 and hip.calls("hipMemcpy") == 0


@case
def batch_waits_once(hip, ct):
    """A batch's results are waited for together, not view by view."""
    scene = ct.HostScene.generate(ct.SCENE_C1, 7)
    opts, _, _ = scene.frame_opts()
    ctx = ct.Context(0)
    ctx.upload(scene)
    cam = scene.camera(8, 8)
    waits = []
    for n in (400, 4, 400):  # the first makes the path buffers
        before = hip.calls("hipStreamSynchronize")
        ctx.render_batch([(cam, 8, 8, 1, i) for i in range(n)], opts)
        waits.append(hip.calls("hipStreamSynchronize") - before)
    assert waits[1] == waits[2], waits


@case
def image_within_the_budget(hip, ct):
    """mem_budget holds for the buffer of a context's first image too: without
    room for it the image comes through the pinned slots."""
    ctx = ct.Context(0, mem_budget=20 * MB)
    ctx.resize(1024, 1024)  # 16 MB
    for read in (ctx.read_image, ctx.read_image, ctx.read_image_rgba8):
        read()
    assert hip.peak() <= 20 * MB


@case
def primitive_order_within_the_budget(hip, ct):
    """So it does for read_trees; without room for the ids' buffer they come by
    a strided copy."""
    scene = ct.HostScene.generate(ct.SCENE_C1, 7)
    budget = 1 << 40
    for _ in range(2):
        ctx = ct.Context(0, mem_budget=budget)
        before = hip.used()
        ctx.upload(scene)
        budget = hip.used() - before + 1024
        hip.peak()
        ids = ctx.read_trees()["prim_indices"]
        peak = hip.peak() - before
        ctx.close()
    assert peak <= budget
    assert np.array_equal(ids, scene.arrays()["prim_indices"])


@case
def results_without_pinned_memory(hip, ct):
    """Results need no pinned memory: where the slots cannot be had they come
    by the runtime's copy."""
    ctx = ct.Context(0)
    ctx.resize(512, 512)  # 4 MB
    acc = np.random.default_rng(1).uniform(0, 4, (512, 512, 4)).astype(np.float32)
    ctx.write_accum(acc, 1)
    for failing in ("hipHostMalloc", "hipHostGetDevicePointer", "hipEventCreateWithFlags"):
        hip.fail(failing, 1000)
        for _ in range(3):
            assert np.array_equal(ctx.read_accum()[0], acc)
            for read in (ctx.read_image, ctx.read_image_rgba8):
                hip.copied(acc)
                image = read()
                assert hip.copied(image) == image.nbytes
        hip.fail(failing, 0)


@case
def pinned_destinations(hip, ct):
    """Results go straight to an array the caller has pinned."""
    ctx = ct.Context(0)
    ctx.resize(512, 512)  # 4 MB
    acc = np.random.default_rng(1).uniform(0, 4, (512, 512, 4)).astype(np.float32)
    ctx.write_accum(acc, 1)
    f, b = hip.pinned((512, 512, 4)), hip.pinned((512, 512, 4), np.uint8)
    fp = f.ctypes.data_as(C.POINTER(C.c_float))
    bp = b.ctypes.data_as(C.POINTER(C.c_uint8))
    n = C.c_int32()
    for read, out in ((lambda: ct.lib.ct_read_accum(ctx.handle, fp, f.size, C.byref(n)), f),
                      (lambda: ct.lib.ct_read_image(ctx.handle, fp, f.size), f),
                      (lambda: ct.lib.ct_read_image_rgba8(ctx.handle, bp, b.size), b)):
        for k in range(3):
            hip.copied(acc)
            allocated = hip.calls("hipMalloc")
            assert read() == 0
            assert hip.copied(out) == out.nbytes
            assert k == 0 or hip.calls("hipMalloc") == allocated  # the image's buffer is kept
    ctx.read_accum(), ctx.read_image()  # pageable ones in between
    hip.copied(acc)
    assert ct.lib.ct_read_accum(ctx.handle, fp, f.size, C.byref(n)) == 0
    assert hip.copied(f) == f.nbytes and np.array_equal(f, acc)


@case
def parts_of_a_result(hip, ct):
    """One part up to 1.5 MB, parts of 512 KB above: at 2 MB one part took longer
    than the runtime's copy."""
    ctx = ct.Context(0)
    for rows, parts in ((1024, 0), (257, 1), (384, 1), (385, 4), (512, 4), (513, 5)):
        ctx.resize(256, rows)  # 4 KB a row; the first makes the slots due
        before = hip.calls("hipLaunchKernel")
        ctx.read_accum()
        assert hip.calls("hipLaunchKernel") - before == parts, rows


@case
def stages_of_a_small_frame(hip, ct):
    """A frame with statistics has its stages' device times, however small."""
    scene = ct.HostScene.generate(ct.SCENE_C1, 7)
    opts, _, _ = scene.frame_opts()
    opts.rr_start, opts.max_depth = -1, 4
    ctx = ct.Context(0)
    ctx.upload(scene)
    ctx.resize(64, 64)
    for trace in (ctx.trace_frame, ctx.trace_frame_serial):
        st = trace(scene.camera(64, 64), opts)
        # one launch a bounce and one for the last shadow rays
        assert st.chunks == 1 and st.extend_launches == 5
        assert min(st.extend_ms, st.shade_ms, st.connect_ms, st.other_ms) > 0.0 and st.tail_ms == 0.0


@case
def one_wait_a_result(hip, ct):
    """A result is waited for once, by the runtime's copy (the first) or through
    the slots."""
    ctx = ct.Context(0)
    ctx.resize(512, 512)  # 4 MB
    for _ in range(3):
        before = hip.calls("hipStreamSynchronize")
        ctx.read_accum()
        assert hip.calls("hipStreamSynchronize") - before == 1


@case
def one_wait_for_a_few_rays(hip, ct):
    scene = ct.HostScene.generate(ct.SCENE_C1, 7)
    ctx = ct.Context(0)
    ctx.upload(scene)
    opts, _, _ = scene.frame_opts()
    waits = []
    for n in (4096, 1, 64, 4096):  # the first makes the path buffers
        o, d = np.zeros((n, 3), np.float32), np.ones((n, 3), np.float32)
        before = hip.calls("hipStreamSynchronize")
        ctx.trace_rays(o, d, opts)
        waits.append(hip.calls("hipStreamSynchronize") - before)
    assert waits[1:] == [1, 1, 1], waits


@pytest.mark.parametrize("name", list(CASES))
def test_hip_calls(standin, name):
    r = subprocess.run([sys.executable, __file__, str(standin), name], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    sys.path.insert(0, str(HERE.parent))
    hip_ = Hip(sys.argv[1])  # before the library
    import cudatracer_amd

    CASES[sys.argv[2]](hip_, cudatracer_amd)
    assert hip_.calls("hipSetDevice") > 0, "the library did not reach the stand-in"
