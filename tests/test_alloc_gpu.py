"""Calls that run out of device memory part-way: each request for memory of a
call is refused in turn (bs_refuse_allocations) on a context without scratch,
and the volumes it was given must then be what they were."""
import contextlib

import numpy as np
import pytest

import baby_shark_amd as bs
from baby_shark_amd import _lib

pytestmark = pytest.mark.gpu
H = 0.05
AX = np.arange(-60, 60, 9, dtype=np.int32)
Q = np.stack(np.meshgrid(AX, AX, AX, indexing="ij"), -1).reshape(-1, 3)


@contextlib.contextmanager
def refusing(first, count=1 << 40):
    _lib.load().bs_refuse_allocations(first, count)
    try:
        yield
    finally:
        _lib.load().bs_refuse_allocations(0, 0)


def same_volume(g, r):
    for f in ("origins", "masks", "tile_origins", "tile_sizes"):
        assert np.array_equal(getattr(g, f), getattr(r, f)), f
    for f in ("values", "tile_values"):
        assert np.array_equal(getattr(g, f).view(np.uint32), getattr(r, f).view(np.uint32)), f


def operands(ctx, gap, h=H):
    """Two volumes with tiles and upper levels; with a gap between two root
    blocks on a z line, so that those are in the host's form."""
    B = bs.VolumeBuilder(ctx, h)

    def far():
        return bs.volume_from_voxels(np.array([[0, 0, 8192 + 40], [1, 0, 8192 + 40]], np.int32),
                                     np.array([-0.02, 0.03], np.float32), h, ctx)
    a = B.sphere(0.9, (-0.4, 0.0, 0.2)).union(B.sphere(2.0, (0.1, -0.2, 0.3)))
    b = B.sphere(0.6, (1.5, 0.1, 0.0)).union(B.sphere(1.5, (1.6, 0.2, 0.0)))
    assert a.info()["n_tiles"] and b.info()["n_tiles"]
    return (a.union(far()), b.union(far())) if gap else (a, b)


def free_bytes():
    import torch
    bs.release_cached_memory()
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def on_context(v, ctx):
    c = v.clone()
    c._ctx = ctx
    return c


def mesh(ctx, v):
    return bs.MarchingCubesMesher(ctx).with_voxel_size(H).mesh(v).view(np.uint32)


@pytest.mark.parametrize("op", ["union", "subtract", "intersect"])
@pytest.mark.parametrize("form", ["device", "device, gap", "host, gap"])
def test_csg_that_fails_keeps_its_operands(gpu_ctx, op, form):
    a0, b0 = operands(gpu_ctx, form != "device")
    if form == "host, gap":
        a0, b0 = a0.clone().union(b0.clone()), b0.subtract(a0)
    soups = mesh(gpu_ctx, a0.clone()), mesh(gpu_ctx, b0.clone())
    r = getattr(a0.clone(), op)(b0.clone())
    want, signs = r.export(), r.signs_at(Q)
    failed = lost = 0
    for first in range(1, 100):
        print(f"  {op} {form} refused from request {first}", flush=True)
        ctx = bs.Context(0)
        a, b = on_context(a0, ctx), on_context(b0, ctx)
        try:
            with refusing(first):
                r = getattr(a, op)(b)
            break
        except bs.BSError:
            failed += 1
        try:
            got = mesh(ctx, a), mesh(ctx, b)
            assert np.array_equal(got[0], soups[0]) and np.array_equal(got[1], soups[1])
            r = getattr(a, op)(b)
        except bs.BSError as e:  # only where the plan was made in the one form that there was
            assert form == "host, gap" and "upper levels" in str(e)
            assert np.array_equal(a.export().origins, a0.export().origins)
            lost += 1
            continue
        same_volume(r.export(), want)
        assert np.array_equal(r.signs_at(Q), signs)
    else:
        pytest.fail("still refused")
    assert failed > 2 and bool(lost) == (form == "host, gap")
    same_volume(r.export(), want)
    assert np.array_equal(r.signs_at(Q), signs)


@pytest.mark.parametrize("op", ["union", "subtract", "intersect", "offset"])
def test_without_memory_for_the_device_tree(gpu_ctx, op):
    """One request alone is refused: where that is for the upper levels on the
    device, the host's form serves."""
    a0, b0 = operands(gpu_ctx, False)
    a0 = bs.MeshToVolume(gpu_ctx).with_voxel_size(H).with_narrow_band_width(2).convert(mesh(gpu_ctx, a0).view(np.float32))

    def call(a, b):
        return a.offset(0.2) if op == "offset" else getattr(a, op)(b)

    if op == "offset":
        a0 = a0.subtract(b0.clone())
    r = call(a0.clone(), b0.clone())
    want, signs = r.export(), r.signs_at(Q)
    done = failed = 0
    for first in range(1, 100):
        print(f"  {op} refused: request {first}", flush=True)
        ctx = bs.Context(0)
        a, b = on_context(a0, ctx), on_context(b0, ctx)
        _lib.load().bs_refuse_allocations(first, 1)
        try:
            r = call(a, b)
            done += 1
        except bs.BSError:
            failed += 1
            r = call(a, b)
        made = _lib.load().bs_refuse_allocations(0, 0)
        same_volume(r.export(), want)
        assert np.array_equal(r.signs_at(Q), signs)
        assert np.array_equal(mesh(ctx, r), mesh(gpu_ctx, r))
        if made < first:
            break
    # refused for good: the operands' flags and the result's leaves, or what the sweeps need
    assert done > (4 if op == "offset" else 15) and 1 <= failed <= (12 if op == "offset" else 4)


def test_a_result_with_too_many_root_blocks_is_in_the_host_form(gpu_ctx, oracle_lib):
    """256 root blocks are the device form's limit: two operands of 200, their
    union of 400."""
    def line(x0):
        x = x0 + 4096 * np.arange(200)
        idx = np.stack([np.concatenate([x, x + 1]), np.full(400, 3), np.full(400, 5)], 1).astype(np.int32)
        val = np.where(np.arange(400) < 200, -0.02, 0.03).astype(np.float32)
        return bs.volume_from_voxels(idx, val, H, gpu_ctx), oracle_lib.from_voxels(idx, val, H)
    (g, r), (g2, r2) = line(-4096 * 300), line(4096 * 40)
    g, r = g.union(g2), r.union(r2)
    same_volume(g.export(), r.export())
    _lib.load().bs_refuse_allocations(0, 0)
    c = g.clone()
    assert _lib.load().bs_refuse_allocations(0, 0) == 1  # the leaves, and no tree
    g2, r2 = line(-4096 * 300 + 8)
    g, r = c.subtract(g2), r.subtract(r2)
    same_volume(g.export(), r.export())


@pytest.mark.parametrize("gap", [False, True])
def test_offset_that_fails_keeps_its_volume_and_no_memory(gpu_ctx, gap):
    h = H / 2
    v0, _ = operands(gpu_ctx, gap, h)
    v0 = v0.subtract(bs.VolumeBuilder(gpu_ctx, h).sphere(0.9, (0.3, 0.0, 0.2)))
    before = v0.export()
    r = v0.clone().offset(1.0)
    want, signs = r.export(), r.signs_at(Q)
    result_bytes = 2128 * want.origins.shape[0]
    assert result_bytes > 8 << 20
    r.free()

    for _ in range(5):  # the runtime's own memory for kernels, streams and their queues
        ctx = bs.Context(0)
        on_context(v0, ctx).offset(1.0).free()
        ctx.close()
    start = free_bytes()
    failed = 0
    for first in range(1, 100):
        print(f"  gap={gap} refused from request {first}", flush=True)
        ctx = bs.Context(0)
        v = on_context(v0, ctx)
        try:
            with refusing(first):
                v.offset(1.0)
            break
        except bs.BSError:
            failed += 1
        same_volume(v.export(), before)
        if failed % 4 == 0:
            r = v.offset(1.0)
            same_volume(r.export(), want)
            assert np.array_equal(r.signs_at(Q), signs)
            r.free()
        v.free()
        ctx.close()
        assert start - free_bytes() < result_bytes // 2
    else:
        pytest.fail("still refused")
    assert failed > 6  # the blocks and scratch of the sweeps, the leaves


def test_offset_leaves_no_arrays_with_its_context(gpu_ctx):
    """After an offset and release_cached_memory a context holds nothing that
    grew with the leaf pool but the sort's scratch (12 B per pool leaf and side
    buffers): at most 48 B, where the pool's own arrays are 100 B beside the
    values."""
    v0 = bs.VolumeBuilder(gpu_ctx, H / 10).sphere(2.0, (0.1, -0.2, 0.3))
    contexts = []

    def offset():
        contexts.append(bs.Context(0))
        on_context(v0, contexts[-1]).offset(H / 5).free()
        return contexts[-1].last_offset_stats()["n_capacity"]

    for _ in range(5):  # the runtime's own memory for kernels, streams and their queues
        offset()
        contexts[-1].close()
    start = free_bytes()
    pool = offset()
    assert start - free_bytes() < 48 * pool
    contexts[-1].close()


def test_conversion_without_memory_for_the_far_field(gpu_ctx):
    """One request alone is refused: the three buffers of the far field are not
    needed, and the signs are the same without them."""
    from baby_shark_amd import meshgen as mg
    soup = mg.displaced_icosphere(5, radius=0.7, seed=4)
    soup = soup[soup.mean(axis=1)[:, 0] > -0.3]

    def convert(ctx):
        return bs.MeshToVolume(ctx).with_voxel_size(0.02).with_narrow_band_width(2).convert(soup)

    want = convert(gpu_ctx).export()
    done = failed = 0
    for first in range(1, 200):
        ctx = bs.Context(0)
        _lib.load().bs_refuse_allocations(first, 1)
        try:
            v = convert(ctx)
            done += 1
        except bs.BSError:
            failed += 1
            v = convert(ctx)
        made = _lib.load().bs_refuse_allocations(0, 0)
        same_volume(v.export(), want)
        if made < first:
            break
    print(f"  {done} calls made, {failed} failed", flush=True)
    assert done - 1 == 3 and failed > 20  # the last call had nothing refused


@pytest.mark.parametrize("form", ["device", "host, gap"])
def test_densify_that_fails_keeps_its_volume(gpu_ctx, form):
    v0, b = operands(gpu_ctx, form != "device")
    if form == "host, gap":
        v0 = v0.union(b)
    before, soup, signs = v0.export(), mesh(gpu_ctx, v0.clone()), v0.clone().signs_at(Q)
    r = v0.clone().densify_tiles()
    want, want_soup = r.export(), mesh(gpu_ctx, r)
    failed = 0
    for first in range(1, 20):
        ctx = bs.Context(0)
        v = on_context(v0, ctx)
        try:
            with refusing(first):
                v.densify_tiles()
            break
        except bs.BSError:
            failed += 1
        same_volume(v.export(), before)
        assert np.array_equal(mesh(ctx, v), soup) and np.array_equal(v.signs_at(Q), signs)
        v.densify_tiles()
        same_volume(v.export(), want)
        assert np.array_equal(mesh(ctx, v), want_soup)
    assert 3 <= failed < 19
