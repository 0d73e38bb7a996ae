"""A volume's upper levels in the host's form, the device's form and both: calls
that read a volume keep the forms that it has, and threads may read one volume
together."""
import threading

import numpy as np
import pytest

import baby_shark_amd as bs
from baby_shark_amd import _lib
from test_alloc_gpu import H, Q, mesh, operands, same_volume

pytestmark = pytest.mark.gpu


def requests(f):
    """The device allocations that f asks for."""
    _lib.load().bs_refuse_allocations(0, 0)
    f()
    return _lib.load().bs_refuse_allocations(0, 0)


@pytest.mark.parametrize("gap", [False, True])
def test_reading_calls_keep_both_forms(gpu_ctx, gap):
    v, _ = operands(gpu_ctx, gap)
    v = v.subtract(bs.VolumeBuilder(gpu_ctx, H).cuboid((-3.0, -3.0, 0.4), (3.0, 3.0, 3.0))).flood_fill()
    mesher = bs.MarchingCubesMesher(gpu_ctx).with_voxel_size(H)
    soup, signs = mesh(gpu_ctx, v), v.signs_at(Q)
    for _ in range(2):  # the soup is all that a call allocates
        assert requests(lambda: mesher.mesh(v)) == 1
        assert requests(lambda: v.signs_at(Q)) == 0
        assert gap or requests(v.flood_fill) == 0  # a gap is closed in the host's form alone
    assert np.array_equal(mesh(gpu_ctx, v), soup) and np.array_equal(v.signs_at(Q), signs)


@pytest.mark.parametrize("form", ["host", "device", "none"])
def test_a_root_gap_is_seen_before_any_tree_is_made(gpu_ctx, form):
    a, b = operands(gpu_ctx, True)  # results of the device's form
    if form == "host":
        a, b = a.clone().union(b.clone()), a.subtract(b)
    elif form == "none":
        idx = np.array([[0, 0, 0], [0, 0, 8192]], np.int32)
        a = bs.volume_from_voxels(idx, np.array([-0.02, 0.02], np.float32), H, gpu_ctx)
        b = bs.volume_from_voxels(idx + 1, np.array([0.02, 0.02], np.float32), H, gpu_ctx)
    for _ in range(3):
        a0, b0 = a.clone(), b.clone()
        n = requests(lambda: a0.union(b0))
    assert n == 1  # the result's leaves


@pytest.mark.parametrize("gap", [False, True])
def test_flood_fill_of_either_form(gpu_ctx, gap):
    """The device's form alone, the host's alone, both: the same signs, leaves,
    mesh and result of the next operation."""
    v, b = operands(gpu_ctx, gap)
    v = v.subtract(bs.VolumeBuilder(gpu_ctx, H).cuboid((-3.0, -3.0, 0.4), (3.0, 3.0, 3.0)))
    got = []
    for forms in ("as it is", "and the host's", "and the device's", "both"):
        w = v.clone()
        if forms in ("and the host's", "both"):
            w.signs_at(Q)
        if forms in ("and the device's", "both"):
            mesh(gpu_ctx, w)
        w.flood_fill()
        got.append((w.export(), mesh(gpu_ctx, w), w.signs_at(Q), w.union(b.clone()).export()))
    for g in got[1:]:
        same_volume(g[0], got[0][0])
        assert np.array_equal(g[1], got[0][1]) and np.array_equal(g[2], got[0][2])
        same_volume(g[3], got[0][3])


@pytest.mark.parametrize("gap", [False, True])
def test_threads_read_one_volume(gpu_ctx, gap):
    """Threads with a context each mesh, query and clone one volume that has one
    form when they begin."""
    v, _ = operands(gpu_ctx, gap)
    soup, signs = mesh(gpu_ctx, v.clone()), v.clone().signs_at(Q)
    wrong = []

    def read(kind):
        ctx = bs.Context(0)
        for _ in range(8):
            if kind == "mesh":
                ok = np.array_equal(mesh(ctx, v), soup)
            elif kind == "clone":
                ok = np.array_equal(mesh(ctx, v.clone()), soup)
            else:
                out = np.zeros(Q.shape[0], np.uint8)
                q = np.ascontiguousarray(Q)
                s = _lib.load().bs_volume_signs_at(ctx.handle, v._h, q.ctypes.data_as(_lib.C.POINTER(_lib.C.c_int32)),
                                                   q.shape[0], out.ctypes.data_as(_lib.C.POINTER(_lib.C.c_uint8)))
                ok = s == 0 and np.array_equal(out.astype(bool), signs)
            if not ok:
                wrong.append(kind)
        ctx.close()

    threads = [threading.Thread(target=read, args=(k,)) for k in ("mesh", "signs", "clone", "mesh", "signs")]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
