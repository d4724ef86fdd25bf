"""Launches of few rays, whose waves hold fewer than 64 of them: ray counts and
frame sizes around the powers of two where the share changes, bit for bit
against the oracle, and nothing written past the last ray."""
import ctypes as C

import numpy as np
import pytest

import oracle_py as O
from scenes import grid_to_points, scene_grid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(hip_device):
    from pyrit_amd import gpu

    pts = grid_to_points(scene_grid(64))
    cpu = O.build_points(6, pts)
    return gpu.build(6, pts), O.single_scene(cpu), cpu


def _rays(count):
    from pyrit_amd import abi

    rng = np.random.default_rng(count)
    r = np.zeros(count, abi.RAY)
    r["origin"] = rng.uniform(-16, 80, (count, 3))
    r["direction"] = rng.uniform(8, 56, (count, 3)) - r["origin"]
    r["tmax"] = 3.402823466e38
    return r


@pytest.mark.parametrize("count", [1, 2, 127, 4095, 4096, 4097, 8193, 65537, 131071, 131073])
def test_ray_counts(scene, count):
    from pyrit_amd import abi, lib
    from pyrit_amd.device import Buffer, to_device

    built, oracle, _ = scene
    L = lib()
    r = _rays(count)
    rb, hb = to_device(r), Buffer((count + 64) * 16)
    guard = np.full((count + 64) * 4, 0xA5A5A5A5, np.uint32)
    hb.upload(guard)
    d = built.dag()
    abi.check(L, L.pyrhip_trace_dag(C.byref(d), rb.ptr, hb.ptr, count, 0, None), "trace")
    got = hb.download(np.uint32, (count + 64) * 4)
    want = O.trace_rays(oracle, r)
    assert np.array_equal(got[:count * 4], want.view(np.uint32))
    assert (got[count * 4:] == 0xA5A5A5A5).all()
    # the shadow rays of those hits
    sun = np.array([0.3, 0.8, 0.5], np.float32)
    sun /= np.sqrt((sun * sun).sum())
    ob = Buffer((count + 64) * 4)
    ob.upload(guard[:count + 64])
    abi.check(L, L.pyrhip_trace_shadow(C.byref(d), rb.ptr, hb.ptr, (C.c_float * 3)(*[float(v) for v in sun]), ob.ptr, count, None),
              "shadow")
    dark = ob.download(np.uint32, count + 64)
    sr, found = O.shadow_rays(r, want, sun)
    ref = np.full(count, 0xFFFFFFFF, np.uint32)
    sh = O.trace_rays(oracle, sr)
    ref[found] = (sh["instance"][found] == 0).astype(np.uint32)
    assert np.array_equal(dark[:count], ref)
    assert (dark[count:] == 0xA5A5A5A5).all()


@pytest.mark.parametrize("size", [(1, 1), (3, 2), (17, 9), (63, 65), (129, 33), (256, 255), (513, 257)])
def test_frame_sizes(scene, size):
    from pyrit_amd import abi, lib
    from pyrit_amd.device import Buffer

    built, oracle, cpu = scene
    L = lib()
    w, h = size
    eye, tgt, up = (-30.0, 70.0, -40.0), (32.0, 24.0, 32.0), (0.0, 1.0, 0.0)
    cam = abi.PyrCamera()
    L.pyr_camera_look_at(C.byref(cam), (C.c_float * 3)(*eye), (C.c_float * 3)(*tgt), (C.c_float * 3)(*up))
    L.pyr_camera_perspective(C.byref(cam), 0.9, w, h, 0.0)
    rays = O.camera_rays(O.camera(eye, tgt, up, 0.9, w, h))
    want = O.trace_rays(oracle, rays).view(np.uint32)
    guard = np.full(w * h * 4 + 256, 0xA5A5A5A5, np.uint32)
    hb, db = Buffer(guard.nbytes), Buffer(w * h * 4)
    hb.upload(guard)
    d = built.dag()
    abi.check(L, L.pyrhip_trace_camera(C.byref(d), C.byref(cam), hb.ptr, 0, None), "camera")
    got = hb.download(np.uint32, len(guard))
    assert np.array_equal(got[:w * h * 4], want) and (got[w * h * 4:] == 0xA5A5A5A5).all()
    # the same through pyr_render, alone and as the first of many instances far away
    info = abi.PyrCreateInfo()
    info.struct_size, info.version = C.sizeof(abi.PyrCreateInfo), abi.PYR_VERSION
    info.node_pool_bytes = info.leaf_pool_bytes = info.attribute_pool_bytes = 16 << 20
    ctx, dag, geo, view = C.c_void_p(), C.c_void_p(), C.c_void_p(), C.c_void_p()
    abi.check(L, L.pyr_create(C.byref(info), C.byref(ctx)), "create")
    try:
        pts = grid_to_points(scene_grid(64))
        abi.check(L, L.pyr_dag_build_points(6, np.ascontiguousarray(pts).ctypes.data_as(C.c_void_p), len(pts), 0, C.byref(dag)), "dag")
        abi.check(L, L.pyr_geometry_create(ctx, dag, C.byref(geo)), "geometry")
        L.pyr_dag_destroy(dag)
        abi.check(L, L.pyr_view_create(ctx, C.byref(view)), "view")
        t = abi.PyrTargets()
        t.hits, t.depth = hb.ptr, db.ptr
        for more in (1, 11):
            for i in range(more if more == 1 else more - 1):
                inst = C.c_void_p()
                abi.check(L, L.pyr_instance_create(ctx, geo, C.byref(inst)), "instance")
                if more > 1:
                    m = [1, 0, 0, 1e5 + 100 * i, 0, 1, 0, 0, 0, 0, 1, 0]
                    abi.check(L, L.pyr_instance_set_transform(ctx, inst, (C.c_float * 12)(*m)), "transform")
            abi.check(L, L.pyr_commit(ctx, None), "commit")
            hb.upload(guard)
            abi.check(L, L.pyr_render(ctx, view, C.byref(cam), C.byref(t)), "render")
            got = hb.download(np.uint32, len(guard))
            assert np.array_equal(got[:w * h * 4], want) and (got[w * h * 4:] == 0xA5A5A5A5).all()
    finally:
        L.pyr_destroy(ctx)
