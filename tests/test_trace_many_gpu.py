"""Scenes of many instances, bit for bit against the oracle: instance counts
around the ones where the box test of a whole wave begins and where it takes
another round, masked and moved instances, and rays of which a wave's have
nothing in common, infinite and undefined numbers among them; by few rays (one
in a wave) and by enough of them to fill every wave."""
import ctypes as C

import numpy as np
import pytest

import oracle_py as O
from scenes import grid_to_points, scene_grid

pytestmark = pytest.mark.gpu


def _rays(rng, count, span):
    from pyrit_amd import abi

    r = np.zeros(count, abi.RAY)
    r["origin"] = rng.uniform(-span, span, (count, 3))
    r["direction"] = rng.normal(0, 1, (count, 3))
    r["tmax"] = 3.402823466e38
    # a third of them from one eye into a cone, so that whole waves miss most boxes
    k = count // 3
    r["origin"][:k] = (span, span / 3, span)
    r["direction"][:k] = np.array([-1.0, -0.35, -1.0]) + rng.normal(0, 0.1, (k, 3))
    r["direction"][k:k + 64, 1] = 0.0
    r["tmin"][k + 64:k + 128] = span / 2
    r["tmax"][k + 128:k + 256] = span / 2
    for i, value in enumerate([np.inf, -np.inf, np.nan, -0.0, 1e-38, 3e38]):
        r["direction"][-512 + i:-256:16, i % 3] = value
        r["origin"][-256 + i::16, i % 3] = value
    return r


@pytest.mark.parametrize("count", [1, 7, 8, 64, 65, 130])
@pytest.mark.parametrize("rays", [1, 63, 5001])
def test_instances_against_oracle(hip_device, count, rays):
    from pyrit_amd import abi, lib, workloads

    L = lib()
    rng = np.random.default_rng(count)
    grid = scene_grid(32)
    cpu = O.build_points(5, grid_to_points(grid))
    side = int(np.ceil(np.sqrt(count)))
    inst = []
    for i in range(count):
        t = (40.0 * (i % side) - 20.0 * side, 8.0 * rng.normal(), 40.0 * (i // side) - 20.0 * side)
        m = workloads.make_transform(rng.normal(0, 1, 3), 6.28 * rng.random(), 0.3 + rng.random(), t)
        inst.append((m, 0, 0x0F if i % 5 == 2 else 0xFF))
    info = abi.PyrCreateInfo()
    info.struct_size, info.version = C.sizeof(abi.PyrCreateInfo), abi.PYR_VERSION
    info.node_pool_bytes = info.leaf_pool_bytes = info.attribute_pool_bytes = 16 << 20
    info.max_instances, info.max_geometries = 256, 8
    from pyrit_amd.device import Buffer, to_device

    ctx = C.c_void_p()
    abi.check(L, L.pyr_create(C.byref(info), C.byref(ctx)), "create")
    try:
        dag, geo = C.c_void_p(), C.c_void_p()
        abi.check(L, L.pyr_dag_build_dense(5, np.ascontiguousarray(grid).ctypes.data_as(C.c_void_p), 0, C.byref(dag)), "dag")
        abi.check(L, L.pyr_geometry_create(ctx, dag, C.byref(geo)), "geometry")
        L.pyr_dag_destroy(dag)
        for m, _, mask in inst:
            h = C.c_void_p()
            abi.check(L, L.pyr_instance_create(ctx, geo, C.byref(h)), "instance")
            abi.check(L, L.pyr_instance_set_transform(ctx, h, (C.c_float * 12)(*m)), "transform")
            abi.check(L, L.pyr_instance_set_mask(ctx, h, mask), "mask")
        abi.check(L, L.pyr_commit(ctx, None), "commit")
        scene = O.multi_scene([cpu], inst)
        r = _rays(rng, max(rays, 2048), 25.0 * side + 40.0)[:rays]
        rb, hb = to_device(r), Buffer(len(r) * 16)
        for flags, mask in ((0, 0), (0, 0x10), (abi.PYR_TRACE_ANY_HIT, 0), (abi.PYR_TRACE_NO_ATTRIBUTE, 0xF0)):
            abi.check(L, L.pyr_trace(ctx, rb.ptr, hb.ptr, len(r), mask, flags), "trace")
            abi.check(L, L.pyr_synchronize(ctx), "sync")
            got, want = hb.download(abi.HIT, len(r)), O.trace_rays(scene, r, mask, flags)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (flags, mask)
    finally:
        L.pyr_destroy(ctx)


def _limits(r, span):
    """Waves of 64 rays whose limits exclude every box, with rays among them
    whose own limits are undefined or infinite and exclude nothing (an
    undefined limit is none: the larger of it and a number is the number)."""
    n = 20000 // 64 * 64
    lane = np.arange(n) % 64
    for at, field, ordinary, free in ((0, "tmin", 40.0 * span, (np.nan, -np.inf, np.nan, -1.0)),
                                      (n, "tmax", 1e-3, (np.nan, np.inf, np.nan, 3e38))):
        wave = np.arange(n) // 64
        value = np.full(n, ordinary, np.float32)
        for i, v in enumerate(free):
            # one such ray in a wave, at a lane of its own, or every fourth
            value[(wave % 8 == i) & (lane == wave % 64)] = v
            value[(wave % 8 == i + 4) & (lane % 4 == i)] = v
        r[field][at:at + n] = value
    r["tmin"][2 * n:3 * n:3] = np.inf
    r["tmax"][3 * n:4 * n:3] = -np.inf
    return 2 * n


@pytest.mark.parametrize("count", [8, 16, 65])
def test_full_waves_against_oracle(hip_device, count):
    """More than 2^19 rays: 64 of them in every wave."""
    from pyrit_amd import abi, lib, workloads
    from pyrit_amd.device import Buffer, to_device

    L = lib()
    rng = np.random.default_rng(count)
    grid = scene_grid(32)
    cpu = O.build_points(5, grid_to_points(grid))
    side = int(np.ceil(np.sqrt(count)))
    span = 25.0 * side + 40.0
    inst = []
    for i in range(count):
        t = (40.0 * (i % side) - 20.0 * side, 8.0 * rng.normal(), 40.0 * (i // side) - 20.0 * side)
        m = workloads.make_transform(rng.normal(0, 1, 3), 6.28 * rng.random(), 0.3 + rng.random(), t)
        inst.append((m, 0, 0x0F if i % 5 == 2 else 0xFF))
    scene = O.multi_scene([cpu], inst)
    r = _rays(rng, 600001, span)
    rng.shuffle(r[100000:])  # neither the cone's rays nor the undefined ones side by side
    r[:80000] = _rays(rng, 240000, span)[:80000]
    limited = _limits(r, span)
    info = abi.PyrCreateInfo()
    info.struct_size, info.version = C.sizeof(abi.PyrCreateInfo), abi.PYR_VERSION
    info.node_pool_bytes = info.leaf_pool_bytes = info.attribute_pool_bytes = 16 << 20
    info.max_instances, info.max_geometries = 256, 8
    ctx = C.c_void_p()
    abi.check(L, L.pyr_create(C.byref(info), C.byref(ctx)), "create")
    try:
        dag, geo = C.c_void_p(), C.c_void_p()
        abi.check(L, L.pyr_dag_build_dense(5, np.ascontiguousarray(grid).ctypes.data_as(C.c_void_p), 0, C.byref(dag)), "dag")
        abi.check(L, L.pyr_geometry_create(ctx, dag, C.byref(geo)), "geometry")
        L.pyr_dag_destroy(dag)
        for m, _, mask in inst:
            h = C.c_void_p()
            abi.check(L, L.pyr_instance_create(ctx, geo, C.byref(h)), "instance")
            abi.check(L, L.pyr_instance_set_transform(ctx, h, (C.c_float * 12)(*m)), "transform")
            abi.check(L, L.pyr_instance_set_mask(ctx, h, mask), "mask")
        abi.check(L, L.pyr_commit(ctx, None), "commit")
        rb, hb = to_device(r), Buffer(len(r) * 16)
        for flags, mask in ((0, 0), (abi.PYR_TRACE_ANY_HIT, 0x10)):
            abi.check(L, L.pyr_trace(ctx, rb.ptr, hb.ptr, len(r), mask, flags), "trace")
            abi.check(L, L.pyr_synchronize(ctx), "sync")
            got, want = hb.download(abi.HIT, len(r)), O.trace_rays(scene, r, mask, flags)
            # (the rays without limits do hit among those that cannot)
            assert (want["instance"][:limited] != 0xFFFFFFFF).sum() > 100
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (flags, mask)
    finally:
        L.pyr_destroy(ctx)
