"""Scenes of many instances, bit for bit against the oracle: instance counts
around the ones where the box test of a whole wave begins and where it takes
another round, masked and moved instances, and rays of which a wave's have
nothing in common, infinite and undefined numbers among them."""
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
