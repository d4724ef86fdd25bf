"""The work that users of this framework have it do, as cases that can be
timed: DAG builds from voxel records (a prop, a chunk, an edit, a sparse
surface, chunk batches, a whole grid) and traversal (camera frames, shadow
rays, diffuse rays, instanced scenes, picks), each through the C ABI or its
Python mirror with inputs and outputs resident on the GPU.

The sizes of a DAG depend on its voxels, so a build case names its landscape
("land", a generator seed) and a seed turns and mirrors that landscape about
the vertical axis and gives it other materials: every seed has other records
and other arrays of the same sizes. Traversal cases take another landscape or
scene for every seed.

A case is a dict of plain values; "kind" names the call:

  prop       pyrhip_build of a small model's points, in any order
  terrain    pyrhip_build of a solid heightfield grid
  skin       pyrhip_build of a large surface (keys wider than 32 bits from 2^11)
  edit       pyrhip_build of an earlier build's voxels plus some edits
  batch      pyrhip_build_chunks of uneven chunks (world streaming, serving)
  camera     pyrhip_trace_camera, one frame of primary rays
  shadow     pyrhip_trace_shadow, one any-hit ray per primary hit of a frame
  rays       pyrhip_trace_dag of rays that leave a surface in all directions
  instances  pyr_commit + pyr_render of an instanced scene (hits and depth)
  pick       pyr_trace of a few rays in an instanced scene
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

from pyrit_amd import abi, gpu, lib, workloads

ANY_HIT, NO_ATTRIBUTE = abi.PYR_TRACE_ANY_HIT, abi.PYR_TRACE_NO_ATTRIBUTE
EDGES = (32, 64, 128, 256)


def listed():
    return [
        # a prop of a few thousand voxels placed or changed by the user: launch latency counts
        dict(name="prop32", kind="prop", log2=5, shuffled=True),
        # one streamed terrain chunk
        dict(name="chunk64", kind="terrain", land=1, log2=6, caves=0),
        # a brush stroke in a resident chunk: the chunk's voxels again, plus a few hundred edits
        dict(name="edit128", kind="edit", land=5, log2=7, edits=311),
        # an imported surface: few voxels for its edge, separate 64-bit keys
        dict(name="skin2048", kind="skin", land=4, log2=11, caves=2500),
        # one world update: a job of mixed chunk sizes
        dict(name="batch48", kind="batch", land=3, count=48),
        # loading a world: the batch of the benchmark
        dict(name="batch1024", kind="batch", land=3, count=1024),
        # the headline build
        dict(name="grid1024", kind="terrain", land=2, log2=10, caves=2000),
        # one frame of primary rays over a large landscape
        dict(name="camera1080p", kind="camera", log2=12, caves=20000, width=1920, height=1080, flags=0),
        # the sun shadow of that frame
        dict(name="shadow1080p", kind="shadow", log2=12, caves=20000, width=1920, height=1080),
        # ambient light: incoherent rays from the surface, an odd number of them
        dict(name="rays1m", kind="rays", log2=9, count=1_000_003, flags=0),
        # a frame of a scene of instances that moves every frame
        dict(name="instances64", kind="instances", count=64, width=1920, height=1080),
        # what is under the cursor: a handful of rays
        dict(name="pick37", kind="pick", count=64, rays=37),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["prop", "terrain", "skin", "edit", "batch", "camera", "shadow", "rays", "instances", "pick"])
    if kind == "prop":
        return dict(kind=kind, log2=rng.randint(4, 7), shuffled=rng.random() < 0.5)
    land = rng.randint(1, 1 << 20)
    if kind == "terrain":
        return dict(kind=kind, land=land, log2=rng.randint(5, 10), caves=_log_int(rng, 1, 2000))
    if kind == "skin":
        return dict(kind=kind, land=land, log2=rng.randint(8, 11), caves=_log_int(rng, 1, 2500))
    if kind == "edit":
        return dict(kind=kind, land=land, log2=rng.randint(5, 8), edits=_log_int(rng, 1, 4096))
    if kind == "batch":
        return dict(kind=kind, land=land, count=_log_int(rng, 2, 1023))
    if kind in ("camera", "shadow"):
        width = _log_int(rng, 160, 1919)
        case = dict(kind=kind, log2=rng.randint(8, 12), caves=_log_int(rng, 16, 20000), width=width,
                    height=max(90, int(width * rng.uniform(0.4, 0.56))))
        return dict(case, flags=rng.choice([0, 0, NO_ATTRIBUTE])) if kind == "camera" else case
    if kind == "rays":
        return dict(kind=kind, log2=rng.randint(6, 9), count=_log_int(rng, 1, 1_999_999),
                    flags=rng.choice([0, 0, NO_ATTRIBUTE, ANY_HIT | NO_ATTRIBUTE]))
    if kind == "instances":
        width = _log_int(rng, 160, 1919)
        return dict(kind=kind, count=_log_int(rng, 3, 1000), width=width, height=max(90, int(width * rng.uniform(0.4, 0.56))))
    return dict(kind=kind, count=_log_int(rng, 3, 1000), rays=_log_int(rng, 1, 4096))


# ---- device memory as tensors ---------------------------------------------

class _Memory:
    """`count` elements at a device address; keeps their owner alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 2}


def _tensor(owner, ptr, count, typestr, dtype):
    if not count:
        return torch.empty(0, dtype=dtype, device="cuda")
    return torch.as_tensor(_Memory(owner, ptr, (count,), typestr), device="cuda")


def _outputs(b, *more):
    """Everything a build returns, as tensors over its own device arrays."""
    r = b.raw
    return [_tensor(b, r.nodes, r.node_words, "<i4", torch.int32), _tensor(b, r.leaves, r.leaf_count, "<i8", torch.int64),
            _tensor(b, r.keys, r.voxel_count, "<i8", torch.int64), _tensor(b, r.attrs, r.voxel_count, "<i4", torch.int32),
            int(r.root), *more]


def _hits(t):
    """PyrHit records: the distance, and the instance, attribute and face words."""
    return [t.view(torch.float32)[:, 0], t[:, 1:]]


# ---- inputs ----------------------------------------------------------------

def _terrain(case, seed):
    if case["caves"]:
        return workloads.heightfield_grid(seed=seed, log2_size=case["log2"], caves=case["caves"])
    n = 1 << case["log2"]
    ch = workloads.ChunkSpec(log2_size=case["log2"], seed=seed, mean=n // 2, amplitude=n // 4, octaves=2,
                             wavelength_log2=case["log2"] - 1, material_mode=0)
    return workloads.Workload(f"terrain-{n}^3", [ch]).prepare()


def _skin(case, seed):
    return workloads.skin_grid(seed=seed, log2_size=case["log2"], caves=case["caves"])


def _int_tensor(vox, count):
    return _tensor(vox, vox.ptr, count * 4, "<i4", torch.int32).view(-1, 4)


def _turn(records, edge, seed):
    """PyrVoxel records (int32 [n, 4]) of grids of the given edge (a number, or
    one per record) turned, mirrored and given other materials in place."""
    rng = workloads.SplitMix64(seed * 0x9E3779B1 + 17)
    r = rng.next()
    if r & 1:
        records[:, 0], records[:, 2] = records[:, 2].clone(), records[:, 0].clone()
    for axis, bit in ((0, 2), (2, 4)):
        if r & bit:
            records[:, axis] = edge - 1 - records[:, axis]
    solid = (records[:, 3] != 0).int()
    records[:, 3] ^= solid * (((r >> 8) & 0x7FFFFF) << 8)
    return records


@functools.lru_cache(maxsize=4)
def _model(log2):
    """Coordinates (z, y, x) and attributes of the 2^log2 test scene's voxels"""
    grid = workloads.scene_grid(1 << log2)
    z, y, x = np.nonzero(grid)
    return grid, np.stack([x, y, z], 1).astype(np.int32), grid[z, y, x]


def _model_records(log2, seed, shuffled):
    _, xyz, attribute = _model(log2)
    g = np.random.default_rng(seed)
    out = np.zeros(len(xyz), abi.VOXEL)
    # the model turned about the vertical axis, mirrored or not, with this seed's materials
    n = (1 << log2) - 1
    x, z = xyz[:, 0], xyz[:, 2]
    for _ in range(int(g.integers(4))):
        x, z = z, n - x
    out["x"], out["y"], out["z"] = x, xyz[:, 1], z
    out["attribute"] = (attribute ^ np.uint32(g.integers(1 << 24) << 8)) | np.uint32(1)
    if shuffled:
        g.shuffle(out)
    return out


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _surface_rays(records, count, log2, seed):
    """Rays that leave the top faces of a solid grid's surface, cosine
    distributed about the normal; and the grid's occupancy [x, y, z]."""
    n = 1 << log2
    occupied = torch.zeros((n, n, n), dtype=torch.bool, device="cuda")
    v = records[:, :3].long()
    occupied[v[:, 0], v[:, 1], v[:, 2]] = True
    top = occupied.clone()
    top[:, :-1] &= ~occupied[:, 1:]
    cells = top.nonzero()
    g = _generator(seed)
    at = cells[torch.randint(len(cells), (count,), generator=g, device="cuda")].float()
    u = torch.rand((count, 4), generator=g, device="cuda")
    rays = torch.empty((count, 8), dtype=torch.float32, device="cuda")
    rays[:, 0], rays[:, 1], rays[:, 2] = at[:, 0] + u[:, 0], at[:, 1] + 1.001, at[:, 2] + u[:, 1]
    r, phi = u[:, 2].sqrt(), 2 * math.pi * u[:, 3]
    rays[:, 3] = 0.0
    rays[:, 4], rays[:, 5], rays[:, 6] = r * phi.cos(), (1 - u[:, 2]).sqrt().clamp(min=1e-3), r * phi.sin()
    rays[:, 7] = 3.0e38
    return rays, occupied


class _Scene:
    """A context with `count` instances of the 128^3 test scene on a grid,
    each turned and scaled by the seed, a view and a camera that sees them."""

    def __init__(self, count, seed, width=64, height=64):
        L = lib()
        self.lib, self.ctx = L, C.c_void_p()
        rng = workloads.SplitMix64(seed * 0x9E3779B1 + 5)
        info = abi.PyrCreateInfo()
        info.struct_size, info.version = C.sizeof(abi.PyrCreateInfo), abi.PYR_VERSION
        info.max_instances, info.max_geometries = 4096, 16
        info.node_pool_bytes = info.leaf_pool_bytes = info.attribute_pool_bytes = 64 << 20
        abi.check(L, L.pyr_create(C.byref(info), C.byref(self.ctx)), "create")
        dag, geo, self.view = C.c_void_p(), C.c_void_p(), C.c_void_p()
        grid = _model(7)[0]
        abi.check(L, L.pyr_dag_build_dense(7, grid.ctypes.data_as(C.c_void_p), 0, C.byref(dag)), "dag")
        abi.check(L, L.pyr_geometry_create(self.ctx, dag, C.byref(geo)), "geometry")
        L.pyr_dag_destroy(dag)
        xf, eye, target = workloads.instance_grid(count)
        for m in xf:
            inst = C.c_void_p()
            m = workloads.make_transform((rng.uniform() - 0.5, 1, rng.uniform() - 0.5), 2 * math.pi * rng.uniform(),
                                         0.6 + 0.8 * rng.uniform(), (m[3], m[7], m[11]))
            abi.check(L, L.pyr_instance_create(self.ctx, geo, C.byref(inst)), "instance")
            abi.check(L, L.pyr_instance_set_transform(self.ctx, inst, (C.c_float * 12)(*m)), "transform")
        abi.check(L, L.pyr_view_create(self.ctx, C.byref(self.view)), "view")
        turn = 2 * math.pi * rng.uniform()
        eye = (eye[0] * math.cos(turn) - eye[2] * math.sin(turn), eye[1], eye[0] * math.sin(turn) + eye[2] * math.cos(turn))
        self.camera = abi.PyrCamera()
        L.pyr_camera_look_at(C.byref(self.camera), (C.c_float * 3)(*eye), (C.c_float * 3)(*target), (C.c_float * 3)(0, 1, 0))
        L.pyr_camera_perspective(C.byref(self.camera), 0.9, width, height, 0.1)
        abi.check(L, L.pyr_commit(self.ctx, None), "commit")

    def __del__(self):
        if self.ctx:
            self.lib.pyr_destroy(self.ctx)


def prepare(case, seed):
    kind = case["kind"]
    L = lib()
    if kind == "prop":
        rec = torch.from_numpy(_model_records(case["log2"], seed, case["shuffled"]).view(np.int32).reshape(-1, 4)).cuda()
        return dict(case=case, records=rec, ptr=rec.data_ptr(), count=len(rec))
    if kind in ("terrain", "skin"):
        vox, _, total = (_terrain if kind == "terrain" else _skin)(case, case["land"]).generate_device()
        _turn(_int_tensor(vox, total), 1 << case["log2"], seed)
        return dict(case=case, records=vox, ptr=vox.ptr, count=total)
    if kind == "edit":
        n = 1 << case["log2"]
        vox, _, total = _terrain(dict(log2=case["log2"], caves=8), case["land"]).generate_device()
        _turn(_int_tensor(vox, total), n, seed)
        torch.cuda.synchronize()
        old = gpu.build(case["log2"], vox, count=total)
        g = _generator(case["land"])
        # a stroke: voxels around one place, two thirds set, one third removed
        centre = torch.randint(n, (1, 3), generator=g, device="cuda")
        at = (centre + torch.randn((case["edits"], 3), generator=g, device="cuda").mul(n / 16).long()).clamp(0, n - 1)
        attribute = torch.randint(1, 9, (case["edits"], 1), generator=g, device="cuda")
        attribute[torch.rand((case["edits"], 1), generator=g, device="cuda") < 1 / 3] = 0
        rec = _turn(torch.cat([at, attribute], 1).int().contiguous(), n, seed)
        return dict(case=case, old=old, records=rec, ptr=rec.data_ptr(), count=len(rec))
    if kind == "batch":
        w = workloads.uneven_chunks(seed=case["land"], count=case["count"], edges=EDGES)
        vox, offsets, total = w.generate_device()
        log2 = np.array([c.log2_size for c in w.chunks], np.uint8)
        edge = torch.repeat_interleave(torch.from_numpy(1 << log2.astype(np.int32)).cuda(),
                                       torch.from_numpy(np.diff(offsets.astype(np.int64))).cuda(), output_size=total)
        _turn(_int_tensor(vox, total), edge, seed)
        return dict(case=case, records=vox, offsets=offsets.astype(np.uint32), chunk_log2=log2)
    if kind in ("camera", "shadow"):
        w = _skin(case, seed)
        vox, _, total = w.generate_device()
        b = gpu.build(case["log2"], vox, count=total)
        vox.free()
        pixels = case["width"] * case["height"]
        cam = workloads.camera_poses(w, 1, case["width"], case["height"], seed=seed)[0]
        s = dict(case=case, built=b, dag=b.dag(), camera=cam, hits=torch.empty((pixels, 4), dtype=torch.int32, device="cuda"))
        if kind == "shadow":
            s["rays"] = torch.empty((pixels, 8), dtype=torch.float32, device="cuda")
            s["occluded"] = torch.empty(pixels, dtype=torch.int32, device="cuda")
            s["sun"] = (C.c_float * 3)(*[float(x) for x in workloads.normalize(workloads.SUN)])
            abi.check(L, L.pyrhip_camera_rays(C.byref(cam), s["rays"].data_ptr(), None), "rays")
            abi.check(L, L.pyrhip_trace_dag(C.byref(s["dag"]), s["rays"].data_ptr(), s["hits"].data_ptr(), pixels, 0, None), "trace")
        return s
    if kind == "rays":
        vox, _, total = _terrain(dict(log2=case["log2"], caves=200), seed).generate_device()
        b = gpu.build(case["log2"], vox, count=total)
        rays, _ = _surface_rays(_int_tensor(vox, total), case["count"], case["log2"], seed)
        return dict(case=case, built=b, dag=b.dag(), rays=rays,
                    hits=torch.empty((case["count"], 4), dtype=torch.int32, device="cuda"))
    if kind == "instances":
        s = _Scene(case["count"], seed, case["width"], case["height"])
        pixels = case["width"] * case["height"]
        t = abi.PyrTargets()
        out = dict(case=case, scene=s, targets=t, hits=torch.empty((pixels, 4), dtype=torch.int32, device="cuda"),
                   depth=torch.empty(pixels, dtype=torch.float32, device="cuda"))
        t.hits, t.depth = out["hits"].data_ptr(), out["depth"].data_ptr()
        return out
    if kind == "pick":
        s = _Scene(case["count"], seed)
        # rays of the camera through random pixels of its view
        every = torch.empty((64 * 64, 8), dtype=torch.float32, device="cuda")
        abi.check(L, L.pyrhip_camera_rays(C.byref(s.camera), every.data_ptr(), None), "rays")
        torch.cuda.synchronize()
        pick = torch.randint(64 * 64, (case["rays"],), generator=_generator(seed), device="cuda")
        rays = every[pick].contiguous()
        return dict(case=case, scene=s, rays=rays, hits=torch.empty((case["rays"], 4), dtype=torch.int32, device="cuda"))
    raise ValueError(kind)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("prop", "terrain", "skin"):
        return _outputs(gpu.build(case["log2"], state["ptr"], count=state["count"]))
    if kind == "edit":
        return _outputs(gpu.build(case["log2"], state["ptr"], count=state["count"], old=state["old"]))
    if kind == "batch":
        b, roots, first = gpu.build_chunks(8, state["records"], state["offsets"], state["chunk_log2"])
        return _outputs(b, roots.astype(np.int64), first.astype(np.int64))
    L = lib()
    if kind == "camera":
        abi.check(L, L.pyrhip_trace_camera(C.byref(state["dag"]), C.byref(state["camera"]), state["hits"].data_ptr(),
                                           case["flags"], None), "trace")
        return _hits(state["hits"])
    if kind == "shadow":
        abi.check(L, L.pyrhip_trace_shadow(C.byref(state["dag"]), state["rays"].data_ptr(), state["hits"].data_ptr(),
                                           state["sun"], state["occluded"].data_ptr(), len(state["occluded"]), None), "shadow")
        return state["occluded"]
    if kind == "rays":
        abi.check(L, L.pyrhip_trace_dag(C.byref(state["dag"]), state["rays"].data_ptr(), state["hits"].data_ptr(),
                                        case["count"], case["flags"], None), "trace")
        return _hits(state["hits"])
    s = state["scene"]
    if kind == "instances":
        abi.check(L, L.pyr_commit(s.ctx, None), "commit")
        abi.check(L, L.pyr_render(s.ctx, s.view, C.byref(s.camera), C.byref(state["targets"])), "render")
        return _hits(state["hits"]) + [state["depth"]]
    abi.check(L, L.pyr_trace(s.ctx, state["rays"].data_ptr(), state["hits"].data_ptr(), case["rays"], 0, 0), "trace")
    return _hits(state["hits"])


# ---- the work a pass cannot do without ---------------------------------------

def _voxels(case):
    """about how many records the inputs of a build hold"""
    n = float(1 << case["log2"])
    if case["kind"] == "prop":
        return float(len(_model(case["log2"])[1]))
    if case["kind"] == "skin":
        return 3.2 * n * n
    return 0.47 * n ** 3


def work(case):
    kind = case["kind"]
    if kind == "batch":
        # mean occupancy 0.32 of edges 32 / 64 / 128 / 256 with probabilities .4 / .3 / .2 / .1
        v = case["count"] * 0.32 * sum(p * e ** 3 for p, e in zip((0.4, 0.3, 0.2, 0.1), EDGES))
        return {"bytes": v * (16 + 12), "flops": 0}
    if kind in ("prop", "terrain", "skin"):
        return {"bytes": _voxels(case) * (16 + 12), "flops": 0}
    if kind == "edit":
        return {"bytes": _voxels(case) * (12 + 12) + 16 * case["edits"], "flops": 0}
    # a ray in or made in registers, a hit out, and what it touches of the DAG
    # (262 bytes a primary ray on the 4096^3 landscape, counted on the CPU); about
    # 45 cells a ray with 20 floating operations each
    if kind == "pick":
        return {"bytes": case["rays"] * 300.0, "flops": case["rays"] * 900.0}
    rays = case["count"] if kind == "rays" else case["width"] * case["height"]
    own = {"camera": 16, "shadow": 52, "rays": 48, "instances": 20}[kind]
    return {"bytes": rays * (own + 246.0), "flops": rays * 900.0}


def exact(case, seed):
    """Distances of the "rays" kind by a plain walk over a dense grid in 64
    bits, one cell per step; hit records are whole numbers, builds too. The
    landscapes and instanced scenes of the other kinds have no dense grid
    that a plain walk crosses in reasonable time."""
    if case["kind"] != "rays":
        return None
    n = 1 << case["log2"]
    vox, _, total = _terrain(dict(log2=case["log2"], caves=200), seed).generate_device()
    rays, occupied = _surface_rays(_int_tensor(vox, total), case["count"], case["log2"], seed)
    o, d = rays[:, 0:3].double(), rays[:, 4:7].double()
    cell = o.floor().long().clamp(0, n - 1)
    step = torch.where(d < 0, -1, 1)
    inv = 1.0 / torch.where(d.abs() < 1e-30, torch.full_like(d, 1e-30), d)
    side = ((cell + (step > 0)).double() - o) * inv
    delta = inv.abs()
    t = torch.zeros(len(rays), dtype=torch.float64, device="cuda")
    found = torch.full((len(rays),), float(abi.PYR_FLT_MAX), dtype=torch.float64, device="cuda")
    alive = torch.arange(len(rays), device="cuda")
    while len(alive):
        hit = occupied[cell[:, 0], cell[:, 1], cell[:, 2]]
        found[alive[hit]] = t[hit]
        axis = side.argmin(1, keepdim=True)
        t = side.gather(1, axis)[:, 0]
        cell = cell.scatter_add(1, axis, step.gather(1, axis))
        side = side.scatter_add(1, axis, delta.gather(1, axis))
        keep = ~hit & ((cell >= 0) & (cell < n)).all(1)
        alive, cell, side, delta, step, t = (x[keep] for x in (alive, cell, side, delta, step, t))
    return [found, None]
