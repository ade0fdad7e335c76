"""The work whose speed this library is measured by: culls, pyramid builds, batches and served requests, each made
through the C ABI (blitzen_amd.cull.lib()) the way a renderer makes them, with argument structs built once.

A case is a dict of plain values; "kind" says what it is:

    frame      EARLY -> pyramid build -> LATE over one scene, the order in which a renderer's frame makes the calls (the
               early draws are what the depth comes from); the visibility is written out of place
    pass       one PLAIN, ONPC or TEMPORAL pass (TEMPORAL after a pyramid build of its own)
    instanced  the LOD-instanced cull
    clusters   transform updates, then the two-level cluster cull
    views      many uneven views as one graph: pyramid builds and the batched LATE cull
    cascades   a few views of one scene in eager batched calls: shadow cascades (PLAIN) beside cameras (TEMPORAL)
    served     requests submitted to the serving loop, awaited and fetched

Objects are the seeded scenes of the tests and the benchmark: positions U[-500, 500]^3, scale U[0.5, 2], unit
quaternions. With "coherent" neighbouring ids are neighbours in space, as where a level is filled region by region;
otherwise ids are placed at random. With "shared" several objects use one transform.
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

from blitzen_amd import _capi as A
from blitzen_amd import cull as bz

ZNEAR, ZFAR = 0.1, 650.0


def listed():
    return [
        # the smallest scene worth a GPU cull (a single level's props): launches and latency only
        {"name": "frame_1k", "kind": "frame", "objects": 1000, "surfaces": 64, "lods": 4, "w": 512, "h": 512,
         "visible": 0.5, "cache": False, "shared": False, "coherent": False},
        # a game scene, culled the plain way (no frame cache), ids in placement order
        {"name": "frame_65k", "kind": "frame", "objects": 65536, "surfaces": 256, "lods": 8, "w": 1920, "h": 1080,
         "visible": 0.1, "cache": False, "shared": False, "coherent": True},
        # a ragged scene with instanced props (shared transforms), tables too large for LDS, an odd window
        {"name": "frame_262k_odd", "kind": "frame", "objects": 262161, "surfaces": 3001, "lods": 8, "w": 1366,
         "h": 768, "visible": 0.1, "cache": True, "shared": True, "coherent": False},
        # an open world without the frame cache: LATE reads every object again
        {"name": "frame_1m", "kind": "frame", "objects": 1048576, "surfaces": 256, "lods": 8, "w": 2560, "h": 1440,
         "visible": 0.1, "cache": False, "shared": False, "coherent": False},
        # the benchmark's frame: 4 194 304 objects, 1920 x 1080, frame cache
        {"name": "frame_4m", "kind": "frame", "objects": 4194304, "surfaces": 256, "lods": 8, "w": 1920, "h": 1080,
         "visible": 0.5, "cache": True, "shared": False, "coherent": False},
        # the transparent pass of the largest scenes of the benchmark (jobs over 4096 tiles)
        {"name": "plain_16m", "kind": "pass", "pass": A.PASS_PLAIN, "objects": 16777216, "surfaces": 256, "lods": 8,
         "w": 1920, "h": 1080, "pow2": True, "coherent": False},
        # occlusion against a pyramid whose base halves the window (not a power of two: one launch per level)
        {"name": "temporal_500k_odd", "kind": "pass", "pass": A.PASS_TEMPORAL, "objects": 500009, "surfaces": 256,
         "lods": 8, "w": 1600, "h": 900, "pow2": False, "coherent": True},
        # the D3D12 renderer's instanced output at the benchmark's size
        {"name": "instanced_4m", "kind": "instanced", "objects": 4194304, "surfaces": 256, "lods": 8,
         "per_lod": 8192, "coherent": False},
        # cluster mode of the benchmark: 1% of the transforms move, then both levels are culled
        {"name": "clusters_1m", "kind": "clusters", "objects": 1048576, "surfaces": 128, "lods": 8, "moved": 0.01,
         "coherent": False},
        # many uneven views in one replayed graph (the benchmark's distribution, a quarter of its views)
        {"name": "views_64", "kind": "views", "views": 64, "min_objects": 1024, "max_objects": 1048576},
        # a frame's shadow cascades and two cameras over one scene, in eager batched calls
        {"name": "cascades_150k", "kind": "cascades", "objects": 150001, "surfaces": 256, "lods": 8, "cascades": 4,
         "cameras": 2, "size": 1024},
        # a serving node under load: requests of mixed scenes and depth sizes
        {"name": "served_48", "kind": "served", "requests": 48, "scenes": 3, "min_objects": 262144},
    ]


def _log(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]; odd and ragged ones among them."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, n | 1 if rng.random() < 0.5 else n))


def draw(rng):
    kind = rng.choices(["frame", "pass", "instanced", "clusters", "views", "cascades", "served"],
                       [8, 4, 2, 2, 2, 2, 1])[0]
    surfaces, lods = rng.choice([(64, 4), (256, 8), (256, 8), (1000, 6)])
    case = {"kind": kind}
    if kind in ("frame", "pass"):
        w, h = rng.choice([(512, 512), (800, 600), (1024, 768), (1280, 720), (1366, 768), (1600, 900), (1920, 1080),
                           (2048, 1024), (2560, 1440)])
        case.update(surfaces=surfaces, lods=lods, w=w, h=h)
    if kind == "frame":
        n = _log(rng, 1000, 4194304)
        case.update(objects=n, visible=rng.choice([0.1, 0.5]), cache=rng.random() < 0.5, shared=rng.random() < 0.25,
                    coherent=n <= 1048576 and rng.random() < 0.5)
    elif kind == "pass":
        p = rng.choice([A.PASS_PLAIN, A.PASS_ONPC, A.PASS_TEMPORAL])
        n = _log(rng, 1000, 4194304 if p == A.PASS_TEMPORAL else 16777216)
        case.update({"pass": p}, objects=n, pow2=rng.random() < 0.7, coherent=n <= 1048576 and rng.random() < 0.5)
    elif kind == "instanced":
        n = _log(rng, 1000, 4194304)
        case.update(objects=n, surfaces=surfaces, lods=lods, per_lod=rng.choice([256, 1024, 8192]),
                    coherent=n <= 1048576 and rng.random() < 0.5)
    elif kind == "clusters":
        n = _log(rng, 4096, 1048576)
        case.update(objects=n, surfaces=128, lods=8, moved=rng.choice([0.001, 0.01, 0.05]),
                    coherent=rng.random() < 0.5)
    elif kind == "views":
        case.update(views=_log(rng, 8, 64), min_objects=1024, max_objects=rng.choice([65536, 262144, 1048576]))
    elif kind == "cascades":
        case.update(objects=_log(rng, 4096, 400000), surfaces=surfaces, lods=lods, cascades=rng.randint(2, 4),
                    cameras=rng.randint(1, 4), size=rng.choice([512, 1024]))
    else:
        case.update(requests=_log(rng, 8, 48), scenes=rng.randint(1, 3),
                    min_objects=rng.choice([65536, 131072, 262144]))
    return case


# ------------------------------------------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=None)
def _context():
    """The program's context: one for all of its scenes."""
    return bz.Context(0)


def _stream():
    return torch.cuda.current_stream().cuda_stream or None


def _scene(ctx, case, seed, n=None, clusters=(0, 0)):
    n = case["objects"] if n is None else n
    sc = bz.synth_scene(seed, n, case.get("surfaces", 256), case.get("lods", 8), clusters=clusters)
    if case.get("coherent"):
        cell = np.floor((sc.transforms["pos"] + 500.0) / 50.0).astype(np.int32)
        order = np.argsort((cell[:, 0] * 20 + cell[:, 2]) * 20 + cell[:, 1], kind="stable")
        sc.transforms = sc.transforms[order]
    if case.get("shared"):
        sc.objects["transformId"] = np.random.default_rng(seed).integers(0, max(1, n // 2), n, dtype=np.uint32)
    handle = ctx.scene_create(sc.objects, sc.transforms, sc.surfaces, sc.lods)
    if clusters[0]:
        ctx.scene_set_clusters(handle, sc.clusters)
    return handle, sc


def _view(rng, w, h, base_w=0, base_h=0, spread=100.0):
    v = bz.camera_setup(float(rng.uniform(50, 90)), w, h, ZNEAR, ZFAR, tuple(float(x) for x in
                        rng.uniform(-spread, spread, 3)), float(rng.uniform(-math.pi, math.pi)),
                        float(rng.uniform(-0.5, 0.5)))
    v.pyramidWidth, v.pyramidHeight = float(base_w), float(base_h)
    return v


def _depth(seed, w, h, occluders, device="cuda"):
    """A reverse-z depth image: ground below the horizon, sky above it, and boxes in front (the nearest depth wins)."""
    rng = np.random.default_rng([seed, w, h])
    y = torch.arange(h, dtype=torch.float64, device=device)
    ground = ((y + 0.5) / h * 2.0 - 1.0).clamp(min=0.0) * (ZNEAR / 10.0)
    d = ground.float().reshape(h, 1).repeat(1, w)
    x0, y0 = rng.integers(0, w, occluders), rng.integers(0, h, occluders)
    bw, bh = rng.integers(2, max(3, w // 8), occluders), rng.integers(2, max(3, h // 8), occluders)
    for i, z in enumerate(rng.uniform(0.001, 0.2, occluders).astype(np.float32)):
        d[y0[i]:y0[i] + bh[i], x0[i]:x0[i] + bw[i]].clamp_(min=float(z))
    return d


def _extent(case):
    """The pyramid of a window: the reference's power-of-two extent, or half of the window and every level below."""
    if case.get("pow2", True):
        return bz.reference_pyramid_extent(case["w"], case["h"])
    bw, bh = max(1, case["w"] // 2), max(1, case["h"] // 2)
    return bw, bh, min(16, max(bw, bh).bit_length())


def _texels(bw, bh, mips):
    return sum(max(1, bw >> k) * max(1, bh >> k) for k in range(mips))


class _Pyramid:
    """A pyramid and its texels, for as long as the state or a tensor over them is held."""

    def __init__(self, ctx, bw, bh, mips):
        self.ctx, self.handle = ctx, ctx.pyramid_create(bw, bh, mips)

    def values(self):
        """The texels as torch sees memory of another library: the tensor keeps this object."""
        p, n = C.c_void_p(), C.c_uint64()
        self.ctx.check(bz.lib().bz_pyramid_storage(self.ctx.handle, self.handle, C.byref(p), C.byref(n), None),
                       "bz_pyramid_storage")
        self.__cuda_array_interface__ = {"shape": (n.value,), "typestr": "<f4", "data": (p.value, False), "version": 2}
        return torch.as_tensor(self, device="cuda")

    def __del__(self):
        try:
            self.ctx.pyramid_destroy(self.handle)
        except Exception:  # the interpreter is going down
            pass


class _State:
    """What a program holds for one workload: scenes, pyramids, buffers, and its calls with their arguments."""

    def __init__(self, ctx, own_context=False):
        self.ctx, self.own, self.stream = ctx, own_context, _stream()
        self.scenes, self.pyramids, self.graphs, self.keep, self.calls, self.out = [], [], [], [], [], {}

    def zeros(self, *shape):
        t = torch.zeros(shape, dtype=torch.int32, device="cuda")
        self.keep.append(t)
        return t

    def call(self, name, *args):
        self.calls.append((name, getattr(bz.lib(), name), (self.ctx.handle, *args, self.stream)))

    def scene(self, *args, **kw):
        h, sc = _scene(self.ctx, *args, **kw)
        self.scenes.append(h)
        return h, sc

    def pyramid(self, bw, bh, mips):
        self.pyramids.append(_Pyramid(self.ctx, bw, bh, mips))
        return self.pyramids[-1]

    def cull(self, scene, view, pass_, cmds, count, capacity, pyramid=0, flags=0, vis_in=None, vis_out=None):
        a = A.CullArgs(scene=scene, pyramid=pyramid, pass_=pass_, flags=flags, view=C.pointer(view),
                       cmds_dev=cmds.data_ptr(), count_dev=count.data_ptr(), capacity=capacity, object_begin=0,
                       object_count=0, visibility_in_dev=vis_in.data_ptr() if vis_in is not None else None,
                       visibility_out_dev=vis_out.data_ptr() if vis_out is not None else None)
        self.keep += [a, view]
        self.call("bz_cull", C.byref(a))

    def __del__(self):
        try:
            torch.cuda.synchronize()
            if self.own:
                self.ctx.server_stop()
            for g in self.graphs:
                self.ctx.graph_destroy(g)
            for s in self.scenes:
                self.ctx.scene_destroy(s)
            if self.own:
                self.ctx.close()
        except Exception:  # the interpreter is going down
            pass


def prepare(case, seed):
    return {"frame": _prepare_frame, "pass": _prepare_pass, "instanced": _prepare_instanced,
            "clusters": _prepare_clusters, "views": _prepare_views, "cascades": _prepare_cascades,
            "served": _prepare_served}[case["kind"]](case, seed)


def _visibility(seed, n, p):
    return torch.from_numpy(bz.synth_visibility(seed, n, p).view(np.int32)).cuda()


def _prepare_frame(case, seed):
    s, n, rng = _State(_context()), case["objects"], np.random.default_rng(seed)
    scene, _ = s.scene(case, seed)
    bw, bh, mips = _extent(case)
    pyr, depth = s.pyramid(bw, bh, mips), _depth(seed, case["w"], case["h"], 256)
    view = _view(rng, case["w"], case["h"], bw, bh)
    vis, vis_out = _visibility(seed, n, case["visible"]), s.zeros(n)
    early, late, ne, nl = s.zeros(n, 6), s.zeros(n, 6), s.zeros(1), s.zeros(1)
    flags = A.CULL_FRAME_CACHE if case["cache"] else 0
    s.keep += [depth, vis]
    s.cull(scene, view, A.PASS_EARLY, early, ne, n, flags=flags, vis_in=vis)
    s.call("bz_pyramid_build", pyr.handle, depth.data_ptr(), case["w"], case["h"])
    s.cull(scene, view, A.PASS_LATE, late, nl, n, pyramid=pyr.handle, flags=flags, vis_in=vis, vis_out=vis_out)
    s.out = {"early": early, "early_count": ne, "late": late, "late_count": nl, "visibility": vis_out,
             "pyramid": pyr.values()}
    return s


def _prepare_pass(case, seed):
    s, n, rng = _State(_context()), case["objects"], np.random.default_rng(seed)
    scene, _ = s.scene(case, seed)
    bw, bh, mips = _extent(case)
    view = _view(rng, case["w"], case["h"], bw, bh)
    capacity = max(1024, n // 2)  # the benchmark's command buffer for its largest scenes
    cmds, count, handle = s.zeros(capacity, 6), s.zeros(1), 0
    s.out = {"commands": cmds, "count": count}
    if case["pass"] == A.PASS_TEMPORAL:
        pyr, depth = s.pyramid(bw, bh, mips), _depth(seed, case["w"], case["h"], 256)
        s.keep.append(depth)
        s.call("bz_pyramid_build", pyr.handle, depth.data_ptr(), case["w"], case["h"])
        s.out["pyramid"] = pyr.values()
        handle = pyr.handle
    s.cull(scene, view, case["pass"], cmds, count, capacity, pyramid=handle)
    return s


def _prepare_instanced(case, seed):
    s, rng = _State(_context()), np.random.default_rng(seed)
    scene, _ = s.scene(case, seed)
    view, n_lods, per = _view(rng, 1920, 1080), case["surfaces"] * case["lods"], case["per_lod"]
    ids, counters, cmds, count = s.zeros(n_lods * per), s.zeros(n_lods, 2), s.zeros(n_lods, 8), s.zeros(1)
    a = A.InstancedCullArgs(scene=scene, view=C.pointer(view), instances_per_lod=per, capacity=n_lods,
                            instance_ids_dev=ids.data_ptr(), counters_dev=counters.data_ptr(),
                            cmds_dev=cmds.data_ptr(), count_dev=count.data_ptr())
    s.keep += [a, view]
    s.call("bz_cull_instanced", C.byref(a))
    s.out = {"ids": ids, "counters": counters, "commands": cmds, "count": count}
    return s


def _prepare_clusters(case, seed):
    s, n, rng = _State(_context()), case["objects"], np.random.default_rng(seed)
    scene, sc = s.scene(case, seed, clusters=(16, 128))
    w, h = 1920, 1080
    bw, bh, mips = bz.reference_pyramid_extent(w, h)
    pyr, depth, view = s.pyramid(bw, bh, mips), _depth(seed, w, h, 256), _view(rng, w, h, bw, bh)
    s.ctx.pyramid_build(pyr.handle, depth.data_ptr(), w, h, s.stream)  # last frame's
    ids, moved = bz.synth_transform_updates(seed, 1, sc.transforms, max(1, int(n * case["moved"])))
    records = n * 4  # several times what a view expands
    dispatch, cmds, nd, nc = s.zeros(records, 3), s.zeros(n, 6), s.zeros(1), s.zeros(1)
    tests = A.CLUSTER_FRUSTUM | A.CLUSTER_HIZ | A.CLUSTER_CONE
    a = A.ClusterCullArgs(scene=scene, pyramid=pyr.handle, cluster_tests=tests, flags=0, view=C.pointer(view),
                          dispatch_dev=dispatch.data_ptr(), dispatch_count_dev=nd.data_ptr(),
                          dispatch_capacity=records, cmds_dev=cmds.data_ptr(), count_dev=nc.data_ptr(), capacity=n)
    s.keep += [depth, ids, moved, a, view]
    s.call("bz_scene_update_transforms", scene, A.ptr(ids), A.ptr(moved), len(ids))
    s.call("bz_cull_clusters", C.byref(a))
    s.out = {"dispatch": dispatch, "dispatch_count": nd, "commands": cmds, "count": nc}
    return s


def _plan(case, seed):
    """(first object, objects, depth width, depth height) of each view; the sizes follow from the seed."""
    rng = np.random.default_rng(seed)
    n = np.exp(rng.uniform(math.log(case["min_objects"]), math.log(case["max_objects"]), case["views"])).astype(int)
    sizes = [[(512, 512), (1024, 1024), (2048, 1024)][k] for k in rng.integers(0, 3, case["views"])]
    return [(int(b), int(c), *z) for b, c, z in zip(np.cumsum(n) - n, n, sizes)]


def _prepare_views(case, seed):
    s, rng, plan = _State(_context()), np.random.default_rng([seed, 1]), _plan(case, 7)
    total = plan[-1][0] + plan[-1][1]
    scene, _ = s.scene(case, seed, n=total)
    vis, vis_out = _visibility(seed, total, 0.5), s.zeros(total)
    cmds, counts = s.zeros(total, 6), s.zeros(len(plan))
    s.keep.append(vis)
    jobs, builds = [], []
    for k, (begin, n, w, h) in enumerate(plan):
        bw, bh, mips = bz.reference_pyramid_extent(w, h)
        pyr, depth = s.pyramid(bw, bh, mips), _depth(seed + 1000 * k, w, h, 64)
        s.keep.append(depth)
        builds.append((pyr.handle, depth.data_ptr(), w, h))
        jobs.append(A.ViewJob(scene=scene, pyramid=pyr.handle, pass_=A.PASS_LATE, object_begin=begin, object_count=n,
                              capacity=n, view=_view(rng, w, h, bw, bh), visibility_in_dev=vis.data_ptr(),
                              visibility_out_dev=vis_out.data_ptr(), cmds_dev=cmds.data_ptr() + 24 * begin,
                              count_dev=counts.data_ptr() + 4 * k))
    s.graphs.append(s.ctx.batch_graph_create(builds, jobs))
    s.call("bz_graph_launch", s.graphs[0])
    s.out = {"commands": cmds, "counts": counts, "visibility": vis_out}
    return s


def _prepare_cascades(case, seed):
    s, n, rng = _State(_context()), case["objects"], np.random.default_rng(seed)
    scene, _ = s.scene(case, seed)
    size, views = case["size"], case["cascades"] + case["cameras"]
    bw, bh, mips = bz.reference_pyramid_extent(size, size)
    cmds, counts, jobs, builds = s.zeros(views, n, 6), s.zeros(views), [], []
    for k in range(views):
        camera = k >= case["cascades"]
        handle = 0
        if camera:
            pyr, depth = s.pyramid(bw, bh, mips), _depth(seed + 1000 * k, size, size, 64)
            s.keep.append(depth)
            handle = pyr.handle
            builds.append(A.PyramidJob(pyramid=handle, depth_dev=depth.data_ptr(), w=size, h=size))
        jobs.append(A.ViewJob(scene=scene, pyramid=handle, pass_=A.PASS_TEMPORAL if camera else A.PASS_PLAIN,
                              object_begin=0, object_count=n, capacity=n, view=_view(rng, size, size, bw, bh),
                              visibility_in_dev=None, visibility_out_dev=None, cmds_dev=cmds.data_ptr() + 24 * n * k,
                              count_dev=counts.data_ptr() + 4 * k))
    b, j = (A.PyramidJob * len(builds))(*builds), (A.ViewJob * len(jobs))(*jobs)
    s.keep += [b, j]
    s.call("bz_pyramid_build_batch", b, len(builds))
    s.call("bz_cull_batch", j, len(jobs))
    s.out = {"commands": cmds, "counts": counts}
    return s


def _served_scenes(case):
    return [case["min_objects"] << k for k in range(case["scenes"])]


def _served_plan(case):
    """(scene, depth width, depth height) of each request."""
    rng = np.random.default_rng(11)
    sizes = [(512, 512), (800, 600), (1024, 768), (1280, 720), (1600, 900), (1920, 1080)]
    return [(int(rng.integers(case["scenes"])), *sizes[int(rng.integers(len(sizes)))]) for _ in range(case["requests"])]


def _prepare_served(case, seed):
    s, rng = _State(bz.Context(0), own_context=True), np.random.default_rng(seed)
    handles = [s.scene(case, seed + k, n=n)[0] for k, n in enumerate(_served_scenes(case))]
    s.ctx.server_start(4 << 30, inflight=4, max_batch=16)
    s.requests = [bz.Context.request(handles[k], _view(rng, w, h, spread=50.0), depth_seed=seed * 1000 + i, depth_w=w,
                                     depth_h=h, occluders=128, user_tag=i)
                  for i, (k, w, h) in enumerate(_served_plan(case))]
    s.out = {"counts": np.zeros(len(s.requests), np.uint32),
             "commands": [np.zeros((_served_scenes(case)[k] // 4, 6), np.uint32) for k, _, _ in _served_plan(case)]}
    return s


# ------------------------------------------------------------------------------------------------- the work
def run(state):
    if state.own:
        return _serve(state)
    for name, fn, args in state.calls:
        status = fn(*args)
        if status:
            state.ctx.check(status, name)
    return state.out


def _serve(state):
    lib, ctx, counts = bz.lib(), state.ctx, state.out["counts"]
    ticket, result, n = C.c_uint64(), A.Result(), C.c_uint32()
    tickets = []
    for r in state.requests:
        ctx.check(lib.bz_server_submit(ctx.handle, C.byref(r), C.byref(ticket)), "bz_server_submit")
        tickets.append(ticket.value)
    for i, (t, cmds) in enumerate(zip(tickets, state.out["commands"])):
        ctx.check(lib.bz_server_wait(ctx.handle, t, 0, C.byref(result)), "bz_server_wait")
        ctx.check(result.status, "request")
        ctx.check(lib.bz_server_fetch(ctx.handle, t, A.ptr(cmds), len(cmds), C.byref(n)), "bz_server_fetch")
        counts[i] = n.value
    return state.out


def work(case):
    """One pass: a bounding sphere read per object (16 B) and its visibility read and written where the path has it;
    every depth image read, every pyramid texel written; the commands of the objects drawn (about a twentieth)."""
    kind, drawn = case["kind"], 24 / 20
    if kind == "frame":
        depth = 4 * case["w"] * case["h"] + 4 * _texels(*_extent(case))
        return {"bytes": case["objects"] * (16 + 4 + 4 + drawn) + depth, "flops": 60 * case["objects"]}
    if kind == "pass":
        b = case["objects"] * (16 + drawn)
        if case["pass"] == A.PASS_TEMPORAL:
            b += 4 * case["w"] * case["h"] + 4 * _texels(*_extent(case))
        return {"bytes": b, "flops": 60 * case["objects"]}
    if kind == "instanced":
        return {"bytes": case["objects"] * (16 + 4 / 20) + case["surfaces"] * case["lods"] * 40,
                "flops": 60 * case["objects"]}
    if kind == "clusters":  # a record per seven objects, written, its cluster read; the moved transforms over the link
        return {"bytes": case["objects"] * (16 + (12 + 28) / 7 + 36 * case["moved"]), "flops": 70 * case["objects"]}
    if kind == "views":
        plan = _plan(case, 7)
        n = sum(p[1] for p in plan)
        return {"bytes": n * (16 + 4 + 4 + drawn) + sum(4 * w * h + 4 * _texels(*bz.reference_pyramid_extent(w, h))
                                                        for _, _, w, h in plan), "flops": 60 * n}
    if kind == "cascades":  # one scene: its spheres are read once for all views
        e, views = bz.reference_pyramid_extent(case["size"], case["size"]), case["cascades"] + case["cameras"]
        depth = case["cameras"] * 4 * (case["size"] ** 2 + _texels(*e))
        return {"bytes": case["objects"] * (16 + views * drawn) + depth, "flops": 60 * case["objects"] * views}
    plan, sizes = _served_plan(case), _served_scenes(case)
    n = sum(sizes[k] for k, _, _ in plan)
    return {"bytes": sum(sizes) * 16 + n * drawn + sum(4 * w * h + 4 * _texels(*bz.reference_pyramid_extent(w, h))
                                                       for _, w, h in plan), "flops": 60 * n}


def exact(case, seed):
    """The pyramid (the only floating output) from the depth image: the minimum over the texels of each bilinear
    footprint that have weight. The commands, counts, ids and visibility are whole numbers."""
    if case["kind"] not in ("frame", "pass") or (case["kind"] == "pass" and case["pass"] != A.PASS_TEMPORAL):
        return None
    bw, bh, mips = _extent(case)
    src, levels = _depth(seed, case["w"], case["h"], 256, "cpu").numpy().astype(np.float64), []

    def axis(n_dst, n_src):
        f = np.float32  # the sample position is a float32 by definition: its rounding decides which texels have weight
        t = (np.arange(n_dst).astype(f) + f(0.5)) / f(n_dst) * f(n_src) - f(0.5)
        lo = np.floor(t)
        i0 = np.clip(lo, 0, n_src - 1).astype(int)
        return i0, np.where(t - lo > 0, np.clip(lo + 1, 0, n_src - 1).astype(int), i0)

    for k in range(mips):
        (x0, x1), (y0, y1) = axis(max(1, bw >> k), src.shape[1]), axis(max(1, bh >> k), src.shape[0])
        rows = np.minimum(src[y0], src[y1])
        src = np.minimum(rows[:, x0], rows[:, x1])
        levels.append(src.reshape(-1))
    pyramid = np.concatenate(levels)
    if case["kind"] == "pass":
        return {"commands": None, "count": None, "pyramid": pyramid}
    return {"early": None, "early_count": None, "late": None, "late_count": None, "visibility": None,
            "pyramid": pyramid}
