"""What the scene-update path is timed on: single calls and per-frame call
sequences of a renderer that keeps its scene on the device, over the range of
sizes this package is used at.

  cull    one view of one group (dpc_cull through device.cull): a 10,000-object
          scene, where the call itself is the cost, up to millions of objects
  frames  two consecutive frames of a moving camera over a group that keeps its
          result (dpc_cull_diff): mask, changed list, count, and the result's
          updated bits, as culling::Manager::cull runs it
  views   many views in one launch (BatchPlan.cull): shadow cascades, cube map
          faces and cameras over groups of objects
  tree    the transform tree: all nodes propagated and the objects on its leaves
          culled (a scene's first frame, or an animation that moves everything)
  edit    a frame that changes some local matrices: the delta scattered, the
          changes propagated, inverse transposes and the changed-matrix event
          (the call sequence of transform::Tree::compute)
  load    a group's arrays brought into device form, its matrix indices mapped to
          tree slots, the matrices read back, and the group's bounding box
  serve   one tick of the serving loop: each resident scene gets a request with a
          matrix delta and 1-32 views
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from pipeline_amd import _lib, autotune, scenes
from pipeline_amd import device as dev
from pipeline_amd.serving import PinnedArray, Server


def listed():
    return [
        # The smallest call in use: 10,000 objects, one camera.  Call and launch latency.
        {"name": "cull-10k", "kind": "cull", "n": 10_000, "extent": 100.0, "indexed": 0},
        # The single-view scene of a million objects, a matrix each.
        {"name": "cull-1m", "kind": "cull", "n": 1_048_576, "extent": 1000.0, "indexed": 0},
        # The largest single view: an odd count that fills no tile.
        {"name": "cull-5m", "kind": "cull", "n": 4_999_999, "extent": 1000.0, "indexed": 0},
        # Frames of a small interactive scene (four objects share a matrix).
        {"name": "frames-60k", "kind": "frames", "n": 60_001, "extent": 200.0, "indexed": 4},
        # Frames over as many objects as the million-node tree has on its leaves.
        {"name": "frames-2.4m", "kind": "frames", "n": 2_372_871, "extent": 1000.0, "indexed": 4},
        # A few views over a few small groups in the default launch shape.
        {"name": "views-20k", "kind": "views", "n": 20_000, "groups": 8, "frusta": 8, "all": 0, "tuned": 0, "extent": 100.0},
        # The benchmark's multi-view step: 64 views, each of 1-8 of 64 groups.
        {"name": "views-2m", "kind": "views", "n": 2_097_152, "groups": 64, "frusta": 64, "all": 0, "tuned": 1, "extent": 1000.0},
        # Every view sees the whole scene: cascades, cube faces and cameras of one group.
        {"name": "views-whole-500k", "kind": "views", "n": 500_003, "groups": 1, "frusta": 32, "all": 1, "tuned": 0, "extent": 1000.0},
        # The million-node tree: full propagation, then its leaves' objects culled.
        {"name": "tree-1m", "kind": "tree", "nodes": 1_000_000},
        # One percent of a quarter-million-node tree's local matrices edited.
        {"name": "edit-250k", "kind": "edit", "nodes": 250_007, "dirty": 0.01},
        # A group of 600,000 objects loaded; its matrices lie 80 bytes apart.
        {"name": "load-600k", "kind": "load", "n": 600_011, "stride": 80, "extent": 1000.0},
        # Sixteen resident scenes of 10,000-400,000 objects, one request each.
        {"name": "serve-16", "kind": "serve", "scenes": 16, "largest": 400_000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cull", "cull", "frames", "frames", "views", "views", "views", "tree", "edit", "load", "serve"])
    if kind in ("cull", "frames"):
        n = _log(rng, 5_000, 4_900_000 if kind == "cull" else 2_300_000)
        return {"kind": kind, "n": n, "extent": round(100.0 * (n / 1e4) ** 0.5, 1), "indexed": rng.choice([0, 1, 4, 7])}
    if kind == "views":
        while True:
            n, frusta = _log(rng, 5_000, 2_000_000), rng.randint(1, 64)
            groups = _log(rng, 1, 64)
            every = rng.choice([0, 0, 1])
            if n * frusta * (1.0 if every else min(1.0, 4.5 / groups)) <= 16e6:
                return {"kind": kind, "n": n, "groups": groups, "frusta": frusta, "all": every,
                        "tuned": rng.choice([0, 1]), "extent": round(100.0 * (n / 1e4) ** 0.5, 1)}
    if kind == "tree":
        return {"kind": kind, "nodes": _log(rng, 3_000, 980_000)}
    if kind == "edit":
        return {"kind": kind, "nodes": _log(rng, 3_000, 700_000), "dirty": round(math.exp(rng.uniform(math.log(0.001), 0.0)), 4)}
    if kind == "load":
        return {"kind": kind, "n": _log(rng, 5_000, 900_000), "stride": rng.choice([64, 64, 80, 68, 128]), "extent": 500.0}
    return {"kind": kind, "scenes": rng.randint(2, 16), "largest": _log(rng, 20_000, 380_000)}


# ---- inputs ---------------------------------------------------------------------
class Buf:
    """A torch tensor as the package's device functions take a device array."""

    def __init__(self, t):
        self.t = t

    ptr = property(lambda self: C.c_void_p(self.t.data_ptr()))
    addr = property(lambda self: self.t.data_ptr())
    nbytes = property(lambda self: self.t.numel() * self.t.element_size())


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * (hi - lo) + lo


def _boxes(g, n, extent, half=(0.1, 2.0)):
    c, h = _uniform(g, (n, 3), -extent, extent), _uniform(g, (n, 3), *half)
    return torch.cat([c - h, c + h], dim=1).contiguous()


def _trs(g, n, scale=(0.5, 2.0), trans=(-5.0, 5.0)):
    """Rotation x uniform scale x translation, row-vector convention, (n, 4, 4)."""
    q = torch.randn((n, 4), generator=g, device="cuda", dtype=torch.float32)
    x, y, z, w = (q / q.norm(dim=1, keepdim=True)).unbind(1)
    rows = [[1 - 2 * (y * y + z * z), 2 * (x * y + z * w), 2 * (x * z - y * w)],
            [2 * (x * y - z * w), 1 - 2 * (x * x + z * z), 2 * (y * z + x * w)],
            [2 * (x * z + y * w), 2 * (y * z - x * w), 1 - 2 * (x * x + y * y)]]
    m = torch.zeros((n, 4, 4), device="cuda", dtype=torch.float32)
    m[:, :3, :3] = torch.stack([torch.stack(r, dim=1) for r in rows], dim=1) * _uniform(g, (n, 1, 1), *scale)
    m[:, 3, :3] = _uniform(g, (n, 3), *trans)
    m[:, 3, 3] = 1.0
    return m


def _camera(rng, extent):
    return scenes.perspective_vp(rng.uniform(-extent / 20, extent / 20, 3), rng.normal(size=3), 45.0, 16 / 9, 0.1, 2 * extent)


def _empty(n, dtype):
    return Buf(torch.zeros(max(int(n), 1), device="cuda", dtype=dtype))


def _scene(lower_upper, mats, xform=None):
    """A group resident in the backend's layout (mats: (k, 4, 4) as the caller stores them)."""
    lib, n, k = _lib.load(), lower_upper.shape[0], mats.shape[0]
    a, b, p = _empty(4 * n, torch.float32), _empty(2 * n, torch.float32), _empty(16 * k, torch.float32)
    _lib.check(lib.dpc_boxes_from_lower_upper(lower_upper.data_ptr(), n, a.ptr, b.ptr, None))
    _lib.check(lib.dpc_matrices_from_aos(mats.contiguous().data_ptr(), 64, k, p.ptr, k, None))
    torch.cuda.synchronize()
    return dev.DeviceScene(a, b, p, k, n, None if xform is None else Buf(xform))


def _group(case, g):
    """A group of case["n"] objects: a matrix each, or (indexed = s > 0) one for about s objects."""
    n, share = case["n"], case["indexed"]
    k = n if not share else max(n // share, 1)
    xform = None
    if share:
        xform = torch.arange(n, device="cuda", dtype=torch.int64).div(share, rounding_mode="floor").clamp_(max=k - 1).to(torch.int32)
    return _scene(_boxes(g, n, case["extent"]), _trs(g, k), xform)


class State(dict):
    """A case's state; plans and servers are given back with it."""

    def __del__(self):
        for close in self.get("close", ()):
            close()


def prepare(case, seed):
    rng, g = np.random.default_rng(int(seed)), _gen(seed)
    st = State(kind=case["kind"])
    globals()["_prepare_" + case["kind"]](case, rng, g, st)
    torch.cuda.synchronize()
    return st


def run(st):
    return globals()["_run_" + st["kind"]](st)


# ---- cull: one view of one group --------------------------------------------------
def _prepare_cull(case, rng, g, st):
    st.update(scene=_group(case, g), vp=_camera(rng, case["extent"]), mask=_empty(dev.mask_words(case["n"]), torch.int64))


def _run_cull(st):
    return dev.cull(st["scene"], st["vp"], st["mask"]).t


# ---- frames: two frames of a moving camera, with the result's diff ------------------
def _prepare_frames(case, rng, g, st):
    n, e = case["n"], case["extent"]
    words = dev.mask_words(n)
    eye, look = rng.uniform(-e / 20, e / 20, 3), rng.normal(size=3)
    st.update(scene=_group(case, g), old=_empty(words, torch.int64),
              ws=_empty((_lib.load().dpc_cull_diff_workspace(n) + 7) // 8, torch.int64),
              vps=[scenes.perspective_vp(eye, look, 60.0, 16 / 9, 0.1, 2 * e),
                   scenes.perspective_vp(eye + rng.normal(size=3) * e / 200, look / np.linalg.norm(look) + 0.05 * rng.normal(size=3),
                                         60.0, 16 / 9, 0.1, 2 * e)],
              out=[dict(mask=_empty(words, torch.int64), changed=_empty(n, torch.int32), count=_empty(1, torch.int32)) for _ in range(2)])
    _run_frames(st)  # the camera has been moving for a while: the result holds the second frame's bits
    for o in st["out"]:
        o["changed"].t.zero_()


def _run_frames(st):
    lib, s = _lib.load(), st["scene"]
    for vp, o in zip(st["vps"], st["out"]):
        _lib.check(lib.dpc_cull_diff(s.box_a.ptr, s.box_b.ptr, s.xform_addr, s.n_objects, s.planes.ptr, s.ld, dev.vp_arg(vp),
                                     o["mask"].ptr, st["old"].ptr, o["changed"].ptr, o["count"].ptr, 1, st["ws"].ptr, None))
    return [[o["mask"].t, o["changed"].t, o["count"].t] for o in st["out"]] + [st["old"].t]


# ---- views: many views in one launch -------------------------------------------------
def _who_sees_what(case):
    """Group sizes and each view's groups: the case's, so that every seed does the same work."""
    n, F, G = case["n"], case["frusta"], case["groups"]
    r = np.random.default_rng(n * 131 + F)
    sizes = scenes.log_uniform_sizes(r, G, n, 1.0, 500.0)
    return sizes, [range(G) if case["all"] else sorted(r.choice(G, size=min(int(r.integers(1, 9)), G), replace=False)) for _ in range(F)]


def _prepare_views(case, rng, g, st):
    n, e, F, G = case["n"], case["extent"], case["frusta"], case["groups"]
    sizes, seen = _who_sees_what(case)
    first = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    light, cam, centre = rng.normal(size=3), rng.uniform(-e / 20, e / 20, 3), rng.uniform(-e / 4, e / 4, 3)
    light /= np.linalg.norm(light)
    faces = ([1, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0], [0, 0, 1], [0, 0, -1])
    vps = []
    for f in range(F):
        if f < 4:  # shadow cascades
            w = e / 20 * 4.0 ** f
            view = scenes.make_lookat(cam - light * 2 * e, cam, np.array([0.0, 0.0, 1.0]) if abs(light[1]) > 0.95 else np.array([0.0, 1.0, 0.0]))
            vps.append(scenes.view_projection(view, scenes.make_ortho(-w, w, -w, w, 0.1, 4 * e)))
        elif f < 10:  # the faces of a cube map
            vps.append(scenes.perspective_vp(centre, np.array(faces[f - 4], np.float64), 90.0, 1.0, 0.1, 2 * e))
        else:
            vps.append(scenes.perspective_vp(rng.uniform(-e / 2, e / 2, 3), rng.normal(size=3), rng.uniform(30, 90), 16 / 9, 0.1,
                                             rng.uniform(e / 10, 3 * e)))
    vps = np.stack(vps).astype(np.float32)
    pairs, word, tests = [], 0, 0
    for f in range(F):
        for k in seen[f]:
            pairs.append((f, int(k), word))
            word += (int(sizes[k]) + 63) // 64
            tests += int(sizes[k])
    plan = dev.BatchPlan([(0, int(a), int(c)) for a, c in zip(first, sizes)], pairs, F,
                         autotune.best_batch_config(n, tests, F) if case["tuned"] else None)
    st["close"] = [plan.destroy]
    scene = _scene(_boxes(g, n, e), _trs(g, n))
    plan.bind([scene])
    st.update(plan=plan, scene=scene, vps=Buf(torch.from_numpy(vps.reshape(-1, 16)).cuda()), masks=_empty(word, torch.int64))


def _run_views(st):
    st["plan"].cull(st["vps"], st["masks"])
    return st["masks"].t


# ---- the transform tree ---------------------------------------------------------------
def _tree_scene(case, g):
    """The case's tree (its shape is the case's) and its local matrices."""
    ts = scenes.tree_scene(case["nodes"], case["nodes"] % 1009)
    local = _trs(g, ts.n_slots, (0.8, 1.25), (-10.0, 10.0))
    local[0] = torch.eye(4, device="cuda")
    return ts, local


def _tree(case, g, st):
    """The tree on the device: locals, worlds (root = identity), its launch plan, and the objects on its leaves."""
    ts, d_aos = _tree_scene(case, g)
    lib, n = _lib.load(), ts.n_slots
    local, world = _empty(16 * n, torch.float32), _empty(16 * n, torch.float32)
    _lib.check(lib.dpc_matrices_from_aos(d_aos.data_ptr(), 64, n, local.ptr, n, None))
    world.t.view(4, n, 4)[:, 0] = torch.eye(4, device="cuda")
    plan = C.c_void_p()
    parents, offsets = np.ascontiguousarray(ts.parent_slot, np.uint32), np.ascontiguousarray(ts.level_offsets, np.uint64)
    _lib.check(lib.dpc_tree_plan_create(parents.ctypes.data, n, offsets.ctypes.data, len(offsets) - 1, 0, C.byref(plan)))
    st.update(close=[lambda: lib.dpc_tree_plan_destroy(plan)], plan=plan, n=n, local=local, world=world,
              dirty_world=_empty((n + 3) // 4, torch.int32))
    return ts


def _prepare_tree(case, rng, g, st):
    ts = _tree(case, g, st)
    m = ts.obj_slot.size
    a, b = _empty(4 * m, torch.float32), _empty(2 * m, torch.float32)
    lu = _boxes(g, m, 2.0, (0.05, 1.0))
    _lib.check(_lib.load().dpc_boxes_from_lower_upper(lu.data_ptr(), m, a.ptr, b.ptr, None))
    torch.cuda.synchronize()
    st.update(scene=dev.DeviceScene(a, b, st["world"], st["n"], m, Buf(torch.from_numpy(ts.obj_slot.view(np.int32)).cuda())),
              vp=scenes.perspective_vp(rng.uniform(-50, 50, 3), rng.normal(size=3), 60.0, 16 / 9, 0.1, 1000.0), mask=_empty(dev.mask_words(m), torch.int64))


def _run_tree(st):
    _lib.check(_lib.load().dpc_tree_propagate_plan(st["plan"], st["local"].ptr, st["world"].ptr, None, st["dirty_world"].ptr, None))
    return [dev.cull(st["scene"], st["vp"], st["mask"]).t, st["world"].t]


def _prepare_edit(case, rng, g, st):
    ts = _tree(case, g, st)
    lib, n = _lib.load(), st["n"]
    count = max(1, int(round(case["dirty"] * (n - 1))))
    slots = np.sort(rng.choice(np.arange(1, n), count, replace=False)).astype(np.int32)
    dirty = np.zeros(n, np.uint8)
    dirty[slots] = 1
    st.update(count=count, idx=Buf(torch.from_numpy(slots).cuda()), delta=Buf(_trs(g, count, (0.8, 1.25), (-10.0, 10.0))),
              dirty=Buf(torch.from_numpy(dirty).cuda()), index=Buf(torch.from_numpy(ts.index_of_slot.view(np.int32)).cuda()),
              inverse=_empty(16 * n, torch.float32), bits=_empty(2 * dev.mask_words(n), torch.int32))
    # the scene's first frame has been computed
    _lib.check(lib.dpc_tree_propagate_plan(st["plan"], st["local"].ptr, st["world"].ptr, None, st["dirty_world"].ptr, None))
    _lib.check(lib.dpc_inverse_transpose(st["world"].ptr, n, None, n, st["inverse"].ptr, n, None, None))
    _lib.check(lib.dpc_fill_u32(st["dirty_world"].ptr, 0, (n + 3) // 4, None))


def _run_edit(st):
    lib, n = _lib.load(), st["n"]
    _lib.check(lib.dpc_matrices_scatter(st["local"].ptr, n, st["idx"].ptr, st["delta"].ptr, st["count"], None))
    _lib.check(lib.dpc_tree_propagate_plan(st["plan"], st["local"].ptr, st["world"].ptr, st["dirty"].ptr, st["dirty_world"].ptr, None))
    _lib.check(lib.dpc_inverse_transpose(st["world"].ptr, n, st["dirty_world"].ptr, n, st["inverse"].ptr, n, None, None))
    _lib.check(lib.dpc_fill_u32(st["bits"].ptr, 0, st["bits"].nbytes // 4, None))
    _lib.check(lib.dpc_bytes_to_bits_indexed(st["dirty_world"].ptr, st["index"].ptr, n, st["bits"].ptr, n, None))
    _lib.check(lib.dpc_fill_u32(st["dirty_world"].ptr, 0, (n + 3) // 4, None))
    return [st["world"].t, st["inverse"].t, st["bits"].t, st["local"].t]


# ---- load: a group's arrays into device form, and its bounding box ----------------------
def _prepare_load(case, rng, g, st):
    n, e, stride = case["n"], case["extent"], case["stride"]
    k = max(n // 3, 1)
    aos = _uniform(g, (k, stride // 4), -1.0, 1.0)  # (a record's other members lie between the matrices)
    aos[:, :16] = _trs(g, k).reshape(k, 16)
    table = torch.randperm(k, generator=g, device="cuda").to(torch.int32)
    xform = torch.randint(0, k, (n,), generator=g, device="cuda").to(torch.int32)
    st.update(n=n, k=k, stride=stride, lu=Buf(_boxes(g, n, e)), aos=Buf(aos.contiguous()), table=Buf(table), xform=Buf(xform),
              slot=_empty(n, torch.int32), a=_empty(4 * n, torch.float32), b=_empty(2 * n, torch.float32),
              planes=_empty(16 * k, torch.float32), back=_empty(16 * k, torch.float32), box=_empty(6, torch.float32),
              ws=_empty((_lib.load().dpc_bbox_workspace(n) + 7) // 8, torch.int64))


def _run_load(st):
    lib, n, k = _lib.load(), st["n"], st["k"]
    _lib.check(lib.dpc_boxes_from_lower_upper(st["lu"].ptr, n, st["a"].ptr, st["b"].ptr, None))
    _lib.check(lib.dpc_matrices_from_aos(st["aos"].ptr, st["stride"], k, st["planes"].ptr, k, None))
    _lib.check(lib.dpc_gather_u32(st["table"].ptr, k, st["xform"].ptr, n, st["slot"].ptr, None))
    _lib.check(lib.dpc_matrices_to_aos(st["planes"].ptr, k, st["table"].ptr, k, st["back"].ptr, 64, None))
    _lib.check(lib.dpc_bbox(st["a"].ptr, st["b"].ptr, st["slot"].ptr, n, st["planes"].ptr, k, st["box"].ptr, st["ws"].ptr, None))
    return [st["a"].t, st["b"].t, st["planes"].t, st["slot"].t, st["back"].t, st["box"].t]


# ---- serve: one tick over resident scenes ------------------------------------------------
def _prepare_serve(case, rng, g, st):
    srv = Server()
    st["close"] = [srv.close]
    reqs, pinned = [], []
    # (the mix of sizes and views is the case's, so that every seed does about the same work)
    spread = np.random.default_rng(case["scenes"] * 1009 + case["largest"])
    sizes = np.exp(spread.uniform(np.log(10_000), np.log(case["largest"]), case["scenes"])).astype(int)
    sizes[0] = case["largest"]
    for n in map(int, sizes):
        lu = _boxes(g, n, 1000.0).cpu().numpy()
        sid = srv.add_scene(lu[:, :3], lu[:, 3:], _trs(g, n).cpu().numpy())
        F, k = int(spread.integers(1, 33)), max(1, int(round(spread.uniform(0.01, 0.10) * n)))
        arrays = [PinnedArray((srv.mask_words(sid, F),), np.uint64), PinnedArray((k,), np.uint32), PinnedArray((k, 4, 4), np.float32)]
        arrays[0].array[:] = 0
        arrays[1].array[:] = torch.randperm(n, generator=g, device="cuda")[:k].cpu().numpy()
        arrays[2].array[:] = _trs(g, k).cpu().numpy()
        pinned += arrays
        reqs.append((sid, np.stack([_camera(rng, 1000.0) for _ in range(F)])) + tuple(p.array for p in arrays))
    st["close"] += [p.free for p in pinned]
    st.update(server=srv, requests=reqs)


class Masks(list):
    """The requests' masks; they lie in the state's pinned buffers, which live as long as this list."""


def _run_serve(st):
    srv = st["server"]
    ids = [srv.submit(sid, vps, masks, idx, mats) for sid, vps, masks, idx, mats in st["requests"]]
    for rid in ids:
        srv.wait(rid)
    out = Masks(r[2].view(np.int64) for r in st["requests"])
    out.state = st
    return out


# ---- work --------------------------------------------------------------------------------
def work(case):
    """Bytes that have to be read and written and FP32 operations of the transforms and
    corner sums (40 per object, 140 per object and view, 112 per tree node)."""
    kind = case["kind"]
    if kind in ("cull", "frames"):
        n, share = case["n"], case["indexed"]
        k = n if not share else max(n // share, 1)
        one = n * 24 + k * 64 + (4 * n if share else 0) + n / 8
        return {"bytes": one if kind == "cull" else 2 * (one + n / 4), "flops": 180 * n * (1 if kind == "cull" else 2)}
    if kind == "views":
        sizes, seen = _who_sees_what(case)
        objects, tests = sum(int(sizes[k]) for k in set().union(*seen)), sum(int(sizes[k]) for v in seen for k in v)
        return {"bytes": 88 * objects + tests / 8, "flops": 40 * objects + 140 * tests}
    if kind == "tree":
        n = case["nodes"]
        m = 2.37 * n  # objects on the leaves
        return {"bytes": n * (64 + 64 + 4 + 1) + m * (24 + 4 + 1 / 8), "flops": 112 * n + 180 * m}
    if kind == "edit":
        n, d = case["nodes"], case["dirty"]
        changed = min(1.0, 8.5 * d) * n  # (a node's change reaches its subtree)
        return {"bytes": d * n * 132 + n * (4 + 1 + 1 + 1 / 8) + changed * (64 + 64 + 64), "flops": changed * 220}
    if kind == "load":
        n, k = case["n"], max(case["n"] // 3, 1)
        return {"bytes": n * (24 + 24) + k * (64 + 64) + n * 8 + k * 4 + k * (64 + 64) + n * 28 + k * 64, "flops": 100 * n}
    m = case["scenes"] * (case["largest"] - 10_000) / max(math.log(case["largest"] / 10_000), 1e-3)
    return {"bytes": m * (88 + 0.055 * 2 * 68 + 16.5 / 8 * 2), "flops": m * (40 + 140 * 16.5)}


# ---- the same in 64 bits -------------------------------------------------------------------
def _world64(parent, offsets, local):
    """World matrices of a level-major tree (slot 0 = the root, identity)."""
    world = np.zeros_like(local)
    world[0] = np.eye(4)
    for a, b in zip(offsets[:-1], offsets[1:]):
        world[a:b] = np.matmul(local[a:b], world[parent[a:b]])
    return world


def _planes64(m):
    return np.ascontiguousarray(m.transpose(1, 0, 2)).reshape(-1)


def exact(case, seed):
    """The computed numbers in float64 (masks, lists, indices and event bits are whole numbers: None)."""
    rng, g = np.random.default_rng(int(seed)), _gen(seed)
    kind = case["kind"]
    if kind in ("tree", "edit"):
        ts, local = _tree_scene(case, g)
        parent, offsets = ts.parent_slot.astype(np.int64), ts.level_offsets.astype(np.int64)
        local = local.cpu().numpy().astype(np.float64)
        if kind == "tree":
            return [None, _planes64(_world64(parent, offsets, local))]
        n = ts.n_slots
        count = max(1, int(round(case["dirty"] * (n - 1))))
        slots = np.sort(rng.choice(np.arange(1, n), count, replace=False))
        local[slots] = _trs(g, count, (0.8, 1.25), (-10.0, 10.0)).cpu().numpy()
        world = _world64(parent, offsets, local)
        return [_planes64(world), _planes64(np.linalg.inv(world).transpose(0, 2, 1)), None, _planes64(local)]
    if kind == "load":
        n, k = case["n"], max(case["n"] // 3, 1)
        _uniform(g, (k, case["stride"] // 4), -1.0, 1.0)
        mats = _trs(g, k).double()
        table = torch.randperm(k, generator=g, device="cuda").to(torch.int32)
        xform = torch.randint(0, k, (n,), generator=g, device="cuda").to(torch.int32)
        lu = _boxes(g, n, case["extent"]).double()
        lower, ext = lu[:, :3], lu[:, 3:] - lu[:, :3]
        m = mats[table[xform.long()].long()]
        p = (lower[:, :, None] * m[:, :3, :3]).sum(1) + m[:, 3, :3]
        lo = torch.full((3,), math.inf, device="cuda", dtype=torch.float64)
        hi = -lo
        for c in range(8):
            v = p.clone()
            for axis in range(3):
                if c >> axis & 1:
                    v += ext[:, axis:axis + 1] * m[:, axis, :3]
            lo, hi = torch.minimum(lo, v.amin(0)), torch.maximum(hi, v.amax(0))
        return [torch.cat([lower, ext[:, :1]], dim=1).reshape(-1), ext[:, 1:].reshape(-1).contiguous(),
                mats.permute(1, 0, 2).reshape(-1).contiguous(), None, mats[table.long()].reshape(-1), torch.cat([lo, hi])]
    return None
