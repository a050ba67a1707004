"""The work that users of this framework have it do, as cases to be timed.

A case is one pass through the public interface as a user's program calls it
(oibvh_amd.api, or the C ABI for the build over caller-owned memory), with the
default tuning. Every family takes new inputs per pass (vertex positions or
model matrices that lie in device memory) and hands back what the program
reads: the colliding pairs or their triangles, or the tree itself.

  frame      a plain scene: new vertices, every tree refit, then the collision
             query; one frame that is waited for, or (frames > 1) a prescribed
             animation whose frames overlap, read after the last one
  rebuild    the same after a large deformation: every tree built again
  rigid      a plain scene of several rigid meshes that get new matrices
  batch      many scenes of rigid meshes, FP32 filter with the FP64 pass
  precision  scenes of coplanar and edge-touching meshes, FP64 pass
  cloth      a folded sheet against itself
  build      one tree built into caller-owned memory

Entry levels and levels per step are those of the reference's main loop (4, 3)
and of this repository's own measurements (3, 2 for overlapped batches and
cloth, 4, 2 for the coplanar scenes).
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from oibvh_amd import _lib, api
from oibvh_amd import meshgen as M


def listed():
    return [
        # two small bodies in an interactive program, pairs read on the host
        {"name": "frame_ico_1k", "kind": "frame", "shape": "ico", "size": 3, "frames": 1, "fp64": False,
         "entry": 4, "expand": 3, "out": "host"},
        # the demo's size: two bodies of 81,920 triangles, pairs stay on the device
        {"name": "frame_ico_82k", "kind": "frame", "shape": "ico", "size": 6, "frames": 1, "fp64": False,
         "entry": 4, "expand": 3, "out": "pairs"},
        # a detailed deforming pair, 1,000,000 triangles each, frame by frame
        {"name": "frame_uv_1m", "kind": "frame", "shape": "uv", "size": 1000, "frames": 1, "fp64": False,
         "entry": 4, "expand": 3, "out": "pairs"},
        # the same pair played back: the positions of all frames are known
        {"name": "animate_uv_1m", "kind": "frame", "shape": "uv", "size": 1000, "frames": 16, "fp64": False,
         "entry": 4, "expand": 3, "out": "pairs"},
        # trees built again for a new pose, 100,172 triangles each, fine keys
        {"name": "rebuild_uv_100k_63bit", "kind": "rebuild", "shape": "uv", "size": 317, "bits": 63,
         "entry": 4, "expand": 3, "out": "pairs"},
        # a tree for a small body (13,068 triangles) into the caller's memory
        {"name": "build_box_13k", "kind": "build", "shape": "box", "size": 33},
        # the same for a detailed one, 1,000,000 triangles
        {"name": "build_uv_1m", "kind": "build", "shape": "uv", "size": 1000},
        # one scene of 16 rigid bodies, colliding triangles exported for drawing
        {"name": "rigid_16", "kind": "rigid", "meshes": 16, "fp64": False, "entry": 4, "expand": 3,
         "out": "vertices"},
        # simulation of many scenes at once: 128 scenes, about 42M triangles,
        # prescribed motion, four frames
        {"name": "batch_128", "kind": "batch", "scenes": 128, "instanced": False, "frames": 4,
         "entry": 3, "expand": 2},
        # contact tests where FP32 alone does not decide: about 4M triangles
        {"name": "precision_8", "kind": "precision", "scenes": 8, "plane": 354, "box": 144,
         "entry": 4, "expand": 2},
        # a folded cloth against itself, 522,242 triangles
        {"name": "cloth_512", "kind": "cloth", "nv": 512, "frames": 1, "entry": 3, "expand": 2},
        # a fine one, 8,380,418 triangles
        {"name": "cloth_2048", "kind": "cloth", "nv": 2048, "frames": 1, "entry": 3, "expand": 2},
    ]


def _log(rng, lo, hi):
    """a whole number of [lo, hi], even over its logarithm"""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "rebuild", "rigid", "batch", "precision", "cloth", "build", "build"])
    entry, expand = rng.choice([(4, 3), (4, 2), (3, 2)])
    # UV spheres of n x (n // 2 + 1) have about n^2 triangles: 1,000 to 1,000,000
    uv = {"shape": "uv", "size": _log(rng, 33, 1000)}
    if kind == "frame":
        return {"kind": kind, **uv, "frames": rng.choice([1, 1, 16]), "fp64": rng.random() < 0.3,
                "entry": entry, "expand": expand, "out": rng.choice(["host", "pairs", "vertices"])}
    if kind == "rebuild":
        return {"kind": kind, **uv, "bits": rng.choice([30, 63]), "entry": entry, "expand": expand, "out": "pairs"}
    if kind == "rigid":
        return {"kind": kind, "meshes": rng.randint(2, 16), "fp64": rng.random() < 0.5, "entry": entry,
                "expand": expand, "out": rng.choice(["pairs", "vertices"])}
    if kind == "batch":
        return {"kind": kind, "scenes": _log(rng, 4, 128), "instanced": rng.random() < 0.5,
                "frames": rng.choice([1, 4]), "entry": entry, "expand": expand}
    if kind == "precision":
        return {"kind": kind, "scenes": rng.randint(4, 8), "plane": _log(rng, 40, 354), "box": _log(rng, 16, 144),
                "entry": entry, "expand": expand}
    if kind == "cloth":
        return {"kind": kind, "nv": _log(rng, 64, 1448), "frames": rng.choice([1, 4]), "entry": entry,
                "expand": expand}
    if rng.random() < 0.5:
        return {"kind": kind, **uv}
    return {"kind": kind, "shape": "box", "size": _log(rng, 9, 288)}


# ---------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=None)
def _ctx():
    """the context of the program (one per process)"""
    return api.Context(0)


@functools.lru_cache(maxsize=8)
def _shape(shape, size):
    """rest vertices and faces: a unit sphere about the origin or a box"""
    if shape == "ico":
        xyz, faces = M.icosphere_unit(size)
    elif shape == "uv":
        xyz, faces = M.uv_sphere(size, size // 2 + 1)
    else:
        xyz, faces = M.box(size, 0.5)
    return np.asarray(xyz, np.float32), np.asarray(faces, np.uint32)


def _radial(rest, seed, frame, noise, centre):
    """A body whose vertices move along their radius: a travelling wave, or
    with `noise` a fixed uniform roughness and a slow drift."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    d = torch.from_numpy(rest).cuda().double()
    k = (torch.rand(3, generator=g, device="cuda", dtype=torch.float64) * 2 - 1) * 8
    if noise:
        r = 1 + noise * (torch.rand(len(d), generator=g, device="cuda", dtype=torch.float64) * 2 - 1)
        centre = centre + 0.01 * frame
    else:
        omega = 0.05 + 0.2 * torch.rand(1, generator=g, device="cuda", dtype=torch.float64)
        r = 1 + 0.05 * torch.sin(omega * frame + (d * k).sum(1))
    xyz = d * r[:, None]
    xyz[:, 0] += centre
    return xyz.float().contiguous()


def _pair(case, seed, frames):
    """two bodies that interpenetrate: faces, positions[frame][body]"""
    rest, faces = _shape(case["shape"], case["size"])
    noise, apart = (0.02, 1.6) if case["shape"] == "ico" else (0.0, 0.9)
    pos = [[_radial(rest, 2 * seed + m, f, noise, apart * m) for m in range(2)] for f in range(frames)]
    return faces, pos


@functools.lru_cache(maxsize=None)
def _cloth_faces(nv):
    return M._grid_faces(nv, nv).astype(np.uint32)


def _cloth(nv, seed, frame):
    """meshgen.cloth_positions with the sheet's phases drawn from the seed"""
    a, b = M.uniform(seed, 2, 0.0, 2.0 * np.pi)
    t = torch.arange(nv, device="cuda", dtype=torch.float64) / (nv - 1)
    u, v = t[:, None].expand(nv, nv), t[None, :].expand(nv, nv)
    w = 2.0 * np.pi / 0.05
    su = torch.sin(w * u + (a + 0.02 * frame))
    return torch.stack([u + 1.5 / w * su, v, 0.2 * su * torch.sin(w * v + b)], 2).reshape(-1, 3).float().contiguous()


@functools.lru_cache(maxsize=4)
def _rigid(scenes, lo, hi):
    """the scenes' bodies (1k to 200k triangles) and motion"""
    return M.RigidScenes(n_scenes=scenes, meshes=(lo, hi))


def _body(key, seed):
    kind, size = key[:2]
    return M.icosphere(size, 1.0, 0.02, seed) if kind == "ico" else M.box(size, 0.6, 0.02, seed)


def _matrices(rs, seed, frames):
    """column-major matrices of `frames` frames, (frames, meshes, 16), on the device"""
    m = np.stack([rs.transforms(seed % 97 + f) for f in range(frames)])
    return torch.from_numpy(np.ascontiguousarray(m.transpose(0, 1, 3, 2)).reshape(frames, -1, 16)).cuda()


class _Memory:
    """a pair list in the library's device memory as a tensor sees it"""

    def __init__(self, address, n):
        self.__cuda_array_interface__ = {"shape": (n, 4), "typestr": "<i4", "data": (address, False), "version": 2}


@functools.lru_cache(maxsize=None)
def _stream():
    """the library's stream: what the program takes over from the library's
    memory is copied there, before the next frame's work"""
    return torch.cuda.ExternalStream(_ctx().stream)


def _room(case):
    """pairs that the program's own contact list holds"""
    F = max(f for _, f in _sizes(case))
    if case["kind"] in ("frame", "rebuild"):
        return 4096 + 40 * math.isqrt(F)  # two closed curves on each body
    if case["kind"] == "cloth":
        return 65536 + 400 * case["nv"]
    total = sum(f for _, f in _sizes(case))
    return 65536 + (total // 2 if case["kind"] == "precision" else total // 8)


def _scene(trees):
    scene = api.Scene(_ctx())
    for t in trees:
        t.build()
        scene.addOibvhTree(t)
    return scene


def prepare(case, seed):
    ctx, kind = _ctx(), case["kind"]
    s = {"kind": kind, "out": case.get("out", "pairs"), "keep": []}
    if kind != "build":
        s["query"] = (case["entry"], case["expand"])
    s["flags"] = {"fp64_fallback": kind in ("batch", "precision") or case.get("fp64", False),
                  "self_collide": kind == "cloth"}
    frames = case.get("frames", 1)
    if s["out"] == "host":
        s["contacts"] = np.zeros((_room(case), 4), np.uint32)
    elif kind != "build":
        with torch.cuda.stream(_stream()):
            s["contacts"] = (torch.zeros((_room(case), 6, 3), device="cuda") if s["out"] == "vertices" else
                             torch.zeros((_room(case), 4), device="cuda", dtype=torch.int32))
    if kind == "build":
        rest, faces = _shape(case["shape"], case["size"])
        if case["shape"] == "box":
            g = torch.Generator(device="cuda").manual_seed(seed)
            s["xyz"] = torch.from_numpy(rest).cuda()
            s["xyz"] = s["xyz"] + 0.01 * (torch.rand(s["xyz"].shape, generator=g, device="cuda") * 2 - 1)
        else:
            s["xyz"] = _radial(rest, seed, 0, 0.0, 0.0)
        F = len(faces)
        s["faces"] = torch.from_numpy(faces.view(np.int32)).cuda()
        s["nodes"] = torch.empty((_nodes(F), 6), device="cuda")
        s["perm"] = torch.empty(F, device="cuda", dtype=torch.int32)
        s["sorted"] = torch.empty((F, 3), device="cuda", dtype=torch.int32)
    elif kind in ("frame", "rebuild"):
        # the trees are built for the pose before the first frame
        faces, pos = _pair(case, seed, frames + 1)
        torch.cuda.synchronize()
        trees = [api.OibvhTree(ctx, x.cpu().numpy(), faces) for x in pos[0]]
        for t in trees:
            t.set_morton_bits(case.get("bits", 30))
        s["scene"] = _scene(trees)
        s["keep"] = [trees, pos]
        s["positions"] = [api.position_array([x.data_ptr() for x in p]) for p in pos[1:]]
        s["poses"] = [(t, x.data_ptr()) for t, x in zip(trees, pos[1])]
    elif kind == "rigid":
        rs = _rigid(1, case["meshes"], case["meshes"])
        mats = _matrices(rs, seed, 2)
        trees = [api.OibvhTree(ctx, *_body(rs.kinds[lib], 1000 * seed + i)) for i, (_, lib) in enumerate(rs.instances)]
        torch.cuda.synchronize()
        scene = s["scene"] = api.Scene(ctx)
        for t in trees:
            t.build()
            scene.addOibvhTree(t)
        s["keep"] = [trees, mats]
        s["matrices"] = mats[1].data_ptr()
    elif kind == "batch":
        rs = _rigid(case["scenes"], 2, 16)
        mats = _matrices(rs, seed, frames + 1)
        b = s["batch"] = api.Batch(ctx)
        first = {}
        for i, (scene, lib) in enumerate(rs.instances):
            if case["instanced"] and lib in first:
                b.add_instance(scene, first[lib])
            else:
                first[lib] = b.add_mesh(scene, *_body(rs.kinds[lib], 100000 * seed + i))
        torch.cuda.synchronize()
        b.set_transforms_device(mats[0].data_ptr())
        b.build()
        s["keep"] = [mats]
        s["matrices"] = [mats[f].data_ptr() for f in range(1, frames + 1)]
    elif kind == "precision":
        b = s["batch"] = api.Batch(ctx)
        for i, pair in enumerate(M.precision_scenes(case["scenes"], M.CFG4_SEED + seed, case["plane"], case["box"])):
            for xyz, faces in pair:
                b.add_mesh(i, xyz, faces)
        b.build()
    else:
        pos = [_cloth(case["nv"], seed, f) for f in range(frames + 1)]
        torch.cuda.synchronize()
        trees = [api.OibvhTree(ctx, pos[0].cpu().numpy(), _cloth_faces(case["nv"]))]
        s["scene"] = _scene(trees)
        s["keep"] = [trees, pos]
        s["positions"] = [api.position_array([x.data_ptr()]) for x in pos[1:]]
    ctx.synchronize()
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------- a pass
def _result(obj, state):
    """The query's pairs into the program's own list (the library's is valid
    until the next query): from host memory, on the device, or as triangles."""
    contacts = state["contacts"]
    if state["out"] == "vertices":
        n = obj.getIntTriPairCount()
        obj.pair_vertices_device(contacts.data_ptr(), contacts.numel())
        return {"count": n, "contacts": contacts}
    if state["out"] == "host":
        pairs = obj.getIntTriPairs()
        n = len(pairs)
        contacts[:n] = pairs
    else:
        address, n = obj.pairs_device()
        if n:
            with torch.cuda.stream(_stream()):
                contacts[:n].copy_(torch.as_tensor(_Memory(address, n), device="cuda"))
    return {"count": n, "contacts": contacts}


def run(state):
    kind = state["kind"]
    if kind == "build":
        ctx, xyz, faces = _ctx(), state["xyz"], state["faces"]
        status = ctx._lib.oibvh_build_noalloc(ctx.h, xyz.data_ptr(), len(xyz), faces.data_ptr(), len(faces),
                                              state["nodes"].data_ptr(), state["perm"].data_ptr(),
                                              state["sorted"].data_ptr())
        if status != _lib.OK:
            raise _lib.OibvhError(status, "oibvh_build_noalloc")
        return {"nodes": state["nodes"], "perm": state["perm"], "sorted": state["sorted"]}
    entry, expand = state["query"]
    flags = state["flags"]
    if kind in ("batch", "precision"):
        b = state["batch"]
        frames = state.get("matrices", [None])
        overlap = len(frames) > 1
        for m in frames:
            if m is not None:
                b.set_transforms_device(m)
            b.frame(entry, expand, asynchronous=overlap, overlap=overlap, **flags)
        return _result(b, state)
    scene = state["scene"]
    if kind == "rebuild":
        for tree, address in state["poses"]:
            tree.set_positions_device(address)
        scene.build()
        scene.detectCollision(entry, expand, **flags)
    elif kind == "rigid":
        scene.set_transforms(device=state["matrices"], borrow=True)
        scene.frame(None, entry, expand, **flags)
    else:
        overlap = len(state["positions"]) > 1
        for p in state["positions"]:
            scene.frame(p, entry, expand, asynchronous=overlap, overlap=overlap, **flags)
    return _result(scene, state)


# ---------------------------------------------------------------- what a pass needs
def _nodes(F):
    """nodes of a tree of F leaves"""
    return 2 * F + bin((1 << (F - 1).bit_length()) - F).count("1") - 1


def _sizes(case):
    """(vertices, faces) of every tree of the case"""
    kind = case["kind"]
    if kind in ("frame", "rebuild", "build"):
        rest, faces = _shape(case["shape"], case["size"])
        return [(len(rest), len(faces))] * (1 if kind == "build" else 2)
    if kind in ("rigid", "batch"):
        rs = _rigid(1, case["meshes"], case["meshes"]) if kind == "rigid" else _rigid(case["scenes"], 2, 16)
        return [(len(rs.library[lib][0]), len(rs.library[lib][1])) for _, lib in rs.instances]
    if kind == "precision":
        p, b = case["plane"], case["box"]
        plane, box = ((p + 1) ** 2, 2 * p * p), (6 * (b + 1) ** 2, 12 * b * b)
        return [plane if s % 4 < 2 else box for s in range(case["scenes"]) for _ in range(2)]
    return [(case["nv"] ** 2, 2 * (case["nv"] - 1) ** 2)]


def work(case):
    """Per tree and frame: positions and faces read, nodes written; a build
    also writes the permutation and the sorted faces. (The pairs found, 16
    bytes each, are few beside it.) Operations: a leaf box and a merge of two
    boxes per node, 6 each."""
    build = 16 if case["kind"] in ("rebuild", "build") else 0
    frames = case.get("frames", 1)
    trees = _sizes(case)
    return {"bytes": frames * sum(12 * V + (12 + build) * F + 24 * _nodes(F) for V, F in trees),
            "flops": frames * sum(12 * F + 6 * _nodes(F) for _, F in trees)}


def exact(case, seed):
    """The built tree's boxes: minima and maxima of the vertices under each
    node, leaves in the order of their 30-bit Morton keys (which are whole
    numbers that the format defines through 32-bit arithmetic). Pairs are
    whole numbers; exported vertices are the inputs, transformed."""
    if case["kind"] != "build":
        return None
    s = prepare(case, seed)
    xyz, faces = s["xyz"].cpu().numpy(), s["faces"].cpu().numpy()
    tri = xyz[faces]
    lo, hi = tri.min(1), tri.max(1)
    b0, b1 = xyz.min(0), xyz.max(0)
    q = ((lo + hi) * np.float32(0.5) - b0) / (b1 - b0) * np.float32(1024)
    q = np.minimum(np.maximum(q, 0), 1023).astype(np.uint32)
    key = np.zeros(len(faces), np.uint32)
    for bit in range(10):
        for axis in range(3):
            key |= ((q[:, axis] >> bit) & 1) << (3 * bit + 2 - axis)
    order = np.argsort(key, kind="stable")
    lo, hi = lo[order].astype(np.float64), hi[order].astype(np.float64)
    levels = [np.concatenate([lo, hi], 1)]
    while len(lo) > 1:
        if len(lo) % 2:
            lo, hi = np.concatenate([lo, lo[-1:]]), np.concatenate([hi, hi[-1:]])
        lo, hi = np.minimum(lo[0::2], lo[1::2]), np.maximum(hi[0::2], hi[1::2])
        levels.append(np.concatenate([lo, hi], 1))
    return {"nodes": np.concatenate(levels[::-1]), "perm": None, "sorted": None}
