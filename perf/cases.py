"""The work whose time this repository keeps track of.

Each case is one call (or the few calls that belong together) that a program
using isosurface_amd makes over and over: extracting a mesh from a resident
sample grid, from an implicit program, by dual contouring, by the extended and
the octree extractors, for a batch of chunks and inside the narrow band, and
training the band's network.  listed() names the sizes that the benchmark and
the tests use; draw() gives others of the same ranges.

A case's inputs come from its seed alone.  Meshes are the library's promise
bit for bit (vertex order, f32 positions, index lists), so their tolerance is
"exact"; the network's weights are compared in the 2-norm.
"""
from __future__ import annotations

import ctypes as C
import math
import random

import numpy as np
import torch

from isosurface_amd import _abi as A
from isosurface_amd import workloads as W
from isosurface_amd.band import NarrowBand
from isosurface_amd.engine import Context, chunk_desc
from isosurface_amd.sources import (DemoSource, Difference, RectangularPrism, Sphere, Torus,
                                    Translate, smooth_union_all, union_all)

# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # The smallest whole call: MarchingCubes(65) on one sphere into host
        # arrays (what a first program does, and an editor's preview at every
        # change).  Latency, launches and copies.
        {"name": "host_sphere_65", "kind": "host", "size": 65, "spheres": 1},
        # A small chunk already sampled on the GPU: launch-bound.
        {"name": "grid_33", "kind": "grid", "nx": 33, "ny": 33, "nz": 34},
        # The benchmark's headline: MarchingCubes::new(257) over a resident grid.
        {"name": "grid_257", "kind": "grid", "nx": 257, "ny": 257, "nz": 258},
        # A grid above the 256 MB last-level cache.
        {"name": "grid_513", "kind": "grid", "nx": 513, "ny": 513, "nz": 514},
        # The crate's own criterion bench (MarchingCubes::new(128) on a torus)
        # with the normal sink's second pass over the vertices.
        {"name": "torus_128_normals", "kind": "program", "size": 128, "spheres": 0,
         "normals": True},
        # The benchmark's CSG workload sampled on the GPU instead of a grid.
        {"name": "csg_257", "kind": "program", "size": 257, "spheres": 64, "normals": False},
        # Sharp features: dual contouring over central differences, f64 QEF.
        {"name": "dual_128", "kind": "dual", "size": 128, "boxes": 32, "epsilon": 1e-6},
        # Extended marching cubes (directed distances, features, edge flips).
        {"name": "extended_128", "kind": "extended", "size": 128, "boxes": 32, "epsilon": 0.0},
        # Adaptive extraction: the octree of the same boxes.
        {"name": "octree_7", "kind": "octree", "depth": 7, "boxes": 32},
        # A paged terrain's chunks: 16^3 to 64^3 cells, 1 to 8 primitives each.
        {"name": "batch_4096", "kind": "batch", "chunks": 4096},
        # The largest extraction: 1024^3 cells of 1024 smoothly joined spheres
        # through the certified narrow band.
        {"name": "band_1025", "kind": "band", "size": 1025, "spheres": 1024, "brick8": False},
        # Fitting the band's network: forward, backward and Adam.
        {"name": "train_16384", "kind": "train", "samples": 262144, "batch": 16384, "steps": 200},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["host", "grid", "grid", "program", "program", "dual", "extended", "octree",
                       "batch", "band", "train"])
    if kind == "host":
        return {"kind": kind, "size": _log_int(rng, 17, 129), "spheres": _log_int(rng, 1, 16)}
    if kind == "grid":
        return {"kind": kind, "nx": _log_int(rng, 9, 513), "ny": _log_int(rng, 9, 513),
                "nz": _log_int(rng, 9, 513)}
    if kind == "program":
        return {"kind": kind, "size": _log_int(rng, 33, 257),
                "spheres": rng.choice([0, _log_int(rng, 1, 64)]), "normals": rng.random() < 0.5}
    if kind in ("dual", "extended"):
        return {"kind": kind, "size": _log_int(rng, 17, 128), "boxes": _log_int(rng, 1, 32),
                "epsilon": rng.choice([0.0, 1e-6])}
    if kind == "octree":
        return {"kind": kind, "depth": rng.randint(3, 7), "boxes": _log_int(rng, 1, 32)}
    if kind == "batch":
        return {"kind": kind, "chunks": _log_int(rng, 16, 4096)}
    if kind == "band":
        return {"kind": kind, "size": _log_int(rng, 129, 1025), "spheres": _log_int(rng, 16, 1024),
                "brick8": rng.random() < 0.5}
    return {"kind": kind, "samples": _log_int(rng, 16384, 262144),
            "batch": 16 * _log_int(rng, 64, 1024), "steps": _log_int(rng, 20, 200)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _spheres(seed: int, n: int):
    """n seeded spheres: centres U[-0.4, 0.4]^3, radii U[0.03, 0.12]."""
    r = W.SplitMix64(seed)
    return [((r.uniform(-0.4, 0.4), r.uniform(-0.4, 0.4), r.uniform(-0.4, 0.4)),
             r.uniform(0.03, 0.12)) for _ in range(n)]


def _torus(seed: int):
    r = W.SplitMix64(seed ^ 0x70)
    return r.uniform(0.24, 0.31), r.uniform(0.05, 0.1)


def _csg(seed: int, n: int):
    """The union of n spheres minus a torus; without spheres the torus alone."""
    major, minor = _torus(seed)
    if n == 0:
        return DemoSource(Torus(major, minor))
    u = union_all(Translate(c, Sphere(r)) for c, r in _spheres(seed, n))
    return DemoSource(Difference(Torus(major, minor), u))


def _ball(seed: int, n: int):
    """One large sphere near the domain's centre and n - 1 smaller ones."""
    r = W.SplitMix64(seed ^ 0xba11)
    c = tuple(r.uniform(-0.05, 0.05) for _ in range(3))
    parts = [Translate(c, Sphere(r.uniform(0.3, 0.4)))]
    parts += [Translate(c, Sphere(rad)) for c, rad in _spheres(seed, n - 1)]
    return DemoSource(union_all(parts))


def _boxes(seed: int, n: int):
    r = W.SplitMix64(seed)
    parts = []
    for _ in range(n):
        c = tuple(r.uniform(-0.3, 0.3) for _ in range(3))
        h = tuple(r.uniform(0.05, 0.2) for _ in range(3))
        parts.append(Translate(c, RectangularPrism(h)))
    return DemoSource(union_all(parts))


def _blend(seed: int, n: int):
    """n spheres joined by a smooth minimum (k = 0.02); fewer ones are larger,
    so the surface keeps its extent."""
    r = W.SplitMix64(seed)
    scale = min((1024.0 / n) ** (1.0 / 3.0), 4.0)
    parts = []
    for _ in range(n):
        c = tuple(r.uniform(-0.45, 0.45) for _ in range(3))
        parts.append(Translate(c, Sphere(scale * r.uniform(0.01, 0.05))))
    return DemoSource(smooth_union_all(parts, 0.02))


def _axes(case):
    """The grid's f32 coordinates per axis (x, y, z): sample i at i / (m - 1), m
    the longest side of the cross-section, as MarchingCubes::new places them."""
    step = np.float32(1.0) / np.float32(max(case["nx"], case["ny"]) - 1)
    return [torch.arange(case[k], dtype=torch.float32, device="cuda") * float(step)
            for k in ("nx", "ny", "nz")], step


def _field(case, seed):
    """The grid's samples: 64 spheres minus a torus, in plain torch f32."""
    (x, y, z), _ = _axes(case)
    x, y, z = (x - 0.5)[None, None, :], (y - 0.5)[None, :, None], (z - 0.5)[:, None, None]
    v = torch.full((case["nz"], case["ny"], case["nx"]), 10.0, dtype=torch.float32, device="cuda")
    for c, r in _spheres(seed, 64):
        flat = (x - c[0]) ** 2 + (y - c[1]) ** 2
        torch.minimum(v, (flat + (z - c[2]) ** 2).sqrt_().sub_(r), out=v)
    major, minor = _torus(seed)
    ring = ((x * x + y * y).sqrt() - major) ** 2
    torch.maximum(v, (ring + z * z).sqrt_().sub_(minor).neg_(), out=v)
    return v


def _buffers(case):
    """The caller's mesh buffers: room for any mesh of the case's kind and size,
    zeros where no mesh reaches."""
    n = int(2 * _vertices(case)) + 4096
    if case["kind"] == "host":
        return np.zeros((n, 3), np.float32), np.zeros(6 * n, np.int32)
    return (torch.zeros((n, 3), dtype=torch.float32, device="cuda"),
            torch.zeros(6 * n, dtype=torch.int32, device="cuda"))


def prepare(case, seed):
    ctx = Context(0)
    state = {"case": case, "ctx": ctx}
    kind, lib, h = case["kind"], ctx.lib, ctx.handle
    if kind != "train":
        state["vertices"], state["indices"] = _buffers(case)
    if kind == "host":
        ctx.upload_program(_ball(seed, case["spheres"]).program())
        d = ctx.reference_desc(case["size"], A.ISO_SOURCE_PROGRAM)
        state["call"] = lambda out: lib.iso_extract_mc(h, C.byref(d), C.byref(out))
    elif kind == "grid":
        state["grid"] = _field(case, seed)
        _, step = _axes(case)
        d = A.IsoGridDesc()
        d.nx, d.ny, d.nz = case["nx"], case["ny"], case["nz"]
        for i in range(3):
            d.origin[i], d.spacing[i] = 0.0, float(step)
        d.source = A.ISO_SOURCE_GRID
        ctx.check(lib.iso_grid_bind_device(h, state["grid"].data_ptr(), d.nx, d.ny, d.nz), "bind")
        state["call"] = lambda out: lib.iso_extract_mc(h, C.byref(d), C.byref(out))
    elif kind == "program":
        ctx.upload_program(_csg(seed, case["spheres"]).program())
        d = ctx.reference_desc(case["size"], A.ISO_SOURCE_PROGRAM)
        state["call"] = lambda out: lib.iso_extract_mc(h, C.byref(d), C.byref(out))
        if case["normals"]:
            state["normals"] = torch.zeros_like(state["vertices"])
    elif kind in ("dual", "extended"):
        ctx.upload_program(_boxes(seed, case["boxes"]).program())
        d = ctx.reference_desc(case["size"], A.ISO_SOURCE_PROGRAM)
        fn, eps = (lib.iso_extract_dc if kind == "dual" else lib.iso_extract_emc), case["epsilon"]
        state["call"] = lambda out: fn(h, C.byref(d), C.c_float(eps), C.byref(out))
    elif kind == "octree":
        ctx.upload_program(_boxes(seed, case["boxes"]).program())
        depth = case["depth"]
        state["call"] = lambda out: lib.iso_extract_lhmc(h, depth, C.byref(out))
    elif kind == "batch":
        n = case["chunks"]
        ctx.upload_batch([(src, chunk_desc(size)) for src, size in W.batch_chunks(n, seed)])
        voff, ioff = np.zeros(n + 1, np.uint64), np.zeros(n + 1, np.uint64)
        state["offsets"] = (voff, ioff)

        def call(out):
            b = A.IsoBatchOut(out.vertices, out.indices, out.vertex_capacity, out.index_capacity,
                              voff.ctypes.data, ioff.ctypes.data, 0, 0, A.ISO_MEMORY_DEVICE,
                              A.ISO_BATCH_GRAPH)
            st = lib.iso_extract_batch(h, C.byref(b))
            out.vertex_count, out.index_count = b.vertex_count, b.index_count
            return st

        state["call"] = call
    elif kind == "band":
        src = _blend(seed, case["spheres"])
        band = NarrowBand(ctx)
        band.init(seed & 0xffff)
        pts = np.random.default_rng(seed).random((32768, 3), dtype=np.float32)
        band.train(pts, ctx.sample(src, pts), steps=200, batch=4096, overshoot=8.0, lr=2e-3)
        ctx.upload_program(src.program())
        d = ctx.reference_desc(case["size"], A.ISO_SOURCE_PROGRAM)
        flags = A.ISO_BAND_CERTIFY | (A.ISO_BAND_BRICK8 if case["brick8"] else 0)
        state["call"] = lambda out: lib.iso_extract_mc_band(h, C.byref(d), C.c_float(0.008), flags,
                                                            C.byref(out), None)
    elif kind == "train":
        src = _blend(seed, 256)
        band = NarrowBand(ctx)
        band.init(seed & 0xffff)
        pts = np.random.default_rng(seed).random((case["samples"], 3), dtype=np.float32)
        state["points"] = torch.from_numpy(pts).cuda()
        state["sdf"] = torch.from_numpy(ctx.sample(src, pts)).cuda()
        state["start"] = band.get_params()
        state["seed"] = seed & 0xffff
    else:
        raise ValueError(kind)
    torch.cuda.synchronize()  # the library's own stream reads what torch has written
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "train":
        band = NarrowBand(ctx)
        band.set_params(state["start"])
        prm = A.IsoBandTrainParams(case["steps"], case["batch"], 2e-3, 1e-4, 0.05, state["seed"],
                                   8.0)
        loss = C.c_float(0.0)
        ctx.check(ctx.lib.iso_band_train(ctx.handle, state["points"].data_ptr(),
                                         state["sdf"].data_ptr(), None, case["samples"],
                                         A.ISO_MEMORY_DEVICE, C.byref(prm), C.byref(loss)),
                  "iso_band_train")
        return {"parameters": band.get_params(), "loss": float(loss.value)}
    v, i = state["vertices"], state["indices"]
    if kind == "host":
        out = A.IsoMeshOut(v.ctypes.data, i.ctypes.data, v.shape[0], i.shape[0], 0, 0,
                           A.ISO_MEMORY_HOST, 0)
    else:
        out = A.IsoMeshOut(v.data_ptr(), i.data_ptr(), v.shape[0], i.shape[0], 0, 0,
                           A.ISO_MEMORY_DEVICE, 0)
    ctx.check(state["call"](out), kind)
    nv = int(out.vertex_count)
    res = {"vertices": v, "indices": i, "vertex_count": nv, "index_count": int(out.index_count)}
    if kind == "program" and case["normals"]:
        ctx.check(ctx.lib.iso_sample_normals(ctx.handle, v.data_ptr(), nv, C.c_float(1e-4),
                                             state["normals"].data_ptr(), A.ISO_MEMORY_DEVICE),
                  "iso_sample_normals")
        res["normals"] = state["normals"]
    if kind == "batch":
        res["vertex_offsets"], res["index_offsets"] = (o.view(np.int64) for o in state["offsets"])
    return res


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
# Vertices per squared lattice side, fitted to seeds of each kind over the
# ranges of draw(); a mesh has two triangles for each vertex, so its vertices
# and indices take 36 bytes a vertex.
def _vertices(case):
    kind = case["kind"]
    if kind == "host":
        return (2.3 + 0.05 * (case["spheres"] - 1)) * (case["size"] - 1) ** 2
    if kind == "grid":
        m = max(case["nx"], case["ny"]) - 1
        return 6.0 * m * m * min(1.0, case["nx"] * case["ny"] * case["nz"] / float(m + 1) ** 3)
    if kind == "program":
        per = 1.2 if case["spheres"] == 0 else 0.15 + 0.092 * case["spheres"]
        return per * (case["size"] - 1) ** 2
    if kind in ("dual", "extended"):
        return 4.4 * (case["boxes"] / 32.0) ** 0.5 * (case["size"] - 1) ** 2
    if kind == "octree":
        return 4.4 * (case["boxes"] / 32.0) ** 0.5 * 4.0 ** case["depth"]
    if kind == "batch":
        return 2500.0 * case["chunks"]
    return 15.0 * (case["spheres"] / 1024.0) ** 0.34 * (case["size"] - 1) ** 2  # band


def work(case):
    kind = case["kind"]
    if kind == "train":
        # 15,552 weights, a product each way (forward, inputs' and weights' gradients);
        # the samples drawn for the batches, and the weights in and out.
        drawn = case["batch"] * case["steps"]
        return {"bytes": 16.0 * min(drawn, case["samples"]) + 2 * 4 * 15617,
                "flops": 6.0 * 15552 * drawn}
    v = _vertices(case)
    bytes_, flops = 36.0 * v, 0.0
    if kind == "grid":
        bytes_ += 4.0 * case["nx"] * case["ny"] * case["nz"]
        flops = 12.0 * v
    else:
        # Each vertex lies between two samples of the program: at least one
        # primitive (about 10 operations) for either, and the crossing itself.
        flops = 32.0 * v
        prims = {"host": case.get("spheres"), "program": case.get("spheres", 0) + 1,
                 "dual": case.get("boxes"), "extended": case.get("boxes"),
                 "octree": case.get("boxes"), "batch": 4.5 * case.get("chunks", 0),
                 "band": case.get("spheres")}[kind]
        bytes_ += 32.0 * prims
        if kind == "dual":
            flops += v * (8 * 6 * 10 + 2000)  # eight corner normals, one 8x3 f64 SVD
        if kind == "extended":
            flops += v * 500
        if kind == "program" and case["normals"]:
            bytes_ += 24.0 * v
            flops += 60.0 * v
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    if case["kind"] == "train":
        # bf16 products and float atomics: the same call twice, and the same
        # products summed in another order, move the weights by this share.
        return {"rel": 4e-3, "max": 0.05}
    return "exact"


# ---------------------------------------------------------------------------
# The grid cases in 64 bits
# ---------------------------------------------------------------------------
_CORNER = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
_EDGE = [(0, 1), (1, 2), (2, 3), (3, 0), (4, 5), (5, 6), (6, 7), (7, 4), (0, 4), (1, 5), (2, 6),
         (3, 7)]
# The public Lorensen/Bourke triangulation: each case's edges, as hex digits.
_TRIANGLES = """
,083,019,183981,12a,08312a,92a029,2832a8a98,3b2,0b28b0,19023b,1b219b98b,3a1ba3,0a108a8ba,3903b9b
a9,98aa8b,478,430734,019847,419471731,12a847,34730412a,92a902847,2a9297273794,8473b2,b47b24204,9
0184723b,47b94b9b2921,3a13ba784,1ba14b1047b4,47890b9bab03,47b4b99ba,954,954083,054150,854835315,
12a954,30812a495,52a542402,2a5325354348,95423b,0b208b495,05401523b,21525828b485,a3ba13954,495081
8a18ba,54050b5bab03,54858aa8b,978579,930953573,078017157,153357,978957a12,a12950530573,802825857
a52,2a5253357,7957893b2,95797292027b,23b018178157,b21b17715,958857a13a3b,5705097b010aba0,ba0b03a
50807570,ba57b5,a65,0835a6,9015a6,1831985a6,165261,165126308,965906026,598582526328,23ba65,b08b2
0a65,01923b5a6,5a61929b298b,63b653513,08b0b50515b6,3b6036065059,65969bb98,5a6478,43047365a,1905a
6847,a65197173794,612651478,125526304347,847905065026,739794329596269,3b2784a65,5a647242027b,019
47823b5a6,9219b294b7b45a6,8473b53515b6,51b5b610b7b404b,059065036b63847,65969b4797b9,a4964a,4a649
a083,a01a60640,83181686461a,149124264,308129249264,024426,832824426,a49a64b23,08228b49a4a6,3b201
606461a,64161a48121b8b1,964936913b63,8b1810b61914641,3b6360064,648b68,7a678a89a,0730a709a67a,a67
1a7178180,a67a71173,126168189867,269291679093739,780706602,732672,23ba68a89867,20727b09767a9a7,1
801781a767a23b,b21b17a61671,896867916b63136,091b67,7807063b0b60,7b6,76b,308b76,019b76,819831b76,
a126b7,12a3086b7,2902a96b7,6b72a3a83a98,723627,708760620,276237019,162186198876,a76a17137,a7617a
187108,03707a0a96a7,76a7a88a9,684b86,36b306046,86b846901,946963931b36,6846b82a1,12a30b06b046,4b8
46b0292a9,a93a32943b36463,823842462,042462,190234246438,194142246,8138618466a1,a10a06604,4634386
a3039a93,a946a4,49576b,083495b76,50154076b,b76834354315,954a1276b,6b712a083495,76b54a42a402,3483
54325a52b76,723762549,954086062687,362376150540,628687218485158,954a16176137,16a176107870954,40a
4a503a6a737a,76a7a854a48a,6956b9b89,36b063056095,0b805b01556b,6b3635531,12a95b9b8b56,0b306b09656
912a,b85b56805a52025,6b36352a3a53,589528562382,956960062,158180568382628,156216,13616a386569896,
a10a06950560,03856a,a56,b5a75b,b5ab75830,5b75ab190,a75ab7981831,b12b71751,08312717572b,975927902
2b7,75272b592328982,25a235375,820852875a25,9015a35373a2,982921872a25752,135375,087071175,9039355
37,987597,5845a8ab8,5045b05abb30,01984a8aba45,ab4a45b34941314,2512852b8458,04b0b345b2b151b,02505
92b5458b85,9452b3,25a352345384,5a2524420,3a235a385458019,5a2524192942,845853351,045105,845853905
035,945,4b749b9ab,0834979b79ab,1ab1b414074b,3143481a474bab4,4b79b492b912,9749b791b2b1083,b74b422
40,b74b42834324,29a279237749,9a7974a27870207,37a3a274a1a040a,1a2874,491417713,491417081871,40374
3,487,9a8ab8,30939bb9a,01a0a88ab,31ab3a,12b1b99b8,30939b1292b9,02b80b,32b,23828aa89,9a2092,23828
a0181a8,1a2,138918,091,038,
""".replace("\n", "").split(",")


def exact(case, seed):
    """Marching cubes over the grid in float64: the crossings of every lattice
    edge, numbered by the lowest cell that holds the edge and, within a cell, by
    first use in its triangles.  Other cases have no value apart from the f32
    samples that decide their topology, and a network trained on batches that
    the library draws has none either."""
    if case["kind"] != "grid":
        return None
    v = _field(case, seed)
    inside = ~(v > 0)
    _, step = _axes(case)
    first = torch.full((256, 12), 99, dtype=torch.int64)
    for c, edges in enumerate(_TRIANGLES):
        for k, e in enumerate(edges):
            first[c, int(e, 16)] = min(int(first[c, int(e, 16)]), k)
    first = first.cuda()
    n = (case["nx"], case["ny"], case["nz"])

    def corner(k):
        x, y, z = _CORNER[k]
        return (slice(z, n[2] - 1 + z), slice(y, n[1] - 1 + y), slice(x, n[0] - 1 + x))

    keys, points = [], []
    for e, (a, b) in enumerate(_EDGE):
        low = [min(_CORNER[a][d], _CORNER[b][d]) for d in range(3)]
        axis = [d for d in range(3) if _CORNER[a][d] != _CORNER[b][d]][0]
        crossed = inside[corner(a)] != inside[corner(b)]
        # A cell owns an edge on one of its low faces only where no cell lies beyond.
        keep = [slice(0, 1) if d != axis and low[d] == 0 else slice(None) for d in range(3)]
        cell = crossed[keep[2], keep[1], keep[0]].nonzero()
        if not len(cell):
            continue
        z, y, x = cell.unbind(1)
        case_of = torch.zeros_like(x)
        for k, (dx, dy, dz) in enumerate(_CORNER):
            case_of |= inside[z + dz, y + dy, x + dx].long() << k
        keys.append(((z * (n[1] - 1) + y) * (n[0] - 1) + x) * 16 + first[case_of, e])
        ends = []
        for k in (a, b):
            dx, dy, dz = _CORNER[k]
            ends.append((v[z + dz, y + dy, x + dx].double(),
                         torch.stack([x + dx, y + dy, z + dz], 1).double() * float(step)))
        (va, pa), (vb, pb) = ends
        points.append(pa + (va / (va - vb))[:, None] * (pb - pa))
    res = torch.zeros((_buffers(case)[0].shape[0], 3), dtype=torch.float64, device="cuda")
    if keys:
        mesh = torch.cat(points)[torch.cat(keys).argsort()]
        res[:len(mesh)] = mesh
    return {"vertices": res, "indices": None, "vertex_count": None, "index_count": None}
