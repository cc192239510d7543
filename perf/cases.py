"""What a user of the sparse-voxel-octree builder has it do, as cases that can be timed.

A case is a dict of plain values.  "path" names the entry point it goes through:

  build   one mesh resident on the device -> its octree, left on the device
          (svo_build_device)
  host    one mesh in host memory -> its 168-byte node records in host memory
          (svo_build and svo_tree_copy_nodes): what the reference's class and
          command line do with a mesh
  batch   many device meshes in one call (svo_build_batch)
  plan    the same recorded once and replayed as one HIP graph (svo_plan_run)
  query   neighbor lookups on a resident tree from host arrays
          (svo_query_neighbors)
  sort    Morton keys sorted in place on the caller's stream
          (svo_k_radix_sort_noalloc)

Meshes: icospheres with three octaves of value noise, turned tori and triangle
soups ("mesh" numbers the surface, the seed how a file lists it); grids from 32
to 4096 cells an axis, cubic or not; reference and intended semantics; 32-bit
and 64-bit keys; with vertex, edge and face records or the nodes alone.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gpu-svo_amd"))
import svo_amd  # noqa: E402
from svo_amd import meshgen  # noqa: E402

# Device bytes of the one context: what torch and the caller's other data do
# not need of a 288 GB card.
CONTEXT_BYTES = 192 << 30


def _build(name, shape, mesh, res, **more):
    case = {"path": "build", "name": name, "shape": shape, "mesh": mesh, "rx": res[0],
            "ry": res[1], "rz": res[2], "intended": False, "key_bits": 0, "records": True}
    return dict(case, **more)


def listed():
    return [
        # a lookup of a few neighbors between two steps of a program that walks
        # the tree: the smallest call there is
        {"name": "query_1000", "path": "query", "n": 1000, "mesh": 1, "subdiv": 4, "res": 64},
        # one small mesh in an interactive program (the size of the reference's
        # sample at its default resolution): launches and round trips count
        _build("ico4_64", "ico", 2, (64, 64, 64), subdiv=4),
        # the reference's class: host mesh in, node records out, a grid that is
        # no power of two and not cubic
        _build("host_torus_odd", "torus", 3, (101, 77, 90), a=75, b=34, path="host"),
        # neighbors and shared records for a simulation on the octree
        _build("intended_torus_odd", "torus", 4, (150, 150, 67), a=160, b=64, intended=True),
        _build("intended_ico6_512", "ico", 5, (512, 512, 512), subdiv=6, intended=True),
        # a scanned object at the resolution it is scanned at
        _build("ico7_512", "ico", 6, (512, 512, 512), subdiv=7),
        # unstructured geometry that fills its box, largest 32-bit grid
        _build("soup_1024", "soup", 7, (1024, 1024, 1024), tris=100000, edge=256),
        # beyond 32-bit codes, nodes alone
        _build("soup_2048_nodes", "soup", 8, (2048, 2048, 2048), tris=100000, edge=256,
               key_bits=64, records=False),
        # small features in a huge grid: too sparse for the occupancy bitmap
        _build("sparse_4096_nodes", "soup", 9, (4096, 4096, 4096), tris=150000, edge=1024,
               key_bits=64, records=False),
        # a data set of mixed meshes converted in one call, and the same meshes
        # again and again as one graph
        {"name": "batch_64", "path": "batch", "mesh": 3, "n": 64, "top": 256, "intended": False,
         "records": True},
        {"name": "plan_48", "path": "plan", "mesh": 3, "n": 48, "top": 128, "intended": False,
         "records": True},
        # keys of another program, between its own kernels
        {"name": "sort_1m", "path": "sort", "n": 1000003, "key_bytes": 4, "bits": 30},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    path = rng.choice(["build", "build", "build", "build", "soup", "soup", "host", "batch", "plan",
                       "query", "sort"])
    mesh = rng.randrange(1 << 20)
    if path == "query":
        return {"path": "query", "mesh": mesh, "n": log_int(1, 200000),
                "subdiv": rng.randint(2, 5), "res": log_int(32, 256)}
    if path == "sort":
        key_bytes = rng.choice([4, 8])
        return {"path": "sort", "n": log_int(1000, 1 << 22), "key_bytes": key_bytes,
                "bits": rng.randint(12, 8 * key_bytes)}
    if path in ("batch", "plan"):
        return {"path": path, "mesh": mesh, "n": rng.randint(8, 64 if path == "batch" else 48),
                "top": rng.choice([64, 128, 256] if path == "batch" else [64, 128]),
                "intended": rng.random() < 0.3, "records": rng.random() < 0.8}
    if path == "soup":
        if rng.random() < 0.3:
            return {"path": "build", "shape": "soup", "mesh": mesh, "tris": log_int(2000, 150000),
                    "edge": 1024, "rx": log_int(2100, 4096), "ry": log_int(2100, 4096),
                    "rz": log_int(2100, 4096), "intended": False, "key_bits": 64, "records": False}
        tris = log_int(2000, 100000)
        return {"path": "build", "shape": "soup", "mesh": mesh, "tris": tris, "edge": 256,
                "rx": log_int(64, 1024), "ry": log_int(64, 1024), "rz": log_int(64, 1024),
                "intended": tris < 20000 and rng.random() < 0.4,
                "key_bits": rng.choice([0, 0, 64]), "records": rng.random() < 0.7}
    top = 512 if path == "build" else 160
    r = log_int(32, top)
    case = {"path": path, "mesh": mesh, "rx": r, "ry": r, "rz": r}
    if rng.random() < 0.5:  # not cubic
        case["ry"] = max(16, int(r * rng.uniform(0.4, 1.0)))
        case["rz"] = max(16, int(r * rng.uniform(0.4, 1.0)))
    if rng.random() < 0.5:
        case.update(shape="ico", subdiv=rng.randint(2, 6))
    else:
        case.update(shape="torus", a=log_int(16, 256), b=log_int(16, 160))
    case.update(intended=rng.random() < 0.4,
                key_bits=rng.choice([0, 0, 64]) if path == "build" else 0)
    if path == "build":
        case["records"] = rng.random() < 0.8
    return case


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=None)
def _sphere(subdiv):
    return meshgen.icosphere(subdiv)


@functools.lru_cache(maxsize=1)
def _context():
    """The program's one context, with the tuning that the package holds for this card."""
    ctx = svo_amd.Context(0, CONTEXT_BYTES)
    ctx.load_tuning(os.path.join(svo_amd.PKG_ROOT, "tuning", "mi355x.tuning"))
    return ctx


@functools.lru_cache(maxsize=1)
def _stream():
    """The stream that the program sorts its keys on (the sorts share one scratch)."""
    return torch.cuda.Stream()


def _turned(p, rng):
    q, r = np.linalg.qr(rng.standard_normal((3, 3)))
    return (p.astype(np.float64) @ (q * np.sign(np.diag(r))).T).astype(np.float32)


@functools.lru_cache(maxsize=8)
def _shape(shape, number, *sizes):
    """(points float32[P, 3], triangles int32[T, 3]) of shape `number` of a kind."""
    rng = np.random.default_rng(number)
    if shape == "soup":
        return meshgen.soup(sizes[0], seed=number, median=1.0 / sizes[1])
    if shape == "torus":
        v, f = meshgen.torus(rng.uniform(0.3, 0.45), rng.uniform(0.05, 0.2), *sizes)
        return _turned(v, rng), f
    v, f = _sphere(*sizes)
    p = v.astype(np.float64)
    noise = sum(meshgen.value_noise(p, 4.0 * 2 ** k, number + k) / 2 ** k for k in range(3)) / 1.75
    return _turned(p * (1.0 + 0.1 * noise)[:, None], rng), f


def _seeded(mesh, seed):
    """The mesh as another file might hold it: points and triangles listed from
    another one on, in another unit (a power of two).  The surface is the same,
    so that the lengths of the outputs, which follow from the cells it fills,
    do not depend on the seed."""
    v, f = mesh
    rng = np.random.default_rng(seed)
    shift = int(rng.integers(0, len(v)))
    v = np.roll(v, shift, axis=0) * np.float32(2.0 ** (seed % 16 - 8))
    f = np.roll((f + shift) % len(v), int(rng.integers(0, len(f))), axis=0)
    return np.ascontiguousarray(v, np.float32), np.ascontiguousarray(f, np.int32)


_SIZES = {"soup": ("tris", "edge"), "torus": ("a", "b"), "ico": ("subdiv",)}


def _mesh(case, seed):
    sizes = (case[k] for k in _SIZES[case["shape"]])
    return _seeded(_shape(case["shape"], case["mesh"], *sizes), seed)


def _on_device(p, t):
    return torch.from_numpy(p).cuda(), torch.from_numpy(t).cuda()


def _options(case):
    return {"semantics": svo_amd.SEM_INTENDED if case["intended"] else svo_amd.SEM_REFERENCE,
            "key_bits": case.get("key_bits", 0),
            "flags": 0 if case.get("records", True) else svo_amd.BUILD_NO_VERTEX_EDGE}


def prepare(case, seed):
    s = {"case": case, "ctx": _context()}
    path = case["path"]
    if path == "sort":
        rng = np.random.default_rng(seed)
        n, bits = case["n"], case["bits"]
        keys = rng.integers(0, 1 << bits, size=n, dtype=np.uint64)
        # neighboring cells come near each other, as from a program's own walk
        keys = np.where(np.arange(n) % 4 > 0, np.roll(keys, 1) ^ np.uint64(5), keys)
        kind = torch.int32 if case["key_bytes"] == 4 else torch.int64
        s["keys"] = torch.from_numpy(keys.view(np.int64)).to(kind).cuda()
        return s
    if path == "query":
        p, t = _on_device(*_mesh(dict(case, shape="ico"), seed))
        torch.cuda.synchronize()
        tree = s["ctx"].build_device(p.data_ptr(), p.shape[0], t.data_ptr(), t.shape[0],
                                     case["res"], semantics=svo_amd.SEM_INTENDED)
        rng = np.random.default_rng(seed)
        s.update(tree=tree, nodes=rng.integers(0, tree.info.n_nodes, case["n"]).astype(np.uint32),
                 slots=rng.integers(0, 27, case["n"]).astype(np.uint8))
        return s
    s["options"] = _options(case)
    if path in ("batch", "plan"):
        choices = [r for r in (64, 128, 256) if r <= case["top"]]
        s["meshes"], s["descs"] = [], []
        for spec in meshgen.mixed_specs(case["n"], case["mesh"], choices):
            mesh = _sphere(*spec.params) if spec.kind == "ico" else spec.build()
            p, t = _on_device(*_seeded(mesh, seed))
            s["meshes"].append((p, t))
            s["descs"].append((p.data_ptr(), p.shape[0], t.data_ptr(), t.shape[0], spec.res))
        if path == "plan":
            torch.cuda.synchronize()
            s["plan"] = s["ctx"].plan(s["descs"], on_device=True, **s["options"])
        return s
    s["res"] = (case["rx"], case["ry"], case["rz"])
    p, t = _mesh(case, seed)
    s["mesh"] = (p, t) if path == "host" else _on_device(p, t)
    return s


# ------------------------------------------------------------------ passes
# (field, words of a row, type): integers and records by their bytes
_FIELDS = [("code", 0, "<i4"), ("is_leaf", 1, "|u1"), ("origin", 3, "<f4"), ("width", 1, "<f4"),
           ("parent", 1, "<i4"), ("childs", 8, "<i4"), ("neighbors", 27, "<i4"),
           ("voxels", 0, "<i4"), ("vertices", 2, "<i8"), ("edges", 7, "<i4"), ("faces", 7, "<i4")]
_COUNTS = {"voxels": "n_voxels", "vertices": "n_vertices", "edges": "n_edges", "faces": "n_faces"}


class _Rows:
    """A device array of a tree for torch; keeps the trees it lies in."""

    def __init__(self, trees, ptr, shape, kind):
        self.trees = trees
        self.__cuda_array_interface__ = {"shape": shape, "typestr": kind, "data": (ptr, False),
                                         "version": 2}


def _arrays(trees):
    """Every output array of trees that lie one after the other on the device."""
    out = {}
    for field, words, kind in _FIELDS:
        rows = sum(getattr(t.info, _COUNTS.get(field, "n_nodes")) for t in trees)
        if rows:
            if words == 0 and trees[0].info.key_bits == 64:
                kind = "<i8"
            shape = (rows, words) if words > 1 else (rows,)
            out[field] = torch.as_tensor(_Rows(trees, trees[0].device_ptr(field), shape, kind),
                                         device="cuda")
    return out


def _passes(trees):
    """The trees of a batch as runs that lie one after the other (one for each
    of the batch's concurrent passes)."""
    at = {t.device_ptr("width"): t for t in trees}
    ends = {p + 4 * t.info.n_nodes for p, t in at.items()}
    runs = []
    for p in sorted(at):
        if p not in ends:
            run = [at[p]]
            while (p := p + 4 * run[-1].info.n_nodes) in at:
                run.append(at[p])
            runs.append(run)
    # in the order of the meshes, wherever the passes' memory lies
    first = {id(t): i for i, t in enumerate(trees)}
    return sorted(runs, key=lambda run: min(first[id(t)] for t in run))


def run(state):
    case, path = state["case"], state["case"]["path"]
    if path == "sort":
        with torch.cuda.stream(_stream()):
            keys = state["keys"].clone()
            st = svo_amd.lib().svo_k_radix_sort_noalloc(0, keys.data_ptr(), case["n"],
                                                        case["key_bytes"], case["bits"],
                                                        _stream().cuda_stream)
        assert st == svo_amd.OK, st
        return keys
    if path == "query":
        return state["tree"].query_neighbors(state["nodes"], state["slots"])
    if path == "host":
        tree = state["ctx"].build(*state["mesh"], state["res"], **state["options"])
        nodes = tree.field("nodes_aos").view(np.int32)
        tree.free()
        return nodes
    if path == "build":
        p, t = state["mesh"]
        tree = state["ctx"].build_device(p.data_ptr(), p.shape[0], t.data_ptr(), t.shape[0],
                                         state["res"], **state["options"])
        return _arrays([tree])
    if path == "plan":
        trees, statuses, replayed = state["plan"].run()
        assert replayed
    else:
        trees, statuses = state["ctx"].build_batch(state["descs"], on_device=True,
                                                   **state["options"])
    assert not any(statuses), statuses
    return [_arrays(r) for r in _passes(trees)]


# ------------------------------------------------------------------ bounds
def _surface(shape, res):
    """(voxels, nodes) of a closed surface of this kind on a grid, about."""
    a = res[0] * res[1] + res[1] * res[2] + res[0] * res[2]
    voxels = (1.53 if shape == "ico" else 1.1) * a
    return voxels, 2.65 * voxels


def _soup(case):
    """(voxels, nodes) of a soup: triangles of median side h cells fill about
    1.33 h^2 + 2.4 h + 1.5 cells, and h halves from level to level."""
    def crossed(level):
        h = max(case["rx"], case["ry"], case["rz"]) / case["edge"] / 2 ** level
        cells = case["rx"] * case["ry"] * case["rz"] / 8.0 ** level
        return min(cells, case["tris"] * (1.33 * h * h + 2.4 * h + 1.5))
    depth = int(math.ceil(math.log2(max(case["rx"], case["ry"], case["rz"])))) + 1
    return crossed(0), 8 * sum(crossed(level) for level in range(1, depth))


def work(case):
    """Each triangle and point read once, each output array written once (a
    node's arrays are 161 bytes and its code, its reference records 464)."""
    path = case["path"]
    if path == "sort":
        return {"bytes": 2 * case["n"] * case["key_bytes"], "flops": 0}
    if path == "query":  # node, slot, the table's word and the answer
        return {"bytes": 13 * case["n"], "flops": 0}
    if path in ("batch", "plan"):
        choices = [r for r in (64, 128, 256) if r <= case["top"]]
        tris = case["n"] * 14700.0
        sizes = [_surface("ico", (r, r, r)) for r in choices]
        voxels = case["n"] * 0.75 * sum(v for v, _ in sizes) / len(sizes)
        nodes = case["n"] * 0.75 * sum(n for _, n in sizes) / len(sizes)
    elif case["shape"] == "soup":
        tris = case["tris"]
        voxels, nodes = _soup(case)
    else:
        tris = 20 * 4 ** case["subdiv"] if case["shape"] == "ico" else 2 * case["a"] * case["b"]
        voxels, nodes = _surface(case["shape"], (case["rx"], case["ry"], case["rz"]))
    key = 8 if case.get("key_bits") == 64 else 4
    mesh = 12 * tris + (36 if case.get("shape") == "soup" else 6) * tris
    if path == "host":
        return {"bytes": mesh + 168 * nodes, "flops": 44 * voxels}
    records = 0
    if case.get("records", True):
        records = 16 * 1.5 + 28 * 4.0 + 28 * 3.5 if case["intended"] else 16 * 8 + 28 * 12
    return {"bytes": mesh + key * voxels + (161 + key + records) * nodes, "flops": 44 * voxels}


def exact(case, seed):
    """None: which cells a mesh fills is defined by the single-precision tests
    of the reference, and that set gives every later array its length and order
    (in 64 bits a few cells on a triangle's rim fall the other way).  The codes,
    links and records are compared by their bytes."""
    return None
