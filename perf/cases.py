"""Timed cases of the streaming operations and of the gather / scatter operator.

Each case is a dict of plain values:

  kind "cg"     the vector work of one conjugate-gradient iteration on vectors of n entries:
                p.Ap, then x += alpha p, r -= alpha Ap with r.r, then p = r + beta p.
                storage "f64" (streaming.Reducer) or "f32" / "bf16" (streaming.MixedCG, the
                fused x / r update alone: the other two have no reduced-precision form)
  kind "norm"   sum of a_i^2 over n FP64 entries
  kind "ogs"    one call on a box mesh's operator: op "gs" (gather+scatter in place), "gather"
                or "scatter"; element type, box and degree; k fields per node; storage "f64",
                "f32" (FP32 sums), "mixed_f32" or "mixed_bf16" (FP64 sums, rounded once)
  kind "batch"  one step over `count` independent hex boxes: gather+scatter of k fields, then
                the CG update with one r.r per box, in two launches for all of them
"""
import numpy as np
import torch

from streamparanumal_amd import batch as spb
from streamparanumal_amd import streaming
from streamparanumal_amd.device import DeviceArray
from streamparanumal_amd.ogs import Ogs

ALPHA, BETA = 0.015625, 0.3
NUMPY = {"f64": np.float64, "f32": np.float32, "mixed_f32": np.float32, "mixed_bf16": np.uint16, "bf16": np.uint16}
TORCH = {"f64": torch.float64, "f32": torch.float32, "mixed_f32": torch.float32, "mixed_bf16": torch.bfloat16,
         "bf16": torch.bfloat16}
BYTES = {"f64": 8, "f32": 4, "mixed_f32": 4, "mixed_bf16": 2, "bf16": 2}
ELEMENT_DIM = {"Tri": 2, "Quad": 2, "Tet": 3, "Hex": 3}


def listed():
    return [
        # a small mesh's vectors: launches and latency are all there is
        {"name": "cg_small", "kind": "cg", "n": 10007, "storage": "f64", "mode": "reference"},
        # the streaming benchmark's vectors (2^27 entries)
        {"name": "cg_large", "kind": "cg", "n": 134217728, "storage": "f64", "mode": "reference"},
        # an ordinary mesh's vectors in FP32, ragged length
        {"name": "cg_f32", "kind": "cg", "n": 3000003, "storage": "f32", "mode": "fast"},
        # the smallest configured mesh (8^3 elements, degree 7): one short call
        {"name": "gs_hex7_small", "kind": "ogs", "op": "gs", "element": "Hex", "nx": 8, "ny": 8, "nz": 8, "p": 7,
         "k": 1, "storage": "f64"},
        # the benchmark's own mesh
        {"name": "gs_hex7_large", "kind": "ogs", "op": "gs", "element": "Hex", "nx": 64, "ny": 64, "nz": 64, "p": 7,
         "k": 1, "storage": "f64"},
        # low degree: nearly every node is shared, runs are short
        {"name": "gs_hex2", "kind": "ogs", "op": "gs", "element": "Hex", "nx": 101, "ny": 100, "nz": 99, "p": 2,
         "k": 1, "storage": "f64"},
        # simplices: rows of up to 24 members
        {"name": "gs_tet3", "kind": "ogs", "op": "gs", "element": "Tet", "nx": 60, "ny": 60, "nz": 60, "p": 3,
         "k": 1, "storage": "f64"},
        # values kept in BF16, one field
        {"name": "gs_bf16_hex7", "kind": "ogs", "op": "gs", "element": "Hex", "nx": 48, "ny": 48, "nz": 48, "p": 7,
         "k": 1, "storage": "mixed_bf16"},
        # values kept in FP32, a velocity's three fields, an odd row length
        {"name": "gs_f32_hex4_k3", "kind": "ogs", "op": "gs", "element": "Hex", "nx": 48, "ny": 47, "nz": 46, "p": 4,
         "k": 3, "storage": "mixed_f32"},
        # the drivers' default mesh (50^3 elements, degree 3): assembled values out
        {"name": "gather_hex3", "kind": "ogs", "op": "gather", "element": "Hex", "nx": 50, "ny": 50, "nz": 50, "p": 3,
         "k": 1, "storage": "f64"},
        # assembled values back to the elements
        {"name": "scatter_hex7", "kind": "ogs", "op": "scatter", "element": "Hex", "nx": 48, "ny": 48, "nz": 48,
         "p": 7, "k": 1, "storage": "f64"},
        # many uneven meshes served together, three fields in FP32
        {"name": "batch_f32", "kind": "batch", "count": 16, "mesh_seed": 4, "n_lo": 4, "n_hi": 24, "k": 3,
         "storage": "f32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["cg", "norm", "ogs", "ogs", "ogs", "ogs", "ogs", "batch"])
    if kind == "cg":
        storage = rng.choice(["f64", "f64", "f32", "bf16"])
        return {"kind": "cg", "n": _log_int(rng, 3000, 100000000), "storage": storage,
                "mode": rng.choice(["reference", "fast"])}
    if kind == "norm":
        return {"kind": "norm", "n": _log_int(rng, 3000, 130000000), "mode": rng.choice(["reference", "fast"])}
    if kind == "batch":
        return {"kind": "batch", "count": rng.randint(3, 20), "mesh_seed": rng.randint(1, 1000), "n_lo": 3,
                "n_hi": rng.randint(8, 20), "k": rng.choice([1, 2, 3, 4]),
                "storage": rng.choice(["f64", "f32", "f32", "bf16"])}
    element = rng.choice(["Hex", "Hex", "Hex", "Tet", "Tri", "Quad"])
    p = rng.choice([1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 15]) if element in ("Hex", "Quad") else rng.randint(1, 8)
    k = rng.choice([1, 1, 1, 2, 3, 4])
    dim = ELEMENT_DIM[element]
    nodes = _log_int(rng, 20000, 40000000 // k)
    per_cell = {"Tri": (p + 1) * (p + 2), "Quad": (p + 1) ** 2, "Tet": (p + 1) * (p + 2) * (p + 3),
                "Hex": (p + 1) ** 3}[element]
    side = max(2.0, (nodes / per_cell) ** (1.0 / dim))
    box = [max(2, int(side * rng.uniform(0.8, 1.2))) for _ in range(dim)] + [1]
    return {"kind": "ogs", "op": rng.choice(["gs", "gs", "gs", "gather", "scatter"]), "element": element,
            "nx": box[0], "ny": box[1], "nz": box[2], "p": p, "k": k,
            "storage": rng.choice(["f64", "f64", "f32", "mixed_f32", "mixed_bf16"])}


# ------------------------------------------------------------------ sizes --
def _nodes(case):
    """(local nodes, lattice points) of a box."""
    nx, ny, nz, p = case["nx"], case["ny"], case["nz"], case["p"]
    e = case["element"]
    if ELEMENT_DIM[e] == 2:
        return (nx * ny * ((p + 1) * (p + 2) if e == "Tri" else (p + 1) ** 2), (nx * p + 1) * (ny * p + 1))
    per = (p + 1) * (p + 2) * (p + 3) if e == "Tet" else (p + 1) ** 3
    return nx * ny * nz * per, (nx * p + 1) * (ny * p + 1) * (nz * p + 1)


def _ogs_storage(case):
    # the gather and scatter have no reduced-precision form: FP32 values take their FP32 sums
    s = case["storage"]
    return "f32" if case["op"] != "gs" and s.startswith("mixed") else s


def _batch_sizes(case):
    meshes = spb.instances(case["count"], case["mesh_seed"], case["n_lo"], case["n_hi"])
    return meshes, [n ** 3 * (p + 1) ** 3 for n, p in meshes]


def work(case):
    """Values read once and written once; indices, which another layout could do without, are not counted."""
    if case["kind"] == "norm":
        return {"bytes": 8 * case["n"], "flops": 2 * case["n"]}
    if case["kind"] == "cg":
        n, s = case["n"], BYTES[case["storage"]]
        if case["storage"] == "f64":
            return {"bytes": (2 + 6 + 3) * s * n, "flops": (2 + 6 + 3) * n}
        return {"bytes": 6 * s * n, "flops": 6 * n}
    if case["kind"] == "batch":
        total = case["k"] * sum(_batch_sizes(case)[1])
        return {"bytes": (2 + 6) * BYTES[case["storage"]] * total, "flops": 7 * total}
    nl, ng = _nodes(case)
    s = BYTES[_ogs_storage(case)] * case["k"]
    values = 2 * nl if case["op"] == "gs" else nl + ng
    return {"bytes": values * s, "flops": case["k"] * (nl - ng) if case["op"] != "scatter" else 0}


# ----------------------------------------------------------------- inputs --
class _Shared:
    """A DeviceArray's memory as a torch tensor sees it; holds the array."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {"shape": (array.n,), "typestr": array.dtype.str,
                                         "data": (array.ptr, False), "version": 2}


def _tensor(array, storage):
    if storage in ("bf16", "mixed_bf16"):
        view = _Shared(array)
        view.__cuda_array_interface__["typestr"] = "<i2"
        return torch.as_tensor(view, device="cuda").view(torch.bfloat16)
    return torch.as_tensor(_Shared(array), device="cuda")


def _values(n, storage, seed, which):
    """Uniform on [-1, 1) in FP64, rounded to the storage type: the same for prepare() and exact()."""
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * (seed + 1) + which)
    v = torch.rand(n, dtype=torch.float64, device="cuda", generator=g)
    v.mul_(2.0).sub_(1.0)
    return v if storage == "f64" else v.to(TORCH[storage])


def _vector(n, storage, seed, which):
    a = DeviceArray(n, NUMPY[storage])
    t = _tensor(a, storage)
    t.copy_(_values(n, storage, seed, which))
    return a, t


def _mode(case):
    return 0 if case["mode"] == "reference" else 1


def prepare(case, seed):
    from streamparanumal_amd.ogs import platform_open
    platform_open(0)
    s = {"case": case}
    if case["kind"] == "norm":
        s["a"], _ = _vector(case["n"], "f64", seed, 0)
        s["red"] = streaming.Reducer(case["n"], _mode(case))
        s["out"] = {"norm": _tensor(s["red"].out, "f64")}
    elif case["kind"] == "cg":
        st = case["storage"]
        t = {}
        for i, v in enumerate(("p", "Ap", "x", "r")):
            s[v], t[v] = _vector(case["n"], st, seed, i)
        if st == "f64":
            s["dot"] = streaming.Reducer(case["n"], _mode(case))
            s["cg"] = streaming.Reducer(case["n"], _mode(case))
            s["out"] = {"pAp": _tensor(s["dot"].out, "f64"), "rr": _tensor(s["cg"].out, "f64"), "x": t["x"],
                        "r": t["r"], "p": t["p"]}
        else:
            s["cg"] = streaming.MixedCG()
            s["out"] = {"rr": _tensor(s["cg"].out, "f64"), "x": t["x"], "r": t["r"]}
    elif case["kind"] == "batch":
        meshes, _ = _batch_sizes(case)
        b = spb.Batch(meshes, case["k"], NUMPY[case["storage"]])
        b.vectors, t = {}, {}
        for i, v in enumerate(("q", "p", "x", "r")):
            b.vectors[v], t[v] = _vector(case["k"] * b.N, case["storage"], seed, i)
        b.make_plan()
        s["batch"] = b
        s["out"] = {"q": t["q"], "x": t["x"], "r": t["r"], "rr": _tensor(b.plan.rdotr, "f64")}
    else:
        st = _ogs_storage(case)
        nl, ng = _nodes(case)
        s["ogs"] = Ogs.box(case["element"], case["nx"], case["ny"], case["nz"], case["p"], keep_ids=False)
        if case["op"] == "gs":
            s["q"], s["out"] = _vector(nl * case["k"], st, seed, 0)
        elif case["op"] == "gather":
            s["q"], _ = _vector(nl * case["k"], st, seed, 0)
            s["gq"] = DeviceArray(ng * case["k"], NUMPY[st])
            s["out"] = _tensor(s["gq"], st)
        else:
            s["gq"], _ = _vector(ng * case["k"], st, seed, 0)
            s["q"] = DeviceArray(nl * case["k"], NUMPY[st])
            s["out"] = _tensor(s["q"], st)
    torch.cuda.synchronize()  # torch filled the vectors on its own stream
    return s


# -------------------------------------------------------------------- run --
def run(s):
    case = s["case"]
    if case["kind"] == "norm":
        s["red"].norm(s["a"])
    elif case["kind"] == "cg":
        if case["storage"] == "f64":
            s["dot"].dot(s["p"], s["Ap"])
            s["cg"].cg_full(ALPHA, s["p"], s["Ap"], s["x"], s["r"])
            streaming.axpy(1.0, s["r"], BETA, s["p"])
        else:
            s["cg"].cg_full(ALPHA, s["p"], s["Ap"], s["x"], s["r"])
    elif case["kind"] == "batch":
        s["batch"].step(ALPHA)
    elif case["op"] == "gs":
        if case["storage"].startswith("mixed"):
            s["ogs"].gather_scatter_mixed(s["q"], case["k"])
        else:
            s["ogs"].gather_scatter(s["q"], case["k"])
    elif case["op"] == "gather":
        s["ogs"].gather(s["gq"], s["q"], case["k"])
    else:
        s["ogs"].scatter(s["q"], s["gq"], case["k"])
    return s["out"]


# ------------------------------------------------------- the same in 64 bits --
def _axis(n, device="cuda"):
    return torch.arange(n, dtype=torch.int64, device=device)


def _points(element, nx, ny, nz, p):
    """Lattice point of every local node (x fastest), elements and nodes in the mesh's order."""
    gx, gy = nx * p + 1, ny * p + 1
    a = range(p + 1)
    # cells, x fastest: element corners and the three edge vectors of each element of a cell
    if element in ("Hex", "Quad"):
        corners = [((1, 0, 0), (0, 1, 0), (0, 0, 1))]
        nodes = [(i, j, k) for k in (a if element == "Hex" else [0]) for j in a for i in a]
    elif element == "Tri":
        corners = [((1, 0, 0), (1, 1, 0), (0, 0, 0)), ((1, 1, 0), (0, 1, 0), (0, 0, 0))]
        nodes = [(i, j, 0) for j in a for i in range(p + 1 - j)]
    else:
        def cube(c):
            return (c & 1, (c >> 1) & 1, c >> 2)
        corners = [tuple(cube(c) for c in t) for t in ((3, 2, 7), (1, 3, 7), (2, 6, 7), (6, 4, 7), (5, 1, 7), (4, 5, 7))]
        nodes = [(i, j, k) for k in a for j in range(p + 1 - k) for i in range(p + 1 - j - k)]
    offset = []
    for v in corners:
        for m in nodes:
            x, y, z = (sum(m[i] * v[i][d] for i in range(3)) for d in range(3))
            offset.append(x + gx * (y + gy * z))
    offset = torch.tensor(offset, dtype=torch.int64, device="cuda")
    if ELEMENT_DIM[element] == 2:
        nz = 1
    cell = (_axis(nx)[None, None, :] + gx * (_axis(ny)[None, :, None] + gy * _axis(nz)[:, None, None])) * p
    return (cell.reshape(-1, 1) + offset[None, :]).reshape(-1)


def _rows(point, ng):
    """Row of every lattice point: points in order of their first appearance among the local nodes."""
    first = torch.full((ng,), point.numel(), dtype=torch.int64, device="cuda")
    first.scatter_reduce_(0, point, _axis(point.numel()), "amin")
    row = torch.empty_like(first)
    row[torch.argsort(first)] = _axis(ng)
    return row


def _sums(point, ng, q):
    return torch.zeros((ng, q.shape[1]), dtype=torch.float64, device="cuda").index_add_(0, point, q)


def exact(case, seed):
    if case["kind"] == "norm":
        return {"norm": _values(case["n"], "f64", seed, 0).square_().sum().reshape(1)}
    if case["kind"] == "cg":
        p, ap, x, r = (_values(case["n"], case["storage"], seed, i).double() for i in range(4))
        out = {}
        if case["storage"] == "f64":
            out["pAp"] = (p * ap).sum().reshape(1)
        out["x"] = x.add_(p, alpha=ALPHA)
        out["r"] = r.sub_(ap, alpha=ALPHA)
        # r.r is the sum over the stored r
        out["rr"] = r.to(TORCH[case["storage"]]).double().square().sum().reshape(1)
        if case["storage"] == "f64":
            out["p"] = p.mul_(BETA).add_(r)
        return out
    if case["kind"] == "batch":
        st, k = case["storage"], case["k"]
        meshes, sizes = _batch_sizes(case)
        n = k * sum(sizes)
        q, p, x, r = (_values(n, st, seed, i).double() for i in range(4))
        at = 0
        for (m, deg), nl in zip(meshes, sizes):
            point, ng = _points("Hex", m, m, m, deg), (m * deg + 1) ** 3
            part = q[at:at + k * nl].view(nl, k)
            part.copy_(_sums(point, ng, part)[point])
            at += k * nl
        stored = q.to(TORCH[st]).double()
        x.add_(p, alpha=ALPHA)
        r.sub_(stored, alpha=ALPHA)
        ends = [0]
        for nl in sizes:
            ends.append(ends[-1] + k * nl)
        held = r.to(TORCH[st]).double()
        rr = torch.stack([held[a:b].square().sum() for a, b in zip(ends, ends[1:])])
        return {"q": q, "x": x, "r": r, "rr": rr}
    st, k = _ogs_storage(case), case["k"]
    nl, ng = _nodes(case)
    point = _points(case["element"], case["nx"], case["ny"], case["nz"], case["p"])
    if case["op"] == "gs":
        return _sums(point, ng, _values(nl * k, st, seed, 0).double().view(nl, k))[point].reshape(-1)
    row = _rows(point, ng)[point]
    if case["op"] == "gather":
        return _sums(row, ng, _values(nl * k, st, seed, 0).double().view(nl, k)).reshape(-1)
    return _values(ng * k, st, seed, 0).double().view(ng, k)[row].reshape(-1)
