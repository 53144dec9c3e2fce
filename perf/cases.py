"""What a user of the partitioner has it do: one call (or one batch) per case.

Graphs are made on the GPU from the seed alone: triangulated 2-D meshes (each
grid cell split by a diagonal of random direction), 7-point 3-D stencils with
random edge weights, and R-MAT graphs (a=.57, b=.19, c=.19; symmetrised, no
duplicates, no self-loops). Every output is a whole number.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("jet-partitioner-official-fork_amd"))
import jet_amd  # noqa: E402

TWO_HOP, HEC, MATCHING = 0, 1, 2  # coarsening_alg
WORKERS = 16  # of the batched mode


def _case(name, graph, size, k, imb, alg, entry="device", wmax=1, ef=0, ultra=False):
    c = {"graph": graph, "size": "x".join(str(s) for s in size), "k": k, "imb": imb, "alg": alg, "entry": entry,
         "wmax": wmax, "ef": ef, "ultra": ultra}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest calls: a domain decomposition of a small mesh, where
        # launches and latency are all there is
        _case("mesh2d-64", "mesh2d", (64, 64), 8, 1.03, TWO_HOP),
        # the ordinary small call: 65,536 vertices, unit weights, 8 parts
        _case("mesh2d-256", "mesh2d", (256, 256), 8, 1.03, TWO_HOP),
        # ragged sizes, a prime number of parts, a tight balance, pure
        # matching, and host arrays with 32-bit offsets
        _case("mesh2d-501x333-host", "mesh2d", (501, 333), 37, 1.01, MATCHING, "host", wmax=4),
        # quality mode: eighteen filter temperatures per level
        _case("stencil3d-40-ultra", "stencil3d", (40, 40, 40), 16, 1.03, HEC, wmax=10, ultra=True),
        # a bisection of a large mesh (nested dissection starts so)
        _case("stencil3d-101x97x89-k2", "stencil3d", (101, 97, 89), 2, 1.03, TWO_HOP, wmax=10),
        # the benchmark's default: 2.1 M vertices into 64 parts
        _case("stencil3d-128", "stencil3d", (128, 128, 128), 64, 1.03, HEC, wmax=10),
        # a small irregular graph: hubs and isolated vertices, 2-hop matching
        _case("rmat-16", "rmat", (16,), 32, 1.03, TWO_HOP, ef=8),
        # a social-network-like graph through the 64-bit-weight entry point
        _case("rmat-19-big", "rmat", (19,), 64, 1.10, HEC, "big", ef=16),
        # the benchmark's large irregular graph: 64 M edges into 256 parts
        _case("rmat-22", "rmat", (22,), 256, 1.10, HEC, ef=16),
        # many small graphs at once, the batched mode
        _case("batch-60", "mixed", (60,), 0, 0.0, 0, "batch", wmax=4),
        # the quality report of a given partition: cut, communication volume,
        # and the cut between every two parts
        _case("quality-64", "stencil3d", (64, 64, 64), 256, 0.0, 0, "quality", wmax=10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mesh2d", "mesh2d", "stencil3d", "stencil3d", "rmat", "rmat", "mixed", "quality"])
    if kind == "mixed":
        return _case(None, "mixed", (rng.randint(12, 60),), 0, 0.0, 0, "batch", wmax=4)
    graph = rng.choice(["mesh2d", "stencil3d"]) if kind == "quality" else kind
    ef = 0
    if graph == "mesh2d":
        side = _log(rng, 48, 1400)
        size = (side, max(32, side + rng.randint(-side // 3, side // 3)))
        n = size[0] * size[1]
    elif graph == "stencil3d":
        side = _log(rng, 13, 126)
        size = tuple(max(8, side - rng.randint(0, side // 4)) for _ in range(3))
        n = size[0] * size[1] * size[2]
    else:
        size = (rng.randint(12, 20),)
        ef = rng.choice([6, 8, 12, 16])
        n = 1 << size[0]
    k = min(_log(rng, 2, 256), max(2, n // 64))
    wmax = rng.choice([1, 4, 10]) if graph != "rmat" else rng.choice([1, 1, 4])
    entry = "quality" if kind == "quality" else rng.choice(["device", "device", "device", "host", "big"])
    imb = rng.choice([1.01, 1.03, 1.03, 1.10]) if graph != "rmat" else rng.choice([1.03, 1.10])
    ultra = entry != "quality" and n < 200000 and rng.random() < 0.15
    return _case(None, graph, size, k, imb, rng.choice([TWO_HOP, HEC, HEC, MATCHING]) if graph != "rmat"
                 else rng.choice([TWO_HOP, HEC]), entry, wmax, ef, ultra)


# ---------------------------------------------------------------- graphs
def _sizes(c):
    return [int(s) for s in c["size"].split("x")]


def _mix(x, seed):
    """A hash of int64 keys (wrapping products)."""
    x = (x + seed) * 0x1E3779B97F4A7C15
    x = (x ^ ((x >> 29) & 0x7FFFFFFFF)) * 0x3F58476D1CE4E5B9
    return (x >> 20) & 0x7FFFFFFF


def _csr(n, u, v, wmax, seed):
    """Symmetric CSR of the undirected edges (u, v) without duplicates and
    self-loops; weights 1 .. wmax by hash of the unordered pair."""
    keep = u != v
    u, v = u[keep], v[keep]
    key = torch.unique(torch.cat([u * n + v, v * n + u]))
    src, dst = torch.div(key, n, rounding_mode="floor"), key % n
    rp = torch.zeros(n + 1, dtype=torch.int64, device=key.device)
    rp[1:] = torch.cumsum(torch.bincount(src, minlength=n), 0)
    ew = torch.ones(len(key), dtype=torch.int32, device=key.device)
    if wmax > 1:
        ew = (1 + _mix(torch.minimum(src, dst) * n + torch.maximum(src, dst), seed) % wmax).to(torch.int32)
    vw = torch.ones(n, dtype=torch.int32, device=key.device)
    return {"rowptr": rp, "col": dst.to(torch.int32), "ew": ew, "vw": vw, "uniform": wmax <= 1}


def _mesh2d(nx, ny, wmax, seed, dev):
    gen = torch.Generator(device=dev).manual_seed(seed)
    ids = torch.arange(nx * ny, device=dev).reshape(nx, ny)
    flip = torch.rand((nx - 1, ny - 1), generator=gen, device=dev) < 0.5
    a, b, c, d = ids[:-1, :-1], ids[1:, 1:], ids[1:, :-1], ids[:-1, 1:]
    u = torch.cat([ids[:-1].reshape(-1), ids[:, :-1].reshape(-1), torch.where(flip, a, c).reshape(-1)])
    v = torch.cat([ids[1:].reshape(-1), ids[:, 1:].reshape(-1), torch.where(flip, b, d).reshape(-1)])
    return _csr(nx * ny, u, v, wmax, seed)


def _stencil3d(nx, ny, nz, wmax, seed, dev):
    ids = torch.arange(nx * ny * nz, device=dev).reshape(nx, ny, nz)
    u = torch.cat([ids[:-1].reshape(-1), ids[:, :-1].reshape(-1), ids[:, :, :-1].reshape(-1)])
    v = torch.cat([ids[1:].reshape(-1), ids[:, 1:].reshape(-1), ids[:, :, 1:].reshape(-1)])
    return _csr(nx * ny * nz, u, v, wmax, seed)


def _rmat(scale, ef, wmax, seed, dev):
    gen = torch.Generator(device=dev).manual_seed(seed)
    n, e = 1 << scale, ef << scale
    u = torch.zeros(e, dtype=torch.int64, device=dev)
    v = torch.zeros(e, dtype=torch.int64, device=dev)
    for _ in range(scale):
        r = torch.rand(e, generator=gen, device=dev)
        u = 2 * u + (r >= 0.76)
        v = 2 * v + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    return _csr(n, u, v, wmax, seed)


def _graph(c, seed, dev="cuda"):
    s = _sizes(c)
    if c["graph"] == "mesh2d":
        return _mesh2d(*s, c["wmax"], seed, dev)
    if c["graph"] == "stencil3d":
        return _stencil3d(*s, c["wmax"], seed, dev)
    return _rmat(s[0], c["ef"], c["wmax"], seed, dev)


def _mix_of(c):
    """The batched mix, the same shapes for every seed: half meshes and
    stencils, half R-MAT; 1 K to 200 K vertices, 2 to 64 parts."""
    rng = random.Random(_sizes(c)[0])
    out = []
    for i in range(_sizes(c)[0]):
        n = math.exp(rng.uniform(math.log(1e3), math.log(2e5)))
        k, imb, alg = rng.choice([2, 4, 8, 16, 32, 64]), rng.choice([1.01, 1.03, 1.10]), rng.choice([TWO_HOP, HEC])
        if i % 2:
            out.append(_case(None, "rmat", (max(10, round(math.log2(n))),), k, imb, alg, wmax=4, ef=8))
        elif rng.random() < 0.5:
            side = round(n ** 0.5)
            out.append(_case(None, "mesh2d", (side, side + rng.randint(0, 5)), k, imb, alg, wmax=4))
        else:
            side = round(n ** (1 / 3))
            out.append(_case(None, "stencil3d", (side, side, side + rng.randint(0, 3)), k, imb, alg, wmax=4))
    return out


def _host(g):
    return {k: (v.cpu().numpy() if torch.is_tensor(v) else v) for k, v in g.items()}


def _config(c):
    return jet_amd.Config(num_parts=c["k"], max_imb_ratio=c["imb"], coarsening_alg=c["alg"],
                          ultra_settings=c["ultra"])


def prepare(c, seed):
    if c["entry"] == "batch":
        parts = _mix_of(c)
        graphs = [_host(_graph(p, seed + 31 * i)) for i, p in enumerate(parts)]
        return {"entry": "batch", "graphs": graphs, "cfgs": [_config(p) for p in parts],
                "seeds": [(seed + i) & 0xFFFFFFFF for i in range(len(parts))], "ctx": jet_amd.Context(workers=WORKERS)}
    g = _graph(c, seed)
    st = {"entry": c["entry"], "seed": seed & 0xFFFFFFFF}
    if c["entry"] == "quality":
        # slabs of consecutive ids, one vertex in sixteen in a random part
        gen = torch.Generator(device="cuda").manual_seed(seed)
        n = len(g["vw"])
        part = (torch.arange(n, device="cuda") * c["k"]) // n
        odd = torch.rand(n, generator=gen, device="cuda") < 1 / 16
        other = torch.randint(0, c["k"], (n,), generator=gen, device="cuda")
        part = torch.where(odd, other, part).to(torch.int32)
        return {**st, "g": _host(g), "part": part.cpu().numpy(), "k": c["k"]}
    st["cfg"] = _config(c)
    if c["entry"] == "device":
        st.update(g=g, n=len(g["vw"]), part=torch.empty(len(g["vw"]), dtype=torch.int32, device="cuda"))
        torch.cuda.synchronize()
    else:
        st["g"] = _host(g)
        if c["entry"] == "big":
            for a in ("ew", "vw"):
                st["g"][a] = st["g"][a].astype(np.int64)
        else:
            st["g"]["rowptr"] = st["g"]["rowptr"].astype(np.int32)
    return st


def run(st):
    e = st["entry"]
    if e == "device":
        g = st["g"]
        cut, _ = jet_amd.partition_device(st["n"], g["rowptr"].data_ptr(), g["col"].data_ptr(), g["ew"].data_ptr(),
                                          g["vw"].data_ptr(), st["part"].data_ptr(), st["cfg"], st["seed"],
                                          g["uniform"])
        return {"part": st["part"], "cut": cut}
    if e == "host":
        part, cut, _ = jet_amd.partition(st["g"], st["cfg"], st["g"]["uniform"], st["seed"])
        return {"part": part, "cut": cut}
    if e == "big":
        part, cut, _ = jet_amd.partition_big(st["g"], st["cfg"], st["g"]["uniform"], st["seed"])
        return {"part": part, "cut": cut}
    if e == "batch":
        parts, cuts = st["ctx"].batch(st["graphs"], st["cfgs"], st["seeds"])
        return {"parts": parts, "cuts": cuts}
    q = jet_amd.partition_quality(st["g"], st["part"], st["k"])
    return {"edge_cut": q.edge_cut, "comm_size": q.comm_size, "max_part_cut": q.max_part_cut,
            "largest_part": q.largest_part, "smallest_part": q.smallest_part,
            "heatmap": jet_amd.cut_heatmap(st["g"], st["part"], st["k"])}


def exact(c, seed):
    return None  # parts and cuts are whole numbers


# ---------------------------------------------------------------- work
def _counts(c):
    """(vertices, stored edges); R-MAT's after duplicates are dropped, about."""
    s = _sizes(c)
    if c["graph"] == "mesh2d":
        x, y = s
        return x * y, 2 * (x * (y - 1) + y * (x - 1) + (x - 1) * (y - 1))
    if c["graph"] == "stencil3d":
        x, y, z = s
        return x * y * z, 2 * (x * y * (z - 1) + x * z * (y - 1) + y * z * (x - 1))
    return 1 << s[0], int(1.9 * c["ef"] * (1 << s[0]))


def work(c):
    """The graph read once and the partition written (or read) once: offsets
    8 (4 on the 32-bit entry point), column 4, weights 4 (8 on the 64-bit
    one), part 4; an add or compare per stored edge."""
    total, ops = 0, 0
    for p in _mix_of(c) if c["entry"] == "batch" else [c]:
        n, m = _counts(p)
        off, w = (4 if c["entry"] == "host" else 8), (8 if c["entry"] == "big" else 4)
        total += off * (n + 1) + (4 + w) * m + w * n + 4 * n
        ops += m
    return {"bytes": total, "flops": ops}
