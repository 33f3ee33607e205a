"""The library's everyday work as measurable cases: training a guiding field,
recording paths into training samples, and guided sampling.

  listed()             the cases, as plain dicts
  draw(rng)            another case of the same ranges
  prepare(case, seed)  what a renderer holds before the call (on the GPU, or in
                       host memory where the entry point takes host data)
  run(state)           one pass through the public entry points; its outputs
  work(case)           bytes and flops the pass cannot do without
  exact(case, seed)    the outputs in 64 bits, where they have such a value

A training pass is a whole session on a kept Field handle: reset, then the
session's frames, then one batch of guided queries on the trained field.  The
queries (four or more per hundred samples, spread over the scene) return the
trained mixtures through the calls a renderer reads them with; the kd tree
comes back beside them.  Training has no 64-bit value of its own: the split,
merge and stop decisions of a region depend on its rounded sums.
"""
import ctypes
import math

import numpy as np
import torch

import openpgl_amd as pgl
from openpgl_amd.hip_runtime import pinned_copy, pinned_empty
from openpgl_amd.synth import SAMPLE_DTYPE

_LOBES = 4


def listed():
    return [
        # guided sampling of one small tile: a thousand shading points, launch and latency count
        dict(name="query_tile", kind="query", n=1000, volume=0.0, knn=True, vmm=False, regions=8),
        # a wavefront of a scene with participating media, ragged size
        dict(name="query_mixed", kind="query", n=50021, volume=0.3, knn=True, vmm=False, regions=64),
        # all shading points of a full-HD frame on a well refined field
        dict(name="query_frame", kind="query", n=2073600, volume=0.0, knn=True, vmm=False, regions=400),
        # a query server under a burst of requests of log-uniform size, page-locked host arrays in and out
        dict(name="serve_burst", kind="serve", requests=24, smallest=1000, largest=65536, volume=0.3, regions=64),
        # an interactive preview: few samples per frame, host storage, small leaves
        dict(name="preview", kind="render", n=20011, frames=2, queries=4096, leaf=2000),
        # the render loop a drop-in user has: host storage in, host queries out, a million samples per frame
        dict(name="render_loop", kind="render", n=1000000, frames=2, queries=262144, leaf=32000),
        # progressive training from device-resident records, default settings
        dict(name="train_frames", kind="train", n=1000000, frames=4, queries=98304, leaf=32000, vmm=False,
             deterministic=True),
        # the plain von Mises-Fisher field, arrival order kept, thousands of small regions
        dict(name="train_fine", kind="train", n=700001, frames=2, queries=65536, leaf=1000, vmm=True,
             deterministic=False),
        # a large frame of surface and volume records in one array
        dict(name="train_large", kind="route", n=10000000, frames=2, volume=0.2, queries=524288, leaf=32000),
        # training straight from recorded paths
        dict(name="train_paths", kind="path_train", paths=150000, length=12, frames=2, queries=131072, leaf=32000),
        # training samples of one tile's paths
        dict(name="paths_tile", kind="paths", paths=3001, length=8, nee=False, direct=False, rr=True),
        # training samples of a whole frame's paths
        dict(name="paths_frame", kind="paths", paths=1000000, length=12, nee=True, direct=True, rr=False),
    ]


def _log_int(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["query", "query", "serve", "render", "train", "train", "route", "path_train", "paths", "paths"])
    if kind == "query":
        return dict(kind=kind, n=_log_int(rng, 1000, 2000000), volume=rng.choice([0.0, 0.3, 0.5]),
                    knn=rng.random() < 0.75, vmm=rng.random() < 0.25, regions=_log_int(rng, 8, 400))
    if kind == "serve":
        return dict(kind=kind, requests=rng.randint(4, 32), smallest=1000, largest=_log_int(rng, 4000, 100000),
                    volume=rng.choice([0.0, 0.3]), regions=_log_int(rng, 8, 400))
    if kind == "render":
        n = _log_int(rng, 10000, 1000000)
        return dict(kind=kind, n=n, frames=rng.randint(1, 3), queries=max(4096, n // rng.randint(4, 10)),
                    leaf=rng.choice([2000, 8000, 32000]))
    if kind == "train":
        n = _log_int(rng, 20000, 1500000)
        leaf = rng.choice([1000, 4000, 32000])
        return dict(kind=kind, n=n, frames=rng.randint(1, 4), queries=max(4096, n // 12), leaf=leaf,
                    vmm=rng.random() < 0.3, deterministic=rng.random() < 0.7)
    if kind == "route":
        n = _log_int(rng, 100000, 8000000)
        return dict(kind=kind, n=n, frames=rng.randint(1, 2), volume=rng.choice([0.1, 0.2, 0.5]),
                    queries=max(4096, n // 19), leaf=32000)
    if kind == "path_train":
        return dict(kind=kind, paths=_log_int(rng, 5000, 200000), length=rng.randint(5, 12), frames=rng.randint(1, 2),
                    queries=163840, leaf=rng.choice([4000, 32000]))
    return dict(kind=kind, paths=_log_int(rng, 1000, 1000000), length=rng.randint(4, 12), nee=rng.random() < 0.5,
                direct=rng.random() < 0.5, rr=rng.random() < 0.5)


# ------------------------------------------------------------------- inputs
def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1009 + stream)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda")


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _randint(g, lo, hi, n):
    return torch.randint(lo, hi, (n,), generator=g, device="cuda")


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True)


class _Scene:
    """Blobs of shading points that drift from frame to frame; each blob is lit
    by four vMF lobes of concentration 5 to 500."""

    def __init__(self, seed, blobs=16):
        g = _gen(seed, 0)
        self.blobs = blobs
        self.centre = 0.1 + 0.8 * _rand(g, blobs, 3)
        self.drift = 0.01 * _unit(_randn(g, blobs, 3))
        self.mu = _unit(_randn(g, blobs * _LOBES, 3))
        self.kappa = torch.exp(math.log(5.0) + math.log(100.0) * _rand(g, blobs * _LOBES))

    def positions(self, g, n, frame=0, spread=0.05, loose=0.2):
        """Four of five points in a blob, the others anywhere; and each point's blob."""
        centre = self.centre + frame * self.drift
        blob = _randint(g, 0, self.blobs, n)
        pos = centre[blob] + spread * _randn(g, n, 3)
        free = _rand(g, n) < loose
        pos = torch.where(free[:, None], _rand(g, n, 3), pos)
        for a in range(0, n, 1 << 20):
            b = min(n, a + (1 << 20))
            near = torch.cdist(pos[a:b], centre).argmin(1)
            blob[a:b] = torch.where(free[a:b], near, blob[a:b])
        return pos, blob

    def directions(self, g, blob):
        lobe = blob * _LOBES + _randint(g, 0, _LOBES, len(blob))
        mu, kappa = self.mu[lobe], self.kappa[lobe]
        u = _rand(g, len(blob))
        c = (1.0 + torch.log(u + (1.0 - u) * torch.exp(-2.0 * kappa)) / kappa).clamp(-1.0, 1.0)
        phi = 2.0 * math.pi * _rand(g, len(blob))
        axis = torch.zeros_like(mu)
        flip = mu[:, 0].abs() > 0.9
        axis[:, 0] = torch.where(flip, 0.0, 1.0)
        axis[:, 1] = torch.where(flip, 1.0, 0.0)
        t = _unit(torch.linalg.cross(mu, axis))
        s = (1.0 - c * c).clamp_min(0.0).sqrt()[:, None]
        return _unit(s * (phi.cos()[:, None] * t + phi.sin()[:, None] * torch.linalg.cross(mu, t)) + c[:, None] * mu)

    def records(self, seed, stream, n, frame=0, volume=0.0):
        """n training records (40 bytes each) as a (n, 10) tensor of 32-bit words."""
        g = _gen(seed, stream)
        out = torch.zeros(n, 10, device="cuda")
        pos, blob = self.positions(g, n, frame)
        out[:, 0:3] = pos
        out[:, 3:6] = self.directions(g, blob)
        out[:, 6] = _randn(g, n).exp()
        out[:, 7] = 1.0 / (4.0 * math.pi)
        out[:, 8] = -torch.log1p(-_rand(g, n))
        if volume:
            out.view(torch.int32)[:, 9] = torch.where(_rand(g, n) < volume, 2, 0).to(torch.int32)
        return out

    def queries(self, seed, n, volume=0.0, knn=True):
        """Shading points with their outgoing normal or direction, random numbers and HG mean cosine."""
        g = _gen(seed, 900)
        q = {"pos": self.positions(g, n, loose=0.02)[0].contiguous(), "nrm": _unit(_randn(g, n, 3)).contiguous(),
             "u2": _rand(g, n, 2), "u1": _rand(g, n) if knn else None, "g": None, "vol": None}
        if volume:
            q["g"] = 1.8 * _rand(g, n) - 0.9
            q["vol"] = (_rand(g, n) < volume).to(torch.uint8)
        return q


def _paths(seed, stream, scene, count, length):
    """Recorded paths: vertices near the scene's blobs joined by their
    directions; diffuse, glossy and delta vertices, some refractive, some in a
    medium; sparse emission; Russian roulette after the third vertex.  (vertices
    as (n, 34) 32-bit words of the 136-byte record, path offsets)"""
    g = _gen(seed, stream)
    lengths = _randint(_gen(length, stream), 0, length + 1, count)  # the same for every seed
    lengths[0] = length
    off = torch.zeros(count + 1, dtype=torch.int64, device="cuda")
    off[1:] = lengths.cumsum(0)
    n = int(off[-1])
    path = torch.repeat_interleave(torch.arange(count, device="cuda"), lengths)
    at = torch.arange(n, device="cuda")
    depth = at - off[path]
    last = depth == lengths[path] - 1
    pos = scene.centre[_randint(g, 0, scene.blobs, n)] + 0.08 * _randn(g, n, 3)
    loose = _randn(g, n, 3)
    v = torch.zeros(n, 34, device="cuda")
    v[:, 0:3] = pos
    v[:, 3:6] = _unit(torch.where(last[:, None], loose, pos[torch.where(last, at, at + 1)] - pos))
    v[:, 6:9] = _unit(torch.where((depth == 0)[:, None], loose, pos[(at - 1).clamp_min(0)] - pos))
    v[:, 9:12] = _unit(_randn(g, n, 3))
    delta = _rand(g, n) < 0.15
    words = v.view(torch.int32)
    words[:, 12] = (_rand(g, n) < 0.2).to(torch.int32)
    v[:, 13] = torch.exp(math.log(0.01) + math.log(500.0) * _rand(g, n))
    words[:, 14] = delta.to(torch.int32)
    v[:, 15:18] = 1.5 * _rand(g, n, 3)
    v[:, 18:21] = torch.where(_rand(g, n, 1) < 0.7, 1.0, 0.3 + 0.7 * _rand(g, n, 3))
    v[:, 21:24] = 4.0 * _rand(g, n, 3) * (_rand(g, n, 1) < 0.2)
    v[:, 24] = _rand(g, n)
    v[:, 25:28] = 2.0 * _rand(g, n, 3) * (_rand(g, n, 1) < 0.3)
    rr = torch.where(depth < 3, 1.0, 0.2 + 0.8 * _rand(g, n))
    v[:, 28] = torch.where((depth >= 3) & (_rand(g, n) < 0.05), 0.0, rr)
    v[:, 29] = torch.where(delta & (_rand(g, n) < 0.5), 1.5, 1.0)
    v[:, 30] = torch.where(_rand(g, n) < 0.1, 0.005, _rand(g, n))
    return v, off


# ----------------------------------------------------------------- the cases
_device = None


def _dev():
    global _device
    if _device is None:
        _device = pgl.Device()
    return _device


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def _field(leaf, deterministic=True, vmm=False):
    kind = pgl.PGL_DIRECTIONAL_DISTRIBUTION_VMM if vmm else pgl.PGL_DIRECTIONAL_DISTRIBUTION_PARALLAX_AWARE_VMM
    return pgl.Field(_dev(), max_samples_per_leaf=leaf, deterministic=deterministic, directional_type=kind)


def _query_outputs(n):
    return (torch.zeros(n, 3, device="cuda"), torch.zeros(n, device="cuda"),
            torch.zeros(n, dtype=torch.int32, device="cuda"), torch.zeros(n, device="cuda"))


def _sample_device(field, q, out):
    """pglFieldSampleBatchDevice: all arrays in device memory, queued on the default stream."""
    d, pdf, ids, integral = out
    field.lib.pglFieldSampleBatchDevice(field.h, len(pdf), _ptr(q["pos"]), _ptr(q["nrm"]), _ptr(q["g"]),
                                        _ptr(q["u2"]), _ptr(q["u1"]), _ptr(q["vol"]), _ptr(d), _ptr(pdf), _ptr(ids),
                                        _ptr(integral), None)
    return out


def _host(q):
    return {k: None if t is None else t.cpu().numpy() for k, t in q.items()}


def _trained(scene, seed, regions, volume, vmm=False):
    """A field of about `regions` regions of a kind, trained on two frames."""
    leaf = max(1000, min(32000, 400000 // regions))
    n = max(20000, leaf * regions // 4)
    field = _field(leaf, vmm=vmm)
    for frame in range(2):
        a = scene.records(seed, 20 + frame, n, frame)
        field.update_surface_device(a.data_ptr(), n)
        b = None
        if volume:
            b = scene.records(seed, 30 + frame, n, frame, volume=1.1)
            field.update_volume_device(b.data_ptr(), n)
        torch.cuda.synchronize()
    field.num_regions()
    return field


def prepare(case, seed):
    kind = case["kind"]
    scene = _Scene(seed)
    s = {"case": case, "kind": kind}
    if kind == "query":
        s["field"] = _trained(scene, seed, case["regions"], case["volume"], case["vmm"])
        s["q"] = scene.queries(seed, case["n"], case["volume"], case["knn"])
        s["out"] = _query_outputs(case["n"])
    elif kind == "serve":
        field = _trained(scene, seed, case["regions"], case["volume"])
        # sizes spread evenly over their logarithm, large and small in turn
        r = (7 * np.arange(case["requests"]) % 31 + 0.5) / 31.0
        sizes = np.floor(case["smallest"] * (case["largest"] / case["smallest"]) ** r).astype(np.int64)
        ends = np.cumsum(sizes)
        n = int(ends[-1])
        q = _host(scene.queries(seed, n, case["volume"], knn=False))
        q = {k: None if a is None else pinned_copy(a) for k, a in q.items()}
        out = (pinned_empty((n, 3), np.float32), pinned_empty(n, np.float32), pinned_empty(n, np.uint32),
               pinned_empty(n, np.float32))
        s["requests"] = []
        for a, b in zip(ends - sizes, ends):
            cut = {k: None if t is None else t[a:b] for k, t in q.items()}
            s["requests"].append((cut, tuple(o[a:b] for o in out)))
        s["out"] = out
        s["server"] = pgl.Server(field, memory_budget=1 << 29, slots=4)
    elif kind == "render":
        s["field"] = _field(case["leaf"])
        s["frames"] = []
        for frame in range(case["frames"]):
            rec = scene.records(seed, 40 + frame, case["n"], frame)
            s["frames"].append(pgl.SampleStorage(rec.cpu().numpy().view(SAMPLE_DTYPE).reshape(-1)))
        s["q"] = _host(scene.queries(seed, case["queries"]))
    elif kind in ("train", "route"):
        volume = case.get("volume", 0.0)
        s["field"] = _field(case["leaf"], case.get("deterministic", True), case.get("vmm", False))
        s["frames"] = [scene.records(seed, 40 + f, case["n"], f, volume) for f in range(case["frames"])]
        s["q"] = scene.queries(seed, case["queries"], volume)
        s["out"] = _query_outputs(case["queries"])
    elif kind == "path_train":
        s["field"] = _field(case["leaf"])
        s["frames"] = []
        for f in range(case["frames"]):
            v, off = _paths(seed, 60 + f, scene, case["paths"], case["length"])
            s["frames"].append((v, off.to(torch.int32)))
        s["q"] = scene.queries(seed, case["queries"], 0.2)
        s["out"] = _query_outputs(case["queries"])
    elif kind == "paths":
        v, off = _paths(seed, 60, scene, case["paths"], case["length"])
        s["paths"] = (v, off.to(torch.int32))
        s["surface"] = torch.zeros(len(v), 10, device="cuda")
        s["volume"] = torch.zeros(len(v), 10, device="cuda")
        s["batch"] = pgl.PathSegmentBatch()
    else:
        raise ValueError(kind)
    return s


def _tree(case, field, kind=0):
    """The kd tree's nodes, in arrays with room for the largest tree of the case."""
    pivots, dims, children = field.nodes(kind)
    room = 64 + 16 * case.get("n", 3 * case.get("paths", 0)) * case["frames"] // case["leaf"]
    out = np.zeros(room, np.float32), np.zeros(room, np.uint32), np.zeros(room, np.uint32)
    for o, a in zip(out, (pivots, dims, children)):
        o[:len(a)] = a
    return out


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "query":
        return _sample_device(s["field"], s["q"], s["out"])
    if kind == "serve":
        server = s["server"]
        ids = []
        for q, out in s["requests"]:
            rid, _ = server.submit(q["pos"], q["nrm"], q["u2"], g=q["g"], is_volume=q["vol"], out=out)
            ids.append(rid)
        server.drain()
        for rid in ids:
            server.release(rid)
        return s["out"]
    if kind == "paths":
        v, off = s["paths"]
        ns, nv = s["batch"].prepare_device(v.data_ptr(), len(v), off.data_ptr(), case["paths"],
                                           s["surface"].data_ptr(), len(v), s["volume"].data_ptr(), len(v),
                                           use_nee_mi_weights=case["nee"], guide_direct_light=case["direct"],
                                           rr_affects_direct=case["rr"])
        return {"surface": s["surface"][:, :9], "volume": s["volume"][:, :9], "counts": (ns, nv),
                "surface_flags": s["surface"].view(torch.int32)[:, 9],
                "volume_flags": s["volume"].view(torch.int32)[:, 9]}
    # a training session
    field = s["field"]
    field.reset()
    out = {}
    for f, frame in enumerate(s["frames"]):
        if kind == "render":
            q = s["q"]
            field.update(frame)
            out["queries%d" % f] = field.sample_batch(q["pos"], q["nrm"], q["u2"], u1=q["u1"])
        elif kind == "train":
            field.update_surface_device(frame.data_ptr(), len(frame))
        elif kind == "route":
            field.update_device(frame.data_ptr(), len(frame))
        else:
            v, off = frame
            field.update_from_path_segments_device(v.data_ptr(), len(v), off.data_ptr(), case["paths"])
    if kind != "render":
        out["queries"] = _sample_device(field, s["q"], s["out"])
    out["tree"] = _tree(case, field)
    if kind in ("route", "path_train"):
        out["volume_tree"] = _tree(case, field, 1)
    return out


# A query reads 36 bytes (position, normal, two random numbers, one for the
# neighbour pick) and writes 24; the mixture has about 12 components, a product,
# a share of the integral and a pdf term each (67 flops on a surface, 171 for
# the three lobes of a phase function).
def _query_work(n, volume):
    return 60.0 * n, n * (60.0 + 12.0 * (67.0 * (1.0 - volume) + 171.0 * volume))


def work(case):
    kind = case["kind"]
    if kind == "query":
        b, f = _query_work(case["n"], case["volume"])
    elif kind == "serve":
        lo, hi = case["smallest"], case["largest"]
        b, f = _query_work(case["requests"] * (hi - lo) / math.log(hi / lo), case["volume"])
    elif kind == "paths":
        n = 0.5 * case["paths"] * case["length"]
        b, f = n * (136.0 + 0.45 * 40.0), n * 0.25 * case["length"] * 30.0
    else:
        # a frame's records are read once, a query batch follows; the EM fit of a
        # sample takes about 100 evaluations of a component at 30 flops
        if kind == "path_train":
            v = 0.5 * case["paths"] * case["length"]
            per, b = 0.45 * v, 136.0 * v
        else:
            per, b = float(case["n"]), 40.0 * case["n"]
        f = per * 3100.0
        batches = case["frames"] if kind == "render" else 1
        qb, qf = _query_work(case["queries"], case.get("volume", 0.0))
        b, f = b * case["frames"] + qb * batches, f * case["frames"] + qf * batches
    return {"bytes": b, "flops": f}


def exact(case, seed):
    """Training and what is sampled from a trained field have no 64-bit value
    (see above); the samples of recorded paths do."""
    if case["kind"] != "paths":
        return None
    v32, off = _paths(seed, 60, _Scene(seed), case["paths"], case["length"])
    n, words, v = len(v32), v32.view(torch.int32), v32.double()
    path = torch.repeat_interleave(torch.arange(case["paths"], device="cuda"), off[1:] - off[:-1])
    end = off[1:][path]
    at = torch.arange(n, device="cuda")
    delta, medium = words[:, 14] != 0, words[:, 12] != 0

    # distances: from a path's end backwards, carried through specular vertices
    distance = torch.zeros(n, dtype=torch.float64, device="cuda")
    carried = torch.zeros(n, dtype=torch.float64, device="cuda")  # what vertex i hands to vertex i - 1
    for back in range(2, case["length"] + 1):
        i = (off[1:] - back)[off[1:] - back >= off[:-1]]
        a, b = v[i], v[i + 1]
        d = ((b[:, 0:3] - a[:, 0:3]).norm(dim=1) + carried[i + 1]).clamp_max(2e6)
        distance[i] = d
        bend = ((a[:, 9:12] * a[:, 6:9]).sum(1) / ((a[:, 9:12] * a[:, 3:6]).sum(1) * a[:, 29])).abs()
        rough = ~delta[i] & (v32[i, 30] >= torch.tensor(0.3, device="cuda"))
        carried[i] = torch.where(rough, 0.0, torch.where(a[:, 29] != 1.0, d * bend, d))

    # radiance carried back to vertex i from the later vertices of its path
    light = torch.zeros(n, 3, dtype=torch.float64, device="cuda")
    t = torch.ones(n, 3, dtype=torch.float64, device="cuda")
    before = torch.ones(n, 1, dtype=torch.float64, device="cuda")
    for step in range(1, case["length"]):
        i = at[at + step < end]
        w = v[i + step]
        ti = t[i] * v[i + step - 1, 18:21]
        ct = ti.clamp_max(10.0)
        direct = w[:, 21:24] if case["rr"] else w[:, 21:24] * before[i]
        add = ct * w[:, 25:28]
        if step == 1 and not case["nee"]:
            if case["direct"]:
                add = add + ct * direct
        elif step > 1 or case["direct"]:
            add = add + ct * w[:, 24:25] * direct
        light[i] += add
        rr = w[:, 28:29]
        t[i] = torch.where(rr > 0.0, ti * w[:, 15:18] / rr, 0.0)
        before[i] = rr

    keep = ~delta & (v32[:, 30] > torch.tensor(0.01, device="cuda")) & (at + 1 < end)
    keep &= (light > 0.0).any(1) & (distance > 0.0)
    pdf = torch.maximum(v[:, 13], torch.tensor(0.1, device="cuda").double())
    rec = torch.cat([v[:, 0:6], (light.sum(1) / 3.0 / pdf)[:, None], pdf[:, None], distance[:, None]], 1)
    order = torch.argsort(path * (case["length"] + 1) + (end - 1 - at))  # paths in order, each from its end
    out = {"counts": (None, None), "surface_flags": None, "volume_flags": None}
    for name, side in (("surface", ~medium), ("volume", medium)):
        i = order[(keep & side)[order]]
        out[name] = torch.zeros_like(rec)  # the records, then the buffer's unused end
        out[name][:len(i)] = rec[i]
    return out
