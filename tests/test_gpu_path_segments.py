"""Batched path segments -> training samples on the GPU
(pglPathSegmentBatchPrepareSamplesDevice, pglFieldUpdateFromPathSegmentsDevice)
against the oracle's PathSegmentDataStorage::prepareSamples applied path by
path: the records must be identical bit for bit (same float operations, no
contraction), in per-path propagation order, surface and volume apart; a
field trained from path segments on the device must equal, state for state,
the field trained from the same samples through a host sample storage.
"""
import numpy as np
import pytest

from oracle_ctypes import oracle_path_samples
from openpgl_amd.synth import PATH_SEGMENT_DTYPE, SAMPLE_DTYPE, random_paths

pytestmark = pytest.mark.gpu


def _device_samples(batch, seg, off, **opt):
    from openpgl_amd.hip_runtime import DeviceArray
    dseg = DeviceArray.from_numpy(seg if len(seg) else np.zeros(1, PATH_SEGMENT_DTYPE))
    doff = DeviceArray.from_numpy(off)
    cap = max(1, len(seg))
    ds, dv = DeviceArray(cap * 40), DeviceArray(cap * 40)
    r = batch.prepare_device(dseg.value, len(seg), doff.value, len(off) - 1, ds.value, cap, dv.value, cap, **opt)
    assert r is not None
    ns, nv = r
    s = ds.to_numpy(SAMPLE_DTYPE, (ns,)) if ns else np.zeros(0, SAMPLE_DTYPE)
    v = dv.to_numpy(SAMPLE_DTYPE, (nv,)) if nv else np.zeros(0, SAMPLE_DTYPE)
    return s, v


@pytest.mark.parametrize("nee,guide,rr_direct,max_distance", [(False, False, True, 1e6), (True, False, True, 1e6),
                                                              (False, True, False, 2.0), (True, True, True, 0.5)])
def test_batch_equals_oracle(nee, guide, rr_direct, max_distance):
    import openpgl_amd as pgl
    seg, off = random_paths(40000, seed=7, max_len=16)
    print("paths", len(off) - 1, "vertices", len(seg), "options", nee, guide, rr_direct, max_distance, flush=True)
    batch = pgl.PathSegmentBatch()
    opt = dict(max_distance=max_distance, use_nee_mi_weights=nee, guide_direct_light=guide,
               rr_affects_direct=rr_direct)
    s, v = _device_samples(batch, seg, off, **opt)
    ws, wv = oracle_path_samples(seg, off, **opt)
    assert len(s) == len(ws) and len(v) == len(wv)
    assert len(s) > 1000 and len(v) > 100
    assert s.tobytes() == ws.tobytes()
    assert v.tobytes() == wv.tobytes()


def test_batch_long_and_empty_paths():
    """Paths reaching far beyond a 256-vertex tile (read from global memory
    past the staged vertices) and tiles holding more paths than the offsets
    kept in LDS (runs of empty paths) give the oracle's records too."""
    import openpgl_amd as pgl
    batch = pgl.PathSegmentBatch()
    seg, off = random_paths(300, seed=11, max_len=700)
    print("long paths", len(off) - 1, "vertices", len(seg), "longest", int(np.diff(off).max()), flush=True)
    s, v = _device_samples(batch, seg, off)
    ws, wv = oracle_path_samples(seg, off)
    assert len(s) == len(ws) and len(v) == len(wv) and len(s) > 1000
    assert s.tobytes() == ws.tobytes() and v.tobytes() == wv.tobytes()
    seg, off = random_paths(3000, seed=12, max_len=10)
    off2 = np.concatenate([np.repeat(off[:-1], 25), off[-1:]]).astype(np.uint32)  # 24 empty paths before each
    print("with empty paths", len(off2) - 1, "vertices", len(seg), flush=True)
    s, v = _device_samples(batch, seg, off2)
    ws, wv = oracle_path_samples(seg, off2)
    assert len(s) == len(ws) and len(v) == len(wv) and len(s) > 1000
    assert s.tobytes() == ws.tobytes() and v.tobytes() == wv.tobytes()


def test_batch_edge_cases():
    import openpgl_amd as pgl
    from openpgl_amd.hip_runtime import DeviceArray
    batch = pgl.PathSegmentBatch()
    # no paths; only empty and one-vertex paths
    s, v = _device_samples(batch, np.zeros(0, PATH_SEGMENT_DTYPE), np.zeros(1, np.uint32))
    assert len(s) == 0 and len(v) == 0
    seg, _ = random_paths(10, seed=1)
    one = seg[:3]
    off = np.array([0, 0, 1, 1, 2, 3, 3], np.uint32)
    s, v = _device_samples(batch, one, off)
    assert len(s) == 0 and len(v) == 0
    # too small an output: refused, nothing written
    seg, off = random_paths(2000, seed=2)
    ws, wv = oracle_path_samples(seg, off)
    dseg, doff = DeviceArray.from_numpy(seg), DeviceArray.from_numpy(off)
    ds, dv = DeviceArray(40 * len(ws)), DeviceArray(40 * len(wv))
    assert batch.prepare_device(dseg.value, len(seg), doff.value, len(off) - 1, ds.value, len(ws) - 1, dv.value,
                                len(wv)) is None
    # a range beyond the vertices (or a decreasing one): refused, nothing read
    assert batch.prepare_device(dseg.value, len(seg) - 1, doff.value, len(off) - 1, ds.value, len(ws), dv.value,
                                len(wv)) is None
    r = batch.prepare_device(dseg.value, len(seg), doff.value, len(off) - 1, ds.value, len(ws), dv.value, len(wv))
    assert r == (len(ws), len(wv))
    assert ds.to_numpy(SAMPLE_DTYPE, (len(ws),)).tobytes() == ws.tobytes()


def test_field_update_from_path_segments():
    """Three frames of path segments on the device train the field exactly as
    the same samples through a host sample storage do."""
    import openpgl_amd as pgl
    from openpgl_amd.hip_runtime import DeviceArray
    dev = pgl.Device()
    a = pgl.Field(dev, max_samples_per_leaf=2000)
    b = pgl.Field(dev, max_samples_per_leaf=2000)
    for frame in range(3):
        seg, off = random_paths(60000, seed=100 + frame, max_len=10)
        print("frame", frame, "paths", len(off) - 1, "vertices", len(seg), flush=True)
        dseg, doff = DeviceArray.from_numpy(seg), DeviceArray.from_numpy(off)
        a.update_from_path_segments_device(dseg.value, len(seg), doff.value, len(off) - 1)
        dseg.free()  # the path arrays are consumed when the call returns
        doff.free()
        ws, wv = oracle_path_samples(seg, off)
        st = pgl.SampleStorage(np.concatenate([ws, wv]))
        b.update(st)
        assert a.iteration() == b.iteration() == frame + 1
    assert a.num_regions(0) > 4 and a.num_regions(1) > 1
    assert a.compare(b)
    for kind in (0, 1):
        for i in range(0, a.num_regions(kind), 7):
            ra, rb = a.region(i, kind), b.region(i, kind)
            for key in ("K", "weights", "kappas", "meanDirections", "ssMean", "numSamplesThisUpdate"):
                assert np.array_equal(np.asarray(ra[key]), np.asarray(rb[key])), (kind, i, key)


@pytest.mark.parametrize("lengths", [[64, 65, 64], [8, 300, 8]])
def test_field_update_with_and_without_long_paths(lengths):
    """Frames whose longest path has lengths[frame] vertices, so that the one
    pass and the counting launches alternate on one field: the states of a field
    trained from the oracle's records of the same paths."""
    import openpgl_amd as pgl
    from openpgl_amd.hip_runtime import DeviceArray
    dev = pgl.Device()
    a = pgl.Field(dev, max_samples_per_leaf=2000)
    b = pgl.Field(dev, max_samples_per_leaf=2000)
    for frame, longest in enumerate(lengths):
        seg, off = random_paths(20000, seed=200 + frame, max_len=8)
        at = int(off[7000])  # one path of `longest` vertices, empty paths behind it
        off = np.where((off > at) & (off < at + longest), at + longest, off).astype(np.uint32)
        print("frame", frame, "vertices", len(seg), "longest", int(np.diff(off).max()), flush=True)
        assert longest <= np.diff(off).max() < longest + 8
        dseg, doff = DeviceArray.from_numpy(seg), DeviceArray.from_numpy(off)
        a.update_from_path_segments_device(dseg.value, len(seg), doff.value, len(off) - 1)
        ws, wv = oracle_path_samples(seg, off)
        b.update(pgl.SampleStorage(np.concatenate([ws, wv])))
        assert a.iteration() == b.iteration() == frame + 1
    assert a.num_regions(0) > 4 and a.num_regions(1) > 1
    assert a.compare(b)


def test_field_update_without_room_for_every_vertex():
    """Where outputs for every vertex cannot be allocated, the records are counted
    first: same states, whichever frames it happens in (the failure is set from
    the host, nothing runs out of memory)."""
    import openpgl_amd as pgl
    from openpgl_amd.hip_runtime import DeviceArray
    dev = pgl.Device()
    a, b = pgl.Field(dev, max_samples_per_leaf=2000), pgl.Field(dev, max_samples_per_leaf=2000)
    for frame, fail in enumerate((True, False, True, True, False)):
        seg, off = random_paths(10000 + 3000 * frame, seed=300 + frame, max_len=8)
        print("frame", frame, "vertices", len(seg), "no room" if fail else "", flush=True)
        dseg, doff = DeviceArray.from_numpy(seg), DeviceArray.from_numpy(off)
        for f in (a, b):
            if fail and f is a:
                f.debug_fail_next_path_outputs()
            f.update_from_path_segments_device(dseg.value, len(seg), doff.value, len(off) - 1)
        assert a.iteration() == b.iteration() == frame + 1
        assert a.validate() and a.compare(b)


_SHAPES = {
    "one vertex": ([1], 0, 0),
    "two vertices": ([2], 0, 0),
    "last path begins at a tile's last vertex": ([3] * 85 + [64] + [5] * 3, 0, 0),
    "paths end with the tiles": ([64] * 8, 0, 0),
    "longest one-pass path, then one more": ([64, 65, 7], 0, 0),
    "read-ahead ends inside a path": ([16] * 15 + [15, 17, 2], 0, 0),
    "vertices of no path": ([12] * 60, 300, 300),
    "long runs of them": ([12] * 60, 70 * 256, 70 * 256),
    "tiles of two passes of the sums": ([8] * (520 * 32), 0, 0),
    "most paths of a tile taken one by one": ([4] * 32 + [0] * 1984 + [4] * 112, 0, 0),
    "one more": ([4] * 32 + [0] * 1985 + [4] * 112, 0, 0),
    "a tile of empty paths, then a path into the next": ([0] * 3000 + [7] * 30 + [0] * 3000 + [64, 7], 11, 5),
}


@pytest.mark.parametrize("shape", list(_SHAPES))
def test_one_pass_equals_counting(shape):
    """Outputs with room for every vertex (one pass) and outputs of just the
    records' size (counting first) hold the oracle's records, bit for bit; with
    survival probabilities and throughputs from denormal to huge, where a
    quotient is not formed from a kept reciprocal."""
    import openpgl_amd as pgl
    from openpgl_amd.hip_runtime import DeviceArray
    lengths, lead, trail = _SHAPES[shape]
    n = lead + sum(lengths) + trail
    rng = np.random.Generator(np.random.PCG64([n, 99]))
    seg, _ = random_paths(n // 5 + 8, seed=31, max_len=12)
    seg = seg[:n].copy()
    assert len(seg) == n
    seg["roughness"] = np.maximum(seg["roughness"], 0.02)
    rr = "russianRouletteProbability"
    seg[rr] = rng.choice(np.array([1.0, 0.7, 0.95, 3e-39, 1e-30, 2e-18, 9e-19, 1e6, 2e6, 1e30], np.float32), n,
                         p=[.3, .3, .2] + [.2 / 7] * 7)
    seg["scatteringWeight"] *= rng.choice(np.array([1.0, 0.0, 1e-20, 1e-38, 1e25], np.float32), (n, 1),
                                          p=[.8, .05, .05, .05, .05])
    off = (lead + np.concatenate([[0], np.cumsum(lengths)])).astype(np.uint32)
    print(shape, "paths", len(lengths), "vertices", n, flush=True)
    batch = pgl.PathSegmentBatch()
    ws, wv = oracle_path_samples(seg, off)
    s, v = _device_samples(batch, seg, off)
    assert s.tobytes() == ws.tobytes() and v.tobytes() == wv.tobytes()
    dseg, doff = DeviceArray.from_numpy(seg), DeviceArray.from_numpy(off)
    ds, dv = DeviceArray(40 * max(1, len(ws))), DeviceArray(40 * max(1, len(wv)))
    r = batch.prepare_device(dseg.value, n, doff.value, len(lengths), ds.value, len(ws), dv.value, len(wv))
    assert r == (len(ws), len(wv))
    assert ds.to_numpy(SAMPLE_DTYPE, (len(ws),)).tobytes() == ws.tobytes()
    assert dv.to_numpy(SAMPLE_DTYPE, (len(wv),)).tobytes() == wv.tobytes()


def test_runs_of_empty_paths_cost_little():
    """Half a million empty paths between the paths of a small frame (rays that
    left the scene): the call stays in the time of the frame without them."""
    import time
    import openpgl_amd as pgl
    from openpgl_amd.hip_runtime import DeviceArray
    seg, off = random_paths(2000, seed=5, max_len=12)
    mid = len(off) // 2
    batch = pgl.PathSegmentBatch()
    best, counts = [], []
    for empty in (0, 500000):
        o = np.concatenate([off[:mid], np.full(empty, off[mid], np.uint32), off[mid:]]).astype(np.uint32)
        print("empty paths", empty, flush=True)
        n = len(seg)
        dseg, doff = DeviceArray.from_numpy(seg), DeviceArray.from_numpy(o)
        ds, dv = DeviceArray(40 * n), DeviceArray(40 * n)
        times = []
        for _ in range(20):
            t = time.perf_counter()
            r = batch.prepare_device(dseg.value, n, doff.value, len(o) - 1, ds.value, n, dv.value, n)
            times.append(time.perf_counter() - t)
        best.append(min(times))
        counts.append((r, ds.to_numpy(SAMPLE_DTYPE, (r[0],)).tobytes()))
    assert counts[0] == counts[1]
    assert best[1] < 4 * best[0], best
