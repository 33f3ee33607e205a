"""The region kernel at the edges of its loops: sample counts around a wave, a
workgroup and a chunk, component counts of every number of groups, directions
on both sides of the length from which the exponent itself is bounded, and
launches on either side of the default grid's rule.

Against the oracle (as the batched launch, tests/parity_checks.py) and bit for
bit between schedules: how a region's samples are shared out changes no result.
"""
import numpy as np
import pytest

from field_compare import unit_dirs
from parity_checks import assert_mixture_parity
from test_gpu_batch import _oracle_regions, _state
from openpgl_amd.synth import batched_regions

pytestmark = pytest.mark.gpu

EDGES = [64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2047, 2048, 2049, 4097]


def _regions(counts, ks, seed):
    """region r: the first counts[r] of its samples, ks[r] initial components"""
    n = int(max(counts))
    full, have, _, _ = batched_regions(len(counts), seed=seed, nmin=n, nmax=n + 0.5)
    assert (have == n).all()
    recs = np.concatenate([full[r * n:r * n + c] for r, c in enumerate(counts)])
    stats = np.zeros((len(counts), 7), np.float32)
    at = 0
    for r, c in enumerate(counts):
        p = recs["pos"][at:at + c].astype(np.float64)
        stats[r, 0:3] = p.mean(axis=0)
        stats[r, 3:6] = ((p - p.mean(axis=0)) ** 2).sum(axis=0)
        stats[r, 6] = c
        at += c
    return recs, np.asarray(counts, np.uint32), stats, np.asarray(ks, np.uint32)


def _run(recs, counts, stats, init_k, deterministic=True, **schedule):
    import openpgl_amd as pgl
    from openpgl_amd.hip_runtime import DeviceArray
    batch = pgl.RegionBatch(pgl.Device(), max_samples_per_leaf=32000, deterministic=deterministic)
    if schedule:
        batch.set_schedule(**schedule)
    print("regions", len(counts), "samples", len(recs), "schedule", schedule, flush=True)
    batch.samples = DeviceArray.from_numpy(recs)  # kept with the batch, which reads it after the call
    batch.step_device(batch.samples.value, counts, stats, init_k)
    return batch


@pytest.mark.parametrize("k", [8, 9, 12, 16, 20, 24, 28, 31, 32])
def test_sample_counts_and_groups(k):
    recs, counts, stats, init_k = _regions(EDGES, [k] * len(EDGES), seed=40 + k)
    batch = _run(recs, counts, stats, init_k)
    records = [batch.region(r) for r in range(len(counts))]
    o32 = _oracle_regions(recs, counts, stats, init_k, [(recs, stats)], 0)
    o64 = _oracle_regions(recs, counts, stats, init_k, [(recs, stats)], 1)
    assert_mixture_parity(records, [o.record() for o in o32], [o.record() for o in o64], unit_dirs(512), "K %d" % k)
    assert _state(batch) == _state(_run(recs, counts, stats, init_k, per_region_launches=1))
    assert _state(batch) == _state(_run(recs, counts, stats, init_k, per_region_launches=0, balance=8.0, max_team=64))


def _odd_directions(scale, weight):
    """three regions; some samples of the middle one, in the second and fourth of
    its five chunks, have directions `scale` times a unit vector (at infinite
    distance, so that the reprojection keeps them)"""
    recs, c, stats, init_k = _regions([300, 5000, 300], [8, 20, 32], seed=7)
    recs = recs.copy()
    odd = 300 + np.array([1024 + 5, 1024 + 77, 3072 + 900, 3072 + 901, 3072 + 1023])
    recs["dir"][odd] *= np.float32(scale)
    recs["distance"][odd] = np.inf
    if weight is not None:
        recs["weight"][odd] = weight
    return recs, c, stats, init_k


@pytest.mark.parametrize("weight", [None, 0.0])
@pytest.mark.parametrize("scale", [1.5, 30.0, 1e13, 1e30, np.inf, np.nan])
def test_directions_out_of_range(scale, weight):
    """directions longer than one, on either side of the length from which a
    chunk takes the loops that bound the exponent itself: the same bits alone and
    in teams, the neighbours' bits unchanged"""
    plain = _state(_run(*_odd_directions(1.0, weight), deterministic=False))
    args = _odd_directions(scale, weight)
    ref = _state(_run(*args, deterministic=False, per_region_launches=1))
    assert ref[0] == plain[0] and ref[2] == plain[2]
    assert ref == _state(_run(*args, deterministic=False))
    assert ref == _state(_run(*args, deterministic=False, per_region_launches=0, balance=8.0, max_team=64))


def test_bounded_loops_equal_ordinary_ones():
    """Directions 1e11 times a unit vector take the ordinary loops and 1e13 times
    one the bounded loops, for every sample of their chunks; with weight 0 those
    samples count alike, as every lobe is saturated at both lengths, so the
    regions have the same bits, and finite ones."""
    for schedule in (dict(per_region_launches=1), dict(), dict(per_region_launches=0, balance=8.0, max_team=64)):
        a, b = (_run(*_odd_directions(scale, 0.0), deterministic=False, **schedule) for scale in (1e11, 1e13))
        assert _state(a) == _state(b)
        r = b.region(1)
        assert r["valid"] and r["K"] > 4
        for key in ("weights", "kappas", "meanDirections", "distances", "sumOfWeightedStats", "chiSquareMCEstimates"):
            assert np.all(np.isfinite(np.asarray(r[key]))), key


@pytest.mark.parametrize("counts", [[96 + r % 5 for r in range(511)], [96 + r % 5 for r in range(700)],
                                    [100000 + 777 * r for r in range(36)]])
def test_default_grid_rule(counts):
    """fewer and more regions than the default grid has workgroups, and more
    chunks than it takes at once, against a small fixed grid"""
    recs, c, stats, init_k = _regions(counts, [(8, 16, 32)[r % 3] for r in range(len(counts))], seed=3)
    assert _state(_run(recs, c, stats, init_k)) == _state(_run(recs, c, stats, init_k, grid=96))


@pytest.mark.parametrize("max_team", [16, 64, 65, 128, 200, 256, 1000])
@pytest.mark.parametrize("regions,samples", [(800, 96), (400, 8200)])
def test_default_grid_leaves_the_largest_team(max_team, regions, samples):
    """a batch of more regions, or more samples, than the default grid takes
    leaves as many of the resident workgroups as its largest team has, 64 at the
    least, down to the default grid (two of three workgroups of a compute unit)"""
    resident = _run(*_regions([96] * 800, [8] * 800, seed=5), grid=1 << 20).last_info()["grid"]
    batch = _run(*_regions([samples] * regions, [8] * regions, seed=5), max_team=max_team)
    assert batch.last_info()["grid"] == max(resident * 2 // 3, resident - max(64, max_team))


def test_default_grid_of_updates():
    """Updates of a field keep to the default grid, however many regions there
    are, and take the larger one for a first fit of many regions or for many
    samples."""
    import openpgl_amd as pgl
    from openpgl_amd.synth import generate
    f = pgl.Field(pgl.Device(), max_samples_per_leaf=200, deterministic=True)
    grids = []
    for frame in range(3):
        print("frame", frame, flush=True)
        f.update(pgl.SampleStorage(generate(200000, seed=1, frame=frame)))
        assert f.num_regions(0) > 1000
        grids.append(f.last_update_info()["grid"])
    resident = grids[0] + 64
    assert resident % 3 == 0 and grids[1:] == [resident * 2 // 3] * 2
    f = pgl.Field(pgl.Device(), deterministic=True)
    f.update(pgl.SampleStorage(np.tile(generate(200000, seed=1), 17)))
    assert f.num_regions(0) < 1000 and f.last_update_info()["grid"] == grids[0]
