"""The query kernel for surface batches against the one for mixed batches: the
same surface queries give the same bits from both, and from every batch size,
inside the field and outside it; and a query's result does not depend on its
neighbours in the wave.  Lengths and weights at the ends of the exponent range
give the bits that the same field gives in its middle.
"""
import numpy as np
import pytest

import field_file as ff
from openpgl_amd.synth import generate, queries

pytestmark = pytest.mark.gpu

SIZES = [1, 3, 4, 15, 16, 17, 63, 64, 65, 255, 256, 257, 1021]


def _bits(r):
    return [np.asarray(a).view(np.uint32) for a in r]


@pytest.mark.parametrize("leaf", [500, 4000])
def test_surface_kernel_equals_mixed_kernel(leaf):
    import openpgl_amd as pgl
    dev = pgl.Device()
    f = pgl.Field(dev, max_samples_per_leaf=leaf, deterministic=True)
    for frame in range(2):
        print("leaf", leaf, "frame", frame, flush=True)
        f.update(pgl.SampleStorage(generate(30000, seed=1, frame=frame)))
    assert len({f.region(i)["K"] for i in range(f.num_regions(0))}) > 2  # several numbers of groups
    n = max(SIZES)
    pos, nrm, u2, _, _ = queries(n, seed=9)
    u1 = np.random.Generator(np.random.PCG64(5)).random(n, np.float32)
    pos[5::97] *= np.float32(1e6)
    pos[7::89] *= np.float32(1e19)  # outside the field: no direction, no region
    nrm[11::83] *= np.float32(-1.0)
    for neighbours in (None, u1):
        whole = _bits(f.sample_batch(pos, nrm, u2, u1=neighbours))
        mixed = _bits(f.sample_batch(np.concatenate([pos, pos[:40]]), np.concatenate([nrm, nrm[:40]]),
                                     np.concatenate([u2, u2[:40]]),
                                     u1=None if neighbours is None else np.concatenate([u1, u1[:40]]),
                                     is_volume=np.repeat(np.uint8([0, 1]), [n, 40])))
        for a, b in zip(whole, mixed):
            assert np.array_equal(a, b[:n])
        for m in SIZES:
            part = _bits(f.sample_batch(pos[:m], nrm[:m], u2[:m], u1=None if neighbours is None else u1[:m]))
            for a, b in zip(whole, part):
                assert np.array_equal(a[:m], b), m


def _one_region(path, lengths=0, weights=0):
    """the field file `path` with one valid region per kind in bounds of +-1;
    every length and every component weight times a power of two"""
    d = ff.read_file(open(path, "rb").read(), 8)
    a, w = np.float32(2.0) ** np.float32(lengths), np.float32(2.0) ** np.float32(weights)
    for kind in ("surface", "volume"):
        f = d[kind]
        assert len(f["regions"]) == 1 and f["regions"][0]["valid"]
        r = f["regions"][0]
        assert r["K"] > 8
        rng = np.random.Generator(np.random.PCG64(1))
        r["distances"] = (0.05 * rng.random(32, np.float32) + np.float32(0.001)) * a
        r["weights"] = r["weights"] * w
        r["pivot"] = np.zeros(3, np.float32)
        f["treeBounds"] = tuple(float(v) for v in np.float32([-1, -1, -1, 1, 1, 1]) * a)
        f["sceneBounds"] = f["treeBounds"]
    return ff.write_file(d, 8)


@pytest.mark.parametrize("lengths", [-61, -50, -44, 30, 59, 61])
@pytest.mark.parametrize("weights", [0, -80, 70])
def test_ends_of_the_exponent_range(tmp_path, lengths, weights):
    """All lengths, or all component weights, of a field times a power of two:
    every step of a query scales exactly (the coordinates are of one size, so no
    square of one leaves the range alone), so directions and pdfs keep their bits
    where roots and quotients need their scaled forms too, and the integral
    follows the weights."""
    import openpgl_amd as pgl
    dev = pgl.Device()
    t = pgl.Field(dev, max_samples_per_leaf=32000, deterministic=True)
    t.update(pgl.SampleStorage(np.concatenate([generate(20000, seed=1), generate(20000, seed=2, flags=2)])))
    trained = str(tmp_path / "trained")
    assert t.store(trained)
    n = 4096
    rng = np.random.Generator(np.random.PCG64(7))
    pos = rng.uniform(0.3, 0.6, (n, 3)).astype(np.float32) * rng.choice(np.float32([-1, 1]), (n, 3))
    _, nrm, u2, _, g = queries(n, seed=9)
    mixed = (np.arange(n) % 3 == 0).astype(np.uint8)
    results = []
    for l, w in ((0, 0), (lengths, weights)):
        name = str(tmp_path / ("f%d_%d" % (l, w)))
        with open(name, "wb") as fh:
            fh.write(_one_region(trained, l, w))
        f = pgl.Field.from_file(dev, name)
        p = pos * np.float32(2.0) ** np.float32(l)
        print("lengths 2^%d weights 2^%d" % (l, w), flush=True)
        results.append((f.sample_batch(p, nrm, u2), f.sample_batch(p, nrm, u2, g=g, is_volume=mixed)))
    for (d0, p0, i0, s0), (d1, p1, i1, s1) in zip(*results):
        assert np.all(i0 == 0) and np.all(i1 == 0) and np.all(p0 > 0)
        assert np.array_equal(d0.view(np.uint32), d1.view(np.uint32))
        assert np.array_equal(p0.view(np.uint32), p1.view(np.uint32))
        assert np.array_equal((s0 * np.float32(2.0) ** np.float32(weights)).view(np.uint32), s1.view(np.uint32))


def test_untrained_field():
    """no direction, no pdf, no region from either kernel"""
    import openpgl_amd as pgl
    f = pgl.Field(pgl.Device())
    pos, nrm, u2, is_vol, g = queries(257, seed=3)
    for r in (f.sample_batch(pos, nrm, u2), f.sample_batch(pos, nrm, u2, g=g, is_volume=is_vol)):
        d, pdf, ids, integral = r
        assert not d.any() and not pdf.any() and not integral.any() and np.all(ids == 0xffffffff)
