"""The query kernel for surface batches against the one for mixed batches: the
same surface queries give the same bits from both, and from every batch size,
also where a lobe is far away, the cosine product is tiny, or nothing was
trained; and a query's result does not depend on its neighbours in the wave.
"""
import numpy as np
import pytest

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
    pos[7::89] *= np.float32(1e19)  # the parallax distances over- and underflow
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
