"""spark_pack / spark_unpack at the limits of a chunk: more blocks than a chunk
has segments, and more data than the staging slots hold at once, so that chunks
are cut by the size of a slot and slots are used again within a call."""
import numpy as np
import pytest

from sparkhip import capi, problems

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield


@pytest.mark.parametrize("ndim,shape,count,extra", [
    (1, (1, 1, 1), 2500, 0),   # interior unpack: 2500 segments of one cell in less than one chunk's cells
    (3, (16, 16, 16), 20, 0),  # 100 MB of whole tuples: chunks of one 8 MiB slot
    (3, (17, 16, 15), 20, 3),  # the same with unk slots that are no variable
])
def test_round_trip(ndim, shape, count, extra):
    nunk = capi.SPARK_NPROP + 3 + extra
    r = np.random.default_rng(7)
    slots = r.permutation(nunk)[: capi.SPARK_NPROP + 3]
    var_index = list(slots) + [0] * (capi.SPARK_MAX_SCALARS - 3)
    cfg = problems.base_cfg(ndim=ndim, nguard=10, nscalars=3, nunk_vars=nunk, var_index=var_index)
    blocks = [dict(nx=shape[0], ny=shape[1], nz=shape[2], level=1, dx=1.0, dy=1.0, dz=1.0)] * count
    arrays = [r.random(problems.gc_shape(cfg, blocks[0]) + (nunk,)) for _ in blocks]
    inner = tuple(slice(10, -10) if d < ndim else slice(None) for d in (2, 1, 0))
    b = capi.Batch(cfg, blocks)
    try:
        b.pack(arrays)
        full = [np.full_like(a, np.nan) for a in arrays]
        part = [np.full_like(a, np.nan) for a in arrays]
        b.unpack(full)
        b.unpack(part, interior_only=True)
    finally:
        b.close()
    for a, f, p in zip(arrays, full, part):
        want = np.full_like(a, np.nan)
        want[..., slots] = a[..., slots]
        assert np.array_equal(f, want, equal_nan=True)
        inside = np.full_like(a, np.nan)
        inside[inner] = want[inner]
        assert np.array_equal(p, inside, equal_nan=True)
