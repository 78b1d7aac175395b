"""spark_pack / spark_unpack move exactly the cells and unk slots they are
given: through one chunk or many, with blocks split between chunks, with and
without unk slots that are no variable of the state."""
import numpy as np
import pytest

from sparkhip import capi, problems

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield


# shapes: one cell wide, below and above the size from which several threads
# and chunks are used, one block larger than a staging slot (8 MiB), many
# small blocks (more than one chunk's 1024 segments)
@pytest.mark.parametrize("ndim,shapes,extra,nscalars", [
    (1, [(1, 1, 1)], 0, 0),
    (1, [(37, 1, 1)] * 1100, 2, 3),
    (2, [(5, 9, 1), (16, 16, 1), (1, 7, 1)] * 3, 0, 2),
    (2, [(300, 301, 1)], 3, 0),
    (3, [(8, 8, 8), (13, 5, 9), (3, 4, 30)] * 2, 0, 8),
    (3, [(40, 37, 41), (8, 8, 8)], 0, 1),
    (3, [(17, 16, 15)] * 9, 4, 2),
])
def test_round_trip(ndim, shapes, extra, nscalars):
    nvar = capi.SPARK_NPROP + nscalars
    nunk = nvar + extra
    r = np.random.default_rng(11)
    slots = r.permutation(nunk)[:nvar]
    var_index = list(slots) + [0] * (capi.SPARK_NPROP + capi.SPARK_MAX_SCALARS - nvar)
    cfg = problems.base_cfg(ndim=ndim, nguard=10, nscalars=nscalars, nunk_vars=nunk, var_index=var_index)
    g = cfg["nguard"]
    blocks = [dict(nx=s[0], ny=s[1], nz=s[2], level=1, dx=1.0, dy=1.0, dz=1.0) for s in shapes]
    arrays = [r.random(problems.gc_shape(cfg, b) + (nunk,)) for b in blocks]
    inner = tuple(slice(g, -g) if d < ndim else slice(None) for d in (2, 1, 0))
    b = capi.Batch(cfg, blocks)
    try:
        for _ in range(2):  # the second pair reuses the staging area
            b.pack(arrays)
            full = [np.full_like(a, np.nan) for a in arrays]
            part = [np.full_like(a, np.nan) for a in arrays]
            b.unpack(full)
            b.unpack(part, interior_only=True)
            for a, f, p in zip(arrays, full, part):
                want = np.full_like(a, np.nan)
                want[..., slots] = a[..., slots]
                assert np.array_equal(f, want, equal_nan=True)
                inside = np.full_like(a, np.nan)
                inside[inner] = want[inner]
                assert np.array_equal(p, inside, equal_nan=True)
            arrays = [a + 1.0 for a in arrays]
    finally:
        b.close()
