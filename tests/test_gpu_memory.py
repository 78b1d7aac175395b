"""Device memory of a batch."""
import ctypes

import numpy as np
import pytest

from sparkhip import capi, problems

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield


def free_bytes():
    """Free memory of the device (the HIP runtime the library is linked to)."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert capi.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("form", ["plain_fp64", "batched_fp64", "fp32_flux"])
def test_a_batch_holds_three_states_and_one_field(form):
    """No form holds more than the solution, two stage states and the
    flattening field over its boxes: rows of at most a third more than their
    cells, and 16 MiB beside them."""
    cfg = problems.base_cfg(nscalars=8, form=form)
    blocks = [dict(nx=16, ny=16, nz=16, level=1, dx=1.0, dy=1.0, dz=1.0)] * 48
    capi.Batch(cfg, blocks[:1]).close()  # the library's own first allocations
    before = free_bytes()
    b = capi.Batch(cfg, blocks)
    try:
        used = before - free_bytes()
    finally:
        b.close()
    fields = 3 * (capi.SPARK_NPROP + 8) + 1
    packed = len(blocks) * 36 ** 3 * fields * 8
    print(f"{form}: {used / packed:.3f} of the packed state", flush=True)
    assert used <= packed * 4 / 3 + (16 << 20)
    assert used >= packed


def test_stage_state_fields_outside_the_update_stay_as_they_were():
    """The sweeps keep their divergence terms in the stage buffers; the fields
    that no stage writes (game, shok, temp) of the stage state stay 0."""
    for kw in (dict(), dict(rk_order=2)):
        prob = problems.batched(nblocks=4, nguard=10, sizes=(8,), probs=(1.0,), nscalars=5, **kw)
        b = capi.Batch(prob.cfg, prob.blocks)
        try:
            b.pack(prob.arrays)
            b.advance(2)
            star = [np.full_like(a, np.nan) for a in prob.arrays]
            b.unpack(star, which=1)
        finally:
            b.close()
        for a in star:
            for v in ("game", "shok", "temp"):
                assert np.all(a[..., capi.VI[v]] == 0.0)
            assert np.all(a[10:-10, 10:-10, 10:-10, capi.VI["dens"]] > 0.0)
