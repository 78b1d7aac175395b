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


@pytest.fixture
def scarce():
    """scarce(n): takes all of the device's memory but n bytes (not touched)."""
    held = ctypes.c_void_p()

    def take(leave):
        assert not held and capi.lib().hipMalloc(ctypes.byref(held), ctypes.c_size_t(free_bytes() - leave)) == 0

    yield take
    if held:
        assert capi.lib().hipFree(held) == 0


def run(prob, form, take=None):
    """dts, solution, stage state and the share of the packed states a batch takes."""
    fields = 3 * (capi.SPARK_NPROP + prob.cfg["nscalars"]) + 1
    packed = sum(int(np.prod(a.shape[:3])) for a in prob.arrays) * fields * 8
    capi.Batch(dict(prob.cfg, form=form), prob.blocks[:1]).close()  # the library's own first allocations
    if take:
        take(packed * 23 // 20 + (64 << 20))
    before = free_bytes()
    b = capi.Batch(dict(prob.cfg, form=form), prob.blocks)
    try:
        share = (before - free_bytes()) / packed
        b.pack(prob.arrays)
        dts = b.advance(2)
        out = []
        for which in (0, 1):
            out.append([np.empty_like(a) for a in prob.arrays])
            b.unpack(out[-1], which=which)
    finally:
        b.close()
    return dts, out, share


@pytest.mark.parametrize("form,rk", [("plain_fp64", 3), ("batched_fp64", 2), ("fp32_flux", 3)])
def test_batches_fit_wherever_their_packed_states_do(form, rk, scarce):
    """With little more memory free than three packed states and one field take,
    a batch holds just those (no padding, no pool for the divergence terms, which
    go into the stage buffers) and computes what it computes with all of the
    GPU free, stage state included."""
    prob = problems.batched(nblocks=24, nguard=10, sizes=(16, 32), probs=(0.5, 0.5), shock_every=2, nscalars=5, rk_order=rk)
    d0, o0, s0 = run(prob, form)
    d1, o1, s1 = run(prob, form, scarce)
    print(f"{form}: {s0:.3f} and {s1:.3f} of the packed states", flush=True)
    assert s0 > 1.2 and s1 < 1.05
    assert np.array_equal(d0, d1)
    for x, y in zip(o0[0] + o0[1], o1[0] + o1[1]):
        assert np.array_equal(x, y)


def test_stage_state_fields_outside_the_update_stay_as_they_were():
    """The fields that no stage writes (game, shok, temp) of the stage state
    stay 0."""
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
