"""WENO5 of the FP64 sweeps on values at and beyond the range in which the
weights take quotients without scaling, against the oracle's IEEE divides
(bit for bit, NaN where the oracle has NaN)."""
import math

import numpy as np
import pytest

from sparkhip import capi, problems
import pyoracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield


def compare(prob, nsteps, form="plain_fp64"):
    b = capi.Batch(dict(prob.cfg, form=form), prob.blocks)
    try:
        b.pack(prob.arrays)
        d = b.advance(nsteps)
        out = [a.copy() for a in prob.arrays]
        b.unpack(out)
    finally:
        b.close()
    ref = [a.copy() for a in prob.arrays]
    dref, _ = pyoracle.batch_advance(prob.cfg, prob.blocks, ref, nsteps)
    assert np.array_equal(d, dref)
    g = prob.cfg["nguard"]
    inner = tuple(slice(g, -g) if n > 1 else slice(None) for n in prob.arrays[0].shape[:3])
    for q in range(prob.arrays[0].shape[-1]):
        nd = sum(int(np.count_nonzero(~((x[inner][..., q] == y[inner][..., q])
                                        | (np.isnan(x[inner][..., q]) & np.isnan(y[inner][..., q])))))
                 for x, y in zip(out, ref))
        assert nd == 0, f"variable {q}: {nd} differing values"
    return [a[inner] for a in ref]


@pytest.mark.parametrize("form", ["plain_fp64", "batched_fp64"])
def test_scalars_of_every_magnitude(form):
    """Indicators far below the 1e-36 added to them, ordinary, on both sides
    of 2^900, constants far above, one whose fourfold overflows although its
    threefold does not."""
    scales = (1e-170, 1.0, 1e100, 2.0 ** 448, 2.0 ** 452, 2.0 ** 999, 2.0 ** 1001, 1.25 * 2.0 ** 1022)
    prob = problems.batched(nblocks=6, nguard=10, sizes=(8, 16), probs=(0.5, 0.5), shock_every=2, nscalars=len(scales))
    r = np.random.default_rng(5)
    for a in prob.arrays:
        for q, s in enumerate(scales):
            vary = 0.0 if s >= 2.0 ** 999 else 0.5
            a[..., capi.SPARK_NPROP + q] = s * (1.0 + vary * r.random(a.shape[:-1]))
    ref = compare(prob, 2, form)
    assert all(np.isfinite(x[..., : capi.SPARK_NPROP + 4]).all() for x in ref)


@pytest.mark.parametrize("n", [(64, 4, 1), (128, 4, 1), (8, 8, 4), (16, 8, 6)])
def test_slopes_hidden_by_rounding(n):
    """A scalar that falls and rises by one ulp a cell around each block's
    last interior cell in y (2D) or z (3D): there 3 u0 rounds the one-sided
    slopes away, beta1 = beta3 = 0, and beta2 overflows.  The cells beside it
    come out NaN in the reference too, so the flux through the block's high
    face, which takes that cell's state, is compared, after the first stage.
    Cells of one position along a y or z pencil fill whole waves, so no other
    lane takes the wave off the short quotients."""
    u0 = float.fromhex("0x1.f4d1520de9a2ap+790")
    ndim = 2 if n[2] == 1 else 3
    cfg = problems.base_cfg(ndim=ndim, nguard=6, rk_order=2, nscalars=1, cfl=0.3, flux_correct=1)
    blk = dict(nx=n[0], ny=n[1], nz=n[2], level=1, dx=0.1, dy=0.1, dz=0.1)
    shape = problems.gc_shape(cfg, blk)
    axis = 1 if ndim == 2 else 0
    line = u0 + np.abs(np.arange(shape[axis]) - (shape[axis] - 7)) * math.ulp(u0)
    U = np.zeros(shape + (capi.SPARK_NPROP + 1,))
    problems.fill_thermo(U, np.ones(shape), np.ones(shape), 0.1, 0.2, 0.3, 1.4,
                         scalars=[np.broadcast_to(line[:, None, None] if axis == 0 else line[None, :, None], shape)])
    dt = 1e-3
    e = [(n[2] + (d == 2), n[1] + (d == 1), n[0] + (d == 0), 6) for d in range(3)]
    b = capi.Batch(cfg, [blk])
    try:
        b.pack([U])
        b.step_begin()
        b.stage(1, dt, 0)
        regs = [[np.zeros(x)] for x in e]
        b.get_flux_registers(*regs)
    finally:
        b.close()
    ref = [np.zeros(x) for x in e]
    pyoracle.shock_detect(cfg, blk, U)
    assert pyoracle.stage(cfg, blk, U, U.copy(), 1, 0, dt, fb=ref) == 0
    d = 2 if ndim == 3 else 1
    high = (-1, slice(None), slice(None), 5) if ndim == 3 else (slice(None), -1, slice(None), 5)
    got, want = regs[d][0][high], ref[d][high]
    assert np.isfinite(want).all() and np.all(want != 0.0)
    assert np.array_equal(got, want)


def test_values_whose_fourfold_overflows():
    """A uniform flow with a constant scalar above 2^1022: 4 u overflows where
    3 u does not, so the reference's indicators are infinite and its face
    states NaN."""
    cfg = problems.base_cfg(ndim=2, nguard=10, nscalars=3, cfl=0.3)
    blk = dict(nx=16, ny=8, nz=1, level=1, dx=0.1, dy=0.1, dz=0.1)
    shape = problems.gc_shape(cfg, blk)
    U = np.zeros(shape + (capi.SPARK_NPROP + 3,))
    problems.fill_thermo(U, np.ones(shape), 1.0, 0.1, 0.2, 0.0, 1.4, scalars=[2.0 ** 999, 2.0 ** 1001, 1.25 * 2.0 ** 1022])
    ref = compare(problems.Problem("constant", cfg, [blk], [U]), 1)[0]
    assert np.isfinite(ref[..., : capi.SPARK_NPROP + 2]).all() and np.isnan(ref[..., -1]).all()
