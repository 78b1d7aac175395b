"""The batched FP64 form against the oracle: it runs the plain form's sweeps,
so comparing the two says nothing about either."""
import numpy as np
import pytest

from sparkhip import capi, problems
import pyoracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield


CASES = {
    "mixed": lambda: problems.batched(nblocks=12, nguard=10, shock_every=4),
    "scalars_gravity": lambda: problems.batched(nblocks=8, nguard=10, sizes=(8, 16), probs=(0.5, 0.5), shock_every=2,
                                                nscalars=8, use_gravity=1, grav=(0.0, 0.0, -1.0)),
    "plm_hll_rk2": lambda: problems.batched(nblocks=8, nguard=6, sizes=(8, 16), probs=(0.5, 0.5), shock_every=2,
                                            recon="plm", riemann="hll", rk_order=2, nstencil=2),
    "refill": lambda: problems.sedov3d(nb=4, n=16, nguard=6, guard_mode="refill"),
    "refill_hybrid": lambda: problems.sedov3d(nb=4, n=16, nguard=6, guard_mode="refill", use_hybrid_riemann=1,
                                              center=(1.0 / 64, 0.5, 0.5), r_cells=4.0),
    "telescope_hybrid": lambda: problems.sedov3d(nb=2, n=16, nguard=10, use_hybrid_riemann=1,
                                                 center=(1.0 / 32, 0.5, 0.5), r_cells=4.0),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_batched_fp64_steps_match_the_oracle(case):
    prob = CASES[case]()
    b = capi.Batch(dict(prob.cfg, form="batched_fp64"), prob.blocks)
    try:
        b.pack(prob.arrays)
        if prob.ug is not None:
            b.set_uniform_grid(*prob.ug)
        d = b.advance(3)
        out = [a.copy() for a in prob.arrays]
        b.unpack(out)
    finally:
        b.close()
    ref = [a.copy() for a in prob.arrays]
    if prob.ug is not None:
        dref, nerr = pyoracle.ug_advance(prob.cfg, prob.blocks[0], prob.ug, ref, 3,
                                         refill=prob.cfg["guard_mode"] == "refill")
    else:
        dref, nerr = pyoracle.batch_advance(prob.cfg, prob.blocks, ref, 3)
    assert nerr == 0 and np.array_equal(d, dref)
    g = prob.cfg["nguard"]
    inner = (slice(g, -g),) * 3
    for x, y in zip(out, ref):
        assert np.array_equal(x[inner], y[inner])


def test_batched_fp64_registers_match_the_oracle():
    """Flux registers of one step of independent blocks."""
    prob = problems.batched(nblocks=4, nguard=10, sizes=(8, 16), probs=(0.5, 0.5), shock_every=2, nscalars=2,
                            flux_correct=1)
    nf, dt = 7, 1e-4
    shape = [[(k["nz"] + (d == 2), k["ny"] + (d == 1), k["nx"] + (d == 0), nf) for k in prob.blocks] for d in range(3)]
    got = [[np.zeros(s) for s in shape[d]] for d in range(3)]
    b = capi.Batch(dict(prob.cfg, form="batched_fp64"), prob.blocks)
    try:
        b.pack(prob.arrays)
        b.hydro_step(dt)
        b.get_flux_registers(*got)
    finally:
        b.close()
    for i, blk in enumerate(prob.blocks):
        fb = [np.zeros(shape[d][i]) for d in range(3)]
        assert pyoracle.hydro_block(prob.cfg, blk, prob.arrays[i].copy(), dt, fb=fb) == 0
        for d in range(3):
            axis = 2 - d
            for side in (0, -1):
                face = tuple(side if a == axis else slice(None) for a in range(3))
                assert np.array_equal(got[d][i][face], fb[d][face])
                assert np.any(fb[d][face] != 0.0)
