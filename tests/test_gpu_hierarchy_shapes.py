"""Steps over hierarchies refined in x, y and z: an L of refined columns, so
that level changes cross x, y and z faces, the refined region has convex
and re-entrant edges and corners, some leaves compute edge or corner sectors
of their own, and some have only an edge without a leaf of their level
across; outflow, periodic and reflecting domain faces in each dimension."""
import numpy as np
import pytest

from sparkhip import capi, problems
import pyoracle

pytestmark = pytest.mark.gpu

BC = problems.BC_OUTFLOW, problems.BC_PERIODIC, problems.BC_REFLECT


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield


def lshape(bc, columns, n=10, nguard=10, **kw):
    """4 x 4 x 3 level-1 blocks of n^3; the blocks of three columns (an L in
    x-y) refined, over all of z (columns) or in the middle layer."""
    nb0 = (4, 4, 3)
    cfg = problems.base_cfg(**{**dict(ndim=3, nguard=nguard, nscalars=2, flux_correct=1, cfl=0.3), **kw})
    w = 1.0 / nb0[0]

    def refine(L, lo, hi):
        i, j, k = (round(x / w) for x in lo)
        return L == 1 and (i, j) in ((1, 1), (2, 1), (1, 2)) and (columns or k == 1)

    blocks, arrays, origins = [], [], []
    for L, b in problems.amr_leaves(nb0, n, 2, refine, nguard):
        dx = w / n / 2 ** (L - 1)
        blk = dict(nx=n, ny=n, nz=n, level=L, dx=dx, dy=dx, dz=dx)
        NZ, NY, NX = problems.gc_shape(cfg, blk)
        Z, Y, X = problems._centers(cfg, blk, tuple(q * n * dx for q in b), NZ, NY, NX)
        s = np.sin(2 * np.pi * X + 1) * np.cos(2 * np.pi * Y) + 0.5 * np.sin(8 * Z + 3 * X)
        hot = (X - 0.45) ** 2 + (Y - 0.4) ** 2 + (Z - 0.4) ** 2 < 0.03
        U = np.zeros((NZ, NY, NX, capi.SPARK_NPROP + cfg["nscalars"]))
        problems.fill_thermo(U, 1.0 + 0.3 * s, np.where(hot, 8.0, 1.0) + 0.1 * s, 0.3 * s, -0.2 * s, 0.25 * np.cos(5 * X),
                             1.4, scalars=[0.5 + 0.4 * np.sin((q + 2) * X + Z + Y) for q in range(cfg["nscalars"])])
        blocks.append(blk)
        arrays.append(U)
        origins.append([q * n for q in b])
    return problems.Problem("lshape", cfg, blocks, arrays,
                            info=dict(nb0=nb0, origins=np.asarray(origins, dtype=np.int32), bc=bc))


def run(prob, nsteps, form, **options):
    b = capi.Batch(dict(prob.cfg, form=form), prob.blocks)
    try:
        for k, v in options.items():
            b.set_option(k, v)
        b.pack(prob.arrays)
        b.set_amr_grid(prob.info["nb0"], prob.info["origins"], prob.info["bc"])
        dts = b.advance(nsteps)
        out = [a.copy() for a in prob.arrays]
        b.unpack(out, interior_only=True)
    finally:
        b.close()
    return dts, out


CASES = [((BC[0], BC[2], BC[1]), True), ((BC[1], BC[0], BC[2]), False), ((BC[2], BC[1], BC[0]), False)]


@pytest.mark.parametrize("hybrid", [0, 1])
@pytest.mark.parametrize("bc,columns", CASES)
def test_same_level_halos_equal_telescoping(bc, columns, hybrid):
    prob = lshape(bc, columns, use_hybrid_riemann=hybrid)
    levels = [b["level"] for b in prob.blocks]
    assert levels.count(2) == (72 if columns else 24) and levels.count(1) == (39 if columns else 45)
    res = {}
    for form in ("plain_fp64", "batched_fp64", "fp32_flux"):
        d_on, on = run(prob, 3, form)
        d_off, off = run(prob, 3, form, same_level_halos=0)
        assert np.array_equal(d_on, d_off)
        for x, y in zip(on, off):
            assert np.array_equal(x, y), form
        res[form] = d_on, on
    assert np.array_equal(res["plain_fp64"][0], res["batched_fp64"][0])
    for x, y in zip(res["plain_fp64"][1], res["batched_fp64"][1]):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("bc,columns", CASES)
def test_plain_steps_match_the_oracle(bc, columns):
    prob = lshape(bc, columns, use_hybrid_riemann=1)
    d, out = run(prob, 2, "plain_fp64")
    ref = [a.copy() for a in prob.arrays]
    dref, nerr = pyoracle.amr_advance(prob.cfg, prob.blocks, prob.info["nb0"], prob.info["origins"], ref, 2, bc=bc)
    assert nerr == 0 and np.array_equal(d, dref)
    inner = (slice(10, -10),) * 3
    for x, y in zip(out, ref):
        assert np.array_equal(x[inner], y[inner])
