"""Guard cells a call leaves in the blocks' own boxes (spark_unpack of whole
boxes): the guard fill of the last step's start in the solution, the
telescoped or refilled sectors in the stage state, also where the steps
themselves read halos from neighbouring blocks and fill none."""
import numpy as np
import pytest

from sparkhip import capi, problems
import pyoracle

pytestmark = pytest.mark.gpu

V = capi.VI
STATE = [V[n] for n in ("dens", "eint", "ener", "gamc", "pres", "velx", "vely", "velz")]
CALLS = {
    "hydro_step": lambda b: [b.hydro_step(0.5 * b.compute_dt()[0]) for _ in range(2)],
    "advance(3)": lambda b: b.advance(3),
    "advance(1) twice": lambda b: [b.advance(1) for _ in range(2)],
}


@pytest.fixture(scope="module", autouse=True)
def _device():
    capi.init(0)
    yield


def boxes(prob, form, call, **options):
    """Whole boxes of the solution and of the stage state after a call."""
    b = capi.Batch(dict(prob.cfg, form=form), prob.blocks)
    try:
        for k, v in options.items():
            b.set_option(k, v)
        b.pack(prob.arrays)
        if prob.ug is not None:
            b.set_uniform_grid(*prob.ug)
        else:
            b.set_amr_grid(prob.info["nb0"], prob.info["origins"], prob.info["bc"])
        CALLS[call](b)
        out = []
        for which in (0, 1):
            out.append([np.empty_like(a) for a in prob.arrays])
            b.unpack(out[-1], which=which)
    finally:
        b.close()
    return out


def within(prob, a, depth):
    g = prob.cfg["nguard"]
    return a[(slice(g - depth, a.shape[0] - g + depth),) * 3]


def bare_sectors(prob):
    """Per block the guard sectors (ox, oy, oz) with no leaf of its level across."""
    n, info = prob.blocks[0]["nx"], prob.info
    org = np.asarray(info["origins"]).reshape(-1, 3) // n
    at = {(b["level"],) + tuple(int(x) for x in o) for b, o in zip(prob.blocks, org)}
    out = []
    for b, o in zip(prob.blocks, org):
        nbl = [x << (b["level"] - 1) for x in info["nb0"]]
        bare = []
        for off in np.ndindex(3, 3, 3):
            q = [int(o[d]) + off[d] - 1 for d in range(3)]
            q = [x % m if bc == problems.BC_PERIODIC else x for x, m, bc in zip(q, nbl, info["bc"])]
            if (b["level"],) + tuple(q) not in at:
                bare.append(tuple(x - 1 for x in off))
        out.append(bare)
    return out


@pytest.mark.parametrize("call", sorted(CALLS))
@pytest.mark.parametrize("form,hybrid,rk", [("plain_fp64", 0, 3), ("plain_fp64", 1, 2), ("plain_fp64", 1, 3),
                                            ("batched_fp64", 0, 3), ("batched_fp64", 1, 3), ("fp32_flux", 0, 2),
                                            ("fp32_flux", 1, 3)])
def test_hierarchy_leaves_the_guards_of_telescoping(form, hybrid, rk, call):
    """Against SPARK_OPT_SAME_LEVEL_HALOS = 0, where every leaf telescopes over
    its own guard cells: all of them in the plain form, in the batched forms
    the sectors with no leaf of the block's level across."""
    prob = problems.rt_amr(nb0=(1, 1, 2), n=16, lmax=3, nscalars=2, rk_order=rk,
                           **(dict(use_hybrid_riemann=1, p_boost=(0.5, 1.0, 10.0)) if hybrid else {}))
    g, n = prob.cfg["nguard"], 16
    on, off = boxes(prob, form, call), boxes(prob, form, call, same_level_halos=0)
    reach = 9 if rk == 3 else 6
    written = STATE + [capi.SPARK_NPROP, capi.SPARK_NPROP + 1]
    for which, depth, var in ((0, reach, written + [V["shok"]] * hybrid), (1, 3, written)):
        if form == "plain_fp64":
            for x, y in zip(on[which], off[which]):
                assert np.array_equal(within(prob, x, depth)[..., var], within(prob, y, depth)[..., var])
            continue
        cells = {-1: slice(g - depth, g), 0: slice(g, g + n), 1: slice(g + n, g + n + depth)}
        count = 0
        for x, y, bare in zip(on[which], off[which], bare_sectors(prob)):
            for ox, oy, oz in bare:
                sl = (cells[oz], cells[oy], cells[ox])
                assert np.array_equal(x[sl][..., var], y[sl][..., var]), (which, ox, oy, oz)
                count += 1
        assert count > 0


@pytest.mark.parametrize("form,hybrid", [("plain_fp64", 0), ("plain_fp64", 1), ("batched_fp64", 0), ("fp32_flux", 1)])
def test_refill_grid_leaves_the_guards_it_fills(form, hybrid):
    """3D refill grid: the solution's guards hold the fill of the step's
    start, in the plain form to the stencil's reach, in the batched forms the
    layers shockDetect reads; the plain form's stage state holds the fill
    between the stages."""
    prob = problems.sedov3d(nb=2, n=8, nguard=6, guard_mode="refill", cfl=0.3, p_amb=1e-2, use_hybrid_riemann=hybrid)
    depth = 3 if form == "plain_fp64" else 1 + hybrid
    b = capi.Batch(dict(prob.cfg, form=form), prob.blocks)
    try:
        b.pack(prob.arrays)
        b.set_uniform_grid(*prob.ug)
        for step in ("hydro", "advance", "advance"):
            before = [a.copy() for a in prob.arrays]
            b.unpack(before, interior_only=True)
            if step == "hydro":
                b.hydro_step(0.5 * b.compute_dt()[0])
            else:
                b.advance(1)
            after, star = ([np.empty_like(a) for a in prob.arrays] for _ in range(2))
            b.unpack(after)
            b.unpack(star, which=1)
            for got, want, layers in ((after, before, depth), (star, [a.copy() for a in star], depth)):
                if got is star and form != "plain_fp64":
                    continue
                pyoracle.ug_fill(prob.cfg, prob.blocks[0], prob.ug, want)
                g = prob.cfg["nguard"]
                for x, y in zip(got, want):
                    x, y = within(prob, x, layers)[..., STATE].copy(), within(prob, y, layers)[..., STATE].copy()
                    inner = (slice(layers, -layers),) * 3
                    x[inner] = y[inner] = 0.0
                    assert np.array_equal(x, y)
    finally:
        b.close()


@pytest.mark.parametrize("form", ["plain_fp64", "batched_fp64", "fp32_flux"])
@pytest.mark.parametrize("grid", ["hierarchy", "refill"])
def test_replays_before_the_last_step_match_eager_steps(grid, form):
    """spark_advance replays a captured step for all but the step the call ends
    with: several calls, with unpacks and eager steps between them, give whole
    boxes equal to those without a graph."""
    if grid == "hierarchy":
        prob = problems.rt_amr(nb0=(1, 1, 2), n=16, lmax=3, nscalars=2)
    else:
        prob = problems.sedov3d(nb=2, n=8, nguard=6, guard_mode="refill", cfl=0.3, p_amb=1e-2)
    seq = {}
    for graph in (0, 1):
        b = capi.Batch(dict(prob.cfg, form=form), prob.blocks)
        try:
            b.set_option("graph", graph)
            b.set_option("autotune", 0)  # tuning writes a stage buffer
            b.pack(prob.arrays)
            if prob.ug is not None:
                b.set_uniform_grid(*prob.ug)
            else:
                b.set_amr_grid(prob.info["nb0"], prob.info["origins"], prob.info["bc"])
            seq[graph] = []
            for n in (3, 1, 4, 2):
                dts = b.advance(n)
                if n == 4:
                    b.hydro_step(0.5 * dts[-1])
                for which in (0, 1):
                    out = [np.empty_like(a) for a in prob.arrays]
                    b.unpack(out, which=which)
                    seq[graph].append((dts, out))
        finally:
            b.close()
    for (d0, o0), (d1, o1) in zip(seq[0], seq[1]):
        assert np.array_equal(d0, d1)
        for x, y in zip(o0, o1):
            assert np.array_equal(x, y)
