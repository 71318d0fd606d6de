"""Deposits that are summed per voxel and added by groups of lanes, against
the same histories scored step by step, every deposit with an atomic of its
own (the statistics loop, production kernels): grouped plain and batched
passes and passes of caller-made vertices, of two to six scorers."""
import numpy as np
import pytest

import phantoms
import refbind as rb
from moquimc_amd import _abi

pytestmark = pytest.mark.gpu

# pairs of lanes, groups of four with three and four sums, groups with one
# and two sums behind them
MASKS = [rb.SC_LETD, rb.SC_LETT, rb.SC_EDEP | rb.SC_DM, rb.SC_STAT, rb.SC_DOSE | rb.SC_LETD, rb.SC_DOSE | rb.SC_STAT,
         rb.SC_LETD | rb.SC_LETT, rb.SC_LETD | rb.SC_STAT, rb.SC_DOSE | rb.SC_LETD | rb.SC_LETT,
         rb.SC_LETD | rb.SC_LETT | rb.SC_EDEP | rb.SC_DM]


def _compare(ctx, mask, scenarios, run):
    ctx.set_scorers(mask, scenarios > 1)
    out = []
    for loops in (_abi.LOOPS_ONCE, _abi.LOOPS_REFERENCE_STAT):
        ctx.zero_scorers()
        res = run(loops)
        out.append((res.histories, res.steps,
                    [ctx.scorer(k, s) for k in range(ctx.scorer_count()) for s in range(scenarios)]))
    (h, steps, got), (h1, steps1, want) = out
    assert (h, steps) == (h1, steps1)
    for a, b in zip(got, want):
        # (the last two scorers of the statistics loop score voxel 0 too)
        fin = np.isfinite(b[1:])
        assert np.array_equal(fin, np.isfinite(a[1:])) and (h < 100 or b[1:].any())
        # positive terms in another order: at most some 1e4 a voxel, 2^-53 each
        np.testing.assert_allclose(a[1:][fin], b[1:][fin], rtol=2e-12, atol=0)


@pytest.mark.parametrize("mask", MASKS)
@pytest.mark.parametrize("histories", [3, 65, 1025])
def test_plans(ctx, mask, histories):
    g = phantoms.slab_box(9, 11, 90)
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    ctx.set_scenarios([[0, 0, 0], [1, 0, 0]], [1.0, 0.9])
    ctx.set_spots(phantoms.spots([90.0, 60.0], histories, sigma=3.0, sigma_e_frac=0.01,
                                 positions=[(0, 0, 0.5), (2, -1, 0.5)]))
    for scenarios in (1, 2):
        for batched in (True, False):
            _compare(ctx, mask, scenarios, lambda loops: ctx.run(ctx.config(seed=3, batched=batched, loops=loops)))
    ctx.set_scenarios()


@pytest.mark.parametrize("mask", MASKS)
def test_vertices(ctx, mask):
    g = phantoms.slab_box(9, 11, 90)
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    rng = np.random.default_rng(2)
    v = np.zeros((2003, 7), np.float32)
    v[:, 0] = rng.uniform(50.0, 110.0, len(v))
    v[:, 1:3] = rng.normal(0.0, 2.0, (len(v), 2))
    v[:, 3] = 0.5
    v[:, 6] = -1.0
    for batched in (True, False):
        _compare(ctx, mask, 1, lambda loops: ctx.run_vertices(v, ctx.config(seed=4, batched=batched, loops=loops)))
