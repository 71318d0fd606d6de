"""Plain launches (a lane per history, consecutive spots sharing a launch up to
2^18 histories): every history of every spot and scenario runs once wherever
the launches are cut, with the results of the batched launch, which draws the
same random numbers per history."""
import numpy as np
import pytest

import phantoms
import refbind as rb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("histories,budgets", [
    ([0, 5, 0, 262145, 0, 7, 0], None),          # one above a launch, empty spots at both ends and behind it
    ([131072, 131072, 1, 262143, 1, 1], None),   # cuts exactly at the launch's size
    ([300000, 0], None),                         # only empty spots behind the last launch
    ([1], None),
    ([90000, 90000, 90000], [1.0, 0.5, 0.01]),   # a spot's scenarios stay in one launch
])
def test_plain_launches_cover_the_plan(ctx, histories, budgets):
    g = phantoms.water_box(11, 9, 23, dz=0.5)
    sp = phantoms.spots([8.0 + i for i in range(len(histories))], 1, sigma=1.5)
    sp["histories"] = histories
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    n = 1
    if budgets:
        n = len(budgets)
        ctx.set_scenarios(np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], np.float32), np.ones(3, np.float32), budgets)
    ctx.set_spots(sp)
    for mask in (rb.SC_DOSE | rb.SC_LETD, rb.SC_DOSE | rb.SC_STAT):
        ctx.set_scorers(mask, per_scenario=n > 1)
        outs, runs = [], []
        for batched in (True, False):
            ctx.zero_scorers()
            runs.append(ctx.run(ctx.config(seed=31, batched=batched)))
            outs.append([ctx.scorer(k, scenario=s) for s in range(n) for k in range(ctx.scorer_count())])
        total = sum(int(np.floor(h * b + 0.5)) for h in histories for b in (budgets or [1.0]))
        assert runs[0].histories == runs[1].histories == total
        assert runs[0].steps == runs[1].steps and runs[0].dropped == runs[1].dropped
        # FP64 sums of the same positive terms in another order: below the
        # terms' number (3e5 histories, a few steps each) times 2^-53
        for a, b in zip(*outs):
            assert np.any(a != 0)
            np.testing.assert_allclose(b, a, rtol=1e-9, atol=0)
