"""Launches of five and six scorers (every slot's deposits summed per voxel)
and grouped scoring of caller-made vertices: each scorer equals the one of a
launch that scores fewer of them, the histories being the same."""
import numpy as np
import pytest

import phantoms
import refbind as rb

pytestmark = pytest.mark.gpu

MASKS = [rb.SC_DOSE | rb.SC_LETD | rb.SC_LETT, rb.SC_DOSE | rb.SC_LETD | rb.SC_LETT | rb.SC_EDEP,
         rb.SC_LETD | rb.SC_EDEP | rb.SC_DM | rb.SC_STAT, rb.SC_EDEP | rb.SC_DM]
# a mask's scorers in their order, as (single-purpose mask, index there)
ORDER = [(rb.SC_DOSE, 1), (rb.SC_LETD, 2), (rb.SC_LETT, 2), (rb.SC_EDEP, 1), (rb.SC_DM, 1), (rb.SC_STAT, 2)]


def _check(ctx, mask, run):
    def scores(m):
        ctx.set_scorers(m)
        ctx.zero_scorers()
        res = run()
        return res, [ctx.scorer(k) for k in range(ctx.scorer_count())]

    res, got = scores(mask)
    k = 0
    for bit, count in ORDER:
        if not mask & bit:
            continue
        alone, want = scores(bit)
        assert (alone.histories, alone.steps, alone.dropped) == (res.histories, res.steps, res.dropped)
        for j in range(count):
            assert np.any(want[j] != 0) or res.histories < 100
            # positive terms in another order: their number (5e3 histories'
            # steps in a voxel) times 2^-53 at most
            fin = np.isfinite(want[j])
            assert np.array_equal(fin, np.isfinite(got[k]))
            np.testing.assert_allclose(got[k][fin], want[j][fin], rtol=1e-11, atol=0)
            k += 1
    assert k == len(got)


@pytest.mark.parametrize("mask", MASKS)
@pytest.mark.parametrize("batched", [True, False])
@pytest.mark.parametrize("n", [1, 63, 5000])
def test_vertices_score_as_fewer_scorers_do(ctx, mask, batched, n):
    g = phantoms.slab_box(33, 31, 100)
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    rng = np.random.default_rng(n)
    v = np.zeros((n, 7), np.float32)
    v[:, 0] = rng.uniform(60.0, 120.0, n)
    v[:, 1:3] = rng.normal(0.0, 3.0, (n, 2))
    v[:, 3] = 0.5
    v[:, 6] = -1.0
    _check(ctx, mask, lambda: ctx.run_vertices(v, ctx.config(seed=12, batched=batched)))


@pytest.mark.parametrize("kw", [dict(batched=True), dict(batched=False), dict(batched=True, physics_debug=True),
                                dict(batched=True, waves_per_simd=5, block_size=64)])
def test_plan_scores_as_fewer_scorers_do(ctx, kw):
    g = phantoms.slab_box(20, 22, 90)
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    ctx.set_spots(phantoms.spots([70.0, 90.0], 800, sigma_e_frac=0.01))
    for mask in MASKS[:3]:
        _check(ctx, mask, lambda: ctx.run(ctx.config(seed=13, **kw)))


def test_dij_beside_five_scorers(ctx):
    """The Dij slot behind the first four."""
    g = phantoms.slab_box(20, 22, 90)
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    ctx.set_spots(phantoms.spots([70.0, 90.0], 800, sigma_e_frac=0.01))
    mats = []
    for mask in (rb.SC_DOSE, rb.SC_DOSE | rb.SC_LETD | rb.SC_LETT, rb.SC_LETD | rb.SC_LETT | rb.SC_EDEP):
        ctx.set_scorers(mask)
        ctx.zero_scorers()
        ctx.run(ctx.config(seed=14, dij=True, dij_capacity=1 << 16))
        ctx.dij_build(0.0)
        mats.append(ctx.dij_csr(0))
    for m in mats[1:]:
        assert np.array_equal(m[0], mats[0][0]) and np.array_equal(m[1], mats[0][1])
        np.testing.assert_allclose(m[2], mats[0][2], rtol=1e-6, atol=0)
