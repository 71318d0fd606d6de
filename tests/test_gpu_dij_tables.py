"""Where a Dij table keeps a voxel does not change the matrix: tables smaller
than a group of slots, of odd sizes, nearly full ones (every probe form) and
roomy ones; one wave of histories and many; a Dij slot that is summed per
voxel and one scored step by step; grids whose extent is not a multiple of a
block's; and an overflow is still reported."""
import numpy as np
import pytest
import scipy.sparse as sps

import phantoms
import refbind as rb

pytestmark = pytest.mark.gpu


def _run(ctx, n_spots, histories, shape=(9, 7, 41), mask=rb.SC_DOSE, **kw):
    g = phantoms.slab_box(*shape)
    sp = phantoms.spots([62.0 + 3 * i for i in range(n_spots)], histories, sigma=1.5, sigma_e_frac=0.01,
                        positions=[((i % 3) - 1.0, (i % 2) - 0.5, 0.5) for i in range(n_spots)])
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    ctx.set_scenarios()
    ctx.set_spots(sp)
    ctx.set_scorers(mask)
    ctx.zero_scorers()
    ctx.run(ctx.config(seed=8, batched=True, dij=True, **kw))
    ctx.dij_build(0.0)
    indptr, idx, val, shape = ctx.dij_csr(0)
    return sps.csr_matrix((val, idx, indptr), shape=shape), ctx.scorer(0)


@pytest.mark.parametrize("n_spots,histories", [(1, 1), (3, 64), (5, 700)])
def test_slot_order_does_not_change_the_matrix(ctx, n_spots, histories):
    ref, dose = _run(ctx, n_spots, histories, dij_capacity=1 << 16)
    # FP64 sums rounded to float once per entry, in another order
    assert np.allclose(np.asarray(ref.astype(np.float64).sum(axis=0)).ravel(), dose, rtol=2e-6, atol=1e-30)
    most = int(np.diff(ref.indptr).max())
    assert most > 0 or histories == 1
    for cap in (most + 1, most + 37, 2 * most + 5, 4 * most + 31, 30011):
        if cap < 1:
            continue
        D, _ = _run(ctx, n_spots, histories, dij_capacity=cap)
        assert np.array_equal(D.indptr, ref.indptr) and np.array_equal(D.indices, ref.indices), cap
        assert np.allclose(D.data, ref.data, rtol=1e-6, atol=0), cap
    if most > 1:
        with pytest.raises(RuntimeError, match="overflowed"):
            _run(ctx, n_spots, histories, dij_capacity=most - 1)


def test_tables_smaller_than_a_group(ctx):
    """A spot of a few histories in a grid of 18 voxels: up to 18 entries, in
    tables of 18 to 33 slots."""
    ref, _ = _run(ctx, 2, 40, shape=(3, 2, 3), dij_capacity=1 << 12)
    most = int(np.diff(ref.indptr).max())
    for cap in (18, 31, 32, 33):
        assert most <= cap
        D, _ = _run(ctx, 2, 40, shape=(3, 2, 3), dij_capacity=cap)
        assert np.array_equal(D.indptr, ref.indptr) and np.array_equal(D.indices, ref.indices), cap
        assert np.allclose(D.data, ref.data, rtol=1e-6, atol=0), cap


def test_step_by_step_scorer_slot(ctx):
    """With four scorers before it the Dij slot is scored per step."""
    ref, dose = _run(ctx, 3, 300, dij_capacity=1 << 14)
    for mask in (rb.SC_DOSE | rb.SC_LETD, rb.SC_DOSE | rb.SC_LETD | rb.SC_LETT):
        D, d = _run(ctx, 3, 300, mask=mask, dij_capacity=1 << 14)
        assert np.array_equal(D.indices, ref.indices)
        assert np.allclose(D.data, ref.data, rtol=1e-6, atol=0)
        assert np.allclose(d, dose, rtol=1e-12, atol=0)
