"""Grids whose edges leave no room in 64 KB of LDS for the sums of five or six
scorers (the Dij is then scored step by step behind the first four) or for the
waves' Dij queues (each lane then inserts its own deposits): the matrix and
the scorers are those of narrower workgroups, whose sums and queues fit."""
import numpy as np
import pytest

import refbind as rb

pytestmark = pytest.mark.gpu

# LDS of a workgroup of 256: 14400 bytes of tables, 4 an edge, 2048 a summed
# scorer and 13376 for the queues; at 6368 edges in all they are 64 KB with
# six scorers, at 7392 with four
NO_SIX_SUMS, NO_QUEUE = 6500, 7600


def _run(ctx, nz, mask, block, batched=True):
    g = rb.Grid(rb.uniform_edges(-100, 100, 1), rb.uniform_edges(-100, 100, 1), rb.uniform_edges(-nz * 0.05, 0.0, nz),
                np.full(nz, 1.0e-3, np.float32))
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    ctx.set_spots(np.array([rb.make_spot(e, 2.0, 150, pos=(0, 0, 0.5), sigma_e=0.5) for e in (70.0, 110.0)],
                           dtype=rb.SPOT_DTYPE))
    ctx.set_scorers(mask)
    ctx.zero_scorers()
    res = ctx.run(ctx.config(seed=6, batched=batched, dij=True, dij_capacity=1 << 14, block_size=block))
    ctx.dij_build(0.0)
    return (res.histories, res.steps), ctx.dij_csr(0), [ctx.scorer(k) for k in range(ctx.scorer_count())]


@pytest.mark.parametrize("batched", [True, False])
@pytest.mark.parametrize("nz", [NO_SIX_SUMS, NO_QUEUE])
@pytest.mark.parametrize("mask", [rb.SC_DOSE, rb.SC_EDEP, rb.SC_LETD | rb.SC_LETT, rb.SC_DOSE | rb.SC_LETD | rb.SC_LETT])
def test_launches_without_room(ctx, nz, mask, batched):
    n0, m0, s0 = _run(ctx, nz, mask, 64, batched)
    n1, m1, s1 = _run(ctx, nz, mask, 256, batched)
    assert n0 == n1 and len(m0[1]) > 2000
    assert np.array_equal(m0[0], m1[0]) and np.array_equal(m0[1], m1[1])
    np.testing.assert_allclose(m1[2], m0[2], rtol=1e-6, atol=0)   # FP64 sums rounded to float
    for a, b in zip(s1, s0):
        fin = np.isfinite(b)
        assert np.array_equal(fin, np.isfinite(a)) and b[fin].any()
        # a few hundred positive terms a voxel in another order
        np.testing.assert_allclose(a[fin], b[fin], rtol=1e-12, atol=0)
    if mask & rb.SC_DOSE:   # voxel 0 is in neither
        d = np.zeros(nz)
        np.add.at(d, m1[1], m1[2].astype(np.float64))
        np.testing.assert_allclose(s1[0], d, rtol=1e-6, atol=0)
