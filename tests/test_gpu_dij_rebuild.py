"""A build over the arrays of the one before gives the matrices and products
of a build in a fresh context: the same sizes again, smaller and larger ones,
other scenarios, after a matrix of the caller's and after a build without an
entry."""
import numpy as np
import pytest

import phantoms
import refbind as rb

pytestmark = pytest.mark.gpu


def _run(ctx, n_spots, histories, shape, n_scen, thr):
    import torch
    from moquimc_amd import dij
    g = phantoms.slab_box(*shape)
    sp = phantoms.spots([62.0 + 3 * i for i in range(n_spots)], histories, sigma=1.5, sigma_e_frac=0.01,
                        positions=[((i % 3) - 1.0, (i % 2) - 0.5, 0.5) for i in range(n_spots)])
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    shifts = np.zeros((n_scen, 3), np.float32)
    shifts[:, 0] = np.arange(n_scen) * 0.5
    ctx.set_scenarios(shifts, np.ones(n_scen, np.float32))
    ctx.set_spots(sp)
    ctx.set_scorers(rb.SC_DOSE)
    ctx.zero_scorers()
    ctx.run(ctx.config(seed=8, dij=True, dij_capacity=1 << 15))
    ctx.dij_build(thr)
    out = []
    w = torch.linspace(0.5, 1.5, n_spots, device="cuda")
    for s in range(n_scen):
        m = dij.DijMatrix(ctx, s)
        out += list(ctx.dij_csr(s)[:3])
        if m.nnz:
            d = m.matvec(w)
            f, grad = m.quadratic(w, torch.full_like(d, 1e-3))
            out += [d.cpu().numpy(), f.cpu().numpy(), m.rmatvec(grad).cpu().numpy()]
    return out


def test_rebuild_equals_a_fresh_build(ctx):
    from moquimc_amd import _abi
    for k, plan in enumerate([(3, 500, (12, 11, 60), 3, 1e-4), (3, 500, (12, 11, 60), 3, 1e-4),
                              (3, 505, (12, 11, 60), 3, 1e-4), (2, 100, (9, 7, 41), 1, 1e-2),
                              (5, 900, (20, 21, 90), 4, 0.0), (5, 900, (20, 21, 90), 4, 2.0),
                              (3, 500, (12, 11, 60), 9, 1e-4)]):
        if k == 3:
            ctx.dij_set_csr(np.array([0, 1], np.int64), np.zeros(1, np.int32), np.ones(1, np.float32), (1, 4),
                            scenario=1)
        got = _run(ctx, *plan)
        fresh = _abi.Context(0)
        want = _run(fresh, *plan)
        fresh.close()
        assert len(got) == len(want)
        for a, b in zip(got, want):
            # entries are FP64 sums in any order, rounded to float
            np.testing.assert_allclose(a, b, rtol=1e-6, atol=0)
