"""Both orders of a Dij matrix, built on the device: at the edges of the
4096-nonzero tiles, with voxels and rows that cross them, with one nonzero,
one row or one column, and from hash tables cut into several chunks, the rows
come back sorted and unchanged and both products equal scipy's in FP64."""
import numpy as np
import pytest
import scipy.sparse as sps

import phantoms
import refbind as rb

pytestmark = pytest.mark.gpu


def _matrix(rows, cols, nnz, seed):
    """nnz distinct (row, column) pairs, a third of them in the last column."""
    rng = np.random.default_rng(seed)
    last = min(rows, nnz // 3)
    pick = rng.choice(rows * (cols - 1), nnz - last, replace=False) if cols > 1 else np.zeros(0, np.int64)
    r = np.r_[pick // max(cols - 1, 1), rng.choice(rows, last, replace=False)]
    c = np.r_[pick % max(cols - 1, 1), np.full(last, cols - 1)]
    if cols == 1:
        r, c = rng.choice(rows, nnz, replace=False), np.zeros(nnz, np.int64)
    D = sps.csr_matrix((rng.uniform(1e-6, 1.0, len(r)).astype(np.float32), (r, c)), shape=(rows, cols))
    D.sort_indices()
    return D


@pytest.mark.parametrize("rows,cols,nnz", [(1, 1, 1), (1, 7000, 4095), (3, 5000, 4096), (3, 5000, 4097),
                                           (5000, 1, 4097), (300, 33, 8192), (65536, 40, 8193), (65537, 40, 12289),
                                           (2, 1 << 20, 4098)])
def test_both_orders_at_tile_edges(ctx, rows, cols, nnz):
    import torch
    D = _matrix(rows, cols, nnz, rows + nnz)
    ctx.dij_set_csr(D.indptr, D.indices, D.data, D.shape, scenario=0)
    ip, ix, v, shape = ctx.dij_csr(0)
    assert shape == D.shape and np.array_equal(ip, D.indptr) and np.array_equal(ix, D.indices)
    assert np.array_equal(v.view(np.uint32), D.data.view(np.uint32))
    rng = np.random.default_rng(1)
    w, g = rng.uniform(0.5, 1.5, rows).astype(np.float32), rng.normal(size=cols).astype(np.float32)
    dev = torch.device("cuda", 0)
    tw, tg = torch.from_numpy(w).to(dev), torch.from_numpy(g).to(dev)
    dose = torch.full((cols,), 7.0, dtype=torch.float64, device=dev)
    grad = torch.full((rows,), 7.0, dtype=torch.float64, device=dev)
    ctx.dij_matvec(0, 0, tw.data_ptr(), dose.data_ptr(), y_double=True)
    ctx.dij_matvec(0, 1, tg.data_ptr(), grad.data_ptr(), y_double=True)
    torch.cuda.synchronize()
    D64 = D.astype(np.float64)
    # sums of at most 5000 terms of size 1 in another order: 5000 half ulps
    assert np.abs(dose.cpu().numpy() - D64.T @ w.astype(np.float64)).max() <= 5000 * 1.2e-16 * 5000
    scale = np.abs(D64) @ np.abs(g).astype(np.float64)
    assert (np.abs(grad.cpu().numpy() - D64 @ g.astype(np.float64)) <= 1e-12 * np.maximum(scale, 1.0)).all()


@pytest.mark.parametrize("n_spots,capacity", [(1, 1 << 17), (7, 30011), (700, 1024)])
def test_tables_in_chunks(ctx, n_spots, capacity):
    """One table in as many chunks as fit, odd table sizes, and more tables
    than get two chunks each: the rows hold what a matrix built without a
    threshold has at or above each row's limit, and sum to the dose."""
    g = phantoms.slab_box(16, 16, 40)
    sp = phantoms.spots(list(np.linspace(60.0, 80.0, n_spots)), 40 if n_spots < 700 else 3, sigma=1.0,
                        sigma_e_frac=0.01, positions=[(0, 0, 0.5)] * n_spots)
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    ctx.set_scenarios()
    ctx.set_spots(sp)
    ctx.set_scorers(rb.SC_DOSE)
    ctx.zero_scorers()
    ctx.run(ctx.config(seed=3, batched=True, dij=True, dij_capacity=capacity))
    dose = ctx.scorer(0)

    def build(thr):
        ctx.dij_build(thr)
        indptr, idx, val, shape = ctx.dij_csr(0)
        return sps.csr_matrix((val, idx, indptr), shape=shape)

    full, cut = build(0.0), build(0.05)
    # FP64 sums rounded to float once per entry
    assert np.allclose(np.asarray(full.astype(np.float64).sum(axis=0)).ravel(), dose, rtol=2e-6, atol=1e-30)
    assert full.nnz > 0 and (full.data > 0).all()
    for D in (full, cut):
        assert all((np.diff(D.indices[a:b]) > 0).all() for a, b in zip(D.indptr[:-1], D.indptr[1:]))
    # values next to the limit may round to it
    for r in range(n_spots):
        a = full[r]
        lim = 0.05 * a.data.max()
        b = cut[r]
        sure = a.data > lim * (1 + 1e-6)
        assert set(a.indices[sure]) <= set(b.indices) <= set(a.indices[a.data >= lim * (1 - 1e-6)])
        assert np.array_equal(np.asarray(a[:, b.indices].todense()).ravel(), b.data)
