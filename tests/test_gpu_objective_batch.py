"""The objective over several scenarios in one pass of launches and the
backward product that reads a double gradient and applies the upstream one:
the same bits as one scenario at a time and as torch's conversions and
products around the plain product."""
import numpy as np
import pytest
import scipy.sparse as sps

pytestmark = pytest.mark.gpu


def _csr(rng, rows, cols, kind):
    """full: a voxel-major copy with rows split over partial segments (more
    than 1024 spots in a voxel) and short ones; sparse: rows of a few entries
    (the product without pieces) and most voxels without any."""
    if kind == "full":
        m = sps.random(rows, cols, density=0.02, format="lil", random_state=int(rng.integers(1 << 30)))
        m[:, 3] = 1.0
        m[:, cols - 5] = 0.5
    else:
        m = sps.random(rows, cols, density=3.0 / cols, format="lil", random_state=int(rng.integers(1 << 30)))
        m[0, 1] = 1.0
    m = sps.csr_matrix(m)
    m.sort_indices()
    m.data = rng.uniform(0.1, 1.0, m.nnz).astype(np.float32)
    return m


def _set(ctx, mats):
    from moquimc_amd import dij
    for s, m in enumerate(mats):
        ctx.dij_set_csr(m.indptr.astype(np.int64), m.indices.astype(np.int32), m.data.astype(np.float32), m.shape,
                        scenario=s)
    return [dij.DijMatrix(ctx, s, scale=1.0 + 0.25 * s) for s in range(len(mats))]


@pytest.mark.parametrize("n", [1, 2, 17])   # 16 matrices a launch
@pytest.mark.parametrize("kind,rows,cols", [("full", 1300, 5001), ("sparse", 40, 511), ("sparse", 7, 70001)])
@pytest.mark.parametrize("weights", [False, True])
def test_values_of_several_scenarios(ctx, n, kind, rows, cols, weights):
    import torch
    from moquimc_amd import dij
    rng = np.random.default_rng(17 * n + cols)
    base = [_csr(rng, rows, cols, kind) for _ in range(min(n, 3))]
    cs = [base[s % len(base)] for s in range(n)]
    mats = _set(ctx, cs)
    w_np = rng.uniform(0.5, 1.5, rows).astype(np.float32)
    p_np = rng.uniform(0.0, 2.0, cols)
    c_np = rng.uniform(0.0, 2.0, cols).astype(np.float32)
    w, p = torch.tensor(w_np, device="cuda"), torch.tensor(p_np, device="cuda")
    c = torch.tensor(c_np, device="cuda") if weights else None
    got = dij._values(mats, w, p, c)
    for s, m in enumerate(mats):
        f, _ = m.quadratic(w, p, c, want_grad=False)
        assert got[s].item() == f.item()
        r = (cs[s].T.astype(np.float64) @ w_np.astype(np.float64)) * m.scale - p_np
        ref = np.mean((c_np.astype(np.float64) if weights else 1.0) * r * r)
        # at most 1e5 positive terms summed in FP64
        assert abs(f.item() - ref) <= 1e5 * 2.0 ** -53 * ref * 4
    # a scenario listed twice is evaluated one at a time
    twice = dij._values([mats[0], mats[0]], w, p, c)
    assert twice[0].item() == twice[1].item() == got[0].item()


def test_more_terms_than_one_workgroup_sums(ctx):
    import torch
    n = 33_700_000   # one spot, more than 32768 segments of 1024 entries
    val = np.linspace(0.5, 1.5, n, dtype=np.float32)
    ctx.dij_set_csr(np.array([0, n], np.int64), np.arange(n, dtype=np.int32), val, (1, n), scenario=0)
    from moquimc_amd import dij
    m = dij.DijMatrix(ctx, 0)
    p = torch.full((n,), 0.25, dtype=torch.float64, device="cuda")
    f, g = m.quadratic(torch.ones(1, device="cuda"), p)
    r = val.astype(np.float64) - 0.25
    # 3.4e7 terms in FP64, rounded independently: far below their number
    assert abs(f.item() - np.mean(r * r)) <= 1e-10 * np.mean(r * r)
    assert np.array_equal(g.cpu().numpy(), (2.0 / n * r).astype(np.float32))
    ctx.dij_set_csr(np.array([0, 1], np.int64), np.zeros(1, np.int32), np.ones(1, np.float32), (1, 1), scenario=0)


@pytest.mark.parametrize("kind,rows,cols", [("full", 1300, 5001), ("full", 3, 4099), ("sparse", 40, 511)])
def test_backward_product_equals_the_composed_one(ctx, kind, rows, cols):
    import torch
    from moquimc_amd import dij
    rng = np.random.default_rng(rows)
    if kind == "full" and rows == 3:   # long rows: products over pieces
        m = sps.csr_matrix(rng.uniform(0.1, 1.0, (rows, cols)).astype(np.float32))
    else:
        m = _csr(rng, rows, cols, kind)
    (mat,) = _set(ctx, [m])
    g = torch.tensor(rng.normal(size=cols), device="cuda")
    y = torch.empty(rows, dtype=torch.float64, device="cuda")
    ctx.dij_matvec(0, 1, g.to(torch.float32).data_ptr(), y.data_ptr(), alpha=mat.scale,
                   stream=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(mat.rmatvec(g), y)
    assert torch.equal(mat.rmatvec(g, torch.float32), y.to(torch.float32))
    assert torch.equal(mat.rmatvec(g.expand(1, -1)[0]), y)
    assert torch.equal(mat.rmatvec(torch.stack([g, g], 1)[:, 0]), y)       # strided
    assert torch.equal(mat.rmatvec(torch._neg_view(g)), -y)
    up = torch.tensor(-0.3, dtype=torch.float64, device="cuda")
    for dt in (torch.float32, torch.float64, torch.float16):
        g32 = g.to(torch.float32)
        assert torch.equal(mat._adjoint(g32, dt, up.data_ptr()), (y * up).to(dt))


def test_quadratic_backward_forms(ctx):
    """An upstream gradient with a graph, a batch of upstream gradients and a
    plain one: the gradient is the objective's times the upstream."""
    import torch
    from moquimc_amd import dij
    rng = np.random.default_rng(2)
    (mat,) = _set(ctx, [_csr(rng, 40, 511, "sparse")])
    p = torch.tensor(rng.uniform(0.0, 2.0, 511), device="cuda")
    for dt in (torch.float32, torch.float64):
        w = torch.tensor(rng.uniform(0.5, 1.5, 40), device="cuda", dtype=dt, requires_grad=True)
        f = dij.quadratic_objective(mat, w, p)
        (g1,) = torch.autograd.grad(f, w, retain_graph=True)
        assert g1.dtype == dt and torch.any(g1 != 0)
        ups = torch.tensor([1.0, -0.5, 3.0], dtype=torch.float64, device="cuda")
        (gb,) = torch.autograd.grad(f, w, ups, is_grads_batched=True, retain_graph=True)
        for k in range(3):
            (gk,) = torch.autograd.grad(f, w, ups[k], retain_graph=True)
            assert torch.equal(gb[k], gk)
        # through the upstream gradient: d(grad . v) / d(up) = grad(up = 1) . v
        up = torch.tensor(2.0, dtype=torch.float64, device="cuda", requires_grad=True)
        (gu,) = torch.autograd.grad(f, w, up, create_graph=True)
        v = torch.linspace(1.0, 2.0, 40, device="cuda", dtype=dt)
        (du,) = torch.autograd.grad((gu * v).sum(), up)
        assert torch.allclose(du, (g1.double() * v.double()).sum(), rtol=40 * 2.0 ** -23, atol=0)


def _big(spots, voxels, seed):
    """Voxel v in (a_v + 7 j) mod spots, j < k_v: 1 to 250 spots, all of them
    (a row split over pieces) in some, none in every tenth."""
    rng = np.random.default_rng(seed)
    k = rng.integers(1, 251, voxels)
    k[::1000] = min(spots, 1300)
    k[5::10] = 0
    k[-1] = 3
    row = np.repeat(np.arange(voxels), k)
    j = np.arange(k.sum()) - np.repeat(np.cumsum(k) - k, k)
    col = (rng.integers(0, spots, voxels)[row] + 7 * j) % spots
    m = sps.csr_matrix((rng.uniform(0.1, 1.0, len(row)).astype(np.float32), (col, row)), shape=(spots, voxels))
    m.sort_indices()
    return m


@pytest.mark.parametrize("spots", [1300, 24576, 24577, 66000])   # x in LDS up to 24576; 32-bit columns from 65537
def test_large_matrices(ctx, spots):
    """More segments than the least for which workgroups stay."""
    import torch
    m = _big(spots, 100003, spots)
    assert m.nnz > 8192 * 1100
    (mat,) = _set(ctx, [m])
    rng = np.random.default_rng(9)
    w_np = rng.uniform(0.5, 1.5, spots).astype(np.float32)
    w = torch.tensor(w_np, device="cuda")
    ref = m.T.astype(np.float64) @ w_np.astype(np.float64) * mat.scale
    # up to 1300 positive FP64 terms a voxel
    tol = 1300 * 2.0 ** -52
    y = mat.matvec(w)
    np.testing.assert_allclose(y.cpu().numpy(), ref, rtol=tol, atol=0)
    st = torch.cuda.current_stream().cuda_stream
    y2 = y.clone()
    ctx.dij_matvec(0, 0, w.data_ptr(), y2.data_ptr(), alpha=mat.scale, accumulate=True, stream=st)
    np.testing.assert_allclose(y2.cpu().numpy(), 2 * ref, rtol=2 * tol, atol=0)
    y3 = torch.full((m.shape[1],), 7.0, dtype=torch.float32, device="cuda")
    ctx.dij_matvec(0, 0, w.data_ptr(), y3.data_ptr(), y_double=False, alpha=mat.scale, stream=st)
    assert torch.equal(y3, y.to(torch.float32))
    p_np, c_np = rng.uniform(0.0, 200.0, m.shape[1]), rng.uniform(0.0, 2.0, m.shape[1]).astype(np.float32)
    p, c = torch.tensor(p_np, device="cuda"), torch.tensor(c_np, device="cuda")
    for cc, c64 in ((None, 1.0), (c, c_np.astype(np.float64))):
        f, g = mat.quadratic(w, p, cc)
        r = y.cpu().numpy() - p_np
        assert abs(f.item() - np.mean(c64 * r * r)) <= 1e5 * 2.0 ** -52 * np.mean(c64 * r * r)
        # the rounded residual of a d and p that may cancel, then one rounding to float
        err = 2.0 / m.shape[1] * c64 * (tol * (np.abs(ref) + p_np) + 2.0 ** -23 * np.abs(r))
        assert np.all(np.abs(g.cpu().numpy() - 2.0 / m.shape[1] * c64 * r) <= err + 1e-37)
    # two matrices side by side: the bits of one
    from moquimc_amd import dij
    mats = _set(ctx, [m, m])
    got = dij._values(mats, w, p, c)
    assert got[0].item() == mats[0].quadratic(w, p, c, want_grad=False)[0].item()
    assert got[1].item() == mats[1].quadratic(w, p, c, want_grad=False)[0].item()
