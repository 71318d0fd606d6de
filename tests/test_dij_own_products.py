"""Matrices with products of their own (a subclass of DijMatrix that overrides
them, or another class with the same methods) keep being asked for them: by
the objective's and the dose's backward passes and by the worst case."""
import pytest
import torch

from moquimc_amd import dij


class Dense:
    """scale * D w of a dense matrix (voxels x spots) in host memory."""

    def __init__(self, d, scale=1.0):
        self.d, self.scale, self.asked = d, scale, []

    def matvec(self, w, out_dtype=torch.float64):
        return (self.scale * (self.d @ w.detach().double())).to(out_dtype)

    def quadratic(self, w, prescription, voxel_weights=None, want_grad=True):
        c = torch.ones(len(self.d)) if voxel_weights is None else voxel_weights
        r = self.matvec(w) - prescription
        f = (c * r * r).mean()
        return f, (2.0 * c * r / len(r)).float() if want_grad else None

    def rmatvec(self, g, out_dtype=torch.float64):
        self.asked.append(out_dtype)
        return (self.scale * (self.d.T @ g.detach().double())).to(out_dtype)


class Derived(Dense, dij.DijMatrix):
    pass


@pytest.mark.parametrize("kind", [Dense, Derived])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_backward_asks_for_the_matrix_own_product(kind, dtype):
    gen = torch.Generator().manual_seed(5)
    mats = [kind(torch.rand(30, 4, generator=gen, dtype=torch.float64), 1.0 + s) for s in range(3)]
    p = torch.rand(30, generator=gen, dtype=torch.float64)
    w = torch.rand(4, generator=gen, dtype=dtype, requires_grad=True)

    dij.dose(mats[0], w).sum().backward()
    assert mats[0].asked == [torch.float64]
    assert torch.allclose(w.grad, mats[0].d.sum(0).to(dtype))   # another order of 30 additions

    w.grad = None
    (3.0 * dij.quadratic_objective(mats[0], w, p)).backward()
    assert mats[0].asked == [torch.float64] * 2
    _, g = mats[0].quadratic(w, p)
    assert torch.equal(w.grad, (mats[0].rmatvec(g) * 3.0).to(dtype))

    w.grad = None
    f, vals = dij.worst_case_objective(mats, w, p)
    f.backward()
    k = int(vals.argmax())
    assert f.item() == vals[k].item() and mats[k].asked[-1] == torch.float64
    _, g = mats[k].quadratic(w, p)
    assert torch.equal(w.grad, mats[k].rmatvec(g).to(dtype))
