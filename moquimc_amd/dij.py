"""Differentiable dose from a dose-influence matrix held on the device.

A Dij built by ``Context.dij_build`` is a CSR matrix with one row per spot
(the orientation of the reference's ``io::save_to_npz``,
moqui/base/mqi_io.hpp:249-320).  With D the voxels x spots influence
matrix, the dose of spot weights w is D w and the gradient of an objective
f(D w) with respect to w is D^T (df/dd).  Both products run in the
library's kernels (FP64 accumulation, float32 inputs, fixed summation
order) on torch's current stream; ``dose`` wraps them in a
``torch.autograd.Function``, and ``quadratic_objective`` forms the
quadratic objective and its dose gradient inside the D w pass.

    mat = DijMatrix(ctx, scenario=0)
    w = torch.rand(mat.n_spots, device="cuda", requires_grad=True)
    f = quadratic_objective(mat, w, prescription)   # fused: one pass, no dose vector
    f.backward()                      # w.grad = 2 D^T (D w - p) / n

Robust optimisation: ``worst_case_objective`` over the Dij of several
scenarios (max over scenarios, subgradient of the worst one).  A scenario
run with a history budget factor b holds b times the dose per unit weight
(the tables sum over histories, as the reference's unit-weight Dij does);
``DijMatrix(ctx, s, scale=1 / b)`` puts every scenario on one scale.
"""
import torch


class DijMatrix:
    """Handle on the device CSR of one scenario of a context's Dij; the
    products use scale * D."""

    def __init__(self, ctx, scenario=0, scale=1.0):
        self.ctx = ctx
        self.scenario = int(scenario)
        self.scale = float(scale)
        self.nnz, self.n_spots, self.n_voxels = ctx.dij_info(self.scenario)

    def _vec(self, x, n):
        if x.dim() != 1 or x.numel() != n:
            raise ValueError("expected a vector of %d entries, got shape %s" % (n, tuple(x.shape)))
        if not x.is_cuda:
            raise ValueError("the sparse products take device tensors")
        return x.detach().to(torch.float32).contiguous()

    def matvec(self, w, out_dtype=torch.float64):
        """Dose scale * D w (n_voxels)."""
        x = self._vec(w, self.n_spots)
        y = torch.empty(self.n_voxels, dtype=torch.float64, device=x.device)
        stream = torch.cuda.current_stream(x.device).cuda_stream
        self.ctx.dij_matvec(self.scenario, 0, x.data_ptr(), y.data_ptr(), y_double=True, alpha=self.scale,
                            stream=stream)
        return y if out_dtype == torch.float64 else y.to(out_dtype)

    def quadratic(self, w, prescription, voxel_weights=None, want_grad=True):
        """f = mean_v c_v (scale (D w)_v - p_v)^2 as a device scalar (float64)
        and, with want_grad, df/dd = 2 c (d - p) / n_voxels (float32, the
        input of rmatvec), in one pass over the matrix (mqi_dij_quadratic)."""
        w, p, c = self._objective_inputs(w, prescription, voxel_weights)
        f = torch.empty((), dtype=torch.float64, device=w.device)
        g = torch.empty(self.n_voxels, dtype=torch.float32, device=w.device) if want_grad else None
        stream = torch.cuda.current_stream(w.device).cuda_stream
        self.ctx.dij_quadratic(self.scenario, w.data_ptr(), p.data_ptr(), c.data_ptr() if c is not None else 0,
                               self.scale, g.data_ptr() if g is not None else 0, f.data_ptr(), stream=stream)
        return f, g

    def _objective_inputs(self, w, prescription, voxel_weights):
        w = self._vec(w, self.n_spots)
        p = prescription.detach().to(device=w.device, dtype=torch.float64).contiguous()
        if p.dim() != 1 or p.numel() != self.n_voxels:
            raise ValueError("expected a prescription of %d voxels, got shape %s" % (self.n_voxels, tuple(p.shape)))
        c = None
        if voxel_weights is not None:
            c = voxel_weights.detach().to(device=w.device, dtype=torch.float32).contiguous()
            if c.dim() != 1 or c.numel() != self.n_voxels:
                raise ValueError("expected voxel weights of %d voxels" % self.n_voxels)
        return w, p, c

    def rmatvec(self, g, out_dtype=torch.float64):
        """scale * D^T g (n_spots)."""
        return self._adjoint(g, out_dtype)

    def _adjoint(self, g, out_dtype, up=0):
        """scale * D^T g in out_dtype, times the device double at up (unless
        0).  A float64 g is rounded to float32 where the product reads it."""
        double = (g.dtype == torch.float64 and g.dim() == 1 and g.numel() == self.n_voxels and g.is_cuda and
                  g.is_contiguous() and not g.is_neg())
        x = g.detach() if double else self._vec(g, self.n_voxels)
        y_dtype = torch.float32 if out_dtype == torch.float32 else torch.float64
        y = torch.empty(self.n_spots, dtype=y_dtype, device=x.device)
        stream = torch.cuda.current_stream(x.device).cuda_stream
        self.ctx.dij_adjoint(self.scenario, x.data_ptr(), double, up, self.scale, y.data_ptr(),
                             y_dtype == torch.float64, stream=stream)
        return y if y_dtype == out_dtype else y.to(out_dtype)


class _Dose(torch.autograd.Function):
    @staticmethod
    def forward(fctx, w, mat):
        fctx.mat = mat
        fctx.w_dtype = w.dtype
        return mat.matvec(w, torch.float64)

    @staticmethod
    def backward(fctx, grad_dose):
        if type(fctx.mat) is DijMatrix:
            return fctx.mat.rmatvec(grad_dose, fctx.w_dtype), None
        return fctx.mat.rmatvec(grad_dose, torch.float64).to(fctx.w_dtype), None


def dose(mat, w):
    """Differentiable dose D w (float64, n_voxels) of spot weights w."""
    return _Dose.apply(w, mat)


class _Quadratic(torch.autograd.Function):
    @staticmethod
    def forward(fctx, w, mat, prescription, voxel_weights):
        f, g = mat.quadratic(w, prescription, voxel_weights, want_grad=fctx.needs_input_grad[0])
        fctx.mat = mat
        fctx.w_dtype = w.dtype
        if g is not None:
            fctx.save_for_backward(g)
        return f

    @staticmethod
    def backward(fctx, grad_f):
        (g,) = fctx.saved_tensors
        # the upstream factor goes into the product, unless the matrix has a
        # product of its own
        up = _device_scalar(grad_f, g) if type(fctx.mat) is DijMatrix else 0
        if up:
            return fctx.mat._adjoint(g, fctx.w_dtype, up), None, None, None
        grad_w = fctx.mat.rmatvec(g, torch.float64) * grad_f
        return grad_w.to(fctx.w_dtype), None, None, None


def _device_scalar(s, like):
    """Address of s when it is a plain float64 scalar on like's device that
    the product may take by its address, else 0: a graph through s (create_graph)
    or a batch of scalars (is_grads_batched, without storage of its own) takes
    torch's product."""
    if (s.dtype != torch.float64 or s.numel() != 1 or s.device != like.device or s.is_neg() or
            (torch.is_grad_enabled() and s.requires_grad)):
        return 0
    try:
        return s.data_ptr()
    except RuntimeError:
        return 0


def quadratic_objective(mat, w, prescription, voxel_weights=None):
    """f(w) = mean_v c_v (D w - p)_v^2 (c = 1 when voxel_weights is None), in
    one pass over the matrix (the dose is not formed); the gradient is
    D^T (2 c (D w - p) / n)."""
    return _Quadratic.apply(w, mat, prescription, voxel_weights)


def _values(mats, w, prescription, voxel_weights):
    """The objective of every scenario (float64 vector), in one pass of
    launches where the scenarios are distinct ones of one context and size."""
    first = mats[0] if len(mats) else None
    if (first is None or any(type(m) is not DijMatrix for m in mats) or len({m.scenario for m in mats}) < len(mats) or
            any(m.ctx is not first.ctx or m.n_spots != first.n_spots or m.n_voxels != first.n_voxels for m in mats)):
        return torch.stack([m.quadratic(w, prescription, voxel_weights, want_grad=False)[0] for m in mats])
    w, p, c = first._objective_inputs(w, prescription, voxel_weights)
    f = torch.empty(len(mats), dtype=torch.float64, device=w.device)
    stream = torch.cuda.current_stream(w.device).cuda_stream
    first.ctx.dij_quadratics([m.scenario for m in mats], [m.scale for m in mats], w.data_ptr(), p.data_ptr(),
                             c.data_ptr() if c is not None else 0, f.data_ptr(), stream=stream)
    return f


def worst_case_objective(mats, w, prescription, voxel_weights=None):
    """max over scenarios of the quadratic objective (differentiable: the
    gradient is the worst scenario's), and the per-scenario values (a
    detached vector).  The values are evaluated without a graph and only the
    worst scenario's objective is formed again with one, so a backward pass
    runs one D^T g and not one per scenario (a graph over every scenario
    would carry zero gradients through the others).  The products are
    deterministic: the returned maximum equals its entry in the values."""
    with torch.no_grad():
        vals = _values(mats, w, prescription, voxel_weights)
    k = int(torch.argmax(vals).item())
    return quadratic_objective(mats[k], w, prescription, voxel_weights), vals
