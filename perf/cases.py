"""The timed work of this framework: transports of spot plans and caller-made
vertices, dose-influence matrices, and the products and objectives over them,
each through the public Python entry points (moquimc_amd._abi.Context,
moquimc_amd.dij).

A case is a dict of plain values.  Its "kind" says which entry points it
drives:

  plan       Context.run of a spot plan (one batched launch, or one launch per
             spot) into dense scorers
  vertices   Context.run_vertices of caller-made vertices into dense scorers
  dij        Context.run with the Dij scorer, then Context.dij_build: one CSR
             matrix per scenario
  product    dij.dose forward and backward (D w, then D^T g) over a caller's
             CSR
  objective  dij.quadratic_objective (one scenario) or
             dij.worst_case_objective (several) forward and backward over a
             caller's CSR

Outputs are the scorers', the matrices' or the gradients' own device arrays.
"""
import ctypes

import numpy as np
import torch

from moquimc_amd import _abi, dij, workloads

DEVICE = "cuda:0"

SCORERS = {
    "dose": _abi.SCORE_DOSE,
    "dose+stat": _abi.SCORE_DOSE | _abi.SCORE_STAT,
    "dose+letd": _abi.SCORE_DOSE | _abi.SCORE_LETD,
    "dose+letd+lett": _abi.SCORE_DOSE | _abi.SCORE_LETD | _abi.SCORE_LETT,
}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # commissioning: one pencil beam in a water tank at 1e5 histories with
        # the phantom build's physics; fewer histories than the device's lanes
        # hold, so the longest track sets the time
        dict(name="water-spot", kind="plan", body="water", nx=200, ny=200, nz=350, spots=1, layers=1, h_lo=100000,
             h_hi=100000, scorers="dose", batched=True),
        # the slab phantom of the dose + LETd workload: 25 spots 70-230 MeV
        # through water, lung and bone
        dict(name="slab-letd", kind="plan", body="slabs", nx=200, ny=200, nz=350, spots=25, layers=25, h_lo=100000,
             h_hi=100000, scorers="dose+letd", batched=True),
        # a whole treatment field on the full-resolution CT: 2000 spots,
        # 1e3-1e5 histories each, dose and the statistics pair
        dict(name="ct-field", kind="plan", body="ct", nx=512, ny=512, nz=200, spots=2000, layers=20, h_lo=1000,
             h_hi=100000, scorers="dose+stat", batched=True),
        # a quick look at a small field on a coarse, odd-sized CT: few
        # histories per spot
        dict(name="ct-preview", kind="plan", body="ct", nx=131, ny=127, nz=67, spots=150, layers=6, h_lo=200,
             h_hi=1500, scorers="dose", batched=True),
        # one launch per spot, the reference's own run loop (run_by_spot)
        dict(name="ct-per-spot", kind="plan", body="ct", nx=256, ny=256, nz=128, spots=40, layers=4, h_lo=2000,
             h_hi=20000, scorers="dose+stat", batched=False),
        # vertices made by the caller (a phase-space file), all LET scorers
        dict(name="vertices-let", kind="vertices", body="slabs", nx=100, ny=100, nz=175, histories=300000,
             scorers="dose+letd+lett"),
        # the influence matrix of one field: transport with the Dij scorer
        # and the CSR built from its tables
        dict(name="dij-field", kind="dij", body="ct", nx=256, ny=256, nz=128, spots=400, layers=20, h_lo=5000,
             h_hi=5000, scenarios=1),
        # influence matrices under nine setup and range scenarios
        dict(name="dij-robust", kind="dij", body="ct", nx=201, ny=211, nz=73, spots=60, layers=6, h_lo=500,
             h_hi=5000, scenarios=9),
        # an optimiser's dose and gradient step over a field's matrix
        dict(name="dose-step", kind="product", nx=256, ny=256, nz=128, rows=1000, layers=25, reach=40.0),
        # the fused quadratic objective with voxel weights over the same
        # kind of matrix
        dict(name="objective-weights", kind="objective", nx=256, ny=256, nz=128, rows=1000, layers=25, reach=40.0,
             scenarios=1, weights=True),
        # a small matrix (a tutorial plan, a coarse preview): launches and
        # host work count
        dict(name="objective-small", kind="objective", nx=41, ny=53, nz=29, rows=60, layers=4, reach=24.0,
             scenarios=1, weights=False),
        # robust optimisation: the worst of nine scenarios and its gradient
        dict(name="worst-case", kind="objective", nx=160, ny=120, nz=90, rows=300, layers=10, reach=40.0,
             scenarios=9, weights=False),
    ]


def _log(rng, lo, hi):
    return int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))


def draw(rng):
    kind = rng.choice(["plan", "plan", "plan", "vertices", "dij", "product", "objective", "objective"])
    if kind in ("plan", "vertices"):
        body = rng.choice(["water", "slabs", "ct"]) if kind == "plan" else rng.choice(["water", "slabs"])
        if body == "ct":
            nx, ny, nz = rng.randint(90, 300), rng.randint(90, 300), rng.randint(40, 140)
        else:
            nx, ny, nz = rng.randint(40, 200), rng.randint(40, 200), rng.randint(100, 350)
        c = dict(kind=kind, body=body, nx=nx, ny=ny, nz=nz,
                 scorers=rng.choice(sorted(SCORERS)) if body != "water" else "dose")
        if kind == "vertices":
            c["histories"] = _log(rng, 3000, 1000000)
            return c
        c["batched"] = rng.random() < 0.8
        c["spots"] = 1 if body == "water" else 25 if body == "slabs" else _log(rng, 20, 800 if c["batched"] else 50)
        c["layers"] = min(c["spots"], rng.randint(1, 20))
        # at most 1e7 histories batched, 1e6 with a launch per spot
        top = (1e5 if body == "water" else 1e7 if c["batched"] else 1e6) / c["spots"]
        c["h_hi"] = max(20, _log(rng, min(500, top), top))
        c["h_lo"] = max(10, int(c["h_hi"] * rng.choice([0.01, 0.1, 1.0])))
        return c
    if kind == "dij":
        n = rng.choice([1, 1, 3, 9])
        spots = _log(rng, 10, 400 if n == 1 else 60)
        return dict(kind=kind, body="ct", nx=rng.randint(90, 256), ny=rng.randint(90, 256), nz=rng.randint(40, 128),
                    spots=spots, layers=min(spots, rng.randint(1, 20)), h_lo=_log(rng, 200, 1000),
                    h_hi=_log(rng, 1000, 5000), scenarios=n)
    n = 1 if kind == "product" else rng.choice([1, 1, 3, 9])
    c = dict(kind=kind, nx=rng.randint(30, 256), ny=rng.randint(30, 256), nz=rng.randint(20, 128),
             rows=_log(rng, 20, 1000 if n == 1 else 300), layers=rng.randint(1, 25), reach=rng.uniform(15.0, 40.0))
    if kind == "objective":
        c["scenarios"] = n
        c["weights"] = rng.random() < 0.5
    return c


# ------------------------------------------------------------------ plans
# extents (mm) of the bodies: a case's voxel counts divide them
CT_X, CT_Y, CT_Z = 501.76, 501.76, 400.0
TANK_XY, TANK_Z = 100.0, 350.0


def _edges(case):
    if case["body"] == "ct":
        return [workloads.uniform_edges(-e / 2, e / 2, n)
                for e, n in ((CT_X, case["nx"]), (CT_Y, case["ny"]), (CT_Z, case["nz"]))]
    return [workloads.uniform_edges(-TANK_XY / 2, TANK_XY / 2, case["nx"]),
            workloads.uniform_edges(-TANK_XY / 2, TANK_XY / 2, case["ny"]),
            workloads.uniform_edges(-TANK_Z, 0, case["nz"])]


def _spots(case, rng):
    """Spots of the case's body with histories log-uniform in [h_lo, h_hi]:
    one 200 MeV spot (water), 70-230 MeV on a square grid (slabs), energy
    layers of 100-180 MeV on a 5 mm hexagonal grid (ct)."""
    n = case["spots"]
    hist = np.round(np.exp(rng.uniform(np.log(case["h_lo"]), np.log(case["h_hi"]), n))).astype(int)
    if case["body"] == "water":
        return [workloads.spot(200.0, 3.0, hist[0], z=0.5)]
    if case["body"] == "slabs":
        side = int(np.ceil(np.sqrt(n)))
        out = []
        for k in range(n):
            e = float(np.float32(rng.uniform(70.0, 230.0)))
            pos = (-20.0 + 40.0 * (k % side) / max(1, side - 1), -20.0 + 40.0 * (k // side) / max(1, side - 1))
            out.append(workloads.spot(e, 4.0, hist[k], pos=pos, z=0.5, sigma_e=0.01 * e))
        return out
    layers = max(1, min(case["layers"], n))
    pos = workloads.hex_positions(-(-n // layers), 5.0)
    out = []
    for k in range(n):
        e = float(np.float32(100.0 + 80.0 * (k % layers + 0.5) / layers))
        p = pos[k // layers]
        out.append(workloads.spot(e, 4.0, hist[k], pos=(float(p[0]), float(p[1])), sigma_e=0.01 * e,
                                  rotation=workloads.ROT_PLUS_Y, translation=(0.0, -130.0, 0.0)))
    return out


def _context(case, seed):
    """A context with the case's body as its grid."""
    xe, ye, ze = _edges(case)
    ctx = _abi.Context(0)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["body"] == "ct":
        hu = workloads.synthetic_ct(nx, ny, nz, CT_X / nx, CT_Y / ny, CT_Z / nz, seed,
                                    z_half=200.0 if case["kind"] == "dij" else None)
        ctx.set_grid_hu(xe, ye, ze, hu)
    elif case["body"] == "slabs":
        ctx.set_grid(xe, ye, ze, workloads.slab_density(ze, nx * ny))
    else:
        ctx.set_grid(xe, ye, ze, np.full(nx * ny * nz, 1.0e-3, np.float32))
    return ctx


class _DeviceArray:
    """An array of a context's device memory; keeps the context alive."""

    def __init__(self, ctx, ptr, shape, typestr):
        self.ctx = ctx
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape), "typestr": typestr,
                                         "version": 2}


def _view(ctx, ptr, shape, typestr):
    return torch.as_tensor(_DeviceArray(ctx, ptr, shape, typestr), device=DEVICE)


def _scorers(ctx):
    return [_view(ctx, ctx.scorer_device_ptr(k), ctx.shape, "<f8") for k in range(ctx.scorer_count())]


# ------------------------------------------------------------------ matrices
def _geometry(case):
    """Per spot of a synthetic influence matrix: lateral centre (voxels) and
    depth reached (voxels), and the half-widths of a spot's box."""
    rows, layers = case["rows"], max(1, min(case["layers"], case["rows"]))
    dx, dz = 500.0 / 256, 4.0   # mm
    hx = max(2, min(int(case["reach"] / dx), case["nx"] // 2))
    hz = max(1, min(int(case["reach"] / dz), case["nz"] // 2))
    pos = workloads.hex_positions(-(-rows // layers), 5.0)
    k = np.arange(rows)
    cx = case["nx"] / 2 + pos[k % len(pos), 0] / dx
    cz = case["nz"] / 2 + pos[k % len(pos), 1] / dz
    depth = np.round(case["ny"] * (0.35 + 0.5 * (k // len(pos) + 0.5) / layers)).astype(int)
    return dx, dz, hx, hz, cx, cz, np.clip(depth, 2, case["ny"])


def _matrix(case, seed, scenario, device=DEVICE):
    """A pencil-beam influence matrix as a CSR (rows = spots, columns = voxels,
    x fastest): a core every spot reaches around its axis and a halo thinning
    out with the distance from it, values falling off laterally.  Made on the
    device from the seed; (indptr int64, indices int32, values float32)."""
    gen = torch.Generator(device=device).manual_seed(1000003 * int(seed) + 101 * scenario + 17)
    dx, dz, hx, hz, cx, cz, depth = _geometry(case)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    rows = case["rows"]
    shift = np.random.default_rng(int(seed) * 31 + scenario).uniform(-1.0, 1.0, 2)
    ox = torch.arange(-hx, hx + 1, device=device)
    oz = torch.arange(-hz, hz + 1, device=device)
    yy = torch.arange(ny, device=device)
    counts, cols, vals = [], [], []
    step = max(1, int(4.0e6 / (ny * len(ox) * len(oz))))
    for r0 in range(0, rows, step):
        r1 = min(rows, r0 + step)
        ax = torch.tensor(cx[r0:r1] + shift[0], device=device, dtype=torch.float32)
        az = torch.tensor(cz[r0:r1] + shift[1], device=device, dtype=torch.float32)
        dp = torch.tensor(depth[r0:r1], device=device)
        ix = ax.round().long()[:, None] + ox[None, :]
        iz = az.round().long()[:, None] + oz[None, :]
        rx = (ix.float() - ax[:, None]) * dx
        rz = (iz.float() - az[:, None]) * dz
        r = torch.sqrt(rz[:, :, None, None] ** 2 + rx[:, None, None, :] ** 2)       # spot, z, 1, x
        core = (12.0 + 10.0 * yy.float() / ny)[None, None, :, None]                # widens with depth
        p = torch.exp(-(r - core).clamp(min=0.0) / 10.0)
        keep = torch.rand(p.shape, generator=gen, device=device) < p
        keep &= (yy[None, :] < dp[:, None])[:, None, :, None]
        keep &= ((iz >= 0) & (iz < nz))[:, :, None, None] & ((ix >= 0) & (ix < nx))[:, None, None, :]
        lin = (iz[:, :, None, None] * ny + yy[None, None, :, None]) * nx + ix[:, None, None, :]
        v = torch.exp(-0.5 * (r / 6.0) ** 2) * (0.2 + torch.rand(p.shape, generator=gen, device=device)) + 1.0e-4
        cols.append(lin[keep].to(torch.int32))
        vals.append(v[keep].to(torch.float32) * 1.0e-7)
        counts.append(keep.sum(dim=(1, 2, 3)))
    indptr = torch.zeros(rows + 1, dtype=torch.int64, device=device)
    indptr[1:] = torch.cumsum(torch.cat(counts), 0)
    return indptr, torch.cat(cols), torch.cat(vals)


def _voxels(case):
    return case["nx"] * case["ny"] * case["nz"]


def _spot_weights(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(7919 * int(seed) + 5)
    return (torch.rand(case["rows"], generator=gen, device=DEVICE) + 0.5).to(torch.float32)


def _dose_gradient(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(7919 * int(seed) + 6)
    # as an objective gives it: float32 residuals over the voxels
    return torch.randn(_voxels(case), generator=gen, device=DEVICE, dtype=torch.float32).double()


def _prescription(case, seed):
    """Dose asked for: a level inside a sphere around the middle, 0 outside;
    and the voxel weights: 1 there, 0.1-0.6 elsewhere."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    dx, dz = 500.0 / 256, 4.0
    z = (torch.arange(nz, device=DEVICE) - nz / 2) * dz
    y = (torch.arange(ny, device=DEVICE) - ny / 2) * dx
    x = (torch.arange(nx, device=DEVICE) - nx / 2) * dx
    inside = z[:, None, None] ** 2 + y[None, :, None] ** 2 + x[None, None, :] ** 2 <= 30.0 ** 2
    inside = inside.reshape(-1)
    gen = torch.Generator(device=DEVICE).manual_seed(7919 * int(seed) + 7)
    level = 1.0e-6 * (1.0 + torch.rand((), generator=gen, device=DEVICE, dtype=torch.float64))
    c = torch.where(inside, 1.0, 0.1 + 0.5 * torch.rand(_voxels(case), generator=gen, device=DEVICE))
    return torch.where(inside, level, torch.zeros_like(level)), c.to(torch.float32)


# ------------------------------------------------------------------ prepare / run
def prepare(case, seed):
    rng = np.random.default_rng(int(seed) * 7 + 3)
    kind = case["kind"]
    if kind in ("plan", "dij"):
        ctx = _context(case, seed)
        debug = case["body"] == "water"
        if case.get("scenarios", 1) > 1:
            shifts, scales, budgets = workloads.robust_scenarios()
            n = case["scenarios"]
            ctx.set_scenarios(shifts[:n], scales[:n], budgets[:n])
        ctx.set_spots(_spots(case, rng))
        ctx.set_scorers(SCORERS[case["scorers"]] if kind == "plan" else _abi.SCORE_DOSE)
        # the tables of a spot's matrix row grow with the root of its histories
        more = dict(dij=True, dij_slots_sqrt=4096) if kind == "dij" else dict(batched=case["batched"])
        state = dict(case=case, ctx=ctx, cfg=ctx.config(seed=int(seed) + 1, physics_debug=debug, **more))
        if kind == "dij":
            # the program's own arrays of every scenario's matrix
            cap = int(case["spots"] * 2200 * np.sqrt(2 * case["h_hi"]))
            state["rows"] = [(torch.empty(cap, dtype=torch.int32, device=DEVICE),
                              torch.empty(cap, dtype=torch.float32, device=DEVICE))
                             for _ in range(case["scenarios"])]
        return state
    if kind == "vertices":
        ctx = _context(case, seed)
        ctx.set_scorers(SCORERS[case["scorers"]])
        n = case["histories"]
        v = np.zeros((n, 7), np.float32)
        v[:, 0] = rng.uniform(70.0, 230.0, n)                   # MeV
        v[:, 1:3] = rng.normal(0.0, 4.0, (n, 2))                # mm
        v[:, 3] = 0.5
        v[:, 4:6] = rng.normal(0.0, 0.003, (n, 2))
        v[:, 6] = -np.sqrt(1.0 - v[:, 4] ** 2 - v[:, 5] ** 2)
        debug = case["body"] == "water"
        return dict(case=case, ctx=ctx, vertices=v, cfg=ctx.config(seed=int(seed) + 1, physics_debug=debug))
    ctx = _abi.Context(0)
    n = case.get("scenarios", 1)
    for s in range(n):
        ip, ix, v = (t.cpu().numpy() for t in _matrix(case, seed, s))
        ctx.dij_set_csr(ip, ix, v, (case["rows"], _voxels(case)), scenario=s)
    state = dict(case=case, ctx=ctx, mats=[dij.DijMatrix(ctx, s) for s in range(n)], w=_spot_weights(case, seed))
    if kind == "product":
        state["g"] = _dose_gradient(case, seed)
    else:
        state["p"], c = _prescription(case, seed)
        state["c"] = c if case["weights"] else None
    return state


def run(state):
    kind, ctx = state["case"]["kind"], state["ctx"]
    if kind == "plan":
        ctx.zero_scorers()
        ctx.run(state["cfg"])
        return _scorers(ctx)
    if kind == "vertices":
        ctx.zero_scorers()
        ctx.run_vertices(state["vertices"], state["cfg"])
        return _scorers(ctx)
    if kind == "dij":
        ctx.zero_scorers()
        ctx.run(state["cfg"])
        ctx.dij_build(1.0e-4)
        out = []
        for s, (cols, vals) in enumerate(state["rows"]):
            nnz, rows, _ = ctx.dij_info(s)
            ip, ix, v = (ctypes.c_void_p() for _ in range(3))
            if _abi.lib().mqi_dij_device_ptrs(ctx.h, s, ctypes.byref(ip), ctypes.byref(ix), ctypes.byref(v)):
                raise RuntimeError("mqi_dij_device_ptrs failed")
            # into the arrays the program keeps (0 behind the last entry)
            cols[:nnz] = _view(ctx, ix.value, (nnz,), "<i4")
            vals[:nnz] = _view(ctx, v.value, (nnz,), "<f4")
            cols[nnz:] = 0
            vals[nnz:] = 0
            out += [_view(ctx, ip.value, (rows + 1,), "<i8"), cols, vals]
        return out + _scorers(ctx)
    w = state["w"].clone().requires_grad_(True)
    if kind == "product":
        d = dij.dose(state["mats"][0], w)
        d.backward(state["g"])
        return [d.detach(), w.grad]
    if len(state["mats"]) == 1:
        f = dij.quadratic_objective(state["mats"][0], w, state["p"], state["c"])
        f.backward()
        return [f.detach(), w.grad]
    f, vals = dij.worst_case_objective(state["mats"], w, state["p"], state["c"])
    f.backward()
    return [f.detach(), vals, w.grad]


# ------------------------------------------------------------------ exact
def exact(case, seed):
    """The products and objectives in 64 bits (plain torch).  A transport has
    no such value: its tracks are sampled in float arithmetic."""
    if case["kind"] not in ("product", "objective"):
        return None
    w = _spot_weights(case, seed).double()
    n = _voxels(case)

    def rows_cols_vals(s):
        ip, ix, v = _matrix(case, seed, s)
        rows = torch.repeat_interleave(torch.arange(case["rows"], device=DEVICE), ip.diff())
        return rows, ix.long(), v.double()

    def dose(m):
        return torch.zeros(n, dtype=torch.float64, device=DEVICE).index_add_(0, m[1], m[2] * w[m[0]])

    def adjoint(m, g):
        return torch.zeros(case["rows"], dtype=torch.float64, device=DEVICE).index_add_(0, m[0], m[2] * g[m[1]])

    if case["kind"] == "product":
        m = rows_cols_vals(0)
        return [dose(m), adjoint(m, _dose_gradient(case, seed))]
    p, c = _prescription(case, seed)
    c = c.double() if case["weights"] else torch.ones_like(p)
    vals, grads = [], []
    for s in range(case["scenarios"]):
        m = rows_cols_vals(s)
        r = dose(m) - p
        vals.append((c * r * r).mean())
        grads.append(adjoint(m, 2.0 * c * r / n))
    k = int(torch.argmax(torch.stack(vals)))
    if case["scenarios"] == 1:
        return [vals[0], grads[0]]
    return [vals[k], torch.stack(vals), grads[k]]


# ------------------------------------------------------------------ work
def work(case):
    """Bytes: each input read once, each output written once.  Operations of
    a transport: about 400 per voxel step, the steps taken as the voxels along
    the primaries' paths."""
    kind = case["kind"]
    if kind in ("plan", "vertices", "dij"):
        nvox = _voxels(case)
        if kind == "vertices":
            hist, n_arrays, scen = float(case["histories"]), {"dose": 1, "dose+stat": 3, "dose+letd": 3,
                                                              "dose+letd+lett": 5}[case["scorers"]], 1.0
        else:
            lo, hi = case["h_lo"], case["h_hi"]
            mean = (hi - lo) / np.log(hi / lo) if hi > lo else float(lo)
            scen = float(case.get("scenarios", 1))
            hist = case["spots"] * mean * (1.0 if scen == 1 else scen + 1.0)   # the nominal one twice
            n_arrays = {"dose": 1, "dose+stat": 3, "dose+letd": 3, "dose+letd+lett": 5}[case.get("scorers", "dose")]
        if case["body"] == "ct":
            path = 180.0 / (CT_Y / case["ny"]) * 1.2
        else:
            path = 200.0 / (TANK_Z / case["nz"]) * 1.2
        bytes_ = nvox * (4.0 + 8.0 * n_arrays)
        if kind == "dij":
            bytes_ += 8.0 * hist / case["spots"] ** 0.5 * 20.0   # the rows, which grow with the root of the histories
        return {"bytes": float(bytes_), "flops": float(hist * path * 400.0)}
    dx, dz, hx, hz, _, _, depth = _geometry(case)
    ox, oz = np.arange(-hx, hx + 1) * dx, np.arange(-hz, hz + 1) * dz
    r = np.hypot(ox[None, :], oz[:, None])
    nnz = float(np.exp(-np.clip(r - 15.0, 0.0, None) / 10.0).sum() * depth.sum()) * case.get("scenarios", 1)
    n, rows = float(_voxels(case)), float(case["rows"])
    if kind == "product":     # both products read the matrix; g and the dose are float64
        return {"bytes": 2 * 8.0 * nnz + 16.0 * n + 16.0 * rows, "flops": 4.0 * nnz}
    # every scenario's objective, and the adjoint of one of them
    adj = nnz / case["scenarios"]
    return {"bytes": 8.0 * (nnz + adj) + (12.0 if case["weights"] else 8.0) * n * case["scenarios"] + 8.0 * rows,
            "flops": 2.0 * (nnz + adj)}
