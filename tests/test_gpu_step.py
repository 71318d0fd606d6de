"""The production kernels' step arithmetic (mqi_prod.hpp) on the device,
through mqi_physics_probe, against the committed values of the reference
(tests/golden/reference_functions.npz) and FP64 restatements on the edges of
its branches and tables.

Tolerances: the stopping power ratio 2e-6 absolute ((rho^-0.7 - 1) cancels
near water), the radiation length 8 float ulp (1e-6 relative), interpolated
tables 1e-4 relative and 1e-6 of the table's maximum (a bin edge at 300 MeV is
rounded to 3e-5 MeV, 6e-5 of the 0.5 MeV bin)."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
FUNCS = os.path.join(HERE, "golden", "reference_functions.npz")
TABLES = os.path.join(HERE, "golden", "reference_tables.npz")


def _near(x):
    """x as float32 with its neighbours."""
    x = np.float32(x)
    return [np.nextafter(x, np.float32(-np.inf)), x, np.nextafter(x, np.float32(np.inf))]


@pytest.mark.parametrize("dbg", [0, 1])
def test_production_spr_and_radiation_length_against_the_reference_values(ctx, dbg):
    g = np.load(FUNCS)
    rho, ek = np.ascontiguousarray(g["rho"]), np.ascontiguousarray(g["ek"])
    s = ctx.physics_probe(0, rho, ek, exact=False, physics_debug=dbg)
    x = ctx.physics_probe(1, rho, exact=False, physics_debug=dbg)
    assert np.abs(s.astype(np.float64) - g["spr_%d" % dbg]).max() <= 2e-6
    assert (np.abs(x.astype(np.float64) - g["x0_%d" % dbg]) <= 1e-6 * g["x0_%d" % dbg]).all()


@pytest.mark.parametrize("dbg", [0, 1])
def test_production_materials_at_branch_edges(ctx, dbg):
    """Densities (g/mm^3) one float around every threshold: 0.0012, 0.26 and
    0.9 g/cm^3, and the phantom build's water window."""
    rho = np.array([v for c in (1.2e-6, 0.26e-3, 0.9e-3, 0.999e-3, 1.001e-3, 1e-3, 2.5e-3, 5e-7) for v in _near(c)],
                   np.float32)
    ek = np.tile(np.array([0.5, 70.0, 230.0], np.float32), 8)
    s = ctx.physics_probe(0, rho, ek, exact=False, physics_debug=dbg)
    x = ctx.physics_probe(1, rho, exact=False, physics_debug=dbg)
    d = (rho * np.float32(1000)).astype(np.float64)   # the float product the branches see
    e = ek.astype(np.float64)
    fit = 1.0123 - 3.386e-5 * e + 0.291 * (1 + e ** -0.3421) * (d ** -0.7 - 1)
    low = 0.8815 + (d - 0.0012) * (0.9925 - 0.8815) / (0.26 - 0.0012)
    mid = 0.9925 + (d - 0.26) * (fit - 0.9925) / (0.9 - 0.26)
    want = np.where(d < 0.0012, 0.0, np.where(d <= 0.26, low, np.where(d < 0.9, mid, fit)))
    f = np.where(d <= 0.26, 0.9857 + 0.0085 * d,
                 np.where(d <= 0.9, 1.0446 - 0.2180 * d, 1.19 + 0.44 * np.log(np.maximum(d - 0.44, 1e-3))))
    x0 = 0.360863 / (d * 0.001 * f)
    if dbg:
        water = np.abs(d - 1.0) < 1e-3
        want = np.where(water, 1.0, want)
        x0 = np.where(water, 360.863, x0)
    assert np.array_equal(s == 0, want == 0)
    assert np.abs(s - want).max() <= 2e-6
    assert (np.abs(x - x0) <= 1e-6 * x0).all()


def test_production_tables_at_their_edges(ctx):
    """The first and last bins of both index grids, bin edges and the
    energies outside them."""
    t = np.load(TABLES)
    e = np.array([v for c in (0.1, 0.5, 0.6, 1.0, 1.1, 100.1, 100.5, 299.1, 299.5) for v in _near(c)]
                 + [0.0, 0.05, 299.7, 300.5, 310.0], np.float32)
    got = ctx.physics_probe(2, np.full(e.size, 1.0, np.float32), e, exact=False)

    def table(name, lo, hi, first):
        y = np.concatenate([t[name].astype(np.float64), [0.0]])
        v = e.astype(np.float64)
        i = np.clip(((e - np.float32(lo)) * 2).astype(np.int64), 0, 599)
        x0 = first + 0.5 * i
        out = y[i] + (v - x0) * (y[i + 1] - y[i]) / 0.5
        return np.where((e >= np.float32(lo)) & (e <= np.float32(hi)), out, 0.0)

    ion = table("cs_p_ion", 0.1, 299.6, float(np.float32(0.1)))
    dedx = table("dedx_restricted", 0.1, 299.6, float(np.float32(0.1)))
    dedx = np.where((e < np.float32(0.1)) & (e > 0), t["dedx_restricted"][0], dedx)
    for k, want in ((0, ion), (1, table("cs_pp_e", 0.5, 300, 0.5)), (2, table("cs_po_e", 0.5, 300, 0.5)),
                    (3, table("cs_po_i", 0.5, 300, 0.5)), (4, -dedx)):
        scale = np.abs(want).max()
        assert (np.abs(got[:, k] - want) <= 1e-4 * np.abs(want) + 1e-6 * scale).all(), k
        assert np.array_equal(got[:, k] == 0, want == 0), k


@pytest.mark.parametrize("shape,dx,dz", [((20, 24, 30), 2.5, 3.0), ((1, 7, 65), 11.0, 0.75), ((64, 3, 2), 0.5, 40.0)])
def test_production_vacuum_traversal_equals_the_oracle(ctx, shape, dx, dz):
    """Voxel exits with both directions of an axis in one expression: rays on
    edges, along axes and from outside, bit for bit (the oracle's traversal is
    pinned to the reference)."""
    import phantoms
    import refbind as rb
    from test_gpu_exact import _assert_trace_equal, _split_ref, _vacuum_rays
    g = phantoms.water_box(*shape, dx=dx, dz=dz, rho=0.0)
    rays = _vacuum_rays(g, 300, 17)
    ref = _split_ref(*rb.oracle_trace(g, rays, debug=1, prec=32, rng=1, math=1), len(rays))
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    ctx.set_scorers(rb.SC_DOSE)
    cnb, rec, nst = ctx.trace(ctx.config(seed=5, exact=False, batched=False), len(rays), 400, vertices=rays)
    _assert_trace_equal(cnb, rec, nst, ref)


@pytest.mark.parametrize("histories", [1, 3, 63, 65, 1025])
@pytest.mark.parametrize("mask", [1, 4, 5, 2, 3, 18, 19, 16 + 32, 32 + 64])
def test_grouped_flush_equals_the_plain_launch(ctx, histories, mask):
    """Every number of grouped scorers (1, the pair, three and four, and five
    with one beyond the deferred slots) at history counts around a group, a
    wave and a workgroup: a batched pass adds the same deposits as one launch
    per spot (the sums differ in FP64 order only)."""
    import phantoms
    g = phantoms.slab_box(9, 11, 90)
    sp = phantoms.spots([90.0, 60.0], histories, sigma=3.0, sigma_e_frac=0.01, positions=[(0, 0, 0.5), (2, -1, 0.5)])
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    ctx.set_scenarios([[0, 0, 0], [1, 0, 0]], [1.0, 0.9])
    ctx.set_spots(sp)
    for per_scenario in (False, True):
        ctx.set_scorers(mask, per_scenario)
        out = []
        for batched in (True, False):
            ctx.zero_scorers()
            r = ctx.run(ctx.config(seed=3, batched=batched))
            assert r.histories == 4 * histories
            out.append([ctx.scorer(k, s) for k in range(ctx.scorer_count()) for s in range(2 if per_scenario else 1)])
        for a, b in zip(*out):
            assert histories == 1 or b.sum() > 0   # a single proton may pass beside the box
            assert np.allclose(a, b, rtol=1e-12, atol=0)
    ctx.set_scenarios()
