"""Memory of the interleaved scoring array that plain passes and passes of
caller-made vertices may take: at most 1 GiB, given back with the scorers, and
the sums are the same with and without it."""
import numpy as np
import pytest
import torch

import phantoms
import refbind as rb
from moquimc_amd import _abi

pytestmark = pytest.mark.gpu

MASK = rb.SC_DOSE | rb.SC_LETD   # three sums: four doubles a voxel


@pytest.fixture
def own():
    c = _abi.Context(0)
    yield c
    c.close()


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _plan(ctx, n):
    g = phantoms.water_box(n, n, n, dx=1.0, dz=1.0)
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    ctx.set_spots(phantoms.spots([100.0, 120.0, 140.0, 160.0], 10000, sigma=4.0, sigma_e_frac=0.01))


def _pass(ctx, vertices, batched=False):
    cfg = ctx.config(seed=5, batched=batched)
    if vertices:
        rng = np.random.default_rng(3)
        v = np.zeros((40000, 7), np.float32)
        v[:, 0] = rng.uniform(60, 160, len(v))
        v[:, 1:3] = rng.normal(0, 4, (len(v), 2))
        v[:, 3] = 0.5
        v[:, 6] = -1.0
        ctx.run_vertices(v, cfg)
    else:
        ctx.run(cfg)
    return [ctx.scorer(k) for k in range(ctx.scorer_count())]


@pytest.mark.parametrize("vertices", [False, True])
def test_a_large_grid_is_scored_without_the_array(own, vertices):
    """340^3 voxels: the array would be 1.26 GB."""
    _plan(own, 340)
    own.set_scorers(rb.SC_DOSE)
    _pass(own, vertices)         # stacks and work lists
    own.set_scorers(MASK)
    before = _free()
    plain = _pass(own, vertices)
    assert before - _free() <= 64 << 20
    if not vertices:
        own.zero_scorers()
        batched = _pass(own, vertices, batched=True)   # which does take it
        assert before - _free() > 1 << 30
        for a, b in zip(plain, batched):
            assert a.any() and np.allclose(a, b, rtol=1e-12, atol=0)


@pytest.mark.parametrize("vertices", [False, True])
def test_the_array_goes_with_the_scorers(own, vertices):
    """200^3 voxels: 256 MB, held until the scorers are set anew."""
    _plan(own, 200)
    own.set_scorers(rb.SC_DOSE)
    _pass(own, vertices)
    before = _free()
    own.set_scorers(MASK)
    _pass(own, vertices)
    assert before - _free() > 300 << 20   # two more scorers and the array
    own.set_scorers(rb.SC_DOSE)
    assert before - _free() <= 64 << 20
