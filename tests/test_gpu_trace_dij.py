"""A trace with a Dij config does not look into the Dij tables: they are the
last Dij run's, of fewer spots here than the traced plan has."""
import numpy as np
import pytest

import phantoms
import refbind as rb
from moquimc_amd import _abi

pytestmark = pytest.mark.gpu


@pytest.fixture
def own():
    c = _abi.Context(0)
    yield c
    c.close()


def _plan(ctx, n_spots):
    g = phantoms.slab_box(9, 7, 41)
    sp = phantoms.spots([62.0 + 3 * i for i in range(n_spots)], 40, sigma=1.5, sigma_e_frac=0.01,
                        positions=[((i % 3) - 1.0, (i % 2) - 0.5, 0.5) for i in range(n_spots)])
    ctx.set_grid(g.xe, g.ye, g.ze, g.density)
    ctx.set_spots(sp)
    ctx.set_scorers(rb.SC_DOSE)


def test_trace_before_any_dij_run_is_refused(own):
    _plan(own, 2)
    with pytest.raises(RuntimeError):
        own.trace(own.config(seed=8, dij=True), 80, 300)


@pytest.mark.parametrize("exact", [True, False])
def test_trace_leaves_the_tables_alone(own, exact):
    _plan(own, 1)
    own.run(own.config(seed=8, batched=True, dij=True, dij_capacity=2048))
    own.dij_build(0.0)
    before = own.dij_csr(0)
    _plan(own, 6)
    want = own.trace(own.config(seed=8, exact=exact), 240, 300)
    got = own.trace(own.config(seed=8, exact=exact, dij=True), 240, 300)
    assert want[2].max() > 1
    for a, b in zip(want, got):
        assert np.array_equal(a, b)
    for a, b in zip(before, own.dij_csr(0)):
        assert np.array_equal(a, b)
