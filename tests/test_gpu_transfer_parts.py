"""Results and states that go through less scratch than they need at once: a
context that finds no room for it (debug_fill_nan=5), and an element state
larger than the scratch grows to (128 MiB)."""
import numpy as np
import pytest

import cppimpact_amd as ci
from cppimpact_amd import _lib as L

from common import E, H, NU, RHO, SY

pytestmark = pytest.mark.gpu


def run(n, quad, **opts):
    x, conn = ci.box_mesh(n, n, n, 0.25, 0.25, 0.25, origin=(0.0, 0.0, 1e-6), quadratic=quad,
                          jitter=0.1, seed=3)
    x = np.vstack([x[:7], [[0.5, 0.5, 0.5]], x[7:]])  # a node of no element
    conn = np.where(conn >= 7, conn + 1, conn).astype(np.int32)
    d = ci.Dynamics(ci.Mesh.from_arrays(x, conn), ci.Elastoplastic(E, RHO, NU, 1.0, H, SY), None,
                    physics=L.PHYSICS_EP, **opts)
    d._x0 = x + np.random.default_rng(1).uniform(-1, 1, x.shape) * 1e-3 / n
    d.vel[:] = np.random.default_rng(2).uniform(-100, 100, x.shape)
    d.init(1e-8)
    d.step(7)
    out = list(d.fetch()) + [d.global_mass] + list(d.element_state())
    st, ss = np.full((len(x), 6), 7.0), np.full((len(x), 6), 8.0)
    L.check(L.lib().cpi_get_stress_strain(d.ctx, L.dptr(st), L.dptr(ss)), d.ctx)
    assert (st[7] == 7.0).all() and (ss[7] == 8.0).all()
    du, only = np.empty_like(x), np.full((len(x), 6), 8.0)
    L.check(L.lib().cpi_get_increment(d.ctx, L.dptr(du)), d.ctx)
    L.check(L.lib().cpi_get_stress_strain(d.ctx, None, L.dptr(only)), d.ctx)
    assert np.array_equal(only, ss)
    ep = np.empty(out[-1].shape)
    L.check(L.lib().cpi_get_element_state(d.ctx, None, L.dptr(ep)), d.ctx)
    assert np.array_equal(ep, out[-1])
    m = np.empty(len(x))
    L.check(L.lib().cpi_get_state(d.ctx, None, None, None, L.dptr(m), None), d.ctx)
    assert np.array_equal(m, out[3])
    d.close()
    return out + [st, ss, du]


@pytest.mark.parametrize("scatter", [L.SCATTER_BLOCK, L.SCATTER_ATOMIC])
@pytest.mark.parametrize("precision", [L.PREC_F64, L.PREC_F32])
@pytest.mark.parametrize("n,quad", [(2, False), (9, False), (4, True)])
def test_results_in_parts_are_the_same(n, quad, precision, scatter):
    """Bit for bit (the atomic scatter adds in any order: 1e-9 of the largest)."""
    opts = dict(precision=precision, scatter=scatter)
    tol = 1e-9 if scatter == L.SCATTER_ATOMIC else 0.0
    if precision == L.PREC_F32:
        tol *= 1e4
    for p, q in zip(run(n, quad, debug_fill_nan=5, **opts), run(n, quad, **opts)):
        assert np.abs(p - q).max() <= tol * np.abs(q).max()


def test_an_element_state_larger_than_the_scratch():
    """623k tet10: 15M words of stress and 2.5M of strain, each below the 16.8M
    that the scratch grows to, and both together above."""
    x, conn = ci.box_mesh(47, 47, 47, 0.25, 0.25, 0.25, quadratic=True)
    d = ci.Dynamics(ci.Mesh.from_arrays(x, conn), ci.Elastoplastic(E, RHO, NU, 1.0, H, SY), None,
                    physics=L.PHYSICS_EP)
    d.vel[:] = np.random.default_rng(2).uniform(-100, 100, x.shape)
    d.init(1e-8)
    d.step(3)
    sig, ep = d.element_state()
    assert sig.size < 16 << 20 < sig.size + ep.size and ep.max() > 0.0
    a, b = np.empty_like(sig), np.empty_like(ep)
    L.check(L.lib().cpi_get_element_state(d.ctx, L.dptr(a), None), d.ctx)
    L.check(L.lib().cpi_get_element_state(d.ctx, None, L.dptr(b)), d.ctx)
    assert np.array_equal(a, sig) and np.array_equal(b, ep)
    d.close()
