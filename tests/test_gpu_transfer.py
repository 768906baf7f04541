"""What leaves and enters the device: nodal strain and stress, nodal state."""
import numpy as np
import pytest

import cppimpact_amd as ci
from cppimpact_amd import _lib as L
from oracle import pyoracle as O

from common import E, NU, RHO, cube, rel, run_gpu, wall_k

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scatter", [L.SCATTER_BLOCK, L.SCATTER_COLOR])
@pytest.mark.parametrize("quad", [False, True])
def test_nodal_stress_takes_the_last_element_and_leaves_loose_nodes(quad, scatter):
    """Every node reports its highest-numbered element, in user order (the
    oracle's element loop), and a node of no element keeps what the caller's
    arrays hold.  Bound: strains of 1e-3 from displacements of 1e-5 carried
    over 10 steps in FP64, rounding below 1e-10 of the largest."""
    x, conn = cube(3, quadratic=quad, jitter=0.1, seed=5, gap=1e-6)
    rng = np.random.default_rng(2)
    conn = np.ascontiguousarray(conn[rng.permutation(len(conn))])
    x = np.vstack([x, [[0.1, 0.1, 0.9]]])  # a node of no element
    k, dt, n = wall_k(0.25, 3), 1e-7, 10
    opts = dict(quadrature=L.QUAD_EXACT4, mass=L.MASS_HRZ) if quad else {}
    g = run_gpu(x, conn, (0, 0, -10.0), dt, n, k, scatter=scatter, **opts)
    o = O.Solver(x, conn, (0, 0, -10.0), E=E, nu=NU, rho=RHO, physics=O.COMPAT,
                 wall=dict(location=0.0, stiffness=k), dt=dt,
                 **(dict(quad_rule=L.QUAD_EXACT4, mass_kind=O.MASS_HRZ) if quad else {}))
    o = o.solve(n, with_strain=True)
    st, ss = np.full((len(x), 6), 7.0), np.full((len(x), 6), 8.0)
    d = g["dyn"]
    L.check(L.lib().cpi_get_stress_strain(d.ctx, L.dptr(st), L.dptr(ss)), d.ctx)
    assert rel(st[:-1], o["strain"][:-1]) < 1e-8 and rel(ss[:-1], o["stress"][:-1]) < 1e-8
    assert (st[-1] == 7.0).all() and (ss[-1] == 8.0).all()
    only = np.zeros_like(st)
    L.check(L.lib().cpi_get_stress_strain(d.ctx, L.dptr(only), None), d.ctx)
    assert np.array_equal(only[:-1], st[:-1])
    d.close()


@pytest.mark.parametrize("n,scatter", [(3, L.SCATTER_BLOCK), (3, L.SCATTER_COLOR),
                                       (24, L.SCATTER_BLOCK), (66, L.SCATTER_ATOMIC)])
def test_state_goes_in_and_comes_out_in_user_order(n, scatter):
    """Without wall and gravity nothing moves the initial state, so x, v and
    v_n come back exactly as set, over the sizes of the one transfer (n = 3),
    of a ring larger (24) and smaller (66: 38 MB) than the result; the state
    of a second initial condition replaces the first."""
    x, conn = cube(n)
    d = ci.Dynamics(ci.Mesh.from_arrays(x, conn), ci.Elastoplastic(E, RHO, NU, 1.0, 7e8, 2.76e8),
                    None, physics=L.PHYSICS_EP, scatter=scatter, gravity=(0.0, 0.0, 0.0))
    for seed in (1, 2):
        rng = np.random.default_rng(seed)
        x0 = x + rng.uniform(-1, 1, x.shape) * 1e-3 * 0.25 / n
        v0 = rng.standard_normal(x.shape)
        d._x0, d.vel = x0, v0.copy()
        d.init(1e-9)
        gx, gv, ga, gm, gvi = d.fetch()
        assert np.array_equal(gx, x0) and np.array_equal(gv, v0) and np.array_equal(gvi, v0)
        assert not ga.any() and (gm > 0).all()
        assert np.array_equal(d.global_mass, np.repeat(gm[:, None], 3, axis=1))
        du = np.full_like(x, 3.0)
        L.check(L.lib().cpi_get_increment(d.ctx, L.dptr(du)), d.ctx)
        assert not du.any()
        sig, ep = d.element_state()
        assert not sig.any() and not ep.any()
    # a refused state leaves the one that was set
    bad = v0.copy()
    bad[-1, 2] = np.inf
    with pytest.raises(L.CpiError) as err:
        L.check(L.lib().cpi_set_state(d.ctx, L.dptr(x), L.dptr(bad)), d.ctx)
    assert err.value.code == -1
    assert np.array_equal(d.fetch()[0], x0)
    d.close()
