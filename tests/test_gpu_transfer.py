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
