"""Resident steps of a mesh with nodes that belong to no element: gravity and
their own velocity move them every step, however the steps are launched."""
import numpy as np
import pytest

import cppimpact_amd as ci
from cppimpact_amd import _lib as L

from common import E, H, NU, RHO, SY

pytestmark = pytest.mark.gpu


def run(cells, quad, rule, loose, **opts):
    x, conn = ci.box_mesh(*cells, *(0.05 * c for c in cells), origin=(0.0, 0.0, 1e-6),
                          quadratic=quad, jitter=0.1, seed=3)
    n = len(x)
    x = np.vstack([x, np.random.default_rng(1).uniform(0.5, 1.0, (loose, 3))])
    # the loose nodes first in the user's order, the last of them held
    order = np.r_[n:n + loose, 0:n]
    inv = np.argsort(order)
    if quad:
        opts.update(quadrature=rule, mass=L.MASS_HRZ)
    d = ci.Dynamics(ci.Mesh.from_arrays(x[order], inv[conn], fixed_nodes=[loose - 1]),
                    ci.Elastoplastic(E, RHO, NU, 1.0, H, SY),
                    ci.Wall("Wall", 0.0, 10 * E * 0.05, None, 0, 1), fixed_bc=1,
                    gravity=(0.0, 0.5, -9.81), **opts)
    v0 = np.random.default_rng(2).uniform(-20, 20, x.shape)
    d.vel[:] = v0
    d.init(2e-7)
    out = []
    for k in (7, 1, 24):
        d.step(k)
        out += list(d.fetch()) + [d.energy()[0]]
    d.close()
    # where the free loose nodes would be without gravity
    way = 32 * 2e-7 * v0[:loose - 1]
    assert np.abs(out[-6][:loose - 1] - x[order][:loose - 1] - way).max(initial=0.0) <= 1e-9
    assert np.array_equal(out[-6][loose - 1], x[order][loose - 1])
    return out


@pytest.mark.parametrize("precision", [L.PREC_F64, L.PREC_F32])
@pytest.mark.parametrize("cells,quad,rule,loose", [
    ((1, 1, 1), False, 0, 2),                 # one block
    ((4, 4, 5), False, 0, 1),                 # two; the one loose node is held
    ((4, 4, 5), False, 0, 900),               # more loose nodes than threads
    ((5, 6, 7), True, L.QUAD_EXACT4, 3),
    ((5, 6, 7), True, L.QUAD_REF5, 3),
])
def test_loose_nodes_move_in_resident_steps(cells, quad, rule, loose, precision):
    """Same bits as steps launched kernel by kernel.  A free node is where its
    velocity took it, to gravity's g t^2 / 2 = 2e-10 and rounding (after 32 steps
    it has gone 1e-4); a held one is where it was."""
    opts = dict(physics=L.PHYSICS_EP, precision=precision)
    a = run(cells, quad, rule, loose, **opts)
    b = run(cells, quad, rule, loose, use_graph=0, **opts)
    for i, (p, q) in enumerate(zip(a, b)):
        if i % 6 == 5:
            assert np.abs(p[:7] - q[:7]).max() <= 1e-12 * np.abs(q[:7]).max()
        else:
            assert np.array_equal(p, q), i
