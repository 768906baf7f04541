"""The stress state in rows per block: rows of every padding (a block smaller
than a memory line, an odd one, a block over a whole line), the short last block."""
import numpy as np
import pytest

import cppimpact_amd as ci
from cppimpact_amd import _lib as L

from common import E, H, NU, RHO, SY

pytestmark = pytest.mark.gpu


def state(quad, **opts):
    x, conn = ci.box_mesh(3, 4, 3, 0.15, 0.2, 0.15, quadratic=quad, jitter=0.1, seed=3)
    if quad:
        opts.update(quadrature=L.QUAD_EXACT4, mass=L.MASS_HRZ)
    d = ci.Dynamics(ci.Mesh.from_arrays(x, conn), ci.Elastoplastic(E, RHO, NU, 1.0, H, SY), None,
                    physics=L.PHYSICS_EP, gravity=(0.0, 0.0, 0.0), **opts)
    d.vel[:] = np.random.default_rng(4).uniform(-300, 300, x.shape)
    d.init(2e-7)
    d.step(7)
    out = d.element_state()
    d.close()
    return out


@pytest.mark.parametrize("precision,tol", [(L.PREC_F64, 1e-10), (L.PREC_F32, 1e-4)])
@pytest.mark.parametrize("quad", [False, True])
def test_element_state_does_not_depend_on_the_blocks(quad, precision, tol):
    """Against the elements in planes (the colour scatter).  The sums at the
    nodes take another order, 1e-16 of a force (1e-7 in FP32) a step over 7
    steps; a state read from another point would differ by its size."""
    a = state(quad, precision=precision, scatter=L.SCATTER_COLOR)
    assert a[1].max() > 0.0
    for be in (1, 2, 7, 8, 9, 33, 64, 128 if quad else 384):
        for graph in (0, 1):
            b = state(quad, precision=precision, block_elements=be, use_graph=graph)
            for p, q in zip(a, b):
                assert np.abs(p - q).max() <= tol * np.abs(p).max(), be
