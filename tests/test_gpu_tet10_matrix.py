"""The FP64 per-point tet10 pass on the matrix units (few blocks) and over quads
of lanes (many), at the edges of its waves of sixteen elements."""
import numpy as np
import pytest

import cppimpact_amd as ci
from cppimpact_amd import _lib as L

from common import E, H, NU, RHO, SY

pytestmark = pytest.mark.gpu


def run(**opts):
    x, conn = ci.box_mesh(5, 5, 5, 0.25, 0.25, 0.25, quadratic=True, jitter=0.1, seed=3)
    d = ci.Dynamics(ci.Mesh.from_arrays(x, conn), ci.Elastoplastic(E, RHO, NU, 1.0, H, SY), None,
                    mass=L.MASS_HRZ, gravity=(0.0, 0.0, 0.0), **opts)
    d.vel[:] = np.random.default_rng(4).uniform(-100, 100, x.shape)
    d.init(1e-7)
    d.step(3)
    out = list(d.fetch()[:3]) + (list(d.element_state()) if opts["physics"] else [])
    e = np.asarray(d.energy()[0][:7])
    d.close()
    return out, e


@pytest.mark.parametrize("rule", [L.QUAD_REF4, L.QUAD_EXACT4])
@pytest.mark.parametrize("physics", [L.PHYSICS_COMPAT, L.PHYSICS_EP])
def test_matrix_and_quad_blocks_match_the_direct_pass(physics, rule):
    """Against one thread per element (the colour scatter); nodes and points
    sum in another order, 1e-15 a step.  750 elements in blocks of one are
    more blocks than the matrix path takes (750), of two fewer (375); then a
    wave's sixteen elements, one more and one less, and a full block."""
    opts = dict(physics=physics, quadrature=rule)
    a, ea = run(scatter=L.SCATTER_COLOR, **opts)
    for be in (1, 2, 15, 16, 17, 128):
        b, eb = run(block_elements=be, **opts)
        for p, q in zip(a, b):
            assert np.abs(p - q).max() <= 1e-11 * np.abs(p).max(), be
        assert np.abs(ea - eb).max() <= 1e-11 * np.abs(ea).max(), be
