"""The five-point tet10 element pass (five lanes per element, twelve elements
per wave) at the edges of its waves, rounds and launch shapes."""
import numpy as np
import pytest

import cppimpact_amd as ci
from cppimpact_amd import _lib as L

from common import E, H, NU, RHO, SY

pytestmark = pytest.mark.gpu


def run(**opts):
    x, conn = ci.box_mesh(6, 6, 6, 0.3, 0.3, 0.3, quadratic=True, jitter=0.1, seed=3)
    d = ci.Dynamics(ci.Mesh.from_arrays(x, conn), ci.Elastoplastic(E, RHO, NU, 1.0, H, SY), None,
                    quadrature=L.QUAD_REF5, mass=L.MASS_HRZ, gravity=(0.0, 0.0, 0.0), **opts)
    d.vel[:] = np.random.default_rng(4).uniform(-100, 100, x.shape)
    d.init(1e-7)
    d.step(3)
    out = list(d.fetch()[:3]) + (list(d.element_state()) if opts["physics"] else [])
    e = d.energy()[0]
    d.close()
    return out, e


@pytest.mark.parametrize("precision,tol", [(L.PREC_F64, 1e-11), (L.PREC_F32, 1e-4)])
@pytest.mark.parametrize("physics", [L.PHYSICS_COMPAT, L.PHYSICS_EP])
def test_five_point_blocks_match_the_direct_pass(physics, precision, tol):
    """Against one thread per element (the colour scatter): nodes sum in
    another order and FP64 factors its products otherwise, 1e-15 a step (FP32:
    the same element bits, but one rounding of 1e-7 in a position's strain).
    1296 elements in blocks of one wave's twelve and one more, of a round of
    384 (72) and of 704 threads (132) and one more, and of several rounds; in
    blocks of four they are more blocks (324) than CUs."""
    opts = dict(physics=physics, precision=precision)
    a, ea = run(scatter=L.SCATTER_COLOR, **opts)
    for be in (0, 4, 12, 13, 72, 73, 132, 133, 150):
        b, eb = run(block_elements=be, **opts)
        for p, q in zip(a, b):
            assert np.abs(p - q).max() <= tol * np.abs(p).max(), be
        assert np.abs(np.asarray(ea[:7]) - eb[:7]).max() <= tol * np.abs(ea[:7]).max(), be
