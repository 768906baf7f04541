"""Which steps the resident kernel takes: the plain steps of a call of five or
more (seven, with more blocks than CUs) where every block fits the chip, none
elsewhere.  A resident path that is silently off gives the same results as the
per-step kernels, so the tests that compare the two say nothing without this
one."""
import pytest

import cppimpact_amd as ci
from cppimpact_amd import _lib as L

from common import E, H, NU, RHO, SY

pytestmark = pytest.mark.gpu

CALLS = (7, 8, 1, 4, 40)
PLAIN = 6 + 7 + 39


def counts(cells, quad, calls=CALLS, **opts):
    x, conn = ci.box_mesh(*cells, *(0.05 * c for c in cells), quadratic=quad, jitter=0.1, seed=3)
    if quad:
        opts.setdefault("quadrature", L.QUAD_EXACT4)
        opts.setdefault("mass", L.MASS_HRZ)
    d = ci.Dynamics(ci.Mesh.from_arrays(x, conn), ci.Elastoplastic(E, RHO, NU, 1.0, H, SY), None,
                    **opts)
    d.vel[:] = (1.0, 0.0, -10.0)
    d.init(2e-7)
    for n in calls:
        d.step(n)
    out = d.resident_steps()
    assert d.energy()[1] == sum(calls) == d.info().step
    d.close()
    return out


@pytest.mark.parametrize("precision", [L.PREC_F64, L.PREC_F32])
@pytest.mark.parametrize("physics", [L.PHYSICS_EP, L.PHYSICS_COMPAT])
@pytest.mark.parametrize("cells,quad,more", [
    ((1, 1, 1), False, {}),
    ((4, 4, 5), False, {}),
    ((9, 7, 11), False, {}),
    ((7, 6, 5), False, dict(block_elements=37)),
    ((32, 32, 32), False, {}),                    # 512 blocks, two per CU
    ((1, 1, 2), True, {}),
    ((5, 6, 7), True, {}),
    ((6, 5, 4), True, dict(block_elements=21)),
    ((1, 1, 2), True, dict(quadrature=L.QUAD_REF5)),
    ((5, 6, 7), True, dict(quadrature=L.QUAD_REF5)),
    ((6, 5, 4), True, dict(quadrature=L.QUAD_REF5, block_elements=13)),
])
def test_small_meshes_are_resident(cells, quad, more, physics, precision):
    assert counts(cells, quad, physics=physics, precision=precision, **more) == (PLAIN, 0)


@pytest.mark.parametrize("cells,quad,more", [
    ((48, 48, 48), False, {}),                                             # 1,728 blocks
    ((6, 6, 6), True, dict(quadrature=L.QUAD_REF5, block_elements=5)),    # 260: more than CUs
    ((5, 5, 5), True, dict(quadrature=L.QUAD_REF5, block_elements=133)),  # a second round
    ((4, 4, 5), False, dict(use_graph=0)),
    ((4, 4, 5), False, dict(scatter=L.SCATTER_COLOR)),
])
def test_other_meshes_are_not(cells, quad, more):
    assert counts(cells, quad, physics=L.PHYSICS_EP, **more) == (0, 0)


def test_short_calls_are_not():
    assert counts((4, 4, 5), False, calls=(1, 2, 3, 4), physics=L.PHYSICS_EP) == (0, 0)
    assert counts((4, 4, 5), False, calls=(5, 6), physics=L.PHYSICS_EP) == (9, 0)
    assert counts((32, 32, 32), False, calls=(5, 6), physics=L.PHYSICS_EP) == (0, 0)


@pytest.mark.parametrize("quad,rule", [(False, -1), (True, L.QUAD_EXACT4), (True, L.QUAD_REF5)])
def test_a_launch_that_gives_up_takes_none(quad, rule):
    """Every wait gives up at its first poll."""
    taken, redone = counts((5, 6, 7), quad, calls=(30, 7, 17), physics=L.PHYSICS_EP,
                           debug_fill_nan=3, **(dict(quadrature=rule) if quad else {}))
    assert taken == 0 and redone >= 29 + 6 + 16
