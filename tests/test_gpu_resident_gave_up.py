"""What calls leave behind whose resident launches gave up (every wait ends at
its first poll, debug_fill_nan=3): the energy rows of each call's own last step,
the state, and the time of the steps that were asked for."""
import numpy as np
import pytest

import cppimpact_amd as ci
from cppimpact_amd import _lib as L

from common import E, H, NU, RHO, SY

pytestmark = pytest.mark.gpu


def make(quad, rule, **opts):
    cells = (5, 6, 7) if quad else (4, 4, 5)
    x, conn = ci.box_mesh(*cells, *(0.05 * c for c in cells), origin=(0.0, 0.0, 1e-6),
                          quadratic=quad, jitter=0.1, seed=3)
    if quad:
        opts.update(quadrature=rule, mass=L.MASS_HRZ)
    d = ci.Dynamics(ci.Mesh.from_arrays(x, conn), ci.Elastoplastic(E, RHO, NU, 1.0, H, SY),
                    ci.Wall("Wall", 0.0, 10 * E * 0.05, None, 0, 1), physics=L.PHYSICS_EP, **opts)
    d.vel[:] = (1.0, 0.0, -40.0)
    d.init(2e-7)
    return d


def run(quad, rule, calls, read, **opts):
    d = make(quad, rule, **opts)
    for i, n in enumerate(calls):
        d.step(n)
        if i in read:
            d.energy()
    out = (d.energy_history(), list(d.fetch()) + list(d.element_state()), d.energy(),
           d.resident_steps()[1])
    d.close()
    return out


@pytest.mark.parametrize("quad,rule", [(False, -1), (True, L.QUAD_EXACT4), (True, L.QUAD_REF5)])
@pytest.mark.parametrize("calls,read", [
    ((25, 25, 25, 25), ()),
    ((30, 1, 6, 3, 17, 2, 1), ()),       # short calls between them
    ((7, 1, 1, 1, 1, 1, 1, 1, 1), ()),    # more queued calls than steps of the first
    ((12, 7, 9), (1,)),                  # read half way
])
def test_every_call_has_the_energies_of_its_own_last_step(quad, rule, calls, read):
    """Row for row against steps launched kernel by kernel: the same launches
    here, so the same bits."""
    a = run(quad, rule, calls, read, debug_fill_nan=3)
    b = run(quad, rule, calls, read, use_graph=0)
    assert a[3] > 0 and b[3] == 0
    assert len(b[0]) == len(calls) + 1
    assert np.array_equal(a[0], b[0])
    assert a[2][1] == b[2][1] == sum(calls) and np.array_equal(a[2][0], b[2][0])
    for p, q in zip(a[1], b[1]):
        assert np.array_equal(p, q)


@pytest.mark.parametrize("more", [dict(debug_fill_nan=3), {}])
def test_more_queued_calls_than_the_context_remembers(more):
    calls = (7,) * 1100
    a = run(False, -1, calls, (), **more)
    b = run(False, -1, calls, (), use_graph=0)
    assert len(a[0]) == len(b[0]) == len(calls) + 1
    assert np.abs(a[0] - b[0])[:, :7].max() <= 1e-12 * np.abs(b[0][:, :7]).max()
    assert np.array_equal(a[1][0], b[1][0])


def test_the_time_of_steps_includes_those_taken_again():
    """The second call runs step by step from the start; the first, which gave
    up, cannot be much shorter."""
    d = make(False, -1, debug_fill_nan=3)
    first = d.time_steps(3000)
    d.energy()
    second = d.time_steps(3000)
    assert d.resident_steps() == (0, 3000) and d.energy()[1] == 6000
    assert first > 0.5 * second
    d.close()
