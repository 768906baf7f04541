"""Calls of more steps than one resident launch takes (1,024), and contexts
whose launches gave up and that start again."""
import threading
import time

import numpy as np
import pytest

import cppimpact_amd as ci
from cppimpact_amd import _lib as L

from common import E, H, NU, RHO, SY

pytestmark = pytest.mark.gpu


def velocities(shape):
    return np.random.default_rng(4).uniform(-5, 5, shape)


def make(n, quad=False, gravity=(0.0, 0.0, 0.0), **opts):
    x, conn = ci.box_mesh(n, n, n + 1, 0.25, 0.25, 0.25, origin=(0.0, 0.0, 1e-6), quadratic=quad,
                          jitter=0.05, seed=3)
    if quad:
        opts.update(quadrature=L.QUAD_EXACT4, mass=L.MASS_HRZ)
    d = ci.Dynamics(ci.Mesh.from_arrays(x, conn), ci.Elastoplastic(E, RHO, NU, 1.0, H, SY), None,
                    physics=L.PHYSICS_EP, gravity=gravity, **opts)
    d.vel[:] = velocities(x.shape)
    d.init(1e-7)
    return d


@pytest.mark.parametrize("quad,precision", [(False, L.PREC_F64), (False, L.PREC_F32),
                                            (True, L.PREC_F64)])
@pytest.mark.parametrize("calls", [(1025, 3), (1026, 5), (3100, 1027)])
def test_a_long_call_has_the_bits_of_single_steps(calls, quad, precision):
    """The launches of a call follow each other at odd and even step counts, with
    one step left for the last."""
    out = []
    for graph in (1, 0):
        d = make(3, quad, block_elements=48, precision=precision, use_graph=graph)
        for n in calls:
            d.step(n)
        taken = d.resident_steps()
        out.append(list(d.fetch()) + list(d.element_state()) + [d.energy()[1]])
        assert taken == ((sum(n - 1 for n in calls if n >= 5), 0) if graph else (0, 0))
        d.close()
    for p, q in zip(*out):
        assert np.array_equal(p, q)


def test_another_context_steps_while_a_long_call_runs():
    """A call that fills the chip for 60,000 steps; the other context needs some
    milliseconds for its ten, and gets them before half of it is over."""
    a, b = make(31), make(4, use_graph=0)
    for d in (a, b):
        d.step(10)
        d.energy()
    assert a.resident_steps() == (9, 0)
    done, start = [], time.perf_counter()
    t = threading.Thread(target=lambda: (a.step(60000), a.synchronize(),
                                         done.append(time.perf_counter() - start)))
    t.start()
    time.sleep(0.01)
    b.step(10)
    b.energy()
    other = time.perf_counter() - start
    t.join()
    assert a.energy()[1] == 60010 and b.energy()[1] == 20
    assert other < 0.5 * done[0]
    a.close()
    b.close()


def test_a_call_of_more_launches_than_are_queued_ahead():
    d = make(1, gravity=(0.0, 0.0, -9.81))
    d.step(140000)  # 137 launches
    assert d.resident_steps() == (139999, 0) and d.energy()[1] == 140000
    x, v = d.fetch()[:2]
    # its centre of mass falls: the half kick and 140,000 steps
    m = d.global_mass
    vz = (m * v).sum(0)[2] / m[:, 2].sum()
    v0 = (m * velocities(v.shape)).sum(0)[2] / m[:, 2].sum()
    assert abs(vz - v0 + 9.81 * 140000.5 * 1e-7) <= 1e-9
    d.close()


def test_a_context_that_gave_up_tries_again_after_init():
    d = make(4, debug_fill_nan=3)
    for _ in range(2):
        d.step(20)
        assert d.resident_steps() == (0, 20)
        d.step(20)  # step by step from there on
        assert d.resident_steps() == (0, 20)
        d.init(1e-7)
        assert d.resident_steps() == (0, 0)
    d.close()
