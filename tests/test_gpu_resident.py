"""Steps taken by the resident kernel (one launch for all the plain steps of a
call, small meshes) against the same steps launched kernel by kernel
(use_graph=0): the same state bit for bit, the cumulative energies to the
rounding of their other order of summation (1e-12 of the largest)."""
import numpy as np
import pytest

import cppimpact_amd as ci
from cppimpact_amd import _lib as L

from common import E, H, NU, RHO, SY

pytestmark = pytest.mark.gpu

EP, COMPAT = L.PHYSICS_EP, L.PHYSICS_COMPAT


def run(cells, quad, calls, speed=40.0, fixed=False, **opts):
    x, conn = ci.box_mesh(*cells, *(0.05 * c for c in cells), origin=(0.0, 0.0, 1e-6),
                          quadratic=quad, jitter=0.1, seed=3)
    low = np.flatnonzero(x[:, 0] < 1e-9)
    mesh = ci.Mesh.from_arrays(x, conn, slave_nodes=np.flatnonzero(x[:, 1] < 0.1),
                               fixed_nodes=low[:3])
    if fixed:
        opts.update(fixed_bc=1, contact_slave_only=1)
    if quad:
        opts.setdefault("quadrature", L.QUAD_EXACT4)
        opts.setdefault("mass", L.MASS_HRZ)
    d = ci.Dynamics(mesh, ci.Elastoplastic(E, RHO, NU, 1.0, H, SY),
                    ci.Wall("Wall", 0.0, 10 * E * 0.05, None, 0, 1), **opts)
    d.vel[:] = (1.0, 0.0, -speed)
    d.init(2e-7)
    out = []
    for n in calls:
        d.step(n)
        out.append(d.energy()[0])
    out += list(d.fetch()) + list(d.element_state()) + list(d.stress_strain())
    out.append(np.array([d.info().step, d.energy()[1]]))
    d.close()
    return len(calls), out


def same(a, b):
    n = a[0]
    for p, q in zip(a[1][:n], b[1][:n]):
        scale = np.abs(q[:7]).max()
        assert np.abs(p[:7] - q[:7]).max() <= 1e-12 * scale and p[7] == q[7]
    for p, q in zip(a[1][n:], b[1][n:]):
        assert np.array_equal(p, q)


@pytest.mark.parametrize("precision", [L.PREC_F64, L.PREC_F32])
@pytest.mark.parametrize("physics", [EP, COMPAT])
@pytest.mark.parametrize("cells,quad,more", [
    ((1, 1, 1), False, {}),                      # one block, one wave with elements
    ((4, 4, 4), False, {}),                      # one full block
    ((4, 4, 5), False, {}),                      # two blocks
    ((9, 7, 11), False, dict(fixed=True)),       # 14 blocks, corners shared by eight
    ((7, 6, 5), False, dict(block_elements=37)),  # many small blocks, idle waves
    ((1, 1, 2), True, {}),
    ((5, 6, 7), True, dict(fixed=True)),
    ((6, 5, 4), True, dict(block_elements=21)),
])
def test_resident_steps_have_the_bits_of_single_steps(cells, quad, more, physics, precision):
    calls = (5, 6, 1, 40)  # the fewest resident ones, even and odd counts, none
    opts = dict(physics=physics, precision=precision, **more)
    a = run(cells, quad, calls, **opts)
    b = run(cells, quad, calls, use_graph=0, **opts)
    same(a, b)
    if physics == EP:
        assert a[1][len(calls) + 6].max() > 0.0  # plastic


@pytest.mark.parametrize("quad", [False, True])
def test_steps_a_resident_launch_gave_up_are_taken_one_by_one(quad):
    """Every wait gives up at its first poll: the launches store nothing and
    the steps asked for are taken all the same."""
    cells, calls = ((9, 7, 11), (30, 6, 17)) if not quad else ((5, 6, 7), (30, 6, 17))
    a = run(cells, quad, calls, physics=EP, debug_fill_nan=3)
    b = run(cells, quad, calls, physics=EP, use_graph=0)
    same(a, b)


def test_resident_contexts_side_by_side():
    """Two contexts' resident launches on two streams, queued alternately
    without waiting in between."""
    def make():
        x, conn = ci.box_mesh(8, 8, 8, 0.4, 0.4, 0.4, origin=(0.0, 0.0, 1e-6), jitter=0.1, seed=1)
        d = ci.Dynamics(ci.Mesh.from_arrays(x, conn), ci.Elastoplastic(E, RHO, NU, 1.0, H, SY),
                        ci.Wall("Wall", 0.0, 10 * E * 0.05, None, 0, 1), physics=EP)
        d.vel[:] = (0.0, 0.0, -30.0)
        d.init(2e-7)
        return d

    d, e, f = make(), make(), make()
    for _ in range(4):
        d.step(25)
        e.step(25)
    f.step(100)
    x = [c.fetch()[:2] for c in (d, e, f)]
    for p in x[1:]:
        assert np.array_equal(x[0][0], p[0]) and np.array_equal(x[0][1], p[1])
    for c in (d, e, f):
        c.close()
