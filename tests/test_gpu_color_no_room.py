"""The colour scatter of a mesh whose corner-force slots find no room on the
device (debug_fill_nan=5): colour by colour, with the bits of the slots."""
import numpy as np
import pytest

import cppimpact_amd as ci
from cppimpact_amd import _lib as L

from common import E, H, NU, RHO, SY

pytestmark = pytest.mark.gpu


def run(quad, physics, **opts):
    n = (3, 4, 5) if quad else (5, 4, 7)
    x, conn = ci.box_mesh(*n, *(0.05 * c for c in n), origin=(0.0, 0.0, 1e-6), quadratic=quad,
                          jitter=0.1, seed=3)
    conn = np.ascontiguousarray(conn[np.random.default_rng(7).permutation(len(conn))])
    x = np.vstack([x, [[0.5, 0.5, 0.5]]])  # a node of no element
    if quad:
        opts.update(mass=L.MASS_HRZ)  # row sums of tet10 corners are negative
    d = ci.Dynamics(ci.Mesh.from_arrays(x, conn), ci.Elastoplastic(E, RHO, NU, 1.0, H, SY),
                    ci.Wall("Wall", 0.0, 10 * E * 0.05, None, 0, 1), physics=physics,
                    scatter=L.SCATTER_COLOR, **opts)
    if physics == L.PHYSICS_EP:
        d.enable_samples(100000)
        d.subsample_samples(0.5, 3)
    d.vel[:] = (1.0, 0.0, -40.0)
    d.init(2e-7)
    d.step(40)
    launches = {k: v[1] for k, v in d.profile_kernels(1).items()}
    smp = d.samples()[0] if physics == L.PHYSICS_EP else np.zeros((1, 1))
    out = list(d.fetch()) + list(d.element_state()) + list(d.stress_strain())
    e, colors = d.energy()[0], d.info().num_colors
    d.close()
    return out, smp[np.lexsort(smp.T)], e, launches["elem_direct"], colors


@pytest.mark.parametrize("precision", [L.PREC_F64, L.PREC_F32])
@pytest.mark.parametrize("physics", [L.PHYSICS_COMPAT, L.PHYSICS_EP])
@pytest.mark.parametrize("quad", [False, True])
def test_colour_by_colour_has_the_bits_of_the_slots(quad, physics, precision):
    """State, recorded samples and mass bit for bit; the energies' sums take
    another order (1e-12 of the largest)."""
    a = run(quad, physics, precision=precision, debug_fill_nan=5)
    b = run(quad, physics, precision=precision)
    for p, q in zip(a[0], b[0]):
        assert np.array_equal(p, q)
    assert len(a[1]) and np.array_equal(a[1], b[1])
    assert np.abs(a[2] - b[2])[:7].max() <= 1e-12 * np.abs(b[2][:7]).max()
    assert a[3] == a[4] > 1 and b[3] == 1
