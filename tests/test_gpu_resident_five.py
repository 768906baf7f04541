"""Resident steps of tet10 on the five-point rule against the same steps launched
kernel by kernel (use_graph=0): the same state bit for bit, the cumulative
energies to the rounding of their other order of summation."""
import numpy as np
import pytest

from cppimpact_amd import _lib as L

from test_gpu_resident import run, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [L.PREC_F64, L.PREC_F32])
@pytest.mark.parametrize("physics", [L.PHYSICS_EP, L.PHYSICS_COMPAT])
@pytest.mark.parametrize("cells,more", [
    ((1, 1, 2), {}),                             # one wave's twelve elements
    ((5, 6, 7), dict(fixed=True)),               # ten blocks of 128
    ((6, 5, 4), dict(block_elements=13)),        # a wave and one more, 56 blocks
    ((6, 6, 6), dict(block_elements=5)),         # 260 blocks: more than CUs
    ((5, 5, 5), dict(block_elements=133)),       # a second round: not resident
])
def test_resident_five_point_steps_have_the_bits_of_single_steps(cells, more, physics, precision):
    calls = (5, 6, 1, 40)
    opts = dict(physics=physics, precision=precision, quadrature=L.QUAD_REF5, **more)
    a = run(cells, True, calls, **opts)
    b = run(cells, True, calls, use_graph=0, **opts)
    same(a, b)


def test_steps_a_five_point_launch_gave_up_are_taken_one_by_one():
    """Every wait gives up at its first poll."""
    calls = (30, 6, 17)
    opts = dict(physics=L.PHYSICS_EP, quadrature=L.QUAD_REF5)
    a = run((5, 6, 7), True, calls, debug_fill_nan=3, **opts)
    b = run((5, 6, 7), True, calls, use_graph=0, **opts)
    same(a, b)
