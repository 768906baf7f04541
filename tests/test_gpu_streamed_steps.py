"""Streamed stress state in plain steps: small meshes take their plain steps in
the resident kernel, where stream_state has no effect, so these runs are launched
kernel by kernel (use_graph=0), as the steps of large meshes are."""
import numpy as np
import pytest

from cppimpact_amd import _lib as L
from oracle import pyoracle as O

from common import cube, rel, run_gpu, run_oracle, wall_k

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [L.PREC_F64, L.PREC_F32])
@pytest.mark.parametrize("npe,block", [
    (4, 0),
    (10, 0),    # FP64: 6 blocks, forces on the matrix units
    (10, 1),    # FP64: 750 blocks, more than the matrix path takes
])
def test_streamed_plain_steps_give_the_same_bits(npe, block, precision):
    """The same bits as cached accesses over a plastic impact, and the oracle's
    state in FP64 (750 elements and 50 steps: 1e-9 as the cached runs)."""
    quad = npe == 10
    x, conn = cube(5 if quad else 8, quadratic=quad, jitter=0.05, seed=4, gap=1e-6)
    k = wall_k(0.25, 10)
    v0, dt, n = (0, 0, -40.0), 1e-7, 50
    opts = dict(quadrature=L.QUAD_EXACT4) if quad else {}
    runs = [run_gpu(x, conn, v0, dt, n, k, physics=L.PHYSICS_EP, precision=precision, use_graph=0,
                    block_elements=block, stream_state=s, **opts) for s in (1, 2)]
    for g in runs:
        assert g["dyn"].resident_steps() == (0, 0)
    if block:
        assert runs[0]["dyn"].info().num_blocks > 512
    for key in ("x", "v", "a", "energy"):
        assert np.array_equal(runs[0][key], runs[1][key]), key
    s1, e1 = runs[0]["dyn"].element_state()
    s2, e2 = runs[1]["dyn"].element_state()
    assert e1.max() > 0.0
    assert np.array_equal(s1, s2) and np.array_equal(e1, e2)
    if precision == L.PREC_F64:
        o = run_oracle(x, conn, v0, dt, n, O.EP, k, **({"quad_rule": L.QUAD_EXACT4} if quad else {}))
        assert rel(runs[0]["x"] - x, o["x"] - x) < 1e-9 and rel(runs[0]["v"], o["v"]) < 1e-9
    for g in runs:
        g["dyn"].close()
