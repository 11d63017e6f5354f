"""Batched GMRES past both lines of the Gram-Schmidt dispatch: more than 16,384
lanes times conditions over four, where the update runs a thread per lane (four
conditions a thread in FP32, one in FP64), and more than 16 groups of 1024
lanes, where a batch's lane sums take two launches.  Each condition's solution
is the bits of its own run."""
import numpy as np
import pytest

from bes_amd import core, meshgen as mg

pytestmark = pytest.mark.gpu


def _state(md, seed, mach):
    P = core.freestream_primitive((mach, 0.0), 2)
    rng = np.random.default_rng(seed)
    return P, core.conserved_from_primitive(P, 2) * (1.0 + 0.01 * rng.uniform(-1, 1, (md.ncell, 4)))


# 263,168 triangles: 32,768 lanes, 32 groups; 16,640 triangles: 2,048 lanes, 2
# groups.  eta 1: the second Gram-Schmidt pass at every step.
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("ni,nj,B", [(512, 257, 2), (512, 257, 4), (128, 65, 64)])
@pytest.mark.parametrize("eta", [0.0, 0.7, 1.0])
def test_batch_is_single_runs(ni, nj, B, precision, eta):
    md = mg.bump_channel(ni, nj)
    PU = [_state(md, 5 + q, 0.3 + 0.4 * q / B) for q in range(B)]
    print("case", md.ncell, B, precision, eta, flush=True)

    def solve(c):
        c.implicit_setup(precision, "ilu0", maxiter=40, rtol=1e-3)
        c.implicit_set_reorth(eta)
        c.implicit_assemble(20.0)
        c.linear_solve(allow_unconverged=True)
        return c.linear_solution(), c.implicit_stats()["reorths"]

    with core.Context(md) as c:
        c.set_batch(B)
        c.set_freestream(np.stack([p for p, _ in PU]))
        c.set_state(np.stack([u for _, u in PU]))
        xb, _ = solve(c)
        its = c.implicit_batch_state()["iters"]
    assert its.min() > 4
    for q in sorted({0, 1, B - 1}):
        with core.Context(md) as c:
            c.set_freestream(PU[q][0])
            c.set_state(PU[q][1])
            x, reorths = solve(c)
            assert np.array_equal(x, xb[q]), f"condition {q}"
            assert eta < 1.0 or reorths >= its[q] - 1
