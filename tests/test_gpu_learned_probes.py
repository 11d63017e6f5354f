"""Learned preconditioner: the Richardson chains of several probes run in groups
of four, two and one.

A probe's chain is the same sums in any group, so the loss over Q probes is the
mean of the Q single-probe losses to the rounding of that mean (Q + 2 additions,
divisions and products: 20 ulp).  The gradient is checked against the CPU
restatement with the 5e-2 of tests/test_gpu_learned.py (BF16 operands on both
sides); a probe left out of Q <= 7 would move it by 1/7 or more.  Cell counts are
no multiple of a wave or of the decoder's 128-node blocks.
"""
import numpy as np
import pytest

from bes_amd import core, meshgen as mg
from oracle import gnn, oracle as orc
from test_gpu_learned import MVEC, _perturbed_params, blocks_from_scalar_csr

pytestmark = pytest.mark.gpu


def _system(nd, precision):
    md = mg.bump_channel(19, 7) if nd == 2 else mg.swept_wing(7, 3, 5)
    mvec = (0.5, 0.0, 0.0) if nd == 2 else MVEC
    c = core.Context(md)
    c.set_freestream(orc.freestream_primitive(mvec, nd))
    c.implicit_setup(precision, "learned", restart=30, maxiter=300, rtol=1e-3)
    c.lp_init(20261202)
    c.set_state(orc.perturbed_state(md.ncell, nd, mvec, seed=8, amp=0.02))
    c.implicit_assemble(10.0)
    return c


@pytest.mark.parametrize("nd,precision,Q,K", [(2, 64, 1, 1), (2, 32, 3, 2), (2, 64, 6, 3), (3, 32, 2, 3),
                                              (3, 64, 5, 2), (3, 64, 7, 3)])
def test_probe_groups(nd, precision, Q, K):
    with _system(nd, precision) as c:
        assert c.ncell % 32 != 0
        theta = _perturbed_params(4)
        c.lp_set_params(theta)
        V = np.random.default_rng(11).standard_normal((Q, c.ncell, c.nv))
        L, grad = c.lp_loss_grad(V, nrich=K)
        one = [c.lp_loss_grad(V[q:q + 1], nrich=K)[0] for q in range(Q)]
        assert abs(L - np.mean(one)) <= 20 * np.finfo(float).eps * L

        rp, col, val, rhs = c.implicit_system()
        g = gnn.Graph.from_geometry(c.geometry())
        D, O = gnn.blocks_from_bsr(*blocks_from_scalar_csr(rp, col, val, c.nv), c.ncell, c.k, g.nbr)
        Lr, gr = gnn.loss_and_grad(theta.astype(np.float64), g, D, O, rhs, V, K=K, bf16_mode=True)
        print("loss %.8e restated %.8e" % (L, Lr))
        assert abs(L - Lr) <= 2e-3 * Lr
        assert np.linalg.norm(grad - gr) <= 5e-2 * np.linalg.norm(gr)
