"""The two forms of the explicit passes, at the sizes where the dispatch changes
(196,608 cell-conditions in 2D, 90,112 in 3D) and at the edges of their blocks, against the CPU
oracle and against each condition's own run, bit for bit."""
import numpy as np
import pytest

from bes_amd import core, meshgen as mg
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _mesh(kind, *n):
    return mg.bump_channel(*n) if kind == "bump" else mg.box_tets(*n, seed=3, slip_faces=("zmin",))


def _case(md, seed=2):
    mach = (0.5, 0.1) if md.ndim == 2 else (0.7, 0.05, 0.1)
    return orc.freestream_primitive(mach, md.ndim), orc.perturbed_state(md.ncell, md.ndim, mach, seed=seed)


# fewer cells than a block's 64, one block, one past it, ragged; the last size of
# the split form and the first of the other, in 2D and 3D
@pytest.mark.parametrize("mesh", [("bump", 5, 4), ("bump", 8, 4), ("bump", 11, 3), ("box", 4, 3, 3), ("box", 5, 5, 3),
                                  ("bump", 384, 256), ("bump", 331, 299), ("box", 25, 24, 25), ("box", 25, 25, 25)])
@pytest.mark.parametrize("graph", [False, True])
def test_steps_equal_the_oracle(mesh, graph):
    md = _mesh(*mesh)
    finf, U = _case(md)
    om = orc.Mesh(md)
    G = om.gradient(U)
    P = om.limiter(U, G)
    R = om.residual(U, G, P, finf)
    alpha = (0.1481, 0.4, 1.0)
    Ur, lr = om.explicit(U, 3, 0.8, finf, alpha=alpha)
    with core.Context(md) as c:
        c.set_freestream(finf)
        c.set_state(U)
        Rg, mx = c.residual()
        Gg, Pg = c.gradient_limiter()
        c.explicit_graph(graph)
        linf = c.explicit_run(3, 0.8, alpha=alpha)
        Ug = c.get_state()
        # once more from the start: the monitors of the run before are gone
        c.set_state(U)
        linf1 = c.explicit_run(1, 0.8, alpha=alpha)
    assert np.array_equal(Gg, G) and np.array_equal(Pg, P)
    assert np.array_equal(Rg, R) and np.array_equal(mx, np.abs(R).max(axis=0))
    assert np.array_equal(Ug, Ur) and np.array_equal(linf, lr)
    assert np.array_equal(linf1, lr[:1])


@pytest.mark.parametrize("alpha", [(1.0,), (0.3, 1.0)])
@pytest.mark.parametrize("local", [True, False])
def test_one_stage_and_global_steps(alpha, local):
    md = _mesh("box", 5, 4, 3)
    finf, U = _case(md)
    Ur, lr = orc.Mesh(md).explicit(U, 4, 0.3, finf, local=local, alpha=alpha)
    with core.Context(md) as c:
        c.set_freestream(finf)
        c.set_state(U)
        linf = c.explicit_run(4, 0.3, local=local, alpha=alpha)
        assert np.array_equal(c.get_state(), Ur) and np.array_equal(linf, lr)


# batches on both sides of the line; frozen limiter values in one condition's place
@pytest.mark.parametrize("mesh,B", [(("bump", 9, 4), 2), (("box", 4, 4, 3), 8), (("bump", 48, 32), 64),
                                    (("bump", 49, 32), 64), (("box", 12, 12, 14), 8)])
def test_batch_equals_single_runs(mesh, B):
    md = _mesh(*mesh)
    PU = [_case(md, 10 + q) for q in range(B)]
    with core.Context(md) as c:
        c.set_batch(B)
        c.set_freestream(np.stack([p for p, _ in PU]))
        c.set_state(np.stack([u for _, u in PU]))
        _, phi = c.gradient_limiter()
        c.freeze_limiter_values(phi)
        linf = c.explicit_run(3, 0.8)
        U = c.get_state()
    for q in sorted({0, 1, B - 1}):
        with core.Context(md) as c:
            c.set_freestream(PU[q][0])
            c.set_state(PU[q][1])
            c.freeze_limiter_values(phi[q])
            l1 = c.explicit_run(3, 0.8)
            assert np.array_equal(c.get_state(), U[q]) and np.array_equal(l1, linf[:, q])
