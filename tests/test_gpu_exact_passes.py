"""The explicit passes with a reconstruction vector per face (geom_mode EXACT),
on both sides of the sizes where the dispatch changes (98,304 cell-conditions
in 2D, 49,152 in 3D), in batches and in the persistent step: against the CPU
oracle, each condition's own run and the launched passes, bit for bit."""
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


@pytest.mark.parametrize("mesh", [("bump", 11, 3), ("box", 5, 5, 3), ("bump", 256, 192), ("bump", 223, 221),
                                  ("box", 32, 16, 16), ("box", 21, 20, 20), ("box", 25, 25, 25)])
def test_steps_equal_the_oracle(mesh):
    md = _mesh(*mesh)
    finf, U = _case(md)
    om = orc.Mesh(md, orc.EXACT)
    G = om.gradient(U)
    P = om.limiter(U, G)
    R = om.residual(U, G, P, finf)
    alpha = (0.1481, 0.4, 1.0)
    Ur, lr = om.explicit(U, 2, 0.8, finf, alpha=alpha)
    print("case", mesh, flush=True)
    with core.Context(md, geom_mode=core.GEOM_EXACT) as c:
        c.set_freestream(finf)
        c.set_state(U)
        Rg, mx = c.residual()
        Gg, Pg = c.gradient_limiter()
        linf = c.explicit_run(2, 0.8, alpha=alpha)
        assert np.array_equal(Gg, G) and np.array_equal(Pg, P)
        assert np.array_equal(Rg, R) and np.array_equal(mx, np.abs(R).max(axis=0))
        assert np.array_equal(c.get_state(), Ur) and np.array_equal(linf, lr)


# batches on both sides of the line
@pytest.mark.parametrize("mesh,B", [(("bump", 9, 4), 2), (("bump", 32, 24), 64), (("bump", 33, 24), 64),
                                    (("box", 4, 4, 3), 8), (("box", 8, 4, 4), 64), (("box", 12, 12, 14), 8)])
def test_batch_equals_single_runs(mesh, B):
    md = _mesh(*mesh)
    PU = [_case(md, 10 + q) for q in range(B)]
    print("case", mesh, B, flush=True)
    with core.Context(md, geom_mode=core.GEOM_EXACT) as c:
        c.set_batch(B)
        c.set_freestream(np.stack([p for p, _ in PU]))
        c.set_state(np.stack([u for _, u in PU]))
        linf = c.explicit_run(3, 0.8)
        U = c.get_state()
    om = orc.Mesh(md, orc.EXACT)
    for q in sorted({0, 1, B - 1}):
        Ur, lr = om.explicit(PU[q][1], 3, 0.8, PU[q][0], alpha=core.RK4_ALPHA)
        assert np.array_equal(U[q], Ur) and np.array_equal(linf[:, q], lr)


# fewer blocks than the grid holds and more, the launched passes split and not
@pytest.mark.parametrize("mesh", [("bump", 40, 20), ("box", 12, 10, 8), ("box", 32, 24, 24)])
def test_persistent_matches_launched(mesh):
    md = _mesh(*mesh)
    finf, U = _case(md)
    print("case", mesh, flush=True)
    out = []
    for persistent in (False, True):
        with core.Context(md, geom_mode=core.GEOM_EXACT) as c:
            c.set_freestream(finf)
            c.set_state(U)
            c.explicit_persistent(persistent)
            linf = c.explicit_run(3, 0.8)
            out.append((c.get_state(), linf))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert not np.array_equal(out[1][0], U)
