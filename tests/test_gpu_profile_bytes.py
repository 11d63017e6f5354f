"""Algorithmic bytes that the profile reports for the explicit passes: every
array a launch touches, once, in the split passes of small meshes and the
separate ones of larger meshes; and for the Gram-Schmidt passes that did work."""
import numpy as np
import pytest

from bes_amd import core, meshgen as mg

pytestmark = pytest.mark.gpu


def _profile(md, mode, B, local):
    P = core.freestream_primitive((0.5,) + (0.0,) * (md.ndim - 1), md.ndim)
    U = core.conserved_from_primitive(P, md.ndim)
    with core.Context(md, geom_mode=mode) as c:
        if B > 1:
            c.set_batch(B)
        shape = (md.ncell, md.ndim + 2) if B == 1 else (B, md.ncell, md.ndim + 2)
        c.set_freestream(P if B == 1 else np.tile(P, (B, 1)))
        c.set_state(np.ascontiguousarray(np.broadcast_to(U, shape)))
        c.set_profiling(True)
        c.explicit_run(2, 0.8, local=local, alpha=(0.5, 1.0))
        return c.profile()


@pytest.mark.parametrize("mode", [core.GEOM_COMPAT, core.GEOM_EXACT])
@pytest.mark.parametrize("local", [True, False])
@pytest.mark.parametrize("mesh,B,split", [(("bump", 20, 10), 1, True), (("box", 5, 4, 3), 1, True),
                                          (("box", 5, 4, 3), 4, True), (("box", 26, 25, 25), 1, False)])
def test_bytes_of_the_explicit_passes(mesh, B, split, local, mode):
    md = mg.bump_channel(*mesh[1:]) if mesh[0] == "bump" else mg.box_tets(*mesh[1:], seed=3)
    nd, N = md.ndim, md.ncell
    nv, k = nd + 2, nd + 1
    F = (N * k + len(md.bfaces)) // 2
    fs = (nv + 1) // 2 * 2 if B == 1 else nv
    pack = 8 * B * (fs if mode == core.GEOM_COMPAT else nv * (1 + nd))
    face = (8 if mode == core.GEOM_COMPAT else 24) * nd
    p = _profile(md, mode, B, local)
    grad = N * (8 * nv * B + k * (16 * nd + 12) + 16 + pack)
    cell = N * (12 * k + 8 + 8 * B + 16 * nv * B)   # faces and areas, V, dt, U0 and U
    got = {q: p[q]["bytes"] / p[q]["launches"] for q in p}
    step = N * (8 * (nv * B + nd + 1) + 8 * B)
    if split:
        dt = N * (8 * nd + 8 * B) if local else 0   # in the first stage's gradient pass
        assert p["gradlim"]["bytes"] == 4 * grad + 2 * dt
        assert got["residual"] == cell + N * (4 * k + 4 + pack) + F * face
        assert "faceflux" not in p and ("timestep" in p) == (not local)
    else:
        assert got["gradlim"] == grad
        assert got["faceflux"] == F * (8 + face + 8 * fs * B) + N * pack
        assert got["residual"] == cell + F * 8 * fs * B
    if "timestep" in p:
        assert got["timestep"] == step


# a second pass that no condition needs moves nothing
@pytest.mark.parametrize("ni,nj,B", [(40, 20, 1), (40, 20, 4), (331, 299, 1)])
def test_bytes_of_an_idle_second_pass(ni, nj, B):
    md = mg.bump_channel(ni, nj)
    P = core.freestream_primitive((0.5, 0.0), 2)
    rng = np.random.default_rng(1)
    U = core.conserved_from_primitive(P, 2) * (1.0 + 0.01 * rng.uniform(-1, 1, (B, md.ncell, 4)))
    print("case", md.ncell, B, flush=True)
    bytes_of, reorths = {}, {}
    for eta in (0.0, 1e-9, 1.0):
        with core.Context(md) as c:
            c.set_batch(B)
            c.set_freestream(np.tile(P, (B, 1)) if B > 1 else P)
            c.set_state(U if B > 1 else U[0])
            c.implicit_setup(64, "ilu0", maxiter=8, rtol=1e-14)
            c.implicit_set_reorth(eta)
            c.implicit_assemble(20.0)
            c.set_profiling(True)
            c.linear_solve(allow_unconverged=True)
            bytes_of[eta] = c.profile()["krylov"]["bytes"]
            reorths[eta] = c.implicit_stats()["reorths"]
    assert reorths == {0.0: 0, 1e-9: 0, 1.0: 8 * B}
    assert bytes_of[1e-9] == bytes_of[0.0] < bytes_of[1.0]
