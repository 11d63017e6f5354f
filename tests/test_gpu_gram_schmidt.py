"""The Gram-Schmidt kernels over the ranges of their dispatch: the number of
reduction lanes follows the vector length (256 lanes up to 16,384 values, then
doubling), and with it the form of the dot products and of the update."""
import numpy as np
import pytest
import scipy.sparse as sp

from bes_amd import core, meshgen as mg

pytestmark = pytest.mark.gpu


def _state(md, seed, mach=(0.5, 0.0)):
    P = core.freestream_primitive(mach, 2)
    rng = np.random.default_rng(seed)
    return P, core.conserved_from_primitive(P, 2) * (1.0 + 0.01 * rng.uniform(-1, 1, (md.ncell, 4)))


def _gmres_iterate(A, b, m):
    """GMRES after m <= restart steps, x0 = 0: the least-squares problem solved directly."""
    beta = np.linalg.norm(b)
    V, H = [b / beta], np.zeros((m + 1, m))
    for j in range(m):
        w = A @ V[j]
        for _ in range(2):
            h = np.array([v @ w for v in V])
            H[:j + 1, j] += h
            w = w - sum(hq * v for hq, v in zip(h, V))
        H[j + 1, j] = np.linalg.norm(w)
        V.append(w / H[j + 1, j])
    e1 = np.zeros(m + 1)
    e1[0] = beta
    y = np.linalg.lstsq(H, e1, rcond=None)[0]
    return sum(yq * v for yq, v in zip(y, V))


# vector lengths 4*cells: one lane group short of and just past 256 lanes,
# ragged lane groups, the last size of the thread-per-group update (16,384
# lanes) and the first past it, the first with 2^17 lanes
@pytest.mark.parametrize("ni,nj", [(12, 8), (64, 32), (41, 50), (183, 83), (512, 256), (512, 257), (1024, 513)])
@pytest.mark.parametrize("eta", [0.0, 0.7])
def test_iterate_matches_numpy(ni, nj, eta):
    steps = 11
    md = mg.bump_channel(ni, nj)
    P, U = _state(md, 3)
    print("case", md.ncell, eta, flush=True)
    with core.Context(md) as c:
        c.set_freestream(P)
        c.set_state(U)
        c.implicit_setup(64, "none", restart=30, maxiter=steps, rtol=1e-14)
        c.implicit_set_reorth(eta)
        c.implicit_assemble(20.0)
        it, rr = c.linear_solve(allow_unconverged=True)
        x = c.linear_solution().ravel()
        rp, col, val, rhs = c.implicit_system()
    A = sp.csr_matrix((val, col, rp), shape=(md.ncell * 4,) * 2)
    b = rhs.ravel()
    xr = _gmres_iterate(A, b, steps)
    assert it == steps
    np.testing.assert_allclose(np.linalg.norm(b - A @ x) / np.linalg.norm(b), rr, rtol=1e-6)
    assert np.linalg.norm(x - xr) <= 1e-8 * np.linalg.norm(xr)


# a condition's iterates are the same bits in a batch as alone: scalar loads
# (B = 2), four conditions a thread (B >= 4), either form of the update
# (both forms for B = 2, the thread-per-group one for larger batches: the other,
# and their lane sums in two launches, are in test_gpu_batch_reductions.py)
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("ni,nj,B", [(20, 11, 2), (20, 11, 4), (64, 33, 8), (90, 47, 64), (300, 221, 2)])
@pytest.mark.parametrize("eta", [0.0, 0.7])
def test_batch_is_single_runs(ni, nj, B, precision, eta):
    md = mg.bump_channel(ni, nj)
    mach = [(0.3 + 0.4 * q / B, 0.0) for q in range(B)]
    PU = [_state(md, 5 + q, mach[q]) for q in range(B)]
    print("case", md.ncell, B, precision, eta, flush=True)

    def solve(c):
        c.implicit_setup(precision, "ilu0", maxiter=40, rtol=1e-4)
        c.implicit_set_reorth(eta)
        c.implicit_assemble(20.0)
        c.linear_solve(allow_unconverged=True)
        return c.linear_solution()

    with core.Context(md) as c:
        c.set_batch(B)
        c.set_freestream(np.stack([p for p, _ in PU]))
        c.set_state(np.stack([u for _, u in PU]))
        xb = solve(c)
        its = c.implicit_batch_state()["iters"]
    assert its.min() > 4
    for q in sorted({0, 1, B - 1}):
        with core.Context(md) as c:
            c.set_freestream(PU[q][0])
            c.set_state(PU[q][1])
            assert np.array_equal(solve(c), xb[q]), f"condition {q}"
