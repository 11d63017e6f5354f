"""Forms of the AMG's kernels that small hierarchies do not reach: the sliced
sweep copy of large coarse levels and the coarsest inverse at the sizes where
its panels change, against the CPU restatement built from the GPU's aggregates."""
import numpy as np
import pytest
import scipy.sparse.linalg as spla

from bes_amd import core, meshgen as mg
from oracle import amg, oracle as orc

pytestmark = pytest.mark.gpu


def _context(md, mach, precision, relax, coarse_enough=500, cfl=20.0):
    finf = orc.freestream_primitive(mach, md.ndim)
    c = core.Context(md)
    c.set_freestream(finf)
    c.implicit_setup(precision, "amg", rtol=1e-8)
    c.amg_set_params(relax=relax, coarse_enough=coarse_enough)
    c.set_state(orc.perturbed_state(md.ncell, md.ndim, mach, seed=3, amp=0.02))
    c.implicit_assemble(cfl, repeat_nv=False)
    rp, col, val, rhs = c.implicit_system()
    return c, amg.BlockCsr.from_scalar_csr(rp, col, val, c.nv)


def _vcycle(c, A, kind, coarse_enough, r):
    rows, _, direct = c.amg_info()
    aggs = [c.amg_level(l)[0] for l in range(len(rows))]
    levels, inv = amg.hierarchy(A, aggregates=lambda l, Al: (int(rows[l + 1]), aggs[l]), kind=kind,
                                coarse_enough=coarse_enough)
    return rows, direct, amg.vcycle(levels, inv, r)


# the first coarse level is past 16,384 rows and no multiple of the 64-row slices
# or the 1024-row windows.  FP16 entries: each block is off by up to 2^-11 of its
# row's scale, which a cycle carries to z at that order
@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("relax,kind", [("block_jacobi", "block"), ("jacobi", "jacobi")])
def test_sliced_level(nd, relax, kind):
    md = mg.bump_channel(331, 167) if nd == 2 else mg.swept_wing(40, 20, 30)
    c, A = _context(md, (0.5, 0.0) if nd == 2 else (0.83, 0.0, 0.04), 32, relax)
    with c:
        r = np.random.default_rng(5).standard_normal(md.ncell * c.nv)
        z = c.amg_apply(r).ravel()
        rows, _, zr = _vcycle(c, A, kind, 500, r)
        print("levels", list(rows))
        assert rows[1] >= 16384 and rows[1] % 64 != 0
        assert np.linalg.norm(z - zr) <= 2e-3 * np.linalg.norm(zr)


# scalar rows of the coarsest system: fewer than a panel's 16 columns, a ragged
# last panel, the whole system (level 0 itself) and past 500, where a panel takes
# fewer columns to fit LDS
@pytest.mark.parametrize("mesh,coarse_enough", [
    (("bump", 24, 12), 12), (("bump", 24, 12), 100), (("bump", 9, 6), 500), (("box", 3, 3, 2), 600),
    (("box", 9, 8, 7), 500), (("bump", 15, 8), 1000), (("box", 11, 3, 1), 1000)])
def test_coarsest_inverse(mesh, coarse_enough):
    md = mg.bump_channel(*mesh[1:]) if mesh[0] == "bump" else mg.box_tets(*mesh[1:], seed=3)
    mach = (0.5, 0.0) if md.ndim == 2 else (0.7, 0.0, 0.05)
    c, A = _context(md, mach, 64, "block_jacobi", coarse_enough)
    with c:
        r = np.random.default_rng(6).standard_normal(md.ncell * c.nv)
        z = c.amg_apply(r).ravel()
        rows, direct, zr = _vcycle(c, A, "block", coarse_enough, r)
        print("levels", list(rows), "scalar rows of the coarsest", rows[-1] * c.nv)
        assert direct and rows[-1] * c.nv <= coarse_enough
        assert np.abs(z - zr).max() <= 1e-9 * np.abs(zr).max()
        if len(rows) == 1:   # the inverse is the whole cycle
            x = spla.spsolve(_csc(A), r)
            assert np.abs(z - x).max() <= 1e-9 * np.abs(x).max()


def _csc(A):
    import scipy.sparse as sp
    return sp.bsr_matrix((A.val, A.col, A.rp), shape=(A.n * A.val.shape[1],) * 2).tocsc()
