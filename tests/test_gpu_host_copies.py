"""Host copies of per-cell arrays: the device-side permutation between the
callers' order and the device layout, against the values themselves."""
import time

import numpy as np
import pytest

from bes_amd import core, meshgen as mg

pytestmark = pytest.mark.gpu


def _states(md, B, seed):
    rng = np.random.default_rng(seed)
    base = core.conserved_from_primitive(core.freestream_primitive((0.4,) + (0.0,) * (md.ndim - 1), md.ndim), md.ndim)
    U = base * (1.0 + 0.01 * rng.uniform(-1, 1, (B, md.ncell, md.ndim + 2)))
    return U[0] if B == 1 else U


# the host loop (up to 512 KiB) and its last size, then the kernel: ragged
# counts, a block's run of every batch size, and an array larger than the
# staging buffer (128 MiB), which goes through it in chunks of cells
@pytest.mark.parametrize("mesh,B", [
    (("bump", 3, 2), 1), (("box", 5, 4, 3), 16), (("bump", 64, 128), 1), (("bump", 129, 64), 1),
    (("bump", 91, 101), 1), (("bump", 91, 47), 2), (("bump", 37, 5), 64), (("box", 13, 11, 9), 4),
    (("box", 7, 5, 5), 32), (("bump", 250, 141), 64),
])
def test_round_trip(mesh, B):
    md = mg.bump_channel(*mesh[1:]) if mesh[0] == "bump" else mg.box_tets(*mesh[1:])
    U = _states(md, B, 7)
    with core.Context(md) as c:
        if B > 1:
            c.set_batch(B)
        c.set_state(U)
        assert np.array_equal(c.get_state(), U)
        # a second state after the first: nothing of it is left behind
        V = _states(md, B, 8)
        c.set_state(V)
        assert np.array_equal(c.get_state(), V)


@pytest.mark.parametrize("n,B", [((5, 4, 3), 1), ((11, 9, 8), 1), ((11, 9, 8), 4)])
def test_gradient_and_limiter_values(n, B):
    """Arrays of more than nv values per cell, frozen limiter values back in."""
    md = mg.box_tets(*n, seed=3)
    U = _states(md, B, 9)
    with core.Context(md) as c:
        if B > 1:
            c.set_batch(B)
        c.set_freestream(core.freestream_primitive((0.4, 0.0, 0.0), 3))
        c.set_state(U)
        G, P = c.gradient_limiter()
        single = []
        for b in range(B):
            with core.Context(md) as d:
                d.set_freestream(core.freestream_primitive((0.4, 0.0, 0.0), 3))
                d.set_state(U if B == 1 else U[b])
                single.append(d.gradient_limiter())
        assert np.array_equal(G, single[0][0] if B == 1 else np.stack([s[0] for s in single]))
        assert np.array_equal(P, single[0][1] if B == 1 else np.stack([s[1] for s in single]))
        c.freeze_limiter_values(0.5 * P)
        assert np.array_equal(c.gradient_limiter()[1], 0.5 * P)


@pytest.mark.parametrize("B", [16, 64])
def test_ragged_counts_copy_in_one_piece(B):
    """A cell count that no block of the permutation divides takes about what its
    neighbour does (cut in two chunks, every condition's part would be a copy of its
    own)."""
    took = {}
    for ni in (640, 641):   # 3,840 cells: whole blocks; 3,846: not
        md = mg.bump_channel(ni, 3)
        U = np.tile(_states(md, 1, 7), (B, 1, 1))
        with core.Context(md) as c:
            c.set_batch(B)
            c.set_state(U)
            ts = []
            for _ in range(15):
                t = time.perf_counter()
                out = c.get_state()
                ts.append(time.perf_counter() - t)
            assert np.array_equal(out, U)
            took[md.ncell] = sorted(ts)[7]
    print("seconds", took)
    assert took[3846] < 3 * took[3840]
