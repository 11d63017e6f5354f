"""A captured step after the state slots changed places: one-stage schemes swap
them at every step, and a capture made before must not run on the old ones."""
import numpy as np
import pytest

from bes_amd import core, meshgen as mg
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("persistent", [False, True])
def test_capture_follows_the_state_slots(persistent):
    md = mg.bump_channel(20, 10)
    finf = orc.freestream_primitive((0.5, 0.1), 2)
    U = orc.perturbed_state(md.ncell, 2, (0.5, 0.1), seed=4)
    om = orc.Mesh(md)
    with core.Context(md) as c:
        c.set_freestream(finf)
        c.set_state(U)
        c.explicit_graph(True)
        c.explicit_run(5, 0.5)   # captured
        U, _ = om.explicit(U, 5, 0.5, finf)
        c.explicit_persistent(persistent)
        c.explicit_run(3, 0.3, alpha=(1.0,))
        U, _ = om.explicit(U, 3, 0.3, finf, alpha=(1.0,))
        c.explicit_persistent(False)
        linf = c.explicit_run(2, 0.5)
        U, lr = om.explicit(U, 2, 0.5, finf)
        assert np.array_equal(c.get_state(), U) and np.array_equal(linf, lr)
