"""k_flux with its three directions in one launch against one launch per direction (which the
timers use): blocks smaller than a workgroup, with odd sides, and with planes of several
workgroups; every order, and FP32 PPM with its near-tie pass."""
import numpy as np
import pytest

from oracle.orc import make_desc
from tests.states import load_state, turbulent_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,precision", [(1, 0), (2, 0), (3, 0), (2, 1), (3, 1)])
@pytest.mark.parametrize("bnx", [(6, 6, 6), (13, 7, 9), (33, 17, 6), (40, 16, 5)])
def test_directions_in_one_launch_identical(agx, bnx, order, precision):
    d = make_desc(nx=tuple(2 * q for q in bnx), bnx=bnx, box=((0.0, 1.0),) * 3, cfl=0.3, nghost=3, xorder=order,
                  precision=precision)
    st = turbulent_state(d, seed=7, mach=2.0)
    out = []
    for timing in (False, True):
        m = agx.Mesh(d)
        load_state(m, st)
        m.initialize()
        m.set_tile(1)
        m.timing(timing)
        m.cycle(1e9, 2)
        out.append([m.get(n) for n in ("u", "b1f", "b2f", "b3f")])
        m.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("order,precision", [(1, 0), (2, 0), (3, 0), (2, 1), (3, 1)])
def test_large_mesh_equals_one_launch_stage(agx, order, precision):
    """arrays beyond the last-level cache, where k_flux takes its workgroups in plain order: the
    split form against the stage that solves its faces itself"""
    d = make_desc(nx=(128, 96, 100), bnx=(32, 24, 20), box=((0.0, 1.28), (0.0, 0.96), (0.0, 1.0)), cfl=0.3, nghost=3,
                  xorder=order, precision=precision)
    st = turbulent_state(d, seed=8, mach=2.0)
    out = []
    for form in (1, 5):
        m = agx.Mesh(d)
        load_state(m, st)
        m.initialize()
        m.set_tile(form)
        m.cycle(1e9, 1)
        out.append([m.get(n) for n in ("u", "b1f", "b2f", "b3f")])
        m.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))
