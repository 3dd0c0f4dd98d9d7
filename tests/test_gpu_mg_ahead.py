"""Threshold solves enqueue several gated V-cycles at a time: a solve that stops after n of them
(none, inside the first chunk, at its end, later, by stalling) equals the solve of n fixed
V-cycles bit for bit, and so does the next solve on the same mesh."""
import numpy as np
import pytest

from oracle.orc import make_desc
from tests.test_oracle_mg_multipole import BOX, gaussian

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mp", [0, 1])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("eps", [1e3, 1e-3, 1e-5, 1e-7, 1e-10, 0.0])
def test_threshold_equals_fixed_count(agx, mp, precision, eps):
    n = 32
    U = np.zeros((5, n, n, n))
    U[0] = gaussian(n, 0.06, c=(0.05, -0.04, 0.03)) + (0.0 if mp else 1.0)
    counts = []

    def run(modes):
        d = make_desc(nx=(n, n, n), bnx=(8, 8, 8), box=BOX, self_gravity=1, mg_bc=mp, mg_mode=0, four_pi_G=1.0, mporder=4,
                      mg_threshold=eps, precision=precision)
        m = agx.Mesh(d)
        m.set("u", agx.scatter_cells(d, U))
        out = []
        for k in range(2):
            m.mg_set_mode(0, *(modes[k] if modes else (eps, 0)))
            m.mg_solve(0)
            counts.append(m.mg_last()[1])
            out.append(m.get("phi"))
        m.close()
        return out

    a = run(None)
    b = run([(-1.0, c) for c in counts[:2]])
    print(f"eps {eps}: V-cycles {counts[:2]}", flush=True)
    assert counts[:2] == counts[2:]
    assert all(np.array_equal(x, y) for x, y in zip(a, b))
