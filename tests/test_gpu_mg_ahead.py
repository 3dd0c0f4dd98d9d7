"""Threshold solves enqueue several gated V-cycles at a time: a solve that stops after n of them
(none, inside the first chunk, at its end, later, by stalling) equals the solve of n fixed
V-cycles bit for bit, and so does the next solve on the same mesh."""
import time

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


def _mesh(agx, mp, precision, eps):
    n = 32
    d = make_desc(nx=(n, n, n), bnx=(8, 8, 8), box=BOX, self_gravity=1, mg_bc=mp, mg_mode=0, four_pi_G=1.0, mporder=4,
                  mg_threshold=eps, precision=precision)
    U = np.zeros((5, n, n, n))
    U[0] = gaussian(n, 0.06, c=(0.05, -0.04, 0.03)) + (0.0 if mp else 1.0)
    m = agx.Mesh(d)
    m.set("u", agx.scatter_cells(d, U))
    return m


@pytest.mark.parametrize("mp", [0, 1])
def test_solve_that_needs_no_vcycle_runs_none(agx, mp):
    """one launch per step, so that a V-cycle, closed gate or not, takes longer than all else a
    read norm can cost: a solve whose first norm meets the threshold against a solve of one fixed
    V-cycle, which does everything the other does and the V-cycle"""
    m = _mesh(agx, mp, 0, 1e30)
    m.set_mg_fuse(0)
    m.set_mg_coarse(0)

    def best():
        out = []
        for _ in range(8):
            m.sync()
            t = time.perf_counter()
            m.mg_solve(0)
            m.sync()
            out.append(time.perf_counter() - t)
        return min(out)

    none = best()
    assert m.mg_last()[1] == 0
    m.mg_set_mode(0, -1.0, 1)
    one = best()
    m.close()
    print(f"mp {mp}: no V-cycle {none * 1e6:.0f} us, one {one * 1e6:.0f} us", flush=True)
    assert none < one


@pytest.mark.parametrize("mp", [0, 1])
@pytest.mark.parametrize("precision", [0, 1])
def test_timers_count_the_passes_that_ran(agx, mp, precision):
    """no pass behind a closed gate is timed: a threshold solve of n V-cycles books the sweeps of
    the solve of n fixed ones"""
    m = _mesh(agx, mp, precision, 1e-5)
    m.timing(True)
    launches = []
    for mode in ((1e-5, 0), (1e-5, 0), None):
        m.mg_set_mode(0, *(mode or (-1.0, m.mg_last()[1])))
        m.timing_reset()
        m.mg_solve(0)
        launches.append(m.timing_get("mg_smooth")[1])
    m.close()
    print(f"mp {mp} precision {precision}: {launches}", flush=True)
    assert launches[0] == launches[1] == launches[2]


def test_prediction_from_a_longer_solve(agx):
    """a solve that needs fewer V-cycles than the last one of its stage (gated passes enqueued
    unread) equals the same solve on a new mesh"""
    for eps in (1e3, 1e-2, 1e-4):
        out = []
        for before in (True, False):
            m = _mesh(agx, 0, 0, 1e-9)
            if before:
                m.mg_solve(0)
                assert m.mg_last()[1] >= 4
                m.mg_coffset(True) if m.mg_coffset() else None
            m.mg_set_mode(0, eps, 0)
            m.mg_solve(0)
            out.append((m.get("phi"), m.mg_last()))
            m.close()
        assert out[0][1] == out[1][1] and np.array_equal(out[0][0], out[1][0])
