"""k_mg_coarse, k_mg_down and k_mg_up against the per-level steps at the edges of their ranges: the
whole hierarchy in the coarse kernel (16^3 cells, and one 8^3 block), root grids that are odd or
flat, levels just above it, levels of one tile, of several and of parts of one, and flat ones; chunks
of two planes (the small shapes), of eight (128^3), and of six with a last one of four (192 x 160 x 40,
the finest level of one shape and a level with a FAS right-hand side of another); the same potential
bit for bit."""
import numpy as np
import pytest

from oracle.orc import Oracle, make_desc
from tests.test_gpu_mg_levels import vcycle_by_steps

pytestmark = pytest.mark.gpu

SHAPES = [((8, 8, 8), 8), ((16, 16, 16), 8), ((24, 8, 8), 8), ((12, 20, 4), 4), ((64, 8, 4), 4), ((32, 32, 32), 8),
          ((40, 24, 56), 8), ((72, 16, 8), 8), ((96, 48, 16), 16), ((128, 128, 4), 4), ((128, 128, 128), 32),
          ((192, 160, 40), 8), ((384, 320, 80), 16)]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,b", SHAPES)
def test_multipole_vcycles_identical(agx, n, b, precision):
    """one launch against one launch per step (a mixed V-cycle is a defect-correction step)"""
    h = 1.0 / max(n)
    d = make_desc(nx=n, bnx=(b, b, b), box=tuple((-0.5 * h * q, 0.5 * h * q) for q in n), self_gravity=1, mg_bc=1,
                  mg_mode=0, four_pi_G=1.0, mporder=4, mg_threshold=-1.0, mg_niter=2, precision=precision)
    U = np.zeros((5, n[2], n[1], n[0]))
    U[0] = np.random.default_rng(3).uniform(0.5, 1.5, n[::-1])
    ub = agx.scatter_cells(d, U)
    out = []
    for on in (1, 0):
        m = agx.Mesh(d)
        m.set("u", ub)
        m.set_mg_coarse(on)
        m.mg_solve(0)
        m.mg_solve(0)   # FMG starts from what the first solve left on the root level
        out.append((m.get("phi"), m.mg_last()))
        m.close()
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]


@pytest.mark.parametrize("n,b", [(8, 8), (16, 8), (16, 16), (32, 16)])
def test_periodic_vcycle_identical(agx, n, b):
    d = make_desc(nx=(n,) * 3, bnx=(b,) * 3, box=((0.0, 1.0),) * 3, self_gravity=1, mg_bc=0, mg_mode=0, four_pi_G=1.0,
                  mg_threshold=-1.0, mg_niter=1)
    U = np.zeros((5, n, n, n))
    U[0] = np.random.default_rng(4).uniform(0.5, 1.5, (n, n, n))
    ub = agx.scatter_cells(d, U)
    a, c = agx.Mesh(d), agx.Mesh(d)
    for m in (a, c):
        m.set("u", ub)
        m.mg_solve(0)
    a.mg_vcycles(2)
    for _ in range(2):
        vcycle_by_steps(c, False)
    assert a.mg_defect_norm() == c.mg_defect_norm()
    for m in (a, c):
        m.mg_step("retrieve")
    assert np.array_equal(a.get("phi"), c.get("phi"))
    a.close()
    c.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,b", [((40, 24, 56), 8), ((64, 64, 64), 32), ((128, 32, 32), 32), ((128, 128, 4), 4),
                                 ((96, 48, 16), 16), ((36, 20, 12), 4), ((128, 128, 128), 32), ((192, 160, 40), 8)])
def test_periodic_passes_identical(agx, n, b, precision):
    """whole passes against one launch per step"""
    h = 1.0 / max(n)
    d = make_desc(nx=n, bnx=(b, b, b), box=tuple((0.0, h * q) for q in n), self_gravity=1, mg_bc=0, mg_mode=0,
                  four_pi_G=1.0, mg_threshold=-1.0, mg_niter=2, precision=precision)
    U = np.zeros((5, n[2], n[1], n[0]))
    U[0] = np.random.default_rng(5).uniform(0.5, 1.5, n[::-1])
    ub = agx.scatter_cells(d, U)
    out = []
    for mode in (1, 0):
        m = agx.Mesh(d)
        m.set("u", ub)
        m.set_mg_fuse(mode)
        m.mg_solve(0)
        out.append((m.get("phi"), m.mg_last()))
        m.close()
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]


@pytest.mark.parametrize("n,b", [((4, 4, 4), 4), ((36, 20, 12), 4), ((64, 4, 8), 4), ((24, 40, 56), 8), ((48, 96, 16), 16)])
def test_defect_norm_matches_oracle(agx, n, b):
    """the finest defect's norm, rows shorter and longer than a workgroup's step: sums of at most
    2e5 squares in another order agree to 1e-9 of the norm (the bar of the parity tests)"""
    h = 1.0 / max(n)
    d = make_desc(nx=n, bnx=(b, b, b), box=tuple((0.0, h * q) for q in n), self_gravity=1, mg_bc=0, mg_mode=0,
                  four_pi_G=1.0, mg_threshold=-1.0, mg_niter=1)
    U = np.zeros((5, n[2], n[1], n[0]))
    U[0] = np.random.default_rng(6).uniform(0.5, 1.5, n[::-1])
    ub = agx.scatter_cells(d, U)
    norms = []
    for m in (agx.Mesh(d), Oracle(d)):
        m.set("u", ub)
        m.mg_solve(0)
        norms.append(m.mg_last()[0])
    print(n, norms, flush=True)
    assert abs(norms[0] - norms[1]) <= 1e-9 * norms[1]
