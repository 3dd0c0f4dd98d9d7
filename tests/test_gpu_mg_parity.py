"""GPU vs oracle parity for the FP64 multigrid self-gravity solve.

The GPU stores each level as one periodic grid; the oracle keeps the reference's
per-MeshBlock hierarchy + root grid with explicit ghost exchanges.  Stencil values
agree exactly; sums (source mean, defect norm) differ in summation order, so the
bar is |phi_gpu - phi_oracle| <= 1e-12 * max|phi| and equal V-cycle counts.
"""
import numpy as np
import pytest

from oracle.orc import Oracle, make_desc
from tests.conftest import load_agx
from tests.test_oracle_mg import blobs, fft_solution

pytestmark = pytest.mark.gpu


def both(N, B, rho, **kw):
    agx = load_agx()
    d = make_desc(nx=(N, N, N), bnx=(B, B, B), box=((0, 1), (0, 1), (0, 1)), self_gravity=1, **kw)
    U = np.zeros((5, N, N, N))
    U[0] = rho
    ub = agx.scatter_cells(d, U)
    o = Oracle(d)
    o.set("u", ub)
    o.mg_solve(0)
    m = agx.Mesh(d)
    m.set("u", ub)
    m.mg_solve(0)
    return (agx.gather_cells(d, m.get("phi"))[0], m.mg_last(), m.get("phi"),
            agx.gather_cells(d, o.get("phi"))[0], o.mg_last(), o.get("phi"))


@pytest.mark.parametrize("N,B", [(32, 8), (32, 32), (64, 16), (16, 4)])
def test_fmg_threshold_parity(N, B):
    rho = blobs(N, 1)
    pg, (ng, ig), pgb, po, (no, io), pob = both(N, B, rho, mg_mode=0, mg_threshold=0.0, four_pi_G=0.7)
    scale = np.abs(po).max()
    err = np.abs(pg - po).max()
    print(f"N={N} B={B}: iters gpu {ig} oracle {io}; norm {ng:.3e} {no:.3e}; max|dphi| {err:.3e}")
    assert ig == io
    assert err <= 1e-12 * scale
    # the one-cell ghost layer written by RetrieveResult agrees too
    g1 = slice(1, -1)
    np.testing.assert_allclose(pgb[:, :, g1, g1, g1], pob[:, :, g1, g1, g1], atol=1e-12 * scale, rtol=0)
    ref = fft_solution(rho, 0.7)
    assert np.abs(pg - ref).max() <= 1e-11 * np.abs(ref).max()


@pytest.mark.parametrize("niter", [1, 3])
def test_mgi_fixed_parity(niter):
    rho = blobs(32, 2)
    pg, (ng, ig), _, po, (no, io), _ = both(32, 16, rho, mg_mode=1, mg_threshold=-1.0, mg_niter=niter)
    assert ig == io == niter
    assert np.abs(pg - po).max() <= 1e-12 * np.abs(po).max()
    assert abs(ng - no) <= 1e-10 * no


def test_absolute_threshold_iterations():
    rho = blobs(32, 3)
    pg, (ng, ig), _, po, (no, io), _ = both(32, 8, rho, mg_mode=0, mg_threshold=1e-9)
    assert ig == io
    assert ng <= 1e-9 and no <= 1e-9
    assert np.abs(pg - po).max() <= 1e-12 * np.abs(po).max()



def test_fused_red_black_levels():
    """A finest level of 2^26 cells, which k_mg_down and k_mg_up walk in one chunk of all its
    planes: 512 x 512 x 256 in MeshBlocks of 256^3.  Fixed V-cycle counts: the oracle's iterate
    sequence, same bar."""
    agx = load_agx()
    N1, N3, B = 512, 256, 256
    d = make_desc(nx=(N1, N1, N3), bnx=(B, B, B), box=((0, 1), (0, 1), (0, 0.5)), self_gravity=1,
                  mg_mode=0, mg_threshold=-1.0, mg_niter=1, four_pi_G=1.0)
    x = (np.arange(N1) + 0.5) / N1
    z = (np.arange(N3) + 0.5) / N1
    Z, Y, X = np.meshgrid(z, x, x, indexing="ij")
    rho = 1.0 + 20.0 * np.exp(-((X - 0.3) ** 2 + (Y - 0.6) ** 2 + (Z - 0.2) ** 2) / 0.05 ** 2) \
        + 5.0 * np.exp(-((X - 0.7) ** 2 + (Y - 0.25) ** 2 + (Z - 0.35) ** 2) / 0.08 ** 2)
    U = np.zeros((5, N3, N1, N1))
    U[0] = rho
    ub = agx.scatter_cells(d, U)
    del U
    o = Oracle(d)
    o.set("u", ub)
    o.mg_solve(0)
    m = agx.Mesh(d)
    m.set("u", ub)
    m.mg_solve(0)
    a, b = m.get("phi"), o.get("phi")
    # the source mean and the final mean of u are sums over 2^26 cells in another order
    # (a constant shift of phi); the rest of the difference is held to the bar
    diff = a - b
    offset = diff.mean()
    scale = np.abs(b).max()
    err = np.abs(diff - offset).max() / scale
    (ng, ig), (no, io) = m.mg_last(), o.mg_last()
    print(f"512x512x256: defect {ng:.6e} vs {no:.6e}; constant offset {offset / scale:.3e}, "
          f"max|dphi - offset|/max|phi| {err:.3e}", flush=True)
    assert abs(offset) <= 1e-11 * scale
    assert err <= 1e-12
    assert ig == io == 1
    assert abs(ng - no) <= 1e-9 * no


@pytest.mark.parametrize("precision", [0, 1])
def test_red_black_pass_forms_identical(precision):
    """Whole passes of a level (k_mg_down, k_mg_up) and one launch per step give the same
    potential bit for bit, in FP64 and in the FP32 correction cycles of the mixed form.  The
    autotuner picks one of the two, so its choice cannot change results."""
    agx = load_agx()
    N, B = 128, 32
    d = make_desc(nx=(N, N, N), bnx=(B, B, B), box=((0, 1),) * 3, self_gravity=1, mg_mode=0,
                  mg_threshold=-1.0, mg_niter=4, four_pi_G=1.0, precision=precision)
    from tests.test_oracle_mg import blobs
    U = np.zeros((5, N, N, N))
    U[0] = blobs(N, 2)
    ub = agx.scatter_cells(d, U)
    out = []
    for mode in (0, 1):
        m = agx.Mesh(d)
        m.set("u", ub)
        m.set_mg_fuse(mode)
        m.mg_solve(0)
        out.append(m.get("phi"))
        m.close()
    d_ = np.abs(out[0] - out[1]).max()
    print(f"precision {precision}: max |phi(steps) - phi(passes)| = {d_:.3e}", flush=True)
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("nb", [(3, 5, 2), (24, 20, 5), (9, 9, 9)])
@pytest.mark.parametrize("precision", [0, 1])
def test_odd_root_grid(nb, precision):
    """root grids whose lowest level has odd extents, of one workgroup and of several: the periodic
    wrap there joins cells of one colour, which a sweep reads as they were before it.  FP64 against
    the oracle at the bar above; both precisions the same bits from run to run."""
    agx = load_agx()
    n = tuple(4 * q for q in nb)
    h = 1.0 / max(n)
    d = make_desc(nx=n, bnx=(4, 4, 4), box=tuple((0.0, h * q) for q in n), self_gravity=1, mg_mode=0, mg_threshold=-1.0,
                  mg_niter=2, four_pi_G=1.0, precision=precision)
    U = np.zeros((5, n[2], n[1], n[0]))
    U[0] = np.random.default_rng(9).uniform(0.5, 1.5, n[::-1])
    ub = agx.scatter_cells(d, U)
    out = []
    for _ in range(3):
        m = agx.Mesh(d)
        m.set("u", ub)
        m.mg_solve(0)
        out.append(m.get("phi"))
        m.close()
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
    if precision == 0:
        o = Oracle(d)
        o.set("u", ub)
        o.mg_solve(0)
        ref = o.get("phi")
        err = np.abs(out[0] - ref).max() / np.abs(ref).max()
        print(f"root {nb}: max|dphi| {err:.3e} of max|phi|", flush=True)
        assert err <= 1e-12
