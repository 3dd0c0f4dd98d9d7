"""Stage kernels whose workgroups walk a chunk of a MeshBlock's k-planes (stage_planes in
agx_mhd.hip): meshes where the chunks are one plane, several, with a shorter last chunk, and
whole columns, each form against the oracle to the parity bar, 1e-12 of each array's maximum (the
cell sizes of these boxes round differently from cell to cell in the oracle, and are one number for a
block on the device), and against the first form run on the same mesh bit for bit."""
import numpy as np
import pytest

from oracle.orc import Oracle, make_desc
from tests.states import load_state, turbulent_state

pytestmark = pytest.mark.gpu

MESHES = {
    "one_plane": dict(nx=(20, 12, 7), bnx=(20, 12, 7)),
    "two_planes_per_block": dict(nx=(16, 8, 8), bnx=(8, 8, 2)),
    "short_last_chunk": dict(nx=(72, 72, 66), bnx=(24, 24, 22)),      # k_vl2: chunks of 4, the last of 2
    "odd_chunks": dict(nx=(66, 99, 75), bnx=(33, 33, 25)),
    "narrow_blocks_few": dict(nx=(32, 32, 48), bnx=(16, 16, 16)),     # default split tile 64 x 4
    "narrow_blocks_many": dict(nx=(64, 32, 32), bnx=(16, 16, 16)),    # 16 x 16
    "whole_columns": dict(nx=(96, 96, 24), bnx=(8, 8, 4)),
}


FIRST = {}   # the arrays of the first form run on each mesh


@pytest.mark.parametrize("form", [None, 0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("name", MESHES)
def test_chunked_stage_matches_oracle(agx, name, form):
    dk = MESHES[name]
    ext = tuple((0.0, n / max(dk["nx"])) for n in dk["nx"])
    desc = make_desc(box=ext, cfl=0.4, **dk)
    st = turbulent_state(desc, seed=29, mach=1.2)
    o = Oracle(desc)
    load_state(o, st)
    o.initialize()
    m = agx.Mesh(desc)
    load_state(m, st)
    if form is not None:
        m.set_tile(form)
    m.initialize()
    assert m.cycle(1e9, 2) == 2
    o.cycle(1e9)
    o.cycle(1e9)
    assert m.time() == o.time()
    for f in ("u", "w", "bcc", "b1f", "b2f", "b3f"):
        a, b = m.get(f), o.get(f)
        err = np.abs(a - b).max()
        print(f"{name} form {form} {f}: max |diff| {err:.2e}", flush=True)
        assert err <= 1e-12 * np.abs(b).max()
        assert np.array_equal(a, FIRST.setdefault((name, f), a))
    m.close()
