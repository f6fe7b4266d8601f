"""dv/dy of columns held in LDS where the two halves of a column meet: the
stencils of each half's innermost three rows reach the other half's rows, which
are overwritten in place.  Every small number of rows (halves of 3 rows, which
are all innermost, upwards; even and odd) and numbers around the unrolled groups of rows, in
blocks enough to fill the chip.  One substep against the oracle to 1e-13 relative L2 per
component, as tests/test_gpu_parity.py holds it, and the same bits every time."""
import numpy as np
import pytest

from cases import rel_l2, tiny
from channel_amd.initial import perturbed_laminar
from channel_amd.solver import RK1, Channel
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny", [8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 18, 19, 24, 25, 39, 40])
def test_halves_of_a_column(ny):
    print("[case] halves", ny, flush=True)
    cfg = tiny(nx=63, ny=ny, nz=63)
    V = perturbed_laminar(cfg, seed=ny, amp=5e-2, kmax=32)
    lam = RK1[0] / cfg.deltat
    g, o = Channel(cfg), orc.Oracle(cfg)
    o.set_field(V)
    o.buildrhs(RK1, False)
    o.linsolve(lam)
    Vo = o.get_field()
    first = None
    for _ in range(4):
        g.set_field(V)
        g.buildrhs(RK1, False)
        g.linsolve(lam)
        Vg = g.get_field()
        for c in range(3):
            assert rel_l2(Vg[..., c], Vo[..., c]) < 1e-13, c
        assert first is None or np.array_equal(Vg, first)
        first = Vg
    g.close()
    o.close()
