"""The solves of columns held in LDS, swept from both walls, at the edges of
their range: even and odd numbers of rows, the fewest and the most that fit,
with and without room for the lower factors, one row past the limit (the
kernels through memory), groups that leave a remainder in a block, moving
walls and the flow-rate correction.  One time step (the oracle takes the wall
velocities there) against the oracle to the step's bar of 1e-12 relative L2 per
component."""
import numpy as np
import pytest

from cases import rel_l2, tiny
from channel_amd.initial import perturbed_laminar
from channel_amd.solver import Channel
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("nx,ny,nz", [(3, 8, 4), (3, 9, 4), (4, 10, 6), (7, 17, 9), (6, 92, 5), (6, 93, 5), (5, 129, 7),
                                      (5, 130, 7), (5, 131, 7), (15, 64, 15)])
def test_solve_at_its_edges(nx, ny, nz, walls):
    print("[case] solve", nx, ny, nz, walls, flush=True)
    kw = dict(meanflowx=0.0, u0=-0.4, uN=0.3) if walls else {}
    cfg = tiny(nx=nx, ny=ny, nz=nz, **kw)
    V = perturbed_laminar(cfg, seed=5, amp=5e-2, kmax=8)
    g, o = Channel(cfg), orc.Oracle(cfg)
    for c in (g, o):
        c.set_field(V)
        c.step()
    Vg, Vo = g.get_field(), o.get_field()
    for c in range(3):
        assert rel_l2(Vg[..., c], Vo[..., c]) < 1e-12
    sg, so = g.scalars(), o.scalars()
    for k in ("fr1", "fr2", "fr3"):
        assert abs(sg[k] - so[k]) <= 1e-12 * max(abs(so["fr1"]), 1.0), k
    if not walls:
        assert np.isclose(sg["corrpx"], so["corrpx"], rtol=0, atol=1e-12 / abs(so["fr3"]))
    g.close()
    o.close()
