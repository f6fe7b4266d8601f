"""The right-hand side kernel at the edges of its row chunks and grids: the
smallest grid, rows that leave a remainder in every chunk length, and enough
pairs for the short chunks of large grids; with and without stored explicit
terms and a body force.  buildrhs against the oracle's to 1e-13 relative L2, as
tests/test_gpu_parity.py holds it."""
import numpy as np
import pytest

from cases import rel_l2, tiny
from channel_amd.body_force import coriolis
from channel_amd.initial import perturbed_laminar
from channel_amd.solver import RK1, RK3, Channel
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("force", ["none", "static", "coriolis"])
@pytest.mark.parametrize("nx,ny,nz", [(3, 8, 4), (7, 33, 9), (15, 98, 15), (255, 19, 128)])
def test_rhs_at_chunk_edges(nx, ny, nz, force):
    print("[case] rhs", nx, ny, nz, force, flush=True)
    cfg = tiny(nx=nx, ny=ny, nz=nz)
    V = perturbed_laminar(cfg, seed=11, amp=5e-2, kmax=8)
    g, o = Channel(cfg), orc.Oracle(cfg)
    g.set_field(V)
    o.set_field(V)
    if force == "static":
        F = perturbed_laminar(cfg, seed=12, amp=5e-2, kmax=8)
        F[[0, 1, -2, -1]] = np.nan  # the wall and ghost rows are the library's
        g.set_body_force(F)
        F[[0, 1, -2, -1]] = 0.0
        o.set_body_force(F)
    elif force == "coriolis":
        g.set_body_force_feedback(*coriolis(cfg, 0.3))
        o.set_body_force_module("coriolis", 0.3, 9999999.0, 1.0)
    for ode in (RK1, RK3):  # without and with the stored explicit terms
        if force == "coriolis":
            o.apply_body_force()
        g.buildrhs(ode)
        o.buildrhs(ode)
        R, Ro = g.get_rhs(), o.get_field()[2:cfg.ny + 1, :, :, 0:2]
        for k in range(2):
            assert rel_l2(R[..., k], Ro[..., k]) < 1e-13
        o.set_field(V)
    g.close()
    o.close()
