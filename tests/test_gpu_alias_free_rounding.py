"""The rounding of the products on the alias-free grids (sizes 9*2^k): FP32 against FP64 on
the same field, next to the physical grid's.  A mode is a mean over the points, so that
its rounding goes with the root of their number; the transforms themselves may not add more
than a quarter to that."""
import numpy as np
import pytest

from cases import rel_l2, tiny
from channel_amd import lib
from channel_amd.initial import perturbed_laminar
from channel_amd.solver import RK1, Channel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz,points", [(47, 47, 192 * 192 / 144 ** 2), (95, 95, 384 * 384 / 288 ** 2),
                                          (95, 16, 384 / 288), (16, 95, 384 / 288), (191, 95, 384 / 288)])
def test_rounding_on_the_smaller_grid(nx, nz, points):
    print("[case] alias-free rounding", nx, nz, flush=True)
    cfg = tiny(nx=nx, ny=100, nz=nz)  # rows enough for every length in x
    V = perturbed_laminar(cfg, seed=5, amp=3e-2, kmax=max(nx, nz))
    R = {}
    for precision in (lib.CHAN_FP64, lib.CHAN_SPLIT):
        g = Channel(cfg, precision)
        for cfl in (False, True):
            g.set_field(V)
            g.buildrhs(RK1, cfl)
            R[precision, cfl] = g.get_rhs()
        g.close()
    for k in range(2):
        small, physical = (rel_l2(R[lib.CHAN_SPLIT, cfl][..., k], R[lib.CHAN_FP64, cfl][..., k]) for cfl in (False, True))
        print("component", k, small, physical, small / physical)
        assert small <= 1.25 * np.sqrt(points) * physical
