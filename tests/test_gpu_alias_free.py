"""Substeps without a CFL maximum form the products on the smallest alias-free
grid (sizes 9*2^k where they are below fftFIT's), which must give the sums of the
physical grid: buildrhs against the oracle, which always uses the physical grid,
for every such size in x and in z, alone and together.  The field has energy in
every mode up to the highest, so that one point too few would show as aliasing.
1e-13 relative L2, as tests/test_gpu_parity.py holds buildrhs; the same for the
physical grid (compute_cfl), whose results must agree with the small grid's."""
import numpy as np
import pytest

from cases import rel_l2, tiny
from channel_amd.solver import RK1, Channel
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def broadband(cfg, seed):
    rng = np.random.default_rng(seed)
    V = 0.05 * (rng.standard_normal(cfg.field_shape) + 1j * rng.standard_normal(cfg.field_shape))
    nz = cfg.nz
    V[:, :nz, 0, :] = np.conj(V[:, :nz:-1, 0, :])  # a real field
    V[:, nz, 0, :] = V[:, nz, 0, :].real
    return np.asfortranarray(V)


@pytest.mark.parametrize("nx,nz", [(11, 4), (23, 8), (47, 8), (95, 8), (191, 8), (383, 8), (4, 11), (7, 23), (7, 47),
                                   (7, 95), (7, 191), (7, 383), (11, 11), (47, 95), (188, 47), (37, 40)])
def test_products_on_the_smallest_grid(nx, nz):
    print("[case] alias-free", nx, nz, flush=True)
    cfg = tiny(nx=nx, ny=9, nz=nz)
    V = broadband(cfg, 100 * nx + nz)
    g, o = Channel(cfg), orc.Oracle(cfg)
    o.set_field(V)
    o.buildrhs(RK1)
    Ro = o.get_field()[2:cfg.ny + 1, :, :, 0:2]
    for cfl in (False, True):
        g.set_field(V)
        g.buildrhs(RK1, cfl)
        R = g.get_rhs()
        for k in range(2):
            assert rel_l2(R[..., k], Ro[..., k]) < 1e-13, (cfl, k)
    g.close()
    o.close()
