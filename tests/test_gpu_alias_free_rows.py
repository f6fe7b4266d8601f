"""The products on the alias-free grids in both precisions: the sizes and mode counts of
tests/test_gpu_alias_free.py and tests/test_gpu_short_rows.py in the split mode, and rows of 72,
144 and 288 points on grids with enough of them to be taken (and one row of planes fewer, where
they are not).  buildrhs and the CFL maximum against the oracle: 1e-13 relative L2 in
FP64; in the split mode 3e-6 and 1e-6 (products and transforms of FP32 samples, about ten
roundings of 6e-8 on the way to a mode of a field whose modes are all alike)."""
import numpy as np
import pytest

from cases import rel_l2, tiny
from channel_amd import lib
from channel_amd.solver import RK1, Channel
from oracle import oracle as orc
from test_gpu_alias_free import broadband

pytestmark = pytest.mark.gpu

SMALL = [(11, 4), (23, 8), (47, 8), (95, 8), (191, 8), (383, 8), (4, 11), (7, 23), (7, 47), (7, 95), (7, 191), (7, 383),
         (11, 11), (47, 95), (188, 47), (37, 40),
         (3, 5), (4, 3), (5, 8), (6, 4), (7, 9), (9, 6), (11, 13), (15, 10), (16, 3), (21, 5), (22, 8), (23, 260), (31, 12),
         (33, 5), (41, 7)]
# nx, ny, nz: z grids of 72 and 288 points; 256 CUs take rows of 144 and 288 from 1024 groups of four
# on, of 144 in FP32 from 2048, and rows of 72 in blocks beyond 2048
ROWS = [(23, 25, 95), (23, 26, 95), (20, 40, 95), (47, 11, 95), (47, 12, 95), (44, 25, 95), (47, 26, 95), (95, 11, 95),
        (95, 12, 95), (90, 54, 23), (94, 30, 94)]


def check(nx, ny, nz, precision):
    cfg = tiny(nx=nx, ny=ny, nz=nz)
    V = broadband(cfg, 100 * nx + nz)
    g, o = Channel(cfg, precision), orc.Oracle(cfg)
    o.set_field(V)
    o.buildrhs(RK1, True)
    Ro = o.get_field()[2:cfg.ny + 1, :, :, 0:2]
    tol, tol_cfl = (1e-13, 1e-13) if precision == lib.CHAN_FP64 else (3e-6, 1e-6)
    for cfl in (False, True):
        g.set_field(V)
        g.buildrhs(RK1, cfl)
        R = g.get_rhs()
        for k in range(2):
            e = rel_l2(R[..., k], Ro[..., k])
            print(nx, ny, nz, precision, cfl, k, e)
            assert e < tol, (cfl, k)
    assert g.scalars()["cfl"] == pytest.approx(o.scalars()["cfl"], rel=tol_cfl)
    g.close()
    o.close()


@pytest.mark.parametrize("nx,nz", SMALL)
def test_split_mode(nx, nz):
    print("[case] alias-free split", nx, nz, flush=True)
    check(nx, 9, nz, lib.CHAN_SPLIT)


@pytest.mark.parametrize("precision", [lib.CHAN_FP64, lib.CHAN_SPLIT])
@pytest.mark.parametrize("nx,ny,nz", ROWS)
def test_long_and_many_rows(nx, ny, nz, precision):
    print("[case] alias-free rows", nx, ny, nz, precision, flush=True)
    check(nx, ny, nz, precision)
