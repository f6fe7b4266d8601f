"""The x pass of short rows (k_xpass_few): buildrhs and the CFL maximum against the
oracle for every row length it takes, at the smallest and largest mode counts of
each and on both sides of the block count where rows of 72 points change kernel.
1e-13 relative L2 for buildrhs and relative for the CFL maximum, as
tests/test_gpu_parity.py holds both; a NaN or an infinity must reach the maximum from
any row."""
import numpy as np
import pytest

from cases import rel_l2, tiny
from channel_amd import lib
from channel_amd.solver import RK1, Channel
from oracle import oracle as orc
from test_gpu_alias_free import broadband

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz", [(3, 5), (4, 3), (5, 8), (6, 4), (7, 9), (9, 6), (11, 13), (15, 10), (16, 3),
                                   (21, 5), (22, 8), (23, 260), (31, 12), (33, 5), (41, 7)])
def test_short_rows(nx, nz):
    print("[case] short rows", nx, nz, flush=True)
    cfg = tiny(nx=nx, ny=9, nz=nz)
    V = broadband(cfg, 31 * nx + nz)
    g, o = Channel(cfg), orc.Oracle(cfg)
    o.set_field(V)
    o.buildrhs(RK1, True)
    Ro = o.get_field()[2:cfg.ny + 1, :, :, 0:2]
    for cfl in (False, True):
        g.set_field(V)
        g.buildrhs(RK1, cfl)
        R = g.get_rhs()
        for k in range(2):
            assert rel_l2(R[..., k], Ro[..., k]) < 1e-13, (cfl, k)
    top = o.scalars()["cfl"]
    assert g.scalars()["cfl"] == pytest.approx(top, rel=1e-13)
    # the running maximum: kept by a read, replaced by a set, raised by a later pass
    assert g.scalars()["cfl"] == pytest.approx(top, rel=1e-13)
    g.set_scalars(cfl=2 * top)
    g.buildrhs(RK1, True)
    assert g.scalars()["cfl"] == 2 * top
    g.set_scalars(cfl=0.0)
    assert g.scalars()["cfl"] == 0.0
    g.close()
    o.close()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_bad_sample_reaches_the_maximum(bad):
    cfg = tiny(nx=15, ny=9, nz=10)
    V = broadband(cfg, 5)
    V[5, cfg.nz, 0, 1] = bad
    g = Channel(cfg)
    g.set_field(V)
    g.buildrhs(RK1, True)
    assert not np.isfinite(g.scalars()["cfl"])
    with pytest.raises(lib.ChanError):
        g.outstats()
    g.close()
