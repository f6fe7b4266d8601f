"""The closure's kernels at the edges of their tiles, against the float64
checkers: rows around the 16-sample tiles, the 64-sample groups and more groups
than blocks; closure grids with ragged sizes, and one whose x phases do not fit
in LDS.  Bounds as in tests/test_gpu_closure.py (forward 1e-4, gradient 1e-3
relative L2) and tests/test_gpu_les.py (features 2e-6 of their scale, force
2e-3)."""
import numpy as np
import pytest

from channel_amd.dns import DnsConfig
from channel_amd.initial import perturbed_laminar
from oracle import les_oracle as lo
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return float(np.linalg.norm(np.ravel(a) - np.ravel(b)) / np.linalg.norm(np.ravel(b)))


def model(n, seed):
    from channel_amd.closure import Mlp
    rng = np.random.default_rng(seed)
    p = (mo.init_params(seed) + 0.05 * rng.standard_normal(mo.NPARAM)).astype(np.float32).astype(np.float64)
    X = rng.standard_normal((n, mo.IN)).astype(np.float32)
    T = rng.standard_normal((n, mo.OUT)).astype(np.float32)
    m = Mlp(n)
    m.set_params(p)
    return m, p, X, T


@pytest.mark.parametrize("n", [1, 15, 17, 63, 65, 32773])
def test_rows_around_the_tiles(n):
    print("[case] closure rows", n, flush=True)
    m, p, X, T = model(n, 4)
    assert rel_l2(m.forward(X), mo.mirrored(p, X.astype(np.float64))[0]) < 1e-4
    m.set_data(X, T)
    loss, g = m.grad(0, n)
    _, lref, gref = mo.mirrored(p, X.astype(np.float64), T.astype(np.float64))
    assert abs(loss - lref) <= 1e-4 * lref
    assert rel_l2(g, gref) < 1e-3
    m.close()


@pytest.mark.parametrize("nx,ny,nz,force", [(13, 25, 12, True), (6, 9, 4, True), (31, 12, 31, True), (300, 9, 4, False)])
def test_closure_grids(nx, ny, nz, force):
    from channel_amd.solver import Channel
    print("[case] closure grid", nx, ny, nz, flush=True)
    cfg = DnsConfig(nx=nx, ny=ny, nz=nz, alfa0=0.5, beta0=1.0, ni=1.0 / 12431.0, a=1.5, cpi=True, cpi_type=1,
                    gamma=0.161436, deltat=0.0, cflmax=1.0)
    V = perturbed_laminar(cfg, seed=7, amp=0.05, kmax=8)
    g = Channel(cfg)
    g.set_field(V)
    X = g.les_features().astype(np.float64)
    y, _, bnd = g.setup()
    Xo = lo.features(cfg, V, y, bnd[1], bnd[6])
    assert np.all(np.max(np.abs(X - Xo), axis=0) < 2e-6 * np.max(np.abs(Xo), axis=0))
    if force:
        m, p, _, _ = model(16, 5)
        norm = np.concatenate([X.mean(0), X.std(0) + 1e-3, 1e-3 * np.arange(6), np.full(6, 2e-3)]).astype(np.float32)
        n32 = norm.astype(np.float64)
        g.les_closure_force(m, norm)
        F = g.get_body_force()
        tau = mo.mirrored(p, (X - n32[:46]) / n32[46:92])[0] * n32[98:104] + n32[92:98]
        tau = np.moveaxis(tau.reshape(cfg.ny + 1, 2 * cfg.nxd, cfg.nzd, 6), -1, 0)
        inner = slice(2, cfg.ny + 1)
        assert rel_l2(F[inner], lo.divergence(cfg, tau, y)[inner]) < 2e-3
        m.close()
    g.close()
