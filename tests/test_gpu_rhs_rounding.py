"""The implicit part of the D2v equation, whose second differences nearly cancel:
no further from an 80-bit evaluation than the plain formula in FP64 is, with a quarter
more for the other order of the sums.  Velocities of 1e-20, so that the products do
not count, and a time step that divides exactly."""
import numpy as np
import pytest

from cases import tiny
from channel_amd.solver import RK1, Channel

pytestmark = pytest.mark.gpu


def implicit(der, v, k2, rdt, ni, kind):
    """rdt (D2 - k2 D0) v + ni (D4 - 2 k2 D2 + k2^2 D0) v, sums in order."""
    d0, d2, d4 = (der[:, k, :].astype(kind) for k in (0, 2, 3))
    v, k2, rdt, ni = v.astype(kind), k2.astype(kind), kind(rdt), kind(ni)
    n = len(der)
    s2, s0, os = (np.zeros((n,) + v.shape[1:], kind) for _ in range(3))
    for j in range(5):
        w = v[j:j + n]
        a0, a2, a4 = (d[:, j, None, None] for d in (d0, d2, d4))
        s2 += a2 * w
        s0 += a0 * w
        os += ni * (a4 - 2 * k2 * a2 + k2 * k2 * a0) * w
    return rdt * (s2 - k2 * s0) + os


@pytest.mark.parametrize("ny", [32, 129, 384])
@pytest.mark.parametrize("wave", [1.0, 8.0])
def test_second_differences_keep_their_digits(ny, wave):
    print("[case] rhs rounding", ny, wave, flush=True)
    cfg = tiny(nx=15, ny=ny, nz=12, alfa0=wave, beta0=wave, deltat=1.0 / 512, meanflowx=0.0)
    g = Channel(cfg)
    y, der, _ = g.setup()
    rng = np.random.default_rng(ny)
    shapes = np.stack([np.cos(n * np.pi * y / 2) for n in range(1, 9)]) / np.arange(1, 9)[:, None]
    c = rng.standard_normal((2, 8, 2 * cfg.nz + 1, cfg.nx + 1))
    v = np.einsum("ny,knzx->kyzx", shapes, c) * 1e-20
    V = np.zeros(cfg.field_shape, dtype=np.complex128, order="F")
    V[..., 1] = v[0] + 1j * v[1]
    g.set_field(V)
    g.buildrhs(RK1)
    R = g.get_rhs()[..., 1]
    g.close()
    kx, kz = cfg.alfa0 * np.arange(cfg.nx + 1), cfg.beta0 * np.arange(-cfg.nz, cfg.nz + 1)
    k2 = kz[:, None] ** 2 + kx[None, :] ** 2
    rdt = RK1[0] * 512
    here = plain = 0.0
    for part, got in ((v[0], R.real), (v[1], R.imag)):
        exact = implicit(der, part, k2, rdt, cfg.ni, np.longdouble)
        here += float(np.sum((got - exact) ** 2))
        plain += float(np.sum((implicit(der, part, k2, rdt, cfg.ni, np.float64) - exact) ** 2))
    print("rms error, here over the plain formula's", np.sqrt(here / plain))
    assert here <= 1.25 ** 2 * plain
