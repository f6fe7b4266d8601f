"""chan_les_closure_force with feature scales at the ends of float's range: the
quotient (x - mean) / scale is IEEE division's, so an infinite scale masks its
feature, a value equal to its mean is 0 over any scale, and a quotient beyond the range
is infinite, not NaN.  The network's inputs cannot be read back, so each case is
compared, bit for bit, with a network or a scale that must give the same force."""
import numpy as np
import pytest

from channel_amd.dns import DnsConfig
from channel_amd.initial import perturbed_laminar
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup():
    from channel_amd.closure import Mlp
    from channel_amd.solver import Channel
    cfg = DnsConfig(nx=7, ny=16, nz=7, alfa0=0.5, beta0=1.0, ni=1.0 / 12431.0, a=1.5, cpi=True, cpi_type=1,
                    gamma=0.161436, deltat=0.0, cflmax=1.0)
    V = perturbed_laminar(cfg, seed=7, amp=0.05, kmax=8)
    g, m = Channel(cfg), Mlp(16)

    def force(params, norm, field=V):
        g.set_field(field)
        m.set_params(params.astype(np.float32))
        g.les_closure_force(m, norm)
        return g.get_body_force()

    yield cfg, V, force
    g.close()
    m.close()


def plain_norm():
    return np.concatenate([np.zeros(46), np.full(46, 0.7), np.zeros(6), np.full(6, 1e-3)]).astype(np.float32)


def params():
    rng = np.random.default_rng(3)
    return (mo.init_params(5) + 0.05 * rng.standard_normal(mo.NPARAM)).astype(np.float32)


def without(p, j):
    q = p.copy()
    q[:46 * 64].reshape(46, 64)[j] = 0.0
    return q


@pytest.mark.parametrize("j", [0, 13, 45])
def test_infinite_scale_masks_the_feature(setup, j):
    cfg, V, force = setup
    p, norm = params(), plain_norm()
    want = force(without(p, j), norm)
    assert not np.array_equal(want, force(p, norm))
    norm[46 + j] = np.inf
    got = force(p, norm)
    assert np.all(np.isfinite(got))
    assert np.array_equal(got, want)


@pytest.mark.parametrize("scale", [1e-39, 1e-45, 2e-38, 1e30, 3e38])
def test_zero_over_any_scale(setup, scale):
    cfg, V, force = setup
    p, norm = params(), plain_norm()
    base = np.zeros_like(V)
    base[:, cfg.nz, 0, 0] = V[:, cfg.nz, 0, 0]  # the mean flow alone: no x or z derivatives
    want = force(p, norm, base)
    norm[46 + 0] = norm[46 + 20] = np.float32(scale)  # du/dx here, du/dz two rows below
    assert np.array_equal(force(p, norm, base), want)


def test_overflow_is_infinite(setup):
    """y+ alone enters; where it is not zero the first layer is huge or infinite, the
    second 0; at the walls they are 0 and 1."""
    cfg, V, force = setup
    W1, b1 = np.zeros((46, 64)), np.zeros(64)
    W1[45] = 1.0
    W2, b2 = np.full((64, 64), -1.0), np.ones(64)
    rng = np.random.default_rng(4)
    rest = [rng.standard_normal((64, 64)) / 8, np.zeros(64), rng.standard_normal((64, 6)) / 8, np.zeros(6)]
    p = np.concatenate([np.ravel(a) for a in [W1, b1, W2, b2] + rest])
    norm = plain_norm()
    norm[46 + 45] = 1e-3
    want = force(p, norm)
    assert np.any(want != 0)
    for scale in (2e-38, 1e-39):
        norm[46 + 45] = np.float32(scale)
        assert np.array_equal(force(p, norm), want)
