"""Transfers of large pageable buffers through the staging of host_copy.hip:
what arrives is bitwise what smaller, direct transfers bring.  Row counts put the
input (184 bytes a row) just below and above the 96 MiB and the output (24) the
8 MiB where the staging begins, with a remainder of a chunk."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [349525, 349526, 547083, 547084, 600001])
def test_forward_rows(n):
    from channel_amd.closure import Mlp, _he_init
    X = np.random.default_rng(n).standard_normal((n, 46)).astype(np.float32)
    m = Mlp(n)
    m.set_params(_he_init(1))
    Ys = [m.forward(X) for _ in range(6)]  # the first ones without the staging
    part = 16384  # multiple of the kernel's tiles: a row's sums do not depend on its place
    Z = np.concatenate([m.forward(X[i:i + part]) for i in range(0, n, part)])
    m.close()
    for Y in Ys:
        assert np.array_equal(Y, Z)


@pytest.mark.parametrize("nx,ny,nz", [(24, 51, 65), (31, 64, 44), (64, 97, 77), (95, 128, 95)])
def test_field_round_trip(nx, ny, nz):
    from channel_amd.dns import DnsConfig
    from channel_amd.solver import Channel
    cfg = DnsConfig(nx=nx, ny=ny, nz=nz, meanflowx=4 / 3., deltat=0.004)
    rng = np.random.default_rng(nx)
    V = np.asfortranarray(rng.standard_normal(cfg.field_shape) + 1j * rng.standard_normal(cfg.field_shape))
    ch = Channel(cfg)
    for k in range(6):  # directly at first, then through slots that hold the last one's data
        ch.set_field(V * (k + 1))
        assert np.array_equal(ch.get_field(), V * (k + 1))
    ch.close()
