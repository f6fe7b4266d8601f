"""chan_mlp_forward_noalloc with outputs that overlap the inputs, in front of
them, in place, inside and behind: bitwise the outputs of chan_mlp_forward, for models
that hold fewer rows than the call and more."""
import numpy as np
import pytest

from oracle import mlp_oracle as mo
from test_zz_no_alloc import _Hip, _model

pytestmark = pytest.mark.gpu

NMAX = 65536


def _offset(where, n):
    """Bytes from dX to dY, of outputs 24 n and inputs 184 n long."""
    return {"before": -24 * n + 4, "in place": 0, "inside": 64 * n, "behind": 184 * n - 4, "apart": 184 * n}[where]


@pytest.mark.parametrize("where", ["before", "in place", "inside", "behind", "apart"])
@pytest.mark.parametrize("n,cap", [(1, 16), (17, 17), (5000, 16), (5000, 6000), (NMAX, 16)])
def test_overlapping_buffers(n, cap, where):
    from channel_amd import lib
    print("[case] noalloc overlap", n, cap, where, flush=True)
    m, rng = _model(cap, 11)
    big, _ = _model(n, 11)  # the same parameters
    X = rng.standard_normal((n, mo.IN)).astype(np.float32)
    want = big.forward(X)
    big.close()
    hip = _Hip()
    front = 24 * n
    buf = hip.alloc(front + 184 * n + 24 * n)
    try:
        base = buf.value + front
        hip.put(base, X)
        lib.check(lib.load().chan_mlp_forward_noalloc(m.h, base, n, base + _offset(where, n)))
        got = np.empty_like(want)
        hip.get(got, base + _offset(where, n))
    finally:
        hip.free(buf)
    m.close()
    np.testing.assert_array_equal(got, want)
