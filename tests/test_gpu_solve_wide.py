"""The solve of wide grids (k_solve_ve_wide): the same as the other kernel's of the same
columns.  A grid of three waves per SIMD and more holds, mode by mode, the systems of a narrower
one, so that with the same right-hand sides in those modes the results must agree; even and odd
rows, past the 130 that LDS takes; walls and the flow-rate correction.  4e-13 relative L2 per
component: both kernels' 1e-13 against the oracle (tests/test_gpu_parity.py) and room for the
derivative."""
import numpy as np
import pytest

from cases import rel_l2, tiny
from channel_amd.initial import perturbed_laminar
from channel_amd.solver import RK1, Channel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,walls", [(131, False), (132, True), (135, False)])
def test_wide_grid_solves_the_narrow_ones_columns(ny, walls):
    print("[case] wide solve", ny, walls, flush=True)
    kw = dict(meanflowx=0.0, u0=-0.4, uN=0.3) if walls else {}
    narrow, wide = tiny(nx=15, ny=ny, nz=15, **kw), tiny(nx=175, ny=ny, nz=170, **kw)
    V = perturbed_laminar(narrow, seed=3, amp=1e-3, kmax=8)
    V[:, :, 9:, :] = 0.0  # modes whose products neither grid drops or aliases
    V[:, :7, :, :] = V[:, 24:, :, :] = 0.0
    W = np.zeros(wide.field_shape, dtype=np.complex128, order="F")
    inner = slice(wide.nz - narrow.nz, wide.nz + narrow.nz + 1)
    W[:, inner, :narrow.nx + 1, :] = V
    out = []
    for cfg, F in ((narrow, V), (wide, W)):
        g = Channel(cfg)
        g.set_field(F)
        g.buildrhs(RK1)
        g.linsolve(RK1[0] / cfg.deltat)
        out.append((g.get_field(), g.scalars()))
        g.close()
    (A, sa), (B, sb) = out
    B = B[:, inner, :narrow.nx + 1, :]
    for c in range(3):
        assert rel_l2(B[..., c], A[..., c]) < 4e-13, c
    for k in ("fr1", "fr2", "fr3"):
        assert abs(sa[k] - sb[k]) <= 1e-12 * max(abs(sa["fr1"]), 1.0), k
