"""Performance cases of the channel DNS step and its learned closure.

``listed()`` names the cases, ``draw(rng)`` gives further ones from the same
ranges, ``prepare`` sets one up on the GPU, ``run`` is one pass through the
public entry points (channel_amd.solver.Channel, channel_amd.closure.Mlp) and
``work`` counts what a pass cannot do without.  ``exact`` computes the outputs
of a pass in 64 bits with plain torch, from the equations: transforms by
torch.fft, the compact stencils by a Vandermonde solve, the wall-normal
systems by a pentadiagonal elimination.

Kinds of a case:

``run``      a simulation leg: ``steps`` time steps, the Runtimedata rows, then
             the field as a restart or snapshot file gets it (in single
             precision in the mixed mode, which carries no more).  Options:
             the precision mode, constant flow rate or CPI, a fixed or CFL-set
             time step, moving walls, the Coriolis body force, and statistics
             profiles every few steps.
``les``      a coarse run with the closure from a given field, as the study of
             it makes them: before every step the body force is renewed from
             the resident field by the network.
``grad``     loss and gradient of one minibatch of resident samples.
``train``    a number of Adam steps over consecutive minibatches.
``forward``  inference on host rows, as the a priori study evaluates a snapshot.
"""
import math

import numpy as np
import torch

from channel_amd import lib
from channel_amd.body_force import coriolis
from channel_amd.closure import Mlp
from channel_amd.dns import DnsConfig
from channel_amd.solver import Channel

IN, HID, OUT = 46, 64, 6
SHAPES = [(IN, HID), (HID,), (HID, HID), (HID,), (HID, HID), (HID,), (HID, OUT), (OUT,)]
NORM_SCALE = 1e-4  # size of the closure's stresses, in squared bulk velocities


def _run(name, nx, ny, nz, steps, **kw):
    c = dict(name=name, kind="run", nx=nx, ny=ny, nz=nz, steps=steps, split=False, alfa0=1.0, beta0=2.0, re=3000.0,
             flow="rate", cflmax=0.0, wall=0.0, omega2=0.0, stats_every=0)
    c.update(kw)
    return c


def listed():
    cpi = dict(alfa0=0.5, beta0=1.0, re=12431.0, flow="cpi", cflmax=1.0)
    return [
        # a host program that looks at the field after every step (control,
        # coupling) on the smallest grid in use: latency and launches
        _run("one step 15x32x15", 15, 32, 15, 1),
        # the small validation grid: a leg between two snapshots
        _run("run 31x64x31", 31, 64, 31, 20),
        # the mid-size grid, constant flow rate, fixed time step
        _run("run 95x128x95", 95, 128, 95, 20),
        # the production grid: CPI, CFL-set time step
        _run("run 191x384x189", 191, 384, 189, 15, **cpi),
        # the same in the mixed-precision mode, whose products are FP32: the
        # snapshot is kept in single precision
        _run("split run 191x384x189", 191, 384, 189, 30, split=True, **cpi),
        # a grid that fits nothing, odd ny, walls that move (Couette)
        _run("walls 100x97x77", 100, 97, 77, 10, wall=0.5, cflmax=0.8),
        # spanwise rotation: the body force is formed from the field
        _run("rotation 63x96x47", 63, 96, 47, 20, omega2=0.02, cflmax=1.0),
        # time-averaged statistics, a profile every other step
        _run("statistics 127x129x127", 127, 129, 127, 10, stats_every=2, cflmax=1.0),
        # the coarse grid of the closure study with its force renewed each step
        dict(name="closure run 31x64x31", kind="les", nx=31, ny=64, nz=31, steps=10, alfa0=0.5, beta0=1.0, re=12431.0),
        # training the closure: one gradient, a run of Adam steps
        dict(name="gradient 16384", kind="grad", n=65536, count=16384),
        dict(name="train 8192", kind="train", n=65536, batch=8192, steps=16),
        # a snapshot of the coarse grid's points through the network
        dict(name="inference 599040", kind="forward", n=599040),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _modes(rng, lo, hi):
    """A number of x modes that the step takes: 3 (nx+1) <= 2 nxd."""
    while True:
        nx = _log(rng, lo, hi)
        if 3 * (nx + 1) <= 2 * _dealiased(nx, 1)[0]:
            return nx


def draw(rng):
    kind = rng.choice(["run"] * 7 + ["les", "grad", "train", "forward"])
    if kind == "run":
        c = _run("", _modes(rng, 11, 191), _log(rng, 24, 384), _log(rng, 11, 189), rng.choice([1, 2, 5, 10, 20]))
        del c["name"]
        c["re"] = round(rng.uniform(1500.0, 12000.0), 1)
        c["alfa0"], c["beta0"] = rng.choice([(1.0, 2.0), (0.5, 1.0)])
        c["flow"] = rng.choice(["rate", "cpi"])
        c["cflmax"] = rng.choice([0.0, 0.5, 1.0])
        c["split"] = rng.random() < 0.2
        extra = rng.random() if not c["split"] else 1.0
        if extra < 0.15:
            c["wall"] = round(rng.uniform(0.1, 0.6), 2)
        elif extra < 0.3:
            c["omega2"] = round(rng.uniform(0.005, 0.05), 3)
        elif extra < 0.45:
            c["stats_every"] = rng.choice([2, 5])
        return c
    if kind == "les":
        return dict(kind="les", nx=_modes(rng, 11, 31), ny=_log(rng, 24, 96), nz=_log(rng, 11, 31), steps=rng.choice([2, 5, 10]),
                    alfa0=0.5, beta0=1.0, re=round(rng.uniform(5000.0, 13000.0), 1))
    if kind == "grad":
        count = _log(rng, 16, 65536)
        return dict(kind="grad", n=max(count, 4096), count=count)
    if kind == "train":
        batch = _log(rng, 512, 32768)
        return dict(kind="train", n=2 * batch + rng.randrange(batch), batch=batch, steps=rng.choice([4, 8, 16]))
    return dict(kind="forward", n=_log(rng, 16, 599040))


# ------------------------------------------------------------------ inputs --
def _fits(i):
    while i % 2 == 0:
        i //= 2
    return i in (1, 3)


def _dealiased(nx, nz):
    a, b = 3 * (nx + 1) // 2, 3 * nz
    while not _fits(a):
        a += 1
    while not _fits(b):
        b += 1
    return a, b


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _config(case):
    cpi = case.get("flow", "cpi") == "cpi"
    wall = case.get("wall", 0.0)
    cflmax = case.get("cflmax", 1.0)
    return DnsConfig(nx=case["nx"], ny=case["ny"], nz=case["nz"], alfa0=case["alfa0"], beta0=case["beta0"],
                     ni=1.0 / case["re"], a=1.5, cpi=cpi, cpi_type=1, gamma=0.161436 if cpi else 0.0,
                     meanflowx=0.0 if cpi or wall else 4.0 / 3.0, u0=-wall, uN=wall,
                     deltat=0.0 if cflmax > 0 else 0.002, cflmax=cflmax)


def _rows(ny):
    """y of the rows -1..ny+1 on the stretched grid (a = 1.5, walls at 0 and 2)."""
    r = 2.0 * np.arange(-1, ny + 2) / ny
    return np.tanh(1.5 * (r - 1)) / math.tanh(1.5) + 1.0


def _field(case, seed):
    """A mean flow and divergence-free fluctuations in every mode, with a
    spectrum that falls off as a resolved turbulent one: V[c][ix][iz][row] on
    the device, which is the memory order of the library's field."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    dev = _device()
    rng = np.random.default_rng(seed)
    y = _rows(ny)
    s, t = 1.0 - (y - 1.0) ** 2, y - 1.0
    shapes_v = np.stack([s * s, s * s * t, s * s * np.cos(6.0 * t)])
    dshapes_v = np.stack([-4.0 * t * s, s * s - 4.0 * t * t * s, -4.0 * t * s * np.cos(6.0 * t) - 6.0 * s * s * np.sin(6.0 * t)])
    shapes_e = np.stack([s, s * t, s * np.cos(9.0 * t)])
    kx = case["alfa0"] * np.arange(nx + 1)[:, None]
    kz = case["beta0"] * np.arange(-nz, nz + 1)[None, :]
    k2 = kx ** 2 + kz ** 2
    fall = (1.0 + k2 / 4.0) ** -1.2 * np.exp(-4.0 * ((kx / kx.max()) ** 2 + (kz / kz.max()) ** 2))
    k2[0, nz] = 1.0

    def coefficients(amp):
        c = amp * fall * (rng.standard_normal((3, nx + 1, 2 * nz + 1)) + 1j * rng.standard_normal((3, nx + 1, 2 * nz + 1)))
        c[:, 0, :nz] = np.conj(c[:, 0, :nz:-1])  # a real field
        c[:, 0, nz] = 0.0
        return c

    def on(a):
        return torch.from_numpy(np.ascontiguousarray(a).astype(np.complex128)).to(dev)

    cv, ce = on(coefficients(0.01)), on(coefficients(0.03))
    kx, kz, k2 = (on(np.broadcast_to(a, k2.shape))[:, :, None] for a in (kx, kz, k2))
    v = torch.einsum("kxz,ky->xzy", cv, on(shapes_v))
    dv = torch.einsum("kxz,ky->xzy", cv, on(dshapes_v))
    eta = torch.einsum("kxz,ky->xzy", ce, on(shapes_e))
    V = torch.empty((3, nx + 1, 2 * nz + 1, ny + 3), dtype=torch.complex128, device=dev)
    V[0] = (1j * kx * dv - 1j * kz * eta) / k2
    V[1] = v
    V[2] = (1j * kz * dv + 1j * kx * eta) / k2
    wall = case.get("wall", 0.0)
    V[0, 0, nz] = on(y * (2.0 - y) + wall * t)
    return V


def _params(seed):
    rng = np.random.default_rng(seed + 77)
    p = [rng.uniform(-1, 1, s) * math.sqrt(6.0 / s[0]) if len(s) == 2 else 0.05 * rng.standard_normal(s) for s in SHAPES]
    return np.concatenate([a.ravel() for a in p]).astype(np.float32)


def _samples(n, seed):
    """Standardised features and targets that depend on them."""
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((n, IN), dtype=np.float32)
    T = np.tanh(X[:, :OUT] * X[:, 9:9 + OUT] + 0.5 * X[:, 18:18 + OUT])
    return X, (T + 0.3 * rng.standard_normal((n, OUT), dtype=np.float32)).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("run", "les"):
        cfg = _config(case)
        V = _field(case, seed).cpu().numpy().transpose(3, 2, 1, 0)
        ch = Channel(cfg, lib.CHAN_SPLIT if case.get("split") else lib.CHAN_FP64)
        ch.set_field(V)
        if case.get("omega2"):
            ch.set_body_force_feedback(*coriolis(cfg, case["omega2"]))
        ch.initial()
        ch.outstats()
        state = dict(case=case, ch=ch)
        if kind == "les":
            state["mlp"] = Mlp(16)
            state["mlp"].set_params(_params(seed))
            state["norm"] = _norm(ch.les_features())
            state["start"] = V
        return state
    n = case["n"]
    m = Mlp(n)
    m.set_params(_params(seed))
    X, T = _samples(n, seed)
    if kind != "forward":
        m.set_data(X, T)
    return dict(case=case, mlp=m, X=X)


def _norm(X):
    """Feature means and scales, and the stresses' means and scales."""
    X = X[::7]
    return np.concatenate([X.mean(0, dtype=np.float64), X.std(0, dtype=np.float64) + 1e-3, np.zeros(OUT),
                           np.full(OUT, NORM_SCALE)]).astype(np.float32)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        ch, n, every = state["ch"], case["steps"], case["stats_every"]
        if case["split"]:
            return dict(rows=ch.steps(n).astype(np.float32), field=ch.get_field().astype(np.complex64))
        if not every:
            return dict(rows=ch.steps(n), field=ch.get_field())
        rows, profiles = [], []
        for k in range(0, n, every):
            rows.append(ch.steps(min(every, n - k)))
            profiles.append(ch.stats())
        return dict(rows=rows, profiles=profiles, field=ch.get_field())
    if kind == "les":
        ch, rows = state["ch"], []
        ch.set_field(state["start"])
        ch.initial()
        ch.outstats()
        for _ in range(case["steps"]):
            ch.les_closure_force(state["mlp"], state["norm"])
            rows.append(ch.step())
        return dict(rows=rows, field=ch.get_field())
    m = state["mlp"]
    if kind == "grad":
        loss, g = m.grad(0, case["count"])
        return dict(loss=loss, grad=g)
    if kind == "train":
        losses, _ = m.train(case["steps"], case["batch"], 1e-3)
        return dict(losses=losses, params=m.get_params())
    return m.forward(state["X"])


def work(case):
    """Bytes and operations of one pass.  A time step is three substeps, each
    of which reads and writes the field and the two stored explicit terms and
    forms nine real 2-D transforms per row (three in, six products out), the
    compact stencils and the solves; the field goes to the host once."""
    kind = case["kind"]
    mlp = IN * HID + 2 * HID * HID + HID * OUT
    if kind in ("run", "les"):
        nxd, nzd = _dealiased(case["nx"], case["nz"])
        pts = 2 * nxd * nzd
        modes, rows = (case["nx"] + 1) * (2 * case["nz"] + 1), case["ny"] + 3
        field = 3 * 16 * modes * rows
        explicit = 2 * (8 if case.get("split") else 16) * modes * rows
        sub_bytes = 2 * field + 2 * explicit
        sub_flops = rows * (9 * 2.5 * pts * math.log2(pts) + 6 * pts + 400 * modes)
        n = case["steps"]
        b, f = 3 * n * sub_bytes + field, 3 * n * sub_flops
        if kind == "les":
            samples = (case["ny"] + 1) * pts
            b += field + n * (field + 4 * (9 + OUT) * samples + field)
            f += n * (samples * 2 * mlp + (case["ny"] + 1) * 15 * 2.5 * pts * math.log2(pts))
        elif case["stats_every"]:
            b += -(-n // case["stats_every"]) * field
        return {"bytes": float(b), "flops": float(f)}
    if kind == "forward":
        return {"bytes": 4.0 * case["n"] * (IN + OUT), "flops": 2.0 * mlp * case["n"]}
    rows = case["count"] if kind == "grad" else case["batch"]
    n = 1 if kind == "grad" else case["steps"]
    return {"bytes": float(n * (rows * (2 * IN + 4 * OUT) + 4 * 4 * mlp)), "flops": float(n * 6 * mlp * rows)}


# --------------------------------------------------- the outputs in 64 bits --
RK = [(120.0 / 32.0, 2.0, 0.0), (120.0 / 8.0, 50.0 / 8.0, 34.0 / 8.0), (120.0 / 20.0, 90.0 / 20.0, 50.0 / 20.0)]


def _stencil(h, right):
    """w with sum_j w_j h_j^(4-i) = right_i, i = 0..4, for offsets of size 1."""
    return np.linalg.solve(np.stack([h ** (4 - i) for i in range(5)]), right)


def _stencils(y):
    """The compact stencils d0, d1, d2, d4 of the interior rows 1..ny-1 and the
    one-sided first derivatives at the walls and ghost rows; y[0] is row -1."""
    ny = len(y) - 3
    d = np.zeros((ny - 1, 4, 5))
    for iy in range(1, ny):
        h = y[iy - 1:iy + 4] - y[iy + 1]
        H = np.abs(h).max()
        h = h / H
        d4 = _stencil(h, np.array([24.0, 0, 0, 0, 0]))
        right = np.array([(d4 * h ** (8 - i)).sum() for i in range(5)])
        d0 = np.linalg.solve(np.stack([(5 - i) * (6 - i) * (7 - i) * (8 - i) * h ** (4 - i) for i in range(5)]), right)
        d2 = _stencil(h, np.array([(d0 * (4 - i) * (3 - i) * h ** max(2 - i, 0)).sum() if i <= 2 else 0.0 for i in range(5)]))
        d1 = _stencil(h, np.array([(d0 * (4 - i) * h ** max(3 - i, 0)).sum() if i <= 3 else 0.0 for i in range(5)]))
        d[iy - 1] = d0, d1 / H, d2 / H ** 2, d4 / H ** 4

    def first(nodes, at):
        h = nodes - at
        H = np.abs(h).max()
        return _stencil(h / H, np.array([0, 0, 0, 1.0, 0])) / H

    lo, hi = y[:5], y[-5:]
    return d, first(lo, y[1]), first(lo, y[0]), first(hi, y[-2]), first(hi, y[-1])


class _Flow:
    """The channel's time step on torch tensors V[c][row][ix][iz]."""

    def __init__(self, case, V):
        self.case, self.dev = case, V.device
        self.cfg = _config(case)
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        self.nx, self.ny, self.nz, self.npair = nx, ny, nz, (nx + 1) * (2 * nz + 1)
        self.nxd, self.nzd = _dealiased(nx, nz)
        self.V = V.permute(0, 3, 1, 2).contiguous()
        self.y = _rows(ny)
        der, *self.one_sided = _stencils(self.y)
        self.der_np = der
        self.der = self.on(der)
        self.kx = self.on(case["alfa0"] * np.arange(nx + 1))[:, None].expand(nx + 1, 2 * nz + 1)
        self.kz = self.on(case["beta0"] * np.arange(-nz, nz + 1))[None, :].expand(nx + 1, 2 * nz + 1)
        self.k2 = self.kx ** 2 + self.kz ** 2
        self.old = [torch.zeros((ny - 1, nx + 1, 2 * nz + 1), dtype=torch.complex128, device=self.dev) for _ in range(2)]
        pi = float(np.float32(math.pi))  # the CFL number's grid spacings carry a single-precision pi
        self.dx, self.dz = pi / (case["alfa0"] * self.nxd), 2.0 * pi / (case["beta0"] * self.nzd)
        self.cfl, self.dt, self.time = 0.0, self.cfg.deltat, 0.0
        self.meanpx = self.corrpx = 0.0
        self.fr = [0.0, 0.0, 0.0]
        self.static = None
        # rows 1..ny-1 of the first-derivative operator's left side, wall columns apart
        n = ny - 1
        A = np.zeros((n, n + 4))
        for r in range(n):
            A[r, r:r + 5] = der[r, 0]
        self.d0 = A
        self.d0_inv = self.on(np.linalg.inv(A[:, 2:-2]))  # a well-conditioned band
        # wall and ghost values eliminated: row 0 / -1 and ny / ny+1 of v and eta
        b0, bm, bn, bp = self.one_sided
        self.walls = {"v": (b0, bn), "eta": (der[0, 3], der[-1, 3])}
        self.weights = self.quadrature()
        self.initial()

    def on(self, a):
        return torch.from_numpy(np.array(a, dtype=np.float64)).to(self.dev)

    def quadrature(self):
        """Weights of the three-point rule over the rows iy-1, iy, iy+1 at odd iy."""
        y, w = self.y, np.zeros(self.ny + 3)
        for i in range(2, self.ny + 1, 2):  # index of row iy is iy + 1
            p, m = y[i + 1] - y[i], y[i - 1] - y[i]
            a1 = -m / 3 + p / 6 + p * p / m / 6
            a3 = p / 3 - m / 6 - m * m / p / 6
            w[i - 1] += a1
            w[i] += p - m - a1 - a3
            w[i + 1] += a3
        return self.on(w)

    def products(self, cfl, keep=True):
        """The six dealiased products, and the CFL maximum of the rows 1..ny-1."""
        nx, nz, ny = self.nx, self.nz, self.ny
        iz = torch.arange(-nz, nz + 1, device=self.dev) % self.nzd
        P = torch.empty((6, ny + 3, nx + 1, 2 * nz + 1), dtype=torch.complex128, device=self.dev) if keep else None
        chunk = max(1, int(2 ** 27 // (2 * self.nxd * self.nzd)) // 4)
        for r0 in range(0, ny + 3, chunk):
            r1 = min(ny + 3, r0 + chunk)
            S = torch.zeros((3, r1 - r0, self.nzd, self.nxd + 1), dtype=torch.complex128, device=self.dev)
            S[:, :, iz, :nx + 1] = self.V[:, r0:r1].transpose(2, 3)
            u, v, w = torch.fft.irfft2(S, s=(self.nzd, 2 * self.nxd), norm="forward")
            if cfl:
                for r in range(max(r0, 2), min(r1, ny + 1)):
                    dy = 0.5 * (self.y[r + 1] - self.y[r - 1])
                    k = r - r0
                    m = (u[k].abs() / self.dx + v[k].abs() / dy + w[k].abs() / self.dz).max()
                    self.cfl = max(self.cfl, float(m))
            if keep:
                for q, p in enumerate((u * u, v * v, w * w, u * v, v * w, u * w)):
                    F = torch.fft.rfft2(p, norm="forward")
                    P[q, r0:r1] = F[:, iz, :nx + 1].transpose(1, 2)
            del S, u, v, w
        return P

    def D(self, k, f):
        """The k-th stencil family (0: d0, 1: d1, 2: d2, 3: d4) of f[row]."""
        n, w = self.ny - 1, self.der[:, k, :, None, None]
        s = w[:, 0] * f[0:n]
        for j in range(1, 5):
            s = s + w[:, j] * f[j:j + n]
        return s

    def force(self):
        om = self.case.get("omega2", 0.0)
        if om:
            F = torch.zeros_like(self.V)
            F[0], F[1] = -om * self.V[1], om * self.V[0]
        elif self.static is not None:
            F = self.static.clone()
        else:
            return None
        F[:, 1] = 0
        F[:, -2] = 0
        lo, hi = self.der_np[0, 3], self.der_np[-1, 3]
        F[:, 0] = -(lo[2] * F[:, 2] + lo[3] * F[:, 3] + lo[4] * F[:, 4]) / lo[0]
        F[:, -1] = -(hi[0] * F[:, -5] + hi[1] * F[:, -4] + hi[2] * F[:, -3]) / hi[4]
        return F

    def substep(self, ode, last):
        uu, vv, ww, uv, vw, uw = self.products(last)
        D, kx, kz, k2, ni, V, dt = self.D, self.kx, self.kz, self.k2, self.cfg.ni, self.V, self.dt
        m = (slice(None), 0, self.nz)
        rhsu = -1j * kx * D(0, uu) - D(1, uv) - 1j * kz * D(0, uw)
        rhsv = -1j * kx * D(0, uv) - D(1, vv) - 1j * kz * D(0, vw)
        rhsw = -1j * kx * D(0, uw) - D(1, vw) - 1j * kz * D(0, ww)
        ev = (1j * kx * (1j * kx * D(1, uu) + D(2, uv) + 1j * kz * D(1, uw))
              + 1j * kz * (1j * kx * D(1, uw) + D(2, vw) + 1j * kz * D(1, ww)) - k2 * rhsv)
        ee = 1j * kz * rhsu - 1j * kx * rhsw
        ee[m] = torch.complex(rhsu[m].real + self.meanpx, rhsw[m].real)
        F = self.force()
        if F is not None:
            ev = ev - k2 * D(0, F[1]) - 1j * kx * D(1, F[0]) - 1j * kz * D(1, F[2])
            fu, fw = D(0, F[0]), D(0, F[2])
            fe = 1j * kz * fu - 1j * kx * fw
            fe[m] = torch.complex(fu[m].real, fw[m].real)
            ee = ee + fe
        eta = 1j * kz * V[0] - 1j * kx * V[2]
        eta[m] = torch.complex(V[0][m].real, V[2][m].real)
        Dv0, Dv2 = D(0, V[1]), D(2, V[1])
        rv = ode[0] / dt * (Dv2 - k2 * Dv0) + ni * (D(3, V[1]) - 2 * k2 * Dv2 + k2 * k2 * Dv0) + ode[1] * ev - ode[2] * self.old[1]
        De0, De2 = D(0, eta), D(2, eta)
        re = ode[0] / dt * De0 + ni * (De2 - k2 * De0) + ode[1] * ee - ode[2] * self.old[0]
        self.old = [ee, ev]
        del uu, vv, ww, uv, vw, uw, rhsu, rhsv, rhsw
        self.solve(ode[0] / dt, re, rv)

    def solve(self, lam, re, rv):
        """eta and v of the rows 1..ny-1 with the wall conditions, for every
        mode at once; one more column holds the mean flow's response to a unit
        force."""
        ny, ni, n, der = self.ny, self.cfg.ni, self.ny - 1, self.der_np
        k2 = torch.cat([self.k2.reshape(-1), torch.zeros(1, dtype=torch.float64, device=self.dev)])
        mean = self.nz  # the column of the mode (0,0)
        wall = {s: torch.zeros((2, self.npair + 1), dtype=torch.complex128, device=self.dev) for s in ("eta", "v")}
        wall["eta"][0, mean], wall["eta"][1, mean] = self.cfg.u0, self.cfg.uN
        out = {}
        for s, rhs, unit in (("eta", re, 1.0), ("v", rv, 0.0)):
            b = torch.cat([rhs.reshape(n, -1), torch.full((n, 1), unit, dtype=torch.complex128, device=self.dev)], 1)
            lo, hi = self.walls[s]

            def band(r):
                d0, d2, d4 = der[r, 0], der[r, 2], der[r, 3]
                if s == "v":
                    return [lam * (d2[j] - k2 * d0[j]) - ni * (d4[j] - 2 * k2 * d2[j] + k2 * k2 * d0[j]) for j in range(5)]
                return [lam * d0[j] - ni * (d2[j] - k2 * d0[j]) for j in range(5)]

            w0, wn = wall[s]
            # ghost value = -(row . the other four) / its own weight
            first, second, x, up = None, None, [None] * n, [None] * n
            for r in range(n):
                a = band(r)
                f = b[r]
                if r == 0:
                    a[1], a[2], a[3], a[4] = (a[j] - a[0] * (lo[j] / lo[0]) for j in (1, 2, 3, 4))
                    f = f - a[1] * w0
                if r == 1:
                    f = f - a[0] * w0
                if r == n - 1:
                    a[0], a[1], a[2], a[3] = (a[j] - a[4] * (hi[j] / hi[4]) for j in (0, 1, 2, 3))
                    f = f - a[3] * wn
                if r == n - 2:
                    f = f - a[4] * wn
                c, d, e = a[2], a[3], a[4]
                l1 = a[1]
                if r >= 2:
                    p1, p2, pf = up[r - 2]
                    l1 = l1 - a[0] * p1
                    c = c - a[0] * p2
                    f = f - a[0] * pf
                if r >= 1:
                    p1, p2, pf = up[r - 1]
                    c = c - l1 * p1
                    d = d - l1 * p2
                    f = f - l1 * pf
                up[r] = (d / c, e / c, f / c)
            for r in range(n - 1, -1, -1):
                p1, p2, pf = up[r]
                v = pf
                if r + 1 < n:
                    v = v - p1 * x[r + 1]
                if r + 2 < n:
                    v = v - p2 * x[r + 2]
                x[r] = v
            glo = -(lo[1] * w0 + lo[2] * x[0] + lo[3] * x[1] + lo[4] * x[2]) / lo[0]
            ghi = -(hi[0] * x[n - 3] + hi[1] * x[n - 2] + hi[2] * x[n - 1] + hi[3] * wn) / hi[4]
            out[s] = torch.stack([glo, w0] + x + [wn, ghi])
        eta, ucor = out["eta"][:, :-1], out["eta"][:, -1].real
        v = out["v"][:, :-1]
        u00, w00 = eta[:, mean].real.clone(), eta[:, mean].imag.clone()
        q = self.weights
        self.fr = [float((q * u00).sum()), float((q * w00).sum()), float((q * ucor).sum())]
        cfg = self.cfg
        if cfg.cpi:
            self.meanpx = 1.5 / cfg.gamma * self.fr[0] * ni
        elif abs(cfg.meanflowx) > 1e-7:
            self.corrpx = (cfg.meanflowx - self.fr[0]) / self.fr[2]
            u00 = u00 + self.corrpx * ucor
        # dv/dy: one-sided at the walls and ghost rows, compact inside
        b0, bm, bn, bp = (self.on(w) for w in self.one_sided)
        lo_v, hi_v = v[:5], v[-5:]
        f0, fm = (b0[:, None] * lo_v).sum(0), (bm[:, None] * lo_v).sum(0)
        fn, fp = (bn[:, None] * hi_v).sum(0), (bp[:, None] * hi_v).sum(0)
        w = self.der[:, 1, :, None]
        f = sum(w[:, j] * v[j:j + n] for j in range(5))
        f = f - self.on(self.d0[:, 0])[:, None] * fm - self.on(self.d0[:, 1])[:, None] * f0
        f = f - self.on(self.d0[:, -2])[:, None] * fn - self.on(self.d0[:, -1])[:, None] * fp
        x = self.d0_inv @ torch.view_as_real(f.contiguous()).reshape(n, -1)
        x = torch.view_as_complex(x.reshape(n, self.npair, 2).contiguous())
        dv = torch.cat([fm[None], f0[None], x, fn[None], fp[None]])
        kx, kz, k2 = self.kx.reshape(-1), self.kz.reshape(-1), self.k2.reshape(-1).clone()
        k2[mean] = 1.0
        U, W = (1j * kx * dv - 1j * kz * eta) / k2, (1j * kz * dv + 1j * kx * eta) / k2
        U[:, mean], W[:, mean] = u00.to(U.dtype), w00.to(U.dtype)
        self.V = torch.stack([U, v, W]).reshape(self.V.shape)

    def initial(self):
        if self.dt == 0:
            self.dt = 1.0
        self.products(True, keep=False)
        m = (slice(None), 0, self.nz)
        self.fr = [float((self.weights * self.V[0][m].real).sum()), float((self.weights * self.V[2][m].real).sum()), 0.0]
        if self.cfg.cpi:
            self.meanpx = 1.5 / self.cfg.gamma * self.fr[0] * self.cfg.ni
        self.outstats()

    def outstats(self):
        cfl, self.cfl = self.cfl, 0.0
        if self.cfg.cflmax > 0:
            self.dt = self.cfg.cflmax / cfl
        u, w = (self.V[c, :, 0, self.nz].real.cpu().numpy() for c in (0, 2))
        b0, _, bn, _ = self.one_sided
        return np.array([self.time, b0 @ u[:5], -(bn @ u[-5:]), b0 @ w[:5], -(bn @ w[-5:]),
                         self.fr[0] + self.corrpx * self.fr[2], self.meanpx + self.corrpx, self.fr[1], 0.0, cfl * self.dt, self.dt])

    def step(self):
        for k, ode in enumerate(RK):
            self.time += 2.0 / ode[0] * self.dt
            self.substep(ode, k == 2)
        return self.outstats()

    def stats(self):
        V = self.V[:, 1:-1].clone()
        mean = V[:, :, 0, self.nz].real.clone()
        V[:, :, 0, self.nz] -= mean
        f = torch.full((self.nx + 1, 1), 2.0, dtype=torch.float64, device=self.dev)
        f[0] = 1.0
        var = (f * V.abs().square()).sum((2, 3))
        uv = (f * (V[0] * V[1].conj()).real).sum((1, 2))
        return {"mean": mean.cpu().numpy(), "var": var.cpu().numpy(), "uv": uv.cpu().numpy()}

    def field(self):
        return self.V.permute(1, 3, 2, 0).cpu().numpy()

    # ---- the closure on the dealiased physical grid, rows 0..ny
    def ddy(self, f):
        """Second-order differences on the stretched rows (axis 0), one-sided at the walls."""
        y = self.on(self.y[1:-1]).reshape((-1,) + (1,) * (f.dim() - 1))
        h = y[1:] - y[:-1]
        a, b = h[:-1], h[1:]
        d = torch.empty_like(f)
        d[1:-1] = -b / (a * (a + b)) * f[:-2] + (b - a) / (a * b) * f[1:-1] + a / (b * (a + b)) * f[2:]
        a, b = h[0], h[1]
        d[0] = -(2 * a + b) / (a * (a + b)) * f[0] + (a + b) / (a * b) * f[1] - a / (b * (a + b)) * f[2]
        a, b = h[-2], h[-1]
        d[-1] = b / (a * (a + b)) * f[-3] - (a + b) / (a * b) * f[-2] + (2 * b + a) / (b * (a + b)) * f[-1]
        return d

    def features(self):
        nx, nz = self.nx, self.nz
        iz = torch.arange(-nz, nz + 1, device=self.dev) % self.nzd
        g = []
        for c in range(3):
            v = self.V[c, 1:-1]
            for d in (1j * self.kx * v, self.ddy(v), 1j * self.kz * v):
                S = torch.zeros((self.ny + 1, self.nzd, self.nxd + 1), dtype=torch.complex128, device=self.dev)
                S[:, iz, :nx + 1] = d.transpose(1, 2)
                g.append(torch.fft.irfft2(S, s=(self.nzd, 2 * self.nxd), norm="forward").transpose(1, 2))
        g = torch.stack(g, -1)  # row, x, z, 9
        rows = torch.arange(self.ny + 1, device=self.dev)
        X = [g[(rows + k).clamp(0, self.ny)] for k in (0, -2, -1, 1, 2)]
        u = self.V[0, :, 0, nz].real.cpu().numpy()
        b0, _, bn, _ = self.one_sided
        utau = math.sqrt(self.cfg.ni * 0.5 * (abs(b0 @ u[:5]) + abs(bn @ u[-5:])))
        yy = self.y[1:-1]
        yp = self.on(np.minimum(yy, 2.0 - yy) * utau / self.cfg.ni)[:, None, None, None].expand(g.shape[:3] + (1,))
        return torch.cat(X + [yp], -1)

    def closure(self, params, norm):
        nx, nz = self.nx, self.nz
        X = (self.features() - norm[:IN]) / norm[IN:2 * IN]
        tau = _net(X.reshape(-1, IN), params)[-1] * norm[2 * IN + OUT:] + norm[2 * IN:2 * IN + OUT]
        tau = tau.reshape(X.shape[:3] + (OUT,)).permute(3, 0, 2, 1)  # q, row, z, x
        iz = torch.arange(-nz, nz + 1, device=self.dev) % self.nzd
        T = torch.fft.rfft2(tau.contiguous(), norm="forward")[:, :, iz, :nx + 1].transpose(2, 3)
        xx, yy, zz, xy, xz, yz = T
        F = torch.zeros_like(self.V)
        for i, (a, b, c) in enumerate(((xx, xy, xz), (xy, yy, yz), (xz, yz, zz))):
            F[i, 1:-1] = -(1j * self.kx * a + self.ddy(b) + 1j * self.kz * c)
        self.static = F


def _net(X, params):
    """Activations of every layer, the last the network's output."""
    acts = [X]
    for k in range(4):
        z = acts[-1] @ params[2 * k] + params[2 * k + 1]
        acts.append(z.relu() if k < 3 else z)
    return acts


def _split_params(p, dev):
    out, o = [], 0
    for s in SHAPES:
        n = int(np.prod(s))
        out.append(torch.from_numpy(p[o:o + n].astype(np.float64).reshape(s)).to(dev))
        o += n
    return out


def _gradient(X, T, params):
    acts = _net(X, params)
    d = acts[-1] - T
    loss = float(d.square().sum()) / (OUT * len(X))
    d = 2.0 * d / (OUT * len(X))
    g = [None] * 8
    for k in (3, 2, 1, 0):
        g[2 * k], g[2 * k + 1] = acts[k].t() @ d, d.sum(0)
        if k:
            d = (d @ params[2 * k].t()) * (acts[k] > 0)
    return loss, g


def exact(case, seed):
    kind, dev = case["kind"], _device()
    if kind in ("run", "les"):
        flow = _Flow(case, _field(case, seed))
        n = case["steps"]
        if kind == "les":
            norm = torch.from_numpy(_norm(flow.features().reshape(-1, IN).float().cpu().numpy()).astype(np.float64)).to(dev)
            params, rows = _split_params(_params(seed), dev), []
            for _ in range(n):
                flow.closure(params, norm)
                rows.append(flow.step())
            return dict(rows=rows, field=flow.field())
        every = case["stats_every"]
        if n > 20 and case["nx"] * case["ny"] * case["nz"] > 10 ** 7:
            return None  # over 20 seconds
        if not every:
            return dict(rows=np.stack([flow.step() for _ in range(n)]), field=flow.field())
        rows, profiles = [], []
        for k in range(0, n, every):
            rows.append(np.stack([flow.step() for _ in range(min(every, n - k))]))
            profiles.append(flow.stats())
        return dict(rows=rows, profiles=profiles, field=flow.field())
    params = _split_params(_params(seed), dev)
    X, T = (torch.from_numpy(a).to(dev).double() for a in _samples(case["n"], seed))
    if kind == "forward":
        return _net(X, params)[-1].cpu().numpy()
    if kind == "grad":
        loss, g = _gradient(X[:case["count"]], T[:case["count"]], params)
        return dict(loss=loss, grad=torch.cat([a.reshape(-1) for a in g]).cpu().numpy())
    losses, first = [], 0
    mom = [[torch.zeros_like(p) for p in params] for _ in range(2)]
    for t in range(1, case["steps"] + 1):
        if first + case["batch"] > case["n"]:
            first = 0
        rows = slice(first, first + case["batch"])
        loss, g = _gradient(X[rows], T[rows], params)
        losses.append(loss)
        for k, p in enumerate(params):
            mom[0][k] = 0.9 * mom[0][k] + 0.1 * g[k]
            mom[1][k] = 0.999 * mom[1][k] + 0.001 * g[k] ** 2
            params[k] = p - 1e-3 * (mom[0][k] / (1 - 0.9 ** t)) / ((mom[1][k] / (1 - 0.999 ** t)).sqrt() + 1e-8)
        first += case["batch"]
    return dict(losses=np.array(losses), params=torch.cat([p.reshape(-1) for p in params]).cpu().numpy())
