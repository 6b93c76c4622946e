"""Timed cases of the engine: what its users have it do, through its public entry points.

Kinds of case (the "kind" of each dict):

  grating   ofd.solve_ofd: a 1D grating swept over frequencies
  pillars   engine.solve_batch: a 2D pillar stack over wavelengths and incidence directions
  designs   surrogate.solve_geometries: many designs of a two-layer grating, one solve each
  uneven    engine.solve_uneven: independent stacks of different sizes
  relief    engine.rcwa_integrate: a z-varying relief as a staircase of slices
  field     engine.field_image: the field of one stack on a slice
  predict   surrogate.MLP.predict: queries answered by the network ensemble
  train     surrogate.MLP.train: epochs of minibatch training
  gradient  surrogate.MLP.gradient: loss and gradient of one batch

Every pass of the solver kinds starts from host arrays, as a program with new
structures does: the plan is built, executed and read back inside the pass.
"""
import functools
import math

import numpy as np
import torch

from openrcwa_amd import engine, ofd, surrogate

C0 = 2.99792458e8
PERIOD = 400e-9
EPS_SUB = 2.25


def listed():
    return [
        # one .ofd file: 5 harmonics, 16 frequencies; the smallest call, all latency
        dict(name="grating-n22-16", kind="grating", nx=5, freqs=16, layers=1, poles=False),
        # a converged 1D spectrum of a dispersive grating
        dict(name="grating-n82-200", kind="grating", nx=20, freqs=200, layers=3, poles=True),
        # a quick look at a 2D structure at few orders
        dict(name="pillars-n98-48", kind="pillars", nx=3, ny=3, layers=4, lams=24, dirs=2,
             mu=False, prec="fp64"),
        # one converged solve: one wavelength, one direction
        dict(name="pillars-n450-1", kind="pillars", nx=7, ny=7, layers=4, lams=1, dirs=1,
             mu=False, prec="fp64"),
        # a spectrum at one direction
        dict(name="pillars-n450-20", kind="pillars", nx=7, ny=7, layers=4, lams=20, dirs=1,
             mu=False, prec="fp64"),
        # a slice of the big sweep (wavelengths x directions): throughput
        dict(name="pillars-n450-320", kind="pillars", nx=7, ny=7, layers=4, lams=40, dirs=8,
             mu=False, prec="fp64"),
        # a large, not square, order count at one wavelength
        dict(name="pillars-n798-1", kind="pillars", nx=10, ny=9, layers=2, lams=1, dirs=1,
             mu=False, prec="fp64"),
        # training data of the learned surrogate, or a design sweep
        dict(name="designs-n242-384", kind="designs", count=384),
        # independent stacks of mixed order and layer counts
        dict(name="uneven-36", kind="uneven", count=36, nmin=3, nmax=6, layers=6),
        # an anti-reflection relief between air and its substrate
        dict(name="relief-n162-24", kind="relief", nx=4, ny=4, slices=24),
        # surrogate inference on a batch of host queries
        dict(name="predict-65536", kind="predict", rows=65536, width=512, depth=4, members=4,
             bf16=False),
        # surrogate training
        dict(name="train-32768", kind="train", rows=32768, batch=4096, epochs=1, width=512,
             depth=4, members=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["grating", "pillars", "pillars", "pillars", "designs", "uneven", "relief",
                       "field", "predict", "train", "gradient"])
    if kind == "grating":
        return dict(kind=kind, nx=rng.randint(3, 30), freqs=_log(rng, 5, 250),
                    layers=rng.randint(1, 4), poles=rng.random() < 0.5)
    if kind == "pillars":
        nx = rng.randint(2, 9)
        ny = max(2, min(9, nx + rng.randint(-2, 2)))
        n = 2 * (2 * nx + 1) * (2 * ny + 1)
        layers, dirs = rng.randint(1, 5), rng.choice([1, 1, 2, 3])
        # up to an eighth of the largest listed sweep's work, and few enough for n > 500
        most = max(1, min(400, int(160 * 450 ** 3 / (n ** 3 * layers * dirs))))
        lams = _log(rng, 1, most) if n <= 500 else 1
        return dict(kind=kind, nx=nx, ny=ny, layers=layers, lams=lams, dirs=dirs,
                    mu=rng.random() < 0.1,
                    prec=rng.choice(["fp64"] * 8 + ["fp32", "bf16x6"]))
    if kind == "designs":
        return dict(kind=kind, count=_log(rng, 3, 380))
    if kind == "uneven":
        nmin = rng.randint(2, 4)
        return dict(kind=kind, count=rng.randint(3, 36), nmin=nmin,
                    nmax=nmin + rng.randint(1, 2), layers=rng.randint(2, 8))
    if kind == "relief":
        nx = rng.randint(2, 5)
        return dict(kind=kind, nx=nx, ny=rng.randint(2, nx), slices=rng.randint(5, 40))
    if kind == "field":
        nx = rng.randint(2, 6)
        return dict(kind=kind, nx=nx, ny=rng.randint(2, nx), layers=rng.randint(1, 4),
                    component=rng.choice(["Ex", "Ey", "Ez", "Hx", "Hy", "Hz"]),
                    plane=rng.choice(["xz", "yz", "xy"]), res=_log(rng, 60, 500))
    net = dict(width=32 * rng.randint(2, 16), depth=rng.randint(2, 5), members=rng.randint(1, 5))
    if kind == "predict":
        return dict(kind=kind, rows=_log(rng, 1, 60000), bf16=rng.random() < 0.4, **net)
    if kind == "train":
        batch = 32 * rng.randint(8, 128)
        return dict(kind=kind, rows=batch * rng.randint(2, 6) + rng.randint(0, 200), batch=batch,
                    epochs=rng.randint(1, 2), **net)
    return dict(kind=kind, rows=_log(rng, 30, 16000), **net)


@functools.lru_cache(None)
def _context(prec="fp64"):
    """The handle that a program makes once (one per star-product precision)."""
    ctx = engine.Context(0)
    ctx.set_gemm_precision(prec)
    return ctx


def _pols(theta, phi):
    """TE and TM transverse amplitudes, angles in degrees."""
    t, p = math.radians(theta), math.radians(phi)
    return np.array([[-math.sin(p), math.cos(p)],
                     [math.cos(t) * math.cos(p), math.cos(t) * math.sin(p)]], dtype=complex)


def _pillar_stack(rs, layers, mu=False):
    """Edges, eps (and mu) grids and thicknesses of `layers` rectangles of lossy
    dielectrics in air, between air and the substrate."""
    rect = [(rs.uniform(0.2, 0.8) * PERIOD, rs.uniform(0.2, 0.8) * PERIOD,
             complex(rs.uniform(2, 12), rs.uniform(0.01, 0.1))) for _ in range(layers)]
    cx = np.array(sorted([0.0, PERIOD] + [r[0] for r in rect]))
    cy = np.array(sorted([0.0, PERIOD] + [r[1] for r in rect]))
    xc, yc = 0.5 * (cx[1:] + cx[:-1]), 0.5 * (cy[1:] + cy[:-1])
    inside = [np.outer(yc < r[1], xc < r[0]) for r in rect]
    air = np.ones((yc.size, xc.size), dtype=complex)
    eps = np.stack([air] + [np.where(i, r[2], 1.0) for i, r in zip(inside, rect)] + [EPS_SUB * air])
    mus = None
    if mu:
        mus = np.stack([air] + [np.where(i, rs.uniform(1.1, 2.0), 1.0) for i in inside] + [air])
    thick = np.concatenate([[0.0], rs.uniform(50e-9, 300e-9, layers), [0.0]])
    return cx, cy, eps, mus, thick


def _pillars(case, seed):
    rs = np.random.RandomState(seed)
    cx, cy, eps, mu, thick = _pillar_stack(rs, case["layers"], case["mu"])
    lam1 = C0 / np.sort(rs.uniform(4.3e14, 7.5e14, case["lams"]))
    ang = [(rs.uniform(0, 35), rs.uniform(0, 45)) for _ in range(case["dirs"])]
    lam = np.repeat(lam1, len(ang))
    th = np.tile([math.radians(a[0]) for a in ang], len(lam1))
    ph = np.tile([math.radians(a[1]) for a in ang], len(lam1))
    k0 = 2 * math.pi / lam
    return dict(nX=case["nx"], nY=case["ny"], coord_x=cx, coord_y=cy, thickness=thick, lam=lam,
                kx0=k0 * np.sin(th) * np.cos(ph), ky0=k0 * np.sin(th) * np.sin(ph), eps=eps,
                pols=np.tile(np.stack([_pols(*a) for a in ang]), (len(lam1), 1, 1)), mu=mu)


def _grating(case, seed):
    rs = np.random.RandomState(seed)
    nl = case["layers"]
    layers = [dict(eps1=1.0, eps2=1.0, fill=0.5, thickness=0.0)]
    layers += [dict(eps1=rs.uniform(2, 6), eps1i=rs.uniform(0.01, 0.05), eps2=1.0,
                    fill=rs.uniform(0.2, 0.8), thickness=rs.uniform(5e-8, 3e-7)) for _ in range(nl)]
    layers += [dict(eps1=EPS_SUB, eps2=EPS_SUB, fill=0.5, thickness=0.0)]
    poles = {}
    if case["poles"]:
        # Lorentz poles well above the swept band: a dielectric with normal dispersion
        poles = {(i, 1): [(rs.uniform(1, 3), rs.uniform(4e15, 8e15), rs.uniform(1e14, 3e14),
                           rs.uniform(6.5e15, 9e15))] for i in range(1, nl + 1)}
    return dict(nX=case["nx"], period=3.0e-7, layers=layers, poles=poles,
                freqs=np.sort(rs.uniform(4.3e14, 7.5e14, case["freqs"])),
                theta=rs.uniform(0, 30), phi=rs.uniform(0, 45))


def _uneven(case, seed):
    rs = np.random.RandomState(seed)
    stacks = []
    # sizes go round the range so that they do not depend on the seed
    for i in range(case["count"]):
        N = case["nmin"] + i % (case["nmax"] - case["nmin"] + 1)
        cx, cy, eps, _, thick = _pillar_stack(rs, 1 + (5 * i) % case["layers"])
        lam, th, ph = rs.uniform(400e-9, 700e-9), rs.uniform(0, 40), rs.uniform(0, 90)
        k0 = 2 * math.pi / lam
        t, p = math.radians(th), math.radians(ph)
        stacks.append(dict(nX=N, nY=N, period=PERIOD, coord_x=cx, coord_y=cy, eps=eps,
                           thickness=thick, lam=lam, kx0=k0 * math.sin(t) * math.cos(p),
                           ky0=k0 * math.sin(t) * math.sin(p), theta=th, phi=ph,
                           pol=_pols(th, ph)))
    return stacks


class _Relief:
    """A rectangular bump that fills the period at the bottom (z = 0) and ends in air at z1."""

    def __init__(self, seed):
        rs = np.random.RandomState(seed)
        self.e = complex(rs.uniform(2, 4), rs.uniform(0.01, 0.05))
        self.ax, self.ay = rs.uniform(0.6, 1.6, 2)
        self.lam = rs.uniform(450e-9, 700e-9)
        self.z1 = rs.uniform(200e-9, 500e-9)
        self.kx0, self.ky0 = 2 * math.pi / self.lam * rs.uniform(0.05, 0.4, 2)

    def __call__(self, z):
        u = 1.0 - z / self.z1
        if u <= 0.0 or u >= 1.0:
            e = np.full((3, 3), self.e if u >= 1.0 else 1.0, dtype=complex)
            c = np.array([0.0, 0.25, 0.75, 1.0]) * PERIOD
            return c, c, e
        wx, wy = 0.5 * u ** self.ax, 0.5 * u ** self.ay
        e = np.ones((3, 3), dtype=complex)
        e[1, 1] = self.e
        return (np.array([0.0, 0.5 - wx, 0.5 + wx, 1.0]) * PERIOD,
                np.array([0.0, 0.5 - wy, 0.5 + wy, 1.0]) * PERIOD, e)


def _field(case, seed):
    rs = np.random.RandomState(seed)
    cx, cy, eps, _, thick = _pillar_stack(rs, case["layers"])
    lam, th, ph = rs.uniform(450e-9, 700e-9), rs.uniform(1, 35), rs.uniform(1, 45)
    k0, t, p = 2 * math.pi / lam, math.radians(th), math.radians(ph)
    z = rs.uniform(0.1, 0.9) * (thick.sum() if case["plane"] == "xy" else PERIOD)
    return dict(nX=case["nx"], nY=case["ny"], coord_x=cx, coord_y=cy, thickness=thick, lam=lam,
                kx0=k0 * math.sin(t) * math.cos(p), ky0=k0 * math.sin(t) * math.sin(p), eps=eps,
                pol=_pols(th, ph)[0], component=case["component"], slice_type=case["plane"],
                coord=z, nres1=case["res"])


def _rows(count, seed):
    """Network inputs of `count` queries and smooth targets in [0, 1]."""
    x = surrogate.features(surrogate.sample_queries(count, seed))
    rs = np.random.RandomState(12)
    a = rs.standard_normal((x.shape[1], surrogate.N_OUT)) * 0.5
    t = 0.25 * (1.0 + np.sin(x[:, :32] @ a[:32])) * (0.5 + 0.5 * np.cos(x @ a * 0.3))
    return x, t.astype(np.float32)


def _net(case, seed):
    return surrogate.MLP(_context(), surrogate.N_FEAT, case["width"], case["depth"],
                         surrogate.N_OUT, case["members"], seed + 1)


def prepare(case, seed):
    kind = case["kind"]
    state = dict(kind=kind, case=case, ctx=_context(case.get("prec", "fp64")))
    if kind == "grating":
        state["args"] = _grating(case, seed)
    elif kind == "pillars":
        state["args"] = _pillars(case, seed)
    elif kind == "designs":
        state["args"] = surrogate.sample_geometries(case["count"], seed)
    elif kind == "uneven":
        state["args"] = _uneven(case, seed)
    elif kind == "relief":
        state["args"] = _Relief(seed)
    elif kind == "field":
        state["args"] = _field(case, seed)
    else:
        state["net"] = _net(case, seed)
        state["x"], state["t"] = _rows(case["rows"], seed)
        if kind == "predict":
            state["net"].set_precision(case["bf16"])
        elif kind == "train":
            state["net"].set_data(state["x"], state["t"])
    return state


def run(state):
    kind, ctx, a = state["kind"], state["ctx"], state.get("args")
    if kind == "grating":
        r = ofd.solve_ofd(ctx, **a)
        return {k: r[k] for k in ("R", "T", "REF", "TRN", "status")}
    if kind == "pillars":
        r = engine.solve_batch(ctx, **a)
        return dict(ref=r.ref, trn=r.trn, amp=r.amp, status=r.status)
    if kind == "designs":
        out, status = surrogate.solve_geometries(ctx, a)
        return dict(out=out, status=status)
    if kind == "uneven":
        r = engine.solve_uneven(ctx, a)
        return dict(ref=np.concatenate([q[0].ravel() for q in r]),
                    trn=np.concatenate([q[1].ravel() for q in r]),
                    status=np.array([q[2] for q in r]))
    if kind == "relief":
        return engine.rcwa_integrate(ctx, state["case"]["nx"], state["case"]["ny"], a, a.lam, 0.0,
                                     a.z1, state["case"]["slices"], a.kx0, a.ky0)
    if kind == "field":
        img, status = engine.field_image(ctx, **a)
        return dict(img=img, status=status)
    if kind == "predict":
        mean, err = state["net"].predict(state["x"])
        return dict(mean=mean, err=err)
    if kind == "train":
        loss = state["net"].train(state["case"]["epochs"], state["case"]["batch"], lr_max=1e-5)
        return dict(loss=loss, params=state["net"].get_params())
    loss, grad = state["net"].gradient(state["x"], state["t"])
    return dict(loss=loss, grad=grad)


def _layer_flops(h, eigs):
    """Complex work of one patterned layer: fe33's inverse, four products, and the eigen solve."""
    return (8.0 / 3 + 16) * h ** 3 + (100.0 * (2 * h) ** 3 if eigs else 0)


def _stack_flops(h, layers, count):
    """`count` solves of `layers` patterned layers between half-spaces: eigen solves and Q W,
    per interface two solves with n columns and the two products of the recursion."""
    n = 2 * h
    return count * (layers * (_layer_flops(h, True) + 8.0 * n ** 3) +
                    (layers + 1) * (2 * (8.0 / 3 + 8) + 24) * n ** 3)


def work(case):
    """Bytes: inputs read and results written.  Flops: the complex arithmetic of the method in
    real operations (100 n^3 for an eigen solve with vectors)."""
    kind = case["kind"]
    if kind == "grating":
        h, b = 2 * case["nx"] + 1, case["freqs"]
        return dict(bytes=b * (16.0 * (case["layers"] + 2) * (case["layers"] + 2) + 4 * 8 * h),
                    flops=_stack_flops(h, case["layers"], b))
    if kind == "pillars":
        h, b = (2 * case["nx"] + 1) * (2 * case["ny"] + 1), case["lams"] * case["dirs"]
        return dict(bytes=b * (4.0 * 8 * h + 8 * 16 * h + 88),
                    flops=_stack_flops(h, case["layers"], b))
    if kind == "designs":
        return dict(bytes=case["count"] * (4 * 9 * 16 + 88 + 8.0 * 36),
                    flops=_stack_flops(121, 2, case["count"]))
    if kind == "uneven":
        f = by = 0.0
        for i in range(case["count"]):
            h = (2 * (case["nmin"] + i % (case["nmax"] - case["nmin"] + 1)) + 1) ** 2
            f += _stack_flops(h, 1 + (5 * i) % case["layers"], 1)
            by += 4.0 * 8 * h + 16 * 8 * 20
        return dict(bytes=by, flops=f)
    if kind == "relief":
        h, s = (2 * case["nx"] + 1) * (2 * case["ny"] + 1), case["slices"]
        n = 2.0 * h
        # per slice: modes, the slab in the outer basis (about 30 n^3 complex) and a star product
        return dict(bytes=8 * 16 * n * n, flops=s * (_layer_flops(h, True) + 8 * n ** 3 +
                                                     8 * 14 * n ** 3 + 8 * 13 * n ** 3))
    if kind == "field":
        h = (2 * case["nx"] + 1) * (2 * case["ny"] + 1)
        return dict(bytes=16.0 * case["res"] ** 2, flops=_stack_flops(h, case["layers"], 1))
    w, nin, nout, m = case["width"], surrogate.N_FEAT, surrogate.N_OUT, case["members"]
    params = nin * w + w + (case["depth"] - 1) * (w * w + w) + w * nout + nout
    rows = case["rows"] * case.get("epochs", 1)
    if kind == "predict":
        return dict(bytes=4.0 * (rows * (nin + nout + 1) + m * params),
                    flops=2.0 * rows * m * params)
    return dict(bytes=4.0 * (rows * (nin + nout) + (3 if kind == "train" else 2) * m * params),
                flops=6.0 * rows * m * params)


# ---------------------------------------------------------------------------
# The same in plain numpy, 64 bits
# ---------------------------------------------------------------------------
def _fourier(edges, f, period, count):
    """Coefficients -(count-1)/2 .. (count-1)/2 of a piecewise constant function."""
    m = np.arange(count) - (count - 1) // 2
    mid, dx = 0.5 * (edges[1:] + edges[:-1]), np.diff(edges)
    e = np.exp(-2j * math.pi * np.outer(m, mid) / period) * np.sinc(np.outer(m, dx) / period)
    return e @ (np.asarray(f) * dx) / period


def _toeplitz(c):
    n = (len(c) + 1) // 2
    i = np.arange(n)
    return c[i[:, None] - i[None, :] + n - 1]


def _convolutions(cx, cy, g, nx, ny):
    """The three convolution matrices of a grid: inverse rule along x, along y, direct rule."""
    px, py = cx[-1] - cx[0], cy[-1] - cy[0]
    one = [_fourier(cy[i:i + 2], [1.0], py, 2 * ny - 1) for i in range(cy.size - 1)]
    f1 = sum(np.kron(np.linalg.inv(_toeplitz(_fourier(cx, 1.0 / g[i], px, 2 * nx - 1))),
                     _toeplitz(one[i])) for i in range(cy.size - 1))
    onx = [_fourier(cx[i:i + 2], [1.0], px, 2 * nx - 1) for i in range(cx.size - 1)]
    f2 = sum(np.kron(_toeplitz(onx[i]),
                     np.linalg.inv(_toeplitz(_fourier(cy, 1.0 / g[:, i], py, 2 * ny - 1))))
             for i in range(cx.size - 1))
    f3 = sum(np.kron(_toeplitz(_fourier(cx, g[i], px, 2 * nx - 1)), _toeplitz(one[i]))
             for i in range(cy.size - 1))
    return f1, f2, f3


def _root(v):
    """The root with a mode's decay or propagation along +z."""
    r = np.sqrt(np.asarray(v, dtype=complex))
    r = np.where(r.imag < 0, -r, r)
    return np.where((np.abs(r.imag) < np.abs(r.real)) & (r.real < 0), -r, r)


class _Modes:
    """Modes of one layer in units of k0: W, V, q, and the direct convolution matrix."""

    def __init__(self, cx, cy, eps, mu, kx, ky, nx, ny):
        h = nx * ny
        eye, kxd, kyd = np.eye(h), np.diag(kx), np.diag(ky)
        if np.all(eps == eps.flat[0]) and (mu is None or np.all(mu == mu.flat[0])):
            e, u = eps.flat[0], 1.0 if mu is None else mu.flat[0]
            f1 = f2 = self.f3 = e * eye
            g1 = g2 = g3 = u * eye
            self.W = np.eye(2 * h, dtype=complex)
            self.q = np.tile(_root(e * u - kx * kx - ky * ky), 2)
        else:
            f1, f2, self.f3 = _convolutions(cx, cy, eps, nx, ny)
            g1, g2, g3 = (eye, eye, eye) if mu is None else _convolutions(cx, cy, mu, nx, ny)
            self.W = None
        ex, ey = np.linalg.solve(self.f3, kxd), np.linalg.solve(self.f3, kyd)
        mx, my = np.linalg.solve(g3, kxd), np.linalg.solve(g3, kyd)
        P = np.block([[kxd @ ey, g2 - kxd @ ex], [kyd @ ey - g1, -kyd @ ex]])
        Q = np.block([[-kxd @ my, kxd @ mx - f2], [f1 - kyd @ my, kyd @ mx]])
        if self.W is None:
            d, self.W = np.linalg.eig(P @ Q)
            self.q = _root(d)
        self.V = Q @ self.W / self.q


def _kvec(nX, nY, px, py, lam, kx0, ky0):
    k0 = 2 * math.pi / lam
    m = np.repeat(np.arange(-nX, nX + 1), 2 * nY + 1)
    n = np.tile(np.arange(-nY, nY + 1), 2 * nX + 1)
    return k0, (kx0 + 2 * math.pi * m / px) / k0, (ky0 + 2 * math.pi * n / py) / k0


def _reflect(modes, thick, k0):
    """Per interface, from the exit side: (upper-side matrix S of the transmitted amplitudes,
    reflection at the upper layer's bottom, reflection at the lower layer's top)."""
    out = []
    R = np.zeros_like(modes[-1].W)
    for a, b, t in zip(modes[-2::-1], modes[:0:-1], thick[:0:-1]):
        ph = np.exp(1j * b.q * k0 * t)
        Rt = ph[:, None] * R * ph[None, :]
        e = np.linalg.solve(a.W, b.W + b.W @ Rt)
        m = np.linalg.solve(a.V, b.V - b.V @ Rt)
        S = 0.5 * (e + m)
        R = np.linalg.solve(S.T, 0.5 * (e - m).T).T
        out.append((S, R, Rt))
    return out[::-1]


def _amplitudes(modes, thick, k0, c):
    """Downward amplitudes at each layer's top, upward ones there and the reflections at the
    layers' bottoms, for the incident c (at the bottom of the first layer)."""
    steps = _reflect(modes, thick, k0)
    down, up, d = [c], [steps[0][1] @ c], c
    for j, (S, _, Rt) in enumerate(steps):
        d = np.linalg.solve(S, d)
        down.append(d)
        up.append(Rt @ d)
        d = np.exp(1j * modes[j + 1].q * k0 * thick[j + 1])[:, None] * d
    return down, up, [R for _, R, _ in steps]


def _stack_modes(nX, nY, cx, cy, eps, mu, kx, ky):
    return [_Modes(cx, cy, e, None if mu is None else mu[i], kx, ky, 2 * nX + 1, 2 * nY + 1)
            for i, e in enumerate(eps)]


def _one(nX, nY, cx, cy, thick, lam, kx0, ky0, eps, pols, mu=None):
    """(ref, trn, amp) of one stack."""
    k0, kx, ky = _kvec(nX, nY, cx[-1] - cx[0], cy[-1] - cy[0], lam, kx0, ky0)
    h = kx.size
    c = np.zeros((2 * h, 2), dtype=complex)
    c[h // 2, 0] = c[h + h // 2, 1] = 1.0
    modes = _stack_modes(nX, nY, cx, cy, eps, mu, kx, ky)
    down, up, _ = _amplitudes(modes, thick, k0, c)
    amp = np.stack([up[0][:h], up[0][h:], down[-1][:h], down[-1][h:]], 0).transpose(2, 0, 1)
    half = [eps[0].flat[0], eps[-1].flat[0]]
    if mu is not None:
        half = [half[0] * mu[0].flat[0], half[1] * mu[-1].flat[0]]
    kz = [np.sqrt(e - kx * kx - ky * ky + 0j) for e in half]
    out = []
    for p in pols:
        a = p[0] * amp[0] + p[1] * amp[1]
        row = []
        for i in (0, 1):
            x, y = a[2 * i], a[2 * i + 1]
            s = abs(x) ** 2 + abs(y) ** 2 + abs((kx * x + ky * y) / kz[i]) ** 2
            row.append(abs(kz[i].real) * s / abs(kz[0][h // 2].real))
        out.append(row)
    out = np.array(out)
    return out[:, 0], out[:, 1], amp


def _exact_grating(a):
    nx, per, out = a["nX"], a["period"], []
    L = a["layers"]
    cx = np.array(sorted({0.0, per, *[q["fill"] * per for q in L]}))
    cy = np.array([0.0, per])
    xc = 0.5 * (cx[1:] + cx[:-1])
    thick = np.array([q["thickness"] for q in L])
    for f in a["freqs"]:
        w, lam = 2 * math.pi * f, C0 / f
        eps = []
        for i, q in enumerate(L):
            e = complex(q["eps1"], q.get("eps1i", 0.0))
            if (i, 1) in a["poles"]:
                e = sum((ae * ae / (ce * ce - w * w - 1j * be * w)
                         for _, ae, be, ce in a["poles"][(i, 1)]), a["poles"][(i, 1)][-1][0])
            eps.append(np.where(xc < q["fill"] * per, e, q["eps2"])[None, :])
        k0, t, p = 2 * math.pi / lam, math.radians(a["theta"]), math.radians(a["phi"])
        pols = _pols(a["theta"], a["phi"])
        kx0, ky0 = k0 * math.sin(t) * math.cos(p), k0 * math.sin(t) * math.sin(p)
        ref, trn, _ = _one(nx, 0, cx, cy, thick, lam, kx0, ky0, eps, pols)
        _, kx, ky = _kvec(nx, 0, per, per, lam, kx0, ky0)
        kt = kx * kx + ky * ky
        out.append((ref.sum(1), trn.sum(1), np.where(kt < 1.0, ref, 0.0),
                    np.where(kt < EPS_SUB, trn, 0.0)))
    R, T, REF, TRN = (np.array(v) for v in zip(*out))
    return dict(R=R, T=T, REF=REF, TRN=TRN, status=None)


def _exact_relief(case, s):
    N, z1 = case["slices"], s.z1
    dz = z1 / N
    k0, kx, ky = _kvec(case["nx"], case["ny"], PERIOD, PERIOD, s.lam, s.kx0, s.ky0)
    zs = [z1] + [(i + 0.5) * dz for i in range(N)][::-1] + [0.0]      # top to bottom
    modes = [_Modes(*s(z), None, kx, ky, 2 * case["nx"] + 1, 2 * case["ny"] + 1) for z in zs]
    thick = np.array([0.0] + [dz] * N + [0.0])
    c = np.eye(2 * kx.size, dtype=complex)
    res = dict(status=None)
    down, up, _ = _amplitudes(modes, thick, k0, c)
    res["Rud"], res["Tdd"] = up[0], down[-1]
    down, up, _ = _amplitudes(modes[::-1], thick[::-1], k0, c)
    res["Rdu"], res["Tuu"] = up[0], down[-1]
    for i, m in ((1, modes[0]), (0, modes[-1])):
        res["W%d" % i], res["V%d" % i], res["gam%d" % i] = m.W, m.V, m.q * k0 ** 2
    return res


def _exact_field(a):
    cx, cy, thick = a["coord_x"], a["coord_y"], a["thickness"]
    nX, nY, comp = a["nX"], a["nY"], a["component"]
    k0, kx, ky = _kvec(nX, nY, PERIOD, PERIOD, a["lam"], a["kx0"], a["ky0"])
    h = kx.size
    c = np.zeros((2 * h, 1), dtype=complex)
    c[h // 2, 0], c[h + h // 2, 0] = a["pol"]
    modes = _stack_modes(nX, nY, cx, cy, a["eps"], None, kx, ky)
    down, _, bottom = _amplitudes(modes, thick, k0, c)
    tops = np.concatenate([[0.0], np.cumsum(thick[1:-1])])

    def harmonics(z):
        j = next(i for i in range(1, len(thick) - 1) if z <= tops[i])
        m, zt = modes[j], z - tops[j - 1]
        ph = np.exp(1j * m.q * k0 * zt)
        back = np.exp(1j * m.q * k0 * (thick[j] - zt))
        # the upward amplitudes at the layer's bottom, so that nothing grows
        u = ph * down[j][:, 0]
        d = back * (bottom[j] @ (np.exp(1j * m.q * k0 * thick[j]) * down[j][:, 0]))
        E, H = m.W @ (u + d), m.V @ (u - d)
        return {"Ex": E[:h], "Ey": E[h:], "Hx": H[:h], "Hy": H[h:],
                "Hz": 1j * (kx * E[h:] - ky * E[:h]) / k0,
                "Ez": 1j * k0 * np.linalg.solve(m.f3, kx * H[h:] - ky * H[:h])}[comp].reshape(
                    2 * nX + 1, 2 * nY + 1)

    mx, my = np.arange(-nX, nX + 1), np.arange(-nY, nY + 1)
    fx = lambda x: np.exp(1j * np.outer(x, 2 * math.pi * mx / PERIOD + a["kx0"]))   # noqa: E731
    fy = lambda y: np.exp(1j * np.outer(y, 2 * math.pi * my / PERIOD + a["ky0"]))   # noqa: E731
    n1 = a["nres1"]
    deep = PERIOD if a["slice_type"] == "xy" else thick.sum()
    n2 = max(1, int(n1 * deep / PERIOD))
    a1, a2 = (np.arange(n1) + 0.5) * PERIOD / n1, (np.arange(n2) + 0.5) * deep / n2
    if a["slice_type"] == "xy":
        return dict(img=fy(a2) @ harmonics(a["coord"]).T @ fx(a1).T, status=None)
    rows = []
    for z in a2:
        H2 = harmonics(z)
        rows.append(fx(a1) @ (H2 @ fy([a["coord"]])[0]) if a["slice_type"] == "xz"
                    else fy(a1) @ (H2.T @ fx([a["coord"]])[0]))
    return dict(img=np.array(rows), status=None)


def _layers_of(case, flat):
    """(weight, bias) of each layer of one member: per layer the weights (in, out), the bias."""
    nin, w, out, at = surrogate.N_FEAT, case["width"], [], 0
    sizes = [(nin, w)] + [(w, w)] * (case["depth"] - 1) + [(w, surrogate.N_OUT)]
    for i, o in sizes:
        out.append((flat[at:at + i * o].reshape(i, o), flat[at + i * o:at + i * o + o]))
        at += i * o + o
    return out


def _forward(case, flat, x):
    layers = _layers_of(case, flat)
    for k, (w, b) in enumerate(layers):
        x = x @ w + b
        if k + 1 < len(layers):
            x = 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))
    return x


def _exact_net(case, seed):
    net = _net(case, seed)
    p = torch.from_numpy(net.get_params().astype(np.float64)).cuda()
    net.close()
    x, t = (torch.from_numpy(v.astype(np.float64)).cuda() for v in _rows(case["rows"], seed))
    if case["kind"] == "predict":
        y = torch.stack([_forward(case, q, x) for q in p])
        return dict(mean=y.mean(0), err=(y.amax(0) - y.amin(0)).amax(1))
    loss, grad = [], []
    for q in p:
        q = q.clone().requires_grad_(True)
        v = ((_forward(case, q, x) - t) ** 2).mean()
        v.backward()
        loss.append(v.detach())
        grad.append(q.grad)
    return dict(loss=torch.stack(loss), grad=torch.stack(grad))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("predict", "gradient"):
        return _exact_net(case, seed)
    # the rows of a training step are in an order that the library draws
    if kind == "train":
        return None
    # numpy takes some 20 s for this much
    if work(case)["flops"] > 5e11:
        return None
    a = prepare(case, seed)["args"]
    if kind == "grating":
        return _exact_grating(a)
    if kind == "relief":
        return _exact_relief(case, a)
    if kind == "field":
        return _exact_field(a)
    if kind == "pillars":
        q = [_one(a["nX"], a["nY"], a["coord_x"], a["coord_y"], a["thickness"], a["lam"][i],
                  a["kx0"][i], a["ky0"][i], a["eps"], a["pols"][i], a["mu"])
             for i in range(a["lam"].size)]
        ref, trn, amp = (np.array(v) for v in zip(*q))
        return dict(ref=ref, trn=trn, amp=amp, status=None)
    if kind == "designs":
        s = surrogate.stack_arrays(a)
        k, out = surrogate.ORDER_IDX, []
        for i in range(a.shape[0]):
            r, t, _ = _one(surrogate.NX, surrogate.NY, s["edges"][i], s["edges"][i],
                           s["thickness"][i], s["lam"][i], s["kx0"][i], s["ky0"][i], s["eps"][i],
                           s["pols"][i])
            out.append(np.concatenate([r[:, k], t[:, k]], 1))
        return dict(out=np.array(out), status=None)
    q = [_one(s["nX"], s["nY"], s["coord_x"], s["coord_y"], s["thickness"], s["lam"], s["kx0"],
              s["ky0"], s["eps"], s["pol"]) for s in a]
    return dict(ref=np.concatenate([v[0].ravel() for v in q]),
                trn=np.concatenate([v[1].ravel() for v in q]), status=None)
