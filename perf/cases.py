"""Workloads of the S-matrix framework, for measuring it on one MI355X.

Every case goes through the package's public Python entry points, as a program that designs
metasurfaces, gratings or waveguide parts calls them. Kinds:

  sweep     one ``batch_stack_rcwa`` call over several stacks of rectangle layers (one wavelength
            each) between homogeneous half-spaces; with ``efficiencies`` followed by
            ``stack_efficiencies`` for a plane wave at normal incidence
  mixed     one ``batch_stack_rcwa_mixed`` call over stacks of different harmonic counts
  gradient  ``batch_stack_rcwa(tape=True)`` and the permittivity cotangent of every slab cell
  rcwa      ``RCWAIntegrator.compute`` on a z-dependent cell (``VarLayerSampler``), PML or periodic
  varrcwa   ``RedhefferIntegrator.compute`` (adaptive trisection) on the same samplers
  fourier   ``assemble_toeplitz`` of pixel-grid layers

S-matrices between homogeneous half-spaces are in the harmonic basis and are returned as they
are. The integrators' S-matrices are in the bases of the end media, whose columns an eigensolver
may order and scale as it likes, so those cases return the field transforms W1 Tuu W0^-1,
W0 Tdd W1^-1, W0 Rdu W0^-1 and W1 Rud W1^-1, which a program compares or plots.

``exact`` restates the formulas (Fourier convolution rules, P and Q, eigen-system, slab
S-matrix, star product, projections, trisection) in 64-bit torch on the CPU.
"""
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

CELL = 0.6  # period of the rectangle stacks, um
PI = 3.1415926535897932


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: one wavelength of a three-layer grating at 5 x 5 harmonics (a unit
        # test, an interactive look, one point of a line search); launches and latency count
        dict(name="one_stack_5x5", kind="sweep", nx=5, ny=5, stacks=1, layers=3, efficiencies=False),
        # a spectrum at few harmonics with its diffraction efficiencies: 64 wavelengths x 10 layers
        dict(name="spectrum_7x7_64", kind="sweep", nx=7, ny=7, stacks=64, layers=10, efficiencies=True),
        # a spectrum at the usual working resolution, 11 x 11
        dict(name="spectrum_11x11_48", kind="sweep", nx=11, ny=11, stacks=48, layers=10, efficiencies=False),
        # a short sweep at 15 x 15: the eigensolver launches do not fill the chip
        dict(name="sweep_15x15_8", kind="sweep", nx=15, ny=15, stacks=8, layers=10, efficiencies=False),
        # one design point at full resolution: one stack, 10 slabs, 21 x 21 (N = 882)
        dict(name="one_stack_21x21", kind="sweep", nx=21, ny=21, stacks=1, layers=10, efficiencies=False),
        # the largest: a batch of stacks at 21 x 21, 250 slabs
        dict(name="sweep_21x21_25", kind="sweep", nx=21, ny=21, stacks=25, layers=10, efficiencies=False),
        # a grating with unequal orders in x and y and an odd number of stacks and layers
        dict(name="grating_27x5_13", kind="sweep", nx=27, ny=5, stacks=13, layers=7, efficiencies=False),
        # a convergence study or adaptive resolution: harmonic counts mixed in one call
        dict(name="mixed_orders_24", kind="mixed", orders="7,11,15", stacks=24, layers=10),
        # inverse design: S and the gradient with respect to every cell of 10 x 10 grayscale slabs
        dict(name="gradient_11x11_6", kind="gradient", nx=11, ny=11, stacks=6, layers=10, grid=10),
        # a PML waveguide taper, plain RCWA with 24 slices at 9 x 7
        dict(name="rcwa_taper_9x7", kind="rcwa", nx=9, ny=7, pml=True, slices=24),
        # the adaptive method on a periodic pillar whose width changes with z, 9 x 9
        dict(name="varrcwa_pillar_9x9", kind="varrcwa", nx=9, ny=9, pml=False, pe=1e-2),
        # convolution matrices of 64 pixel-grid layers (freeform designs, 256 x 256)
        dict(name="pixels_256_11x11", kind="fourier", nx=11, ny=11, layers=64, grid=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _odd(rng, lo, hi):
    """An odd harmonic count in [lo, hi], spread over the logarithm."""
    return 2 * ((_log_int(rng, lo, hi) - 1) // 2) + 1


def draw(rng):
    """One more case of the ranges above; its cost stays below the 250 slabs at N = 882."""
    kind = rng.choice(["sweep", "sweep", "sweep", "mixed", "gradient", "rcwa", "varrcwa", "fourier"])
    if kind == "sweep":
        nx, ny = _odd(rng, 5, 23), _odd(rng, 5, 21)
        layers = _log_int(rng, 2, 30)
        N = 2 * nx * ny
        # slab budget: fewer slabs where a slab costs more; at most 640, and small problems are
        # bounded by latency rather than by N^3
        most = min(640, 0.5 * 250 * (882.0 / max(N, 200)) ** 3)
        stacks = max(1, min(_log_int(rng, 1, 96), int(most / layers)))
        return dict(kind="sweep", nx=nx, ny=ny, stacks=stacks, layers=layers, efficiencies=rng.random() < 0.3)
    if kind == "mixed":
        orders = ",".join(str(o) for o in sorted(rng.sample([5, 7, 9, 11, 13, 15], 3)))
        return dict(kind="mixed", orders=orders, stacks=_log_int(rng, 5, 40), layers=_log_int(rng, 3, 10))
    if kind == "gradient":
        return dict(kind="gradient", nx=_odd(rng, 5, 15), ny=_odd(rng, 5, 11), stacks=_log_int(rng, 1, 8),
                    layers=_log_int(rng, 3, 12), grid=rng.randint(4, 16))
    if kind == "rcwa":
        return dict(kind="rcwa", nx=_odd(rng, 5, 13), ny=_odd(rng, 5, 11), pml=rng.random() < 0.5,
                    slices=_log_int(rng, 4, 48))
    if kind == "varrcwa":
        return dict(kind="varrcwa", nx=_odd(rng, 5, 11), ny=_odd(rng, 5, 9), pml=rng.random() < 0.5,
                    pe=rng.choice([1e-2, 2e-2, 5e-3]))
    return dict(kind="fourier", nx=_odd(rng, 5, 21), ny=_odd(rng, 5, 21), layers=_log_int(rng, 2, 64),
                grid=rng.choice([32, 50, 64, 100, 128, 256]))


# ------------------------------------------------------------------ inputs from the seed
def _rectangles(rng):
    """One layer: 1 to 4 rectangles of eps 4 or 12.25 in air, periodically wrapped, on an exact grid."""
    xs, ys, pieces = {0.0, CELL}, {0.0, CELL}, []
    for _ in range(int(rng.integers(1, 5))):
        w, h = rng.uniform(0.05, 0.3, 2)
        x0, y0 = rng.uniform(0.0, CELL, 2)
        e = (4.0, 12.25)[int(rng.integers(0, 2))]
        for dx in (0.0, -CELL):
            for dy in (0.0, -CELL):
                a, b = max(x0 + dx, 0.0), min(x0 + w + dx, CELL)
                c, d = max(y0 + dy, 0.0), min(y0 + h + dy, CELL)
                if b > a and d > c:
                    pieces.append((a, b, c, d, e))
                    xs.update([a, b])
                    ys.update([c, d])
    x, y = np.array(sorted(xs)), np.array(sorted(ys))
    eps = np.ones((y.size - 1, x.size - 1), complex)
    xm, ym = 0.5 * (x[1:] + x[:-1]), 0.5 * (y[1:] + y[:-1])
    for a, b, c, d, e in pieces:
        eps[np.ix_((ym > c) & (ym < d), (xm > a) & (xm < b))] = e
    return x, y, eps


def _grayscale(rng, grid):
    """One layer of a design under optimisation: grid x grid cells of eps between 1 and 4."""
    x = np.linspace(0.0, CELL, grid + 1)
    return x, x.copy(), rng.uniform(1.0, 4.0, (grid, grid)) + 0j


def _stacks(case, seed):
    """The stacks as plain data: substrate of eps 2.1 below, air above, wavelengths in 0.8 .. 1.6 um."""
    rng = np.random.default_rng(seed)
    edge = np.array([0.0, CELL])
    out = []
    for _ in range(case["stacks"]):
        layer = (lambda: _grayscale(rng, case["grid"])) if case["kind"] == "gradient" else (lambda: _rectangles(rng))
        out.append(dict(lam=float(rng.uniform(0.8, 1.6)), layers=[layer() for _ in range(case["layers"])],
                        thickness=[float(t) for t in rng.uniform(0.05, 0.2, case["layers"])],
                        bottom=(edge, edge, np.array([[2.1 + 0j]])), top=(edge, edge, np.array([[1.0 + 0j]]))))
    return out


def _orders(case, count):
    o = [int(v) for v in case["orders"].split(",")]
    return [(o[i % len(o)],) * 2 for i in range(count)]


def _cell(case, seed):
    """The z-dependent cells: a waveguide taper in PML (its core's right edge moves with z) or a
    periodic square pillar whose right edge follows a cosine. Returns lam, x, y, eps, {x index:
    rule}, z0, z1."""
    rng = np.random.default_rng(seed)
    j = rng.uniform(-1.0, 1.0, 3)
    if case["pml"]:
        x = np.array([0.0, 0.5, 1.5, 2.6, 3.7, 3.9, 5.0, 5.5])
        y = np.array([0.0, 0.5, 1.5, 1.58, 1.8, 2.8, 3.3])
        eps = np.full((6, 7), 1.445 ** 2 + 0j)
        eps[3, 2] = 3.48 ** 2
        a, b = 2.6 + 0.02 * j[0], 3.6 + 0.02 * j[1]
        return (1.55 + 0.02 * j[2], x, y, eps,
                {3: lambda z: a if z < 0.0 else b if z > 4.0 else a + (b - a) * 0.25 * z}, -0.1, 4.1)
    x = np.array([0.0, 0.1, 0.5, 0.65])
    eps = np.ones((3, 3), complex)
    eps[1, 1] = 3.48 ** 2
    w, s = 0.3 + 0.01 * j[0], 0.2 + 0.01 * j[1]
    return (1.55 + 0.02 * j[2], x, x.copy(), eps,
            {2: lambda z: w + s if z <= 1.0 else s * math.cos(0.5 * PI * (z - 1.0)) + w}, 0.0, 2.0)


def _pixels(case, seed):
    """Freeform layers: smooth random patterns thresholded to eps 12.25 in 1 on a grid x grid map."""
    rng = np.random.default_rng(seed)
    g = case["grid"]
    c = (np.arange(g) + 0.5) / g
    x = np.linspace(0.0, CELL, g + 1)
    k = np.arange(1, 4)
    layers = []
    for _ in range(case["layers"]):
        a = np.sin(2 * PI * (np.outer(c, k) + rng.uniform(0, 1, 3)))
        b = np.sin(2 * PI * (np.outer(c, k) + rng.uniform(0, 1, 3)))
        layers.append((x, x.copy(), np.where(a @ rng.normal(size=(3, 3)) @ b.T > 0.0, 12.25 + 0j, 1.0 + 0j)))
    return layers


def _cotangent(case, seed):
    g = np.random.default_rng(seed + 1)
    N = 2 * case["nx"] * case["ny"]
    # the zeroth order of the transmitted blocks, as the usual objectives weigh it
    bar = np.zeros((case["stacks"], 4, N, N), complex)
    c = (N // 2 - 1) // 2
    for i in (c, c + N // 2):
        for k in (c, c + N // 2):
            bar[:, :, i, k] = g.normal(size=(case["stacks"], 4)) + 1j * g.normal(size=(case["stacks"], 4))
    return bar


def prepare(case, seed):
    from varrcwa_amd import api

    ctx = api.default_context()
    kind = case["kind"]
    s = dict(case=case, api=api, ctx=ctx)
    if kind in ("sweep", "mixed", "gradient"):
        s["stacks"] = [dict(i, layers=[api.Layer(*l) for l in i["layers"]], bottom=api.Layer(*i["bottom"]),
                            top=api.Layer(*i["top"])) for i in _stacks(case, seed)]
    if kind == "mixed":
        s["orders"] = _orders(case, case["stacks"])
    if kind == "gradient":
        s["bar"] = torch.from_numpy(_cotangent(case, seed)).cuda()
    if kind == "sweep" and case["efficiencies"]:
        n = case["nx"] * case["ny"]
        s["e_inc"] = torch.zeros((case["stacks"], 2 * n), dtype=torch.complex128, device="cuda")
        s["e_inc"][:, n // 2] = 1.0
    if kind in ("rcwa", "varrcwa"):
        lam, x, y, eps, rules, s["z0"], s["z1"] = _cell(case, seed)
        s["sampler"] = api.VarLayerSampler(lam, case["nx"], case["ny"], x, y, eps, case["pml"], ctx=ctx)
        for k, f in rules.items():
            s["sampler"].addXRule(k, f)
    if kind == "fourier":
        s["layers"] = [api.Layer(*l) for l in _pixels(case, seed)]
    return s


def _transforms(W0, W1, Tdd, Tuu, Rud, Rdu):
    """The S-matrix between field harmonics instead of modes (numpy)."""
    a = np.linalg.solve(W0.T, np.concatenate([W1 @ Tuu, W0 @ Rdu]).T).T
    b = np.linalg.solve(W1.T, np.concatenate([W0 @ Tdd, W1 @ Rud]).T).T
    n = W0.shape[0]
    return dict(Tuu=a[:n], Rdu=a[n:], Tdd=b[:n], Rud=b[n:])


def run(s):
    api, ctx, case = s["api"], s["ctx"], s["case"]
    kind = case["kind"]
    if kind == "sweep":
        out = api.batch_stack_rcwa(ctx, case["nx"], case["ny"], s["stacks"], want_bases=case["efficiencies"])
        if not case["efficiencies"]:
            return dict(S=out["S"])
        ref, trn = api.stack_efficiencies(ctx, case["nx"], case["ny"], s["stacks"], out, s["e_inc"])
        return dict(S=out["S"], ref=ref, trn=trn)
    if kind == "mixed":
        return api.batch_stack_rcwa_mixed(ctx, s["orders"], s["stacks"])["S"]
    if kind == "gradient":
        out = api.batch_stack_rcwa(ctx, case["nx"], case["ny"], s["stacks"], tape=True)
        eps_bar = out["tape"].vjp(s["bar"])
        out["tape"].close()
        return dict(S=out["S"], eps_bar=eps_bar)
    if kind == "fourier":
        return api.assemble_toeplitz(ctx, case["nx"], case["ny"], s["layers"])
    if kind == "rcwa":
        it = api.RCWAIntegrator(s["z0"], s["z1"], s["sampler"])
        it.compute(case["slices"])
    else:
        it = api.RedhefferIntegrator(s["z0"], s["z1"], s["sampler"])
        it.compute(0, pe=case["pe"])
    return _transforms(it.W0(), it.W1(), it.Tdd(), it.Tuu(), it.Rud(), it.Rdu())


# ------------------------------------------------------------------ what the path cannot do without
def _slab_flops(N):
    """Real flops of one slab: eigen-system (Hessenberg, Schur form, vectors) 316/3 N^3, P and Q
    about 6, W^-1 W0 and V^-1 V0 20, slab S-matrix 64/3, star product 248/3."""
    return 235.0 * float(N) ** 3


def work(case):
    kind = case["kind"]
    if kind == "fourier":
        cells, n = case["layers"] * case["grid"] ** 2, case["nx"] * case["ny"]
        g = case["grid"]
        return {"bytes": 16.0 * cells + 48.0 * n * n * case["layers"], "flops": 5.0 * 2 * cells * 2 * math.log2(g)}
    if kind == "mixed":
        Ns = [2 * a * b for a, b in _orders(case, case["stacks"])]
        return {"bytes": sum(64.0 * N * N for N in Ns), "flops": sum(case["layers"] * _slab_flops(N) for N in Ns)}
    N = 2 * case["nx"] * case["ny"]
    if kind in ("rcwa", "varrcwa"):
        # varrcwa: of the order of ten reference systems over these lengths
        slabs = case["slices"] + 2 if kind == "rcwa" else 10
        return {"bytes": 64.0 * N * N, "flops": slabs * _slab_flops(N)}
    slabs = case["stacks"] * case["layers"]
    if kind == "gradient":
        return {"bytes": 128.0 * N * N * case["stacks"], "flops": 2.5 * slabs * _slab_flops(N)}
    return {"bytes": 64.0 * N * N * case["stacks"], "flops": slabs * _slab_flops(N)}


# ------------------------------------------------------------------ the same in 64 bits on the CPU
def _each(f, items):
    """f of every item, side by side: LAPACK's eigensolver runs on one core."""
    items, cores = list(items), torch.get_num_threads()
    if len(items) < 2 or cores < 2:
        return [f(i) for i in items]
    torch.set_num_threads(1)
    try:
        with ThreadPoolExecutor(cores, initializer=torch.set_num_threads, initargs=(1,)) as pool:
            return list(pool.map(f, items))
    finally:
        torch.set_num_threads(cores)


def _t(a):
    return torch.as_tensor(np.asarray(a), dtype=torch.complex128)


def _basis(x, M):
    """Row per order m = -(M-1)/2 ..: the Fourier coefficient of the indicator of every cell of x."""
    d = x[-1] - x[0]
    m = np.arange(M) - (M - 1) // 2
    w = (x[1:] - x[:-1]) / d
    return np.exp(-1j * PI * np.outer(m, x[1:] + x[:-1]) / d) * np.sinc(np.outer(m, w)) * w


def _toeplitz(v):
    n = (v.shape[-1] + 1) // 2
    return v[..., n - 1 + np.arange(n)[:, None] - np.arange(n)[None, :]]


def _convolution(x, y, eps, nx, ny):
    """fe11 (inverse rule along x), fe22 (inverse rule along y), fe33 (Laurent rule)."""
    m, k = np.repeat(np.arange(nx), ny), np.tile(np.arange(ny), nx)
    dm, dk = m[:, None] - m[None, :] + nx - 1, k[:, None] - k[None, :] + ny - 1
    bx, by = _t(_basis(x, 2 * nx - 1)), _t(_basis(y, 2 * ny - 1))
    ix = torch.linalg.inv(_toeplitz((1.0 / eps) @ bx.T))  # per y strip
    iy = torch.linalg.inv(_toeplitz((1.0 / eps).T @ by.T))  # per x cell
    fe11 = torch.einsum("ps,sac->pac", by, ix)[dk, m[:, None], m[None, :]]
    fe22 = torch.einsum("ps,sbd->pbd", bx, iy)[dm, k[:, None], k[None, :]]
    fe33 = (bx @ eps.T @ by.T)[dm, dk]
    return fe11, fe22, fe33


def _sinc(v):
    return np.sinc(v)


def _pml_side(b0, b1, L, n, sign):
    """Fourier coefficients of the complex coordinate stretch of one absorbing side."""
    g = 1.0 / (1.0 - 1.0j)
    w, c = (b1 - b0) / L, (b1 + b0) / L
    ph = np.exp(-1j * PI * n * c)
    r = (8.0 - 2.0 * g) * _sinc(n * w) * ph
    r = r + 4.0 * ph * (_sinc(n * w - 0.5) * np.exp(-0.5j * PI * sign) + _sinc(n * w + 0.5) * np.exp(0.5j * PI * sign))
    r = r + g * ph * (_sinc(n * w - 1.0) * np.exp(-1j * PI * sign) + _sinc(n * w + 1.0) * np.exp(1j * PI * sign))
    return r * w / 16.0


def _stretched(x, M):
    """Per order: the stretch profile along one axis whose first and last cells absorb."""
    L, n = x[-1] - x[0], np.arange(M) - (M - 1) // 2
    mid = (x[-2] - x[1]) / L * _sinc(n * (x[-2] - x[1]) / L) * np.exp(-1j * PI * n * (x[1] + x[-2]) / L)
    return mid + _pml_side(x[0], x[1], L, n, 1.0) + _pml_side(x[-2], x[-1], L, n, -1.0)


def _k_matrices(x, y, nx, ny, pml):
    kx = 2 * PI / (x[-1] - x[0]) * (np.repeat(np.arange(nx), ny) - (nx - 1) // 2)
    ky = 2 * PI / (y[-1] - y[0]) * (np.tile(np.arange(ny), nx) - (ny - 1) // 2)
    if not pml:
        return _t(np.diag(kx)), _t(np.diag(ky))
    m, k = np.repeat(np.arange(nx), ny), np.tile(np.arange(ny), nx)
    dm, dk = m[:, None] - m[None, :] + nx - 1, k[:, None] - k[None, :] + ny - 1
    fx, fy = _stretched(x, 2 * nx - 1)[dm] * (dk == ny - 1), _stretched(y, 2 * ny - 1)[dk] * (dm == nx - 1)
    return _t(fx * kx[None, :]), _t(fy * ky[None, :])


def _pq(x, y, eps, nx, ny, lam, Kx, Ky):
    fe11, fe22, fe33 = _convolution(x, y, eps, nx, ny)
    F = torch.linalg.solve(fe33, torch.cat([Ky, -Kx], 1))
    k2 = (2 * PI / lam) ** 2
    n = nx * ny
    eye = k2 * torch.eye(n, dtype=torch.complex128)
    z = torch.zeros_like(eye)
    P = torch.cat([Kx @ F, Ky @ F]) + torch.cat([torch.cat([z, eye], 1), torch.cat([-eye, z], 1)])
    Q = torch.cat([torch.cat([-Kx @ Ky, Kx @ Kx - k2 * fe22], 1), torch.cat([k2 * fe11 - Ky @ Ky, Ky @ Kx], 1)])
    return P, Q


def _branch(lam):
    g = torch.sqrt(lam)
    g = torch.where(g.imag < 0, -g, g)
    return torch.where((g.imag.abs() < g.real.abs()) & (g.real < 0), -g, g)


def _modes(P, Q):
    lam, W = torch.linalg.eig(P @ Q)
    gam = _branch(lam)
    return W, (Q @ W) / gam, gam


def _free_modes(eps, lam, kx, ky):
    """W = I, V, gamma of a homogeneous medium."""
    k2 = (2 * PI / lam) ** 2
    g = _branch(_t(k2 * (k2 * eps - kx ** 2 - ky ** 2)))
    V = torch.cat([torch.cat([torch.diag(_t(-kx * ky) / g), torch.diag(_t(kx * kx - k2 * eps) / g)], 1),
                   torch.cat([torch.diag(_t(k2 * eps - ky * ky) / g), torch.diag(_t(kx * ky) / g)], 1)])
    return torch.eye(2 * kx.size, dtype=torch.complex128), V, torch.cat([g, g])


def _slab(W, V, gam, s, W0, V0):
    X = torch.exp(1j * gam * s)[:, None]
    F, G = torch.linalg.solve(W, W0), torch.linalg.solve(V, V0)
    A, B = F + G, F - G
    even = torch.linalg.solve(A - X * B, X * A - B)
    odd = torch.linalg.solve(A + X * B, X * A + B)
    return 0.5 * (even + odd), 0.5 * (even - odd)  # Tuu, Rud


def _star(S, t):
    Tdd, Tuu, Rud, Rdu = S
    tdd, tuu, rud, rdu = t
    M = torch.eye(Tdd.shape[0], dtype=torch.complex128) - Rud @ rdu
    Y = torch.linalg.solve(M, torch.cat([Tuu, Rud], 1))
    n = Tdd.shape[0]
    Yt, Yr = Y[:, :n], Y[:, n:]
    K = Yr @ tdd
    return Tdd @ (tdd + rdu @ K), tuu @ Yt, rud + tuu @ K, Rdu + Tdd @ (rdu @ Yt)


def _ab(W, V, W0, V0):
    a, b = torch.linalg.solve(W, W0), torch.linalg.solve(V, V0)
    return 0.5 * (a + b), 0.5 * (a - b)


def _project_left(S, A, B):
    Tdd, Tuu, Rud, Rdu = S
    n = Tdd.shape[0]
    sol = torch.linalg.solve(A - Rdu @ B, torch.cat([Rdu @ A - B, Tdd], 1))
    rdu, tdd = sol[:, :n], sol[:, n:]
    return tdd, Tuu @ (B @ rdu + A), Rud + Tuu @ (B @ tdd), rdu


def _solve_stack(inst, nx, ny, eps_list=None, alone=False):
    Kx, Ky = _k_matrices(np.array([0.0, CELL]), np.array([0.0, CELL]), nx, ny, False)
    kx, ky = Kx.diagonal().real.numpy(), Ky.diagonal().real.numpy()
    lam = inst["lam"]
    W0, V0, _ = _free_modes(inst["bottom"][2][0, 0], lam, kx, ky)
    W1, V1, _ = _free_modes(inst["top"][2][0, 0], lam, kx, ky)

    def slab(i):
        x, y, eps = inst["layers"][i]
        e = _t(eps) if eps_list is None else eps_list[i]
        return _slab(*_modes(*_pq(x, y, e, nx, ny, lam, Kx, Ky)), inst["thickness"][i] * lam / (2 * PI), W1, V1)

    S = None
    for t, r in (_each if alone else map)(slab, range(len(inst["layers"]))):
        S = (t, t, r, r) if S is None else _star(S, (t, t, r, r))
    S = _project_left(S, *_ab(W1, V1, W0, V0))
    return torch.stack([b.T for b in S]), (kx, ky)  # column-major storage, as the library returns it


def _efficiencies(S, inst, kx, ky, e_inc):
    k0 = 2 * PI / inst["lam"]
    n = kx.size

    def power(f, eps, sign):
        kz = sign * np.sqrt(k0 * k0 * eps - kx * kx - ky * ky + 0j)
        ez = (kx * f[:n] + ky * f[n:]) / kz
        return np.abs(kz.real) / (math.sqrt(eps.real) * k0) * (abs(f[:n]) ** 2 + abs(f[n:]) ** 2 + abs(ez) ** 2)

    r, t = (S[3].T @ e_inc).numpy(), (S[1].T @ e_inc).numpy()
    return power(r, inst["bottom"][2][0, 0], -1.0), power(t, inst["top"][2][0, 0], 1.0)


def _sampler(case, seed):
    lam, x, y, eps, rules, z0, z1 = _cell(case, seed)
    Kx, Ky = _k_matrices(x, y, case["nx"], case["ny"], case["pml"])

    def sample(z):
        xz = x.copy()
        for k, f in rules.items():
            xz[k] = f(z)
        return _pq(xz, y, _t(eps), case["nx"], case["ny"], lam, Kx, Ky)

    return lam, sample, z0, z1


def _rcwa(case, seed):
    lam, sample, z0, z1 = _sampler(case, seed)
    W1, V1, _ = _modes(*sample(z1))
    W0, V0, _ = _modes(*sample(z0))
    dz = (z1 - z0) / case["slices"]
    S = None
    for i in range(case["slices"]):
        t, r = _slab(*_modes(*sample(z0 + (i + 0.5) * dz)), dz * lam / (2 * PI), W1, V1)
        S = (t, t, r, r) if S is None else _star(S, (t, t, r, r))
    return W0, W1, _project_left(S, *_ab(W1, V1, W0, V0))


def _varrcwa(case, seed):
    """Trisection with the midpoint's modes as reference, first-order perturbation integrated by
    Simpson's rule, accepted where the largest perturbation entry is at most pe."""
    lam, sample, z0, z1 = _sampler(case, seed)
    k0 = 2 * PI / lam
    W0, V0, _ = _modes(*sample(z0))
    W1, V1, _ = _modes(*sample(z1))
    n = W0.shape[0]
    eye, zero = torch.eye(n, dtype=torch.complex128), torch.zeros((n, n), dtype=torch.complex128)
    S, left = (eye, eye, zero, zero), (W0, V0)

    def segment(ref, modes, a, b, pts):
        W, V, g = modes
        dA, dB = [], []
        for P, Q in pts:
            p, q = torch.linalg.solve(W, (P - ref[0]) @ V), torch.linalg.solve(V, (Q - ref[1]) @ W)
            dA.append(p + q)
            dB.append(p - q)
        ph, pf = torch.exp(0.5j * (b - a) / k0 * g), torch.exp(1j * (b - a) / k0 * g)
        H = 4.0 * ph[:, None] * ph[None, :]
        r, c, k = pf[:, None], pf[None, :], 1j * (b - a) / (12 * k0)
        parts = (k * (dA[0] * c + H * dA[1] + r * dA[2]), k * (r * dA[0] + H * dA[1] + dA[2] * c),
                 -k * (r * dB[0] * c + H * dB[1] + dB[2]), -k * (dB[0] + H * dB[1] + r * dB[2] * c))
        err = max(float(p.abs().max()) for p in parts)
        return (parts[0] + torch.diag(pf), parts[1] + torch.diag(pf), parts[2], parts[3]), err

    def grow(ref, modes, a, b, pts):
        nonlocal S, left
        T, err = segment(ref, modes, a, b, pts)
        if err <= case["pe"]:
            S = _star(S, _project_left(T, *_ab(modes[0], modes[1], *left)))
            left = modes[:2]
            return
        c, d = 2 / 3 * a + 1 / 3 * b, 1 / 3 * a + 2 / 3 * b
        first, last = sample(0.5 * (a + c)), sample(0.5 * (d + b))
        pc, pd = sample(c), sample(d)
        grow(first, _modes(*first), a, c, (pts[0], first, pc))
        grow(ref, modes, c, d, (pc, pts[1], pd))
        grow(last, _modes(*last), d, b, (pd, last, pts[2]))

    mid = sample(0.5 * (z0 + z1))
    grow(mid, _modes(*mid), z0, z1, (sample(z0), mid, sample(z1)))
    Tdd, Tuu, Rud, Rdu = S
    A, B = _ab(*left, W1, V1)
    sol = torch.linalg.solve(A - Rud @ B, torch.cat([Tuu, Rud @ A - B], 1))
    Tuu, Rud = sol[:, :n], sol[:, n:]
    return W0, W1, (Tdd @ (B @ Rud + A), Tuu, Rud, Rdu + Tdd @ (B @ Tuu))


def exact(case, seed):
    kind = case["kind"]
    # about 20 s of eight or more cores: ten slabs at N = 882
    if kind not in ("fourier", "rcwa", "varrcwa") and work(case)["flops"] > 11 * _slab_flops(882) * (
            2.5 if kind == "gradient" else 1.0):
        return None
    if kind == "fourier":
        out = [_convolution(x, y, _t(e), case["nx"], case["ny"]) for x, y, e in _pixels(case, seed)]
        return torch.stack([torch.stack([o[k].T for o in out]) for k in range(3)])
    if kind in ("rcwa", "varrcwa"):
        W0, W1, S = (_rcwa if kind == "rcwa" else _varrcwa)(case, seed)
        return _transforms(*[a.numpy() for a in (W0, W1, *S)])
    stacks = _stacks(case, seed)
    if kind == "mixed":
        return _each(lambda j: _solve_stack(j[0], *j[1])[0], zip(stacks, _orders(case, len(stacks))))
    if kind == "gradient":
        bar = _cotangent(case, seed)

        def one(k):
            eps = [_t(l[2]).requires_grad_(True) for l in stacks[k]["layers"]]
            S, _ = _solve_stack(stacks[k], case["nx"], case["ny"], eps)
            grads = torch.autograd.grad((torch.from_numpy(bar[k]).conj() * S).real.sum(), eps)
            return S.detach(), torch.cat([g.T.reshape(-1) for g in grads])

        out = _each(one, range(len(stacks)))
        return dict(S=torch.stack([o[0] for o in out]), eps_bar=torch.cat([o[1] for o in out]))
    if len(stacks) == 1:
        out = [_solve_stack(stacks[0], case["nx"], case["ny"], alone=True)]
    else:
        out = _each(lambda i: _solve_stack(i, case["nx"], case["ny"]), stacks)
    S = torch.stack([o[0] for o in out])
    if not case["efficiencies"]:
        return dict(S=S)
    e = torch.zeros(2 * case["nx"] * case["ny"], dtype=torch.complex128)
    e[case["nx"] * case["ny"] // 2] = 1.0
    eff = [_efficiencies(o[0], i, *o[1], e) for o, i in zip(out, stacks)]
    return dict(S=S, ref=np.stack([v[0] for v in eff]), trn=np.stack([v[1] for v in eff]))
