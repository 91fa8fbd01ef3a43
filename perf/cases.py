"""Performance cases of tara_amd: the calls a user's program makes, through the
package's public entry points, over the sizes and options it accepts.

A case is a dict of plain values whose "kind" names the path:

  csh      resident 2D vorticity solver (CshSolver): advance, then download the frame
  f2       resident 2D compressible solver (F2Solver; coh: 3 fields, com: 6 fields)
  mhd      resident 3D compressible MHD solver (MhdSolver)
  ens      batched ensemble (Ensemble): advance, then every run's vorticity into
           device memory, as the surrogate's data generation does
  fno      surrogate inference (FNO.forward) on device fields
  fnograd  surrogate loss and gradient (FNO.grads)
  rhs      the allocation-free right-hand side on device arrays
  dropin   the Fortran programs' call: one right-hand side on host arrays

listed() holds the cases, draw(rng) makes more of the same ranges, prepare()
builds what a program holds before the call, run() is one pass, work() what a
pass cannot do without, exact() the same outputs from torch in 64 bits.
"""
import math

import numpy as np
import torch

import tara_amd as T

PI = math.pi
DEV = "cuda"


# --------------------------------------------------------------------- cases
def listed():
    return [
        # The flagship run: 2D hydro at 4096^2, nu 1e-4, dt 2e-4, random-phase
        # initial vorticity; a stretch of steps between two saved frames.
        dict(name="csh_rk4_4096", kind="csh", nx=4096, ny=4096, scheme="rk4", screened=False, ic="spectrum", nu=1e-4,
             dt=2e-4, steps=100, tune=True),
        # The same flow at the configuration's other size, restarted from a
        # real-space field (every mode of the half spectrum present).
        dict(name="csh_rk4_1024", kind="csh", nx=1024, ny=1024, scheme="rk4", screened=False, ic="field", nu=1e-4,
             dt=2e-4, steps=200, tune=True),
        # The reference's default run: 64^2 shear layer, AB2, a snapshot every
        # 1000 steps.  Nothing but the latency of a step counts here.
        dict(name="csh_ab2_64", kind="csh", nx=64, ny=64, scheme="ab2", screened=False, ic="shear", nu=0.01, dt=1e-4,
             steps=1000, tune=False),
        # The screened equations on a box twice as long as it is wide, RK4.
        dict(name="css_rk4_512x256", kind="csh", nx=512, ny=256, scheme="rk4", screened=True, ic="field", nu=1e-3,
             dt=5e-4, steps=100, tune=False),
        # 2D compressible MHD, forced, at the largest grid of that family.
        dict(name="com_ab2_256", kind="f2", family="com", nx=256, ny=256, dt=1e-4, steps=200),
        # 3D MHD with the benchmark's physics and number of steps on a quarter of
        # its grid (the long axis whole), then the state for a restart file.
        dict(name="mhd_ab2_256x128x128", kind="mhd", nx=256, ny=128, nz=128, nu=1e-3, dt=5e-4, steps=500),
        # The same at a size for parameter scans: short launches, little data.
        dict(name="mhd_ab2_64", kind="mhd", nx=64, ny=64, nz=64, nu=1e-2, dt=5e-4, steps=200),
        # Training-data generation: 512 runs of uneven grids and viscosities,
        # sampled into device memory every 20 steps.
        dict(name="ens_rk4_512_runs", kind="ens", n0=128, n1=256, n2=512, runs=512, scheme="rk4", dt=5e-4, steps=20),
        # Surrogate inference over a batch at the production shape.
        dict(name="fno_forward_b16", kind="fno", n=256, width=64, mx=16, my=32, layers=4, batch=16, prec="bf16"),
        # One surrogate loss and gradient at the production shape.
        dict(name="fno_grads_b16", kind="fnograd", n=256, width=64, mx=16, my=32, layers=4, batch=16, prec="bf16"),
        # One right-hand side on device arrays, enqueued on the caller's
        # stream: the smallest call of the library.
        dict(name="rhs_device_256", kind="rhs", nx=256, ny=256, nu=1e-3),
        # A kept Fortran main's call on host arrays, at a grid that is not a
        # power of two (input.ini takes any size).
        dict(name="dropin_rhs_96x80", kind="dropin", nx=96, ny=80, nu=1e-2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _pow2(rng, lo, hi):
    return 1 << rng.randint(int(math.log2(lo)), int(math.log2(hi)))


def draw(rng):
    kind = rng.choice(["csh", "csh", "f2", "mhd", "ens", "fno", "fnograd", "rhs", "dropin"])
    if kind == "csh":
        # any pair of powers of two, both schemes, both equations; as many steps
        # between frames as fit the largest listed case's cost
        nx, ny = _pow2(rng, 64, 4096), _pow2(rng, 32, 4096)
        scheme = rng.choice(["ab2", "rk4"])
        most = max(8, min(300, int(8e8 / (nx * ny))))
        return dict(kind=kind, nx=nx, ny=ny, scheme=scheme, screened=rng.random() < 0.3,
                    ic=rng.choice(["spectrum", "field"]), nu=10.0 ** rng.uniform(-4, -2), dt=1e-4,
                    steps=_log_int(rng, max(4, most // 8), most), tune=rng.random() < 0.5)
    if kind == "f2":
        return dict(kind=kind, family=rng.choice(["coh", "com"]), nx=_pow2(rng, 16, 256), ny=_pow2(rng, 16, 256),
                    dt=1e-4, steps=_log_int(rng, 20, 250))
    if kind == "mhd":
        nx, ny, nz = _pow2(rng, 16, 256), _pow2(rng, 16, 256), _pow2(rng, 16, 256)
        nz = min(nz, 16384 // ny)
        most = min(300, int(2e9 / (nx * ny * nz)))
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, nu=10.0 ** rng.uniform(-3, -2), dt=5e-4,
                    steps=_log_int(rng, most // 8, most))
    if kind == "ens":
        n = [_pow2(rng, 64, 512) for _ in range(3)]
        cap = max(3, min(512, int(4e7 / max(n) ** 2)))
        return dict(kind=kind, n0=n[0], n1=n[1], n2=n[2], runs=_log_int(rng, 3, cap),
                    scheme=rng.choice(["ab2", "rk4"]), dt=5e-4, steps=_log_int(rng, 4, 20))
    if kind in ("fno", "fnograd"):
        n = 8 * _log_int(rng, 8, 32)
        mx = rng.randint(4, 16)
        return dict(kind=kind, n=n, width=rng.choice([16, 24, 32, 48, 64]), mx=mx, my=2 * rng.randint(2, 16),
                    layers=rng.randint(2, 4), batch=_log_int(rng, 1, 16), prec=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "rhs":
        return dict(kind=kind, nx=_pow2(rng, 64, 1024), ny=_pow2(rng, 32, 1024), nu=10.0 ** rng.uniform(-4, -2))
    nx, ny = _log_int(rng, 40, 700), _log_int(rng, 40, 700)
    return dict(kind="dropin", nx=nx, ny=ny, nu=10.0 ** rng.uniform(-3, -2))


# -------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _k(n):
    """derive2csh's full-axis wavenumbers: j for j < n/2, j - n above."""
    j = torch.arange(n, device=DEV, dtype=torch.float64)
    return torch.where(j < n // 2, j, j - n)


def _grids2(nx, ny):
    return torch.arange(nx // 2 + 1, device=DEV, dtype=torch.float64)[None, :], _k(ny)[:, None]


def _vorticity(gen, nx, ny, k0, runs=1):
    """Random-phase vorticity spectra [runs][ny][nx/2+1], E(k) ~ k^4 exp(-(k/k0)^2)
    with no Nyquist modes and unit kinetic energy (the benchmark's initial state)."""
    kx, ky = _grids2(nx, ny)
    k = torch.sqrt(kx * kx + ky * ky)
    k0 = torch.as_tensor(k0, device=DEV, dtype=torch.float64).reshape(-1, 1, 1)
    amp = torch.sqrt(k) * k * k * torch.exp(-0.5 * (k / k0) ** 2)
    if nx % 2 == 0:
        amp = torch.where(kx == nx // 2, torch.zeros_like(amp), amp)
    if ny % 2 == 0:
        amp = torch.where(ky == -(ny // 2), torch.zeros_like(amp), amp)
    z = torch.fft.rfft2(torch.randn((runs, ny, nx), generator=gen, device=DEV, dtype=torch.float64))
    w = z / z.abs().clamp_min(1e-300) * amp
    wt = torch.where((kx == 0), 1.0, 2.0)
    k2 = torch.where(k > 0, k * k, torch.ones_like(k))
    ke = 0.5 * (wt * w.abs() ** 2 / k2).sum((1, 2), keepdim=True) / float(nx * ny) ** 2
    w = w / torch.sqrt(ke)
    w[:, 0, 0] = 0
    return w


def _c2r2(w, nx):
    """FFTW's 2D c2r (y first, Im dropped at kx = 0 and Nx/2), normalised."""
    a = torch.fft.ifft(w, dim=-2)
    a[..., 0].imag = 0
    if nx % 2 == 0:
        a[..., nx // 2].imag = 0
    return torch.fft.irfft(a, n=nx, dim=-1)


def _shear(gen, nx, ny):
    """The reference's shear layer (two opposed layers and a perturbation) whose
    perturbation's size and phase come from the seed."""
    u = torch.rand(2, generator=gen, device=DEV, dtype=torch.float64)
    x = torch.arange(nx, device=DEV, dtype=torch.float64)[None, :] * (2 * PI / nx)
    y = torch.arange(ny, device=DEV, dtype=torch.float64)[:, None] * (2 * PI / ny)
    d, w0 = 3 * PI / 128, 25.0
    w = w0 / torch.cosh((x - PI / 2) / d) ** 2 - w0 / torch.cosh((x - 1.5 * PI) / d) ** 2
    w = w * (1.0 + (0.05 + 0.1 * u[0]) * torch.cos(2.0 * y + 2 * PI * u[1]))
    return torch.fft.rfft2(w)


def _csh_state(case, seed):
    gen = _gen(seed)
    nx, ny = case["nx"], case["ny"]
    ic = case.get("ic", "field")
    if ic == "shear":
        return _shear(gen, nx, ny)
    w = _vorticity(gen, nx, ny, 4.0)[0]
    if ic == "field":  # through real space, as a program that holds the field does
        w = torch.fft.rfft2(_c2r2(w, nx))
    return w


def _smooth(gen, shape, modes=6):
    """Band-limited random real fields (a few low modes), unit variance."""
    f = torch.randn(shape, generator=gen, device=DEV, dtype=torch.float64)
    s = torch.fft.rfftn(f)
    k2 = torch.zeros((), device=DEV, dtype=torch.float64)
    for d, n in enumerate(shape):
        k = torch.arange(n // 2 + 1, device=DEV, dtype=torch.float64) if d == len(shape) - 1 else _k(n)
        k2 = k2 + (k.reshape([-1 if e == d else 1 for e in range(len(shape))])) ** 2
    f = torch.fft.irfftn(s * torch.exp(-k2 / modes), s=shape)
    return f / f.std()


def _f2_state(case, seed):
    gen = _gen(seed)
    shape = (case["ny"], case["nx"])
    f = [1.0 + 0.05 * _smooth(gen, shape)]
    f += [0.2 * _smooth(gen, shape) for _ in range(2)]
    if case["family"] == "com":
        f += [2.0 + 0.1 * _smooth(gen, shape)] + [0.2 * _smooth(gen, shape) for _ in range(2)]
    return [torch.fft.rfft2(a) for a in f]


def _f2_params(case):
    if case["family"] == "coh":
        return T.CohParams(PI, 2 * PI, 2 * PI, 2e-4, 2e-4, 3.77, case["dt"])
    return T.ComParams(PI, 2 * PI, 2 * PI, 1e-3, 1e-4, 2.0, 1.0, 0.3, case["dt"])


def _mhd_grids(nx, ny, nz):
    kx = torch.arange(nx // 2 + 1, device=DEV, dtype=torch.float64)[None, None, :]
    return kx, _k(ny)[None, :, None], _k(nz)[:, None, None]


def _mhd_state(case, seed):
    """Uniform density, random-phase solenoidal u and B with
    E(k) ~ k^4 exp(-2 (k/3)^2), energies 1.0 and 0.5 (the benchmark's state)."""
    gen = _gen(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    K = _mhd_grids(nx, ny, nz)
    k2 = K[0] ** 2 + K[1] ** 2 + K[2] ** 2
    amp = k2 ** 0.5 * torch.exp(-k2 / 9.0)
    inv = torch.where(k2 > 0, 1.0 / k2.clamp_min(1e-30), torch.zeros_like(k2))

    def solenoidal(energy):
        c = [torch.fft.rfftn(torch.randn((nz, ny, nx), generator=gen, device=DEV, dtype=torch.float64)) * amp
             for _ in range(3)]
        div = (K[0] * c[0] + K[1] * c[1] + K[2] * c[2]) * inv
        r = [torch.fft.irfftn(c[i] - K[i] * div, s=(nz, ny, nx)) for i in range(3)]
        s = math.sqrt(energy / float(0.5 * sum((a * a).mean() for a in r)))
        return [a * s for a in r]

    u, b = solenoidal(1.0), solenoidal(0.5)
    rho = torch.ones((nz, ny, nx), device=DEV, dtype=torch.float64)
    e = 1.0 + 0.5 * sum(a * a for a in u) + 0.5 * sum(a * a for a in b)
    return [torch.fft.rfftn(a) for a in [rho] + [rho * a for a in u] + [e] + b]


def _ens_runs(case, seed):
    """(grids, viscosities, k0) of the runs: sizes cycle over n0, n1, n2."""
    r = np.random.default_rng(int(seed))
    sizes = [(case["n0"], case["n1"], case["n2"])[i % 3] for i in range(case["runs"])]
    return sizes, 10.0 ** r.uniform(-4, -2, case["runs"]), r.uniform(3, 8, case["runs"])


def _ens_states(case, seed):
    """{grid: (run indices, spectra [runs][n][n/2+1])}."""
    sizes, _, k0 = _ens_runs(case, seed)
    gen, out = _gen(seed), {}
    for n in sorted(set(sizes)):
        idx = [i for i, s in enumerate(sizes) if s == n]
        out[n] = (idx, _vorticity(gen, n, n, k0[idx], runs=len(idx)))
    return out


def _fno_params(case, seed):
    """A flat parameter vector in the network's layout (lift, spectral weights,
    mixing, projection), of the magnitudes that training reaches."""
    gen = _gen(seed + 7)
    c, m, layers = case["width"], case["mx"] * case["my"], case["layers"]
    h = 2 * c

    def uni(n, s):
        return (2 * torch.rand(n, generator=gen, device=DEV) - 1) * s

    return torch.cat([uni(c, 1.0), uni(c, 0.1), uni(layers * m * 2 * c * c, 2.0 / (c * c)),
                      uni(layers * c * c, 1.0 / math.sqrt(c)), uni(layers * c, 0.1), uni(h * c, 1.0 / math.sqrt(c)),
                      uni(h, 0.1), uni(h, 0.3 / math.sqrt(h)), uni(1, 0.01)])


def _fno_fields(case, seed):
    """(omega, target): float32 vorticity fields [batch][n][n] and what they
    have become a while later (each phase moved on a little)."""
    gen, n, b = _gen(seed), case["n"], case["batch"]
    w = _vorticity(gen, n, n, [3.0 + 5.0 * i / b for i in range(b)], runs=b)
    kx, ky = _grids2(n, n)
    later = w * torch.exp(-1e-3 * (kx * kx + ky * ky)) * torch.exp(1j * 0.1 * kx)
    return _c2r2(w, n).float().contiguous(), _c2r2(later, n).float().contiguous()


def _host(w):
    """Device spectrum [.., ky, kx] -> host array (Nh, Ny[, Nz]) in Fortran order."""
    return w.cpu().numpy().T


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "csh":
        w = _csh_state(case, seed)
        scheme = T.SCHEME_RK4 if case["scheme"] == "rk4" else T.SCHEME_AB2
        s["solver"] = T.CshSolver(case["nx"], case["ny"], case["nu"], case["dt"], scheme, screened=case["screened"])
        s["solver"].upload(_host(w))
        if case["tune"]:
            s["solver"].tune()
    elif kind == "f2":
        s["solver"] = T.F2Solver(case["nx"], case["ny"], _f2_params(case))
        s["solver"].upload([_host(a) for a in _f2_state(case, seed)])
    elif kind == "mhd":
        p = T.MhdParams(2 * PI, 2 * PI, 2 * PI, case["nu"], case["nu"], 10.0, case["dt"])
        s["solver"] = T.MhdSolver(case["nx"], case["ny"], case["nz"], p)
        s["solver"].upload([_host(a) for a in _mhd_state(case, seed)])
    elif kind == "ens":
        sizes, nus, _ = _ens_runs(case, seed)
        scheme = T.SCHEME_RK4 if case["scheme"] == "rk4" else T.SCHEME_AB2
        s["solver"] = T.Ensemble(sizes, nus, case["dt"], scheme)
        s["out"], s["where"] = {}, []
        for n, (idx, w) in _ens_states(case, seed).items():
            w = w.cpu().numpy()
            for q, r in enumerate(idx):
                s["solver"].upload(r, w[q].T)
            s["out"][n] = torch.empty((len(idx), n, n), dtype=torch.float32, device=DEV)
            s["where"] += [(r, s["out"][n][q]) for q, r in enumerate(idx)]
        s["solver"].tune()
    elif kind in ("fno", "fnograd"):
        prec = T.FNO_BF16 if case["prec"] == "bf16" else T.FNO_FP32
        s["net"] = T.FNO(case["n"], case["width"], case["mx"], case["my"], case["layers"], max_batch=case["batch"],
                         precision=prec)
        s["net"].set_params(_fno_params(case, seed).cpu().numpy())
        s["omega"], s["target"] = _fno_fields(case, seed)
        s["out"] = torch.empty_like(s["omega"])
    elif kind == "rhs":
        s["omega"] = torch.view_as_real(_csh_state(case, seed)).contiguous()
        s["out"] = torch.empty_like(s["omega"])
    else:
        s["omega"] = _host(_csh_state(case, seed))
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------- pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("csh", "f2", "mhd"):
        state["solver"].advance(case["steps"])
        w = state["solver"].download()
        return w.T if kind == "csh" else [a.T for a in w]
    if kind == "ens":
        state["solver"].advance(case["steps"])
        for r, out in state["where"]:
            state["solver"].get_omega(r, out)
        return [state["out"][n] for n in sorted(state["out"])]
    if kind == "fno":
        state["net"].forward(case["batch"], state["omega"], state["out"])
        return state["out"]
    if kind == "fnograd":
        loss, g = state["net"].grads(case["batch"], state["omega"], state["target"])
        return [float(loss), g]
    nh = case["nx"] // 2 + 1
    if kind == "rhs":
        T.derive2csh_noalloc(case["nx"], case["ny"], nh, case["nu"], state["omega"].data_ptr(),
                             state["out"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        return state["out"]
    return T.derive2csh(case["nx"], case["ny"], nh, case["nu"], state["omega"]).T


# ---------------------------------------------------------------------- work
def _fno_flops(case):
    n, c, mx, my, layers = (case[k] for k in ("n", "width", "mx", "my", "layers"))
    layer = (4 * mx * n * n * c + 8 * my * n * mx * c + 8 * c * c * mx * my + 8 * n * my * mx * c
             + 4 * c * n * mx * n + 2 * c * c * n * n)
    return case["batch"] * (layers * layer + 4 * c * c * n * n + 4 * c * n * n)


def work(case):
    """Bytes: the state in and out of every step (the least a resident step
    moves), inputs and outputs of the call.  Operations: the transforms (2.5 N
    log2 N each) of every right-hand side, or the network's products."""
    kind = case["kind"]
    if kind in ("csh", "rhs", "dropin"):
        nx, ny = case["nx"], case["ny"]
        s = 16.0 * (nx // 2 + 1) * ny
        fft = 5 * 2.5 * nx * ny * math.log2(nx * ny)
        if kind != "csh":
            return dict(bytes=2 * s, flops=fft)
        rk = case["scheme"] == "rk4"
        return dict(bytes=case["steps"] * (2 if rk else 4) * s + s, flops=case["steps"] * (4 if rk else 1) * fft)
    if kind == "f2":
        nx, ny = case["nx"], case["ny"]
        s = 16.0 * (nx // 2 + 1) * ny
        nf, ntr = (3, 16) if case["family"] == "coh" else (6, 19)
        return dict(bytes=(case["steps"] * 4 + 1) * nf * s,
                    flops=case["steps"] * ntr * 2.5 * nx * ny * math.log2(nx * ny))
    if kind == "mhd":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        s, n = 16.0 * (nx // 2 + 1) * ny * nz, nx * ny * nz
        return dict(bytes=case["steps"] * 28 * s + 8 * s, flops=case["steps"] * 21 * 2.5 * n * math.log2(n))
    if kind == "ens":
        sizes, _, _ = _ens_runs(case, 0)
        rk = case["scheme"] == "rk4"
        s = sum(16.0 * (n // 2 + 1) * n for n in sizes)
        return dict(bytes=case["steps"] * (2 if rk else 4) * s + sum(4.0 * n * n for n in sizes),
                    flops=case["steps"] * (4 if rk else 1) * sum(5 * 2.5 * n * n * math.log2(n * n) for n in sizes))
    c, n, b = case["width"], case["n"], case["batch"]
    npar = c * 2 + case["layers"] * (case["mx"] * case["my"] * 2 * c * c + c * c + c) + 2 * c * c + 4 * c + 1
    wb = 2.0 if case["prec"] == "bf16" else 4.0
    if kind == "fno":
        return dict(bytes=8.0 * b * n * n + wb * npar, flops=_fno_flops(case))
    return dict(bytes=8.0 * b * n * n + (wb + 4.0) * npar, flops=3.0 * _fno_flops(case))


# --------------------------------------------------------------------- exact
def _csh_rhs(w, nx, ny, nu, screened=False, alpha=1.0, lam=T.CSS_LAMBDA):
    """derive2csh / derive2css on spectra [.., ky, kx]; nu broadcasts over runs."""
    kx, ky = _grids2(nx, ny)
    k2 = kx * kx + ky * ky
    if screened:
        psi = w / (k2 + lam)
        psi[..., 0, 0] = 0
        wd = k2 * psi
    else:
        psi = w / torch.where(k2 > 0, k2, torch.ones_like(k2))
        psi[..., 0, 0] = 0
        wd = w
    nl = _c2r2(1j * ky * psi, nx) * _c2r2(1j * kx * wd, nx)
    nl += _c2r2(-1j * kx * psi, nx) * _c2r2(1j * ky * wd, nx)
    nl = torch.fft.rfft2(nl)
    keep = torch.sqrt(k2) < ((nx + ny) / 2.0) / 3.0
    nl = torch.where(keep, nl, torch.zeros_like(nl))
    return -((alpha * nl if screened else nl) + nu * k2 * wd)


def _advance(w, rhs, dt, steps, scheme):
    """AB2 from a zero history, or classic RK4, on one spectrum or a list."""
    many = isinstance(w, list)
    w = w if many else [w]
    f = (lambda z: rhs(z)) if many else (lambda z: [rhs(z[0])])
    old = [torch.zeros_like(a) for a in w]
    for _ in range(steps):
        if scheme == "ab2":
            new = f(w)
            w = [a + (1.5 * n - 0.5 * o) * dt for a, n, o in zip(w, new, old)]
            old = new
        else:
            k1 = f(w)
            k2 = f([a + 0.5 * dt * k for a, k in zip(w, k1)])
            k3 = f([a + 0.5 * dt * k for a, k in zip(w, k2)])
            k4 = f([a + dt * k for a, k in zip(w, k3)])
            w = [a + dt / 6.0 * (p + 2 * q + 2 * r + s) for a, p, q, r, s in zip(w, k1, k2, k3, k4)]
    return w if many else w[0]


def _mask2(case):
    kx, ky = _grids2(case["nx"], case["ny"])
    return torch.sqrt(kx * kx + ky * ky) < ((case["nx"] + case["ny"]) / 2.0) / 3.0


def _coh_rhs(case):
    """derive2coh: n, ux, uy with mux = muy = 2e-4, CS = 3.77, box 2 pi."""
    nx, ny = case["nx"], case["ny"]
    kx, ky = _grids2(nx, ny)
    mu, cs2, keep = 2e-4, 3.77 ** 2, _mask2(case)

    def rhs(st):
        n, ux, uy = (_c2r2(a, nx) for a in st)
        d = lambda k, a: _c2r2(1j * k * a, nx)  # noqa: E731
        d2 = lambda k, a: _c2r2(k * k * a, nx)  # noqa: E731
        nx_, ny_ = d(kx, st[0]), d(ky, st[0])
        uxx, uxy, uyx, uyy = d(kx, st[1]), d(ky, st[1]), d(kx, st[2]), d(ky, st[2])
        t = [ux * nx_ + uy * ny_ + n * (uxx + uyy),
             ux * uxx + uy * uxy + mu * d2(kx, st[1]) / n + mu * d2(ky, st[1]) / n + cs2 * nx_ / n,
             ux * uyx + uy * uyy + mu * d2(kx, st[2]) / n + mu * d2(ky, st[2]) / n + cs2 * ny_ / n]
        return [-torch.where(keep, torch.fft.rfft2(a), 0.0) for a in t]

    return rhs


def _com_rhs(case):
    """derive2com: mu = 1e-3, eta = 1e-4, CS = 2, forcing A = 0.3, kf = 1; its
    curl of B is the velocity gradients' over Nx Ny, as the routine forms it."""
    nx, ny = case["nx"], case["ny"]
    kx, ky = _grids2(nx, ny)
    mu, eta, cs2, amp, kf, keep = 1e-3, 1e-4, 4.0, 0.3, 1.0, _mask2(case)
    x = torch.arange(nx, device=DEV, dtype=torch.float64)[None, :] * (2 * PI / nx)
    y = torch.arange(ny, device=DEV, dtype=torch.float64)[:, None] * (2 * PI / ny)

    def rhs(st):
        rho, rux, ruy, en, bx, by = (_c2r2(a, nx) for a in st)
        ux, uy = rux / rho, ruy / rho
        uxk, uyk = torch.fft.rfft2(ux), torch.fft.rfft2(uy)
        fx, fy = -rho * amp * torch.sin(kf * y), rho * amp * torch.sin(kf * x)
        dudx, dvdy = _c2r2(1j * kx * uxk, nx), _c2r2(1j * ky * uyk, nx)
        b2, p = bx * bx + by * by, cs2 * rho
        curl = (dvdy - dudx) / (nx * ny)
        h = en + p + b2 / 2
        fl = [rux * ux + p + b2 / 2 - bx * bx, rux * uy - bx * by, ruy * uy + p + b2 / 2 - by * by,
              h * ux - ux * bx * bx - uy * bx * by - eta * by * curl,
              h * uy - ux * bx * by - uy * by * by + eta * bx * curl, (dudx + dvdy) ** 2, uy * bx - by * ux]
        m = [torch.where(keep, torch.fft.rfft2(a), 0.0) for a in fl]
        k2 = torch.where(keep, kx * kx + ky * ky, 0.0)
        ik = lambda k, a: 1j * k * a  # noqa: E731
        return [-torch.where(keep, ik(kx, st[1]) + ik(ky, st[2]), 0.0),
                -(ik(kx, m[0]) + ik(ky, m[1])) - mu * k2 * uxk + torch.fft.rfft2(fx),
                -(ik(kx, m[1]) + ik(ky, m[2])) - mu * k2 * uyk + torch.fft.rfft2(fy),
                -(ik(kx, m[3]) + ik(ky, m[4])) + mu * m[5],
                -ik(ky, m[6]) - eta * k2 * st[4], ik(kx, m[6]) - eta * k2 * st[5]]

    return rhs


def _mhd_rhs(case):
    """derive3com's live part (isothermal, CS = 10, box 2 pi); E is frozen."""
    nx, ny, nz, nu = case["nx"], case["ny"], case["nz"], case["nu"]
    K = _mhd_grids(nx, ny, nz)
    k2 = K[0] ** 2 + K[1] ** 2 + K[2] ** 2
    keep = torch.sqrt(k2) < ((nx + ny + nz) / 3.0) / 3.0

    def c2r(a):
        a = torch.fft.ifft(torch.fft.ifft(a, dim=0), dim=1)
        a[..., 0].imag = 0
        a[..., nx // 2].imag = 0
        return torch.fft.irfft(a, n=nx, dim=-1)

    def r2c(a):
        return torch.where(keep, torch.fft.rfftn(a), 0.0)

    def rhs(st):
        rho = c2r(st[0])
        u = [c2r(st[1 + i]) / rho for i in range(3)]
        b = [c2r(st[5 + i]) for i in range(3)]
        pt = 100.0 * rho + 0.5 * (b[0] * b[0] + b[1] * b[1] + b[2] * b[2])
        flux = {(i, j): r2c(rho * u[i] * u[j] - b[i] * b[j] + (pt if i == j else 0.0))
                for i in range(3) for j in range(i, 3)}
        mag = {(i, j): r2c(u[i] * b[j] - u[j] * b[i]) for i in range(3) for j in range(i + 1, 3)}
        out = [-1j * sum(K[i] * torch.where(keep, st[1 + i], 0.0) for i in range(3))]
        for i in range(3):
            div = 1j * sum(K[j] * flux[(min(i, j), max(i, j))] for j in range(3))
            out.append(-div - nu * k2 * r2c(u[i]))
        out.append(torch.zeros_like(st[4]))
        for i in range(3):
            curl = 1j * sum(K[j] * (mag[(i, j)] if i < j else -mag[(j, i)]) for j in range(3) if j != i)
            out.append(curl - nu * k2 * torch.where(keep, st[5 + i], 0.0))
        return out

    return rhs


def _fno_exact(case, seed, grad):
    n, c, mx, my, layers, b = (case[k] for k in ("n", "width", "mx", "my", "layers", "batch"))
    m, h = mx * my, 2 * c
    flat = _fno_params(case, seed).double().requires_grad_(grad)
    omega, target = (a.double() for a in _fno_fields(case, seed))
    shapes = [(c,), (c,), (layers, m, 2, c, c), (layers, c, c), (layers, c), (h, c), (h,), (h,), (1,)]
    p, o = [], 0
    for s in shapes:
        p.append(flat[o:o + math.prod(s)].reshape(s))
        o += math.prod(s)
    wl, bl, r, w, bias, w1, b1, w2, b2 = p
    gelu = lambda x: 0.5 * x * (1.0 + torch.erf(x * math.sqrt(0.5)))  # noqa: E731
    s = torch.sqrt((omega * omega).mean((1, 2), keepdim=True))
    v = wl[None, :, None, None] * (omega / s)[:, None] + bl[None, :, None, None]
    rows = list(range(my // 2)) + list(range(n - my // 2, n))
    for l in range(layers):
        sel = torch.fft.rfft2(v)[:, :, rows, :mx]
        wt = torch.complex(r[l, :, 0], r[l, :, 1]).reshape(my, mx, c, c)
        full = torch.zeros((b, c, n, n // 2 + 1), dtype=torch.complex128, device=DEV)
        full[:, :, rows, :mx] = torch.einsum("bimk,mkio->bomk", sel, wt)
        pre = (torch.fft.irfft2(full, s=(n, n)) + (w[l] @ v.reshape(b, c, n * n)).reshape(b, c, n, n)
               + bias[l][None, :, None, None])
        v = gelu(pre) if l < layers - 1 else pre
    hid = gelu((w1 @ v.reshape(b, c, n * n)) + b1[None, :, None])
    out = omega + s * ((w2 @ hid).reshape(b, n, n) + b2)
    if not grad:
        return out.detach()
    d = torch.sqrt(((out - target) ** 2).sum((1, 2))) / torch.sqrt((target ** 2).sum((1, 2)))
    loss = d.mean()
    loss.backward()
    return [float(loss.detach()), flat.grad]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("rhs", "dropin", "csh"):
        nx, ny, nu = case["nx"], case["ny"], case["nu"]
        w = _csh_state(case, seed)
        if kind == "csh":
            return _advance(w, lambda z: _csh_rhs(z, nx, ny, nu, case["screened"]), case["dt"], case["steps"],
                            case["scheme"])
        f = _csh_rhs(w, nx, ny, nu)
        return f if kind == "dropin" else torch.view_as_real(f)
    if kind == "f2":
        rhs = _coh_rhs(case) if case["family"] == "coh" else _com_rhs(case)
        return _advance(_f2_state(case, seed), rhs, case["dt"], case["steps"], "ab2")
    if kind == "mhd":
        return _advance(_mhd_state(case, seed), _mhd_rhs(case), case["dt"], case["steps"], "ab2")
    if kind == "ens":
        _, nus, _ = _ens_runs(case, seed)
        out = []
        for n, (idx, w) in sorted(_ens_states(case, seed).items()):
            nu = torch.as_tensor(nus[idx], device=DEV).reshape(-1, 1, 1)
            w = _advance(w, lambda z: _csh_rhs(z, n, n, nu), case["dt"], case["steps"], case["scheme"])
            out.append(_c2r2(w, n))
        return out
    return _fno_exact(case, seed, kind == "fnograd")
