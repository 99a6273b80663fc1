"""Timed cases of the framework's main path, through its public entry points.

Every case is one call (or the few calls) that an X-ray inference makes again
and again: the Poisson gradient of the fused model, its sampled KL, the metric
products and the linear solves of the sample draws, the PSF operator in both
directions, the drop-in functions, the Gaussian-process sky and the separate
response chain.  Sizes are those of the benchmark configurations and of the
demos; ``draw`` spreads over the same ranges, odd and ragged sizes among them.

``exact`` restates each case in float64 with plain torch operations.
"""
import math

import numpy as np
import torch

import __graft_entry__

ja = __graft_entry__.load_package()

DTYPES = {"f32": torch.float32, "f64": torch.float64}
GP_GRIDS = (64, 128, 256, 512, 567, 768, 1024, 1134, 2048)
ZERO_MODE, INDEX_MEAN = -2.0, -1.0
POINTS = dict(a=1.995, q=0.8, alpha_mean=-1.5, alpha_std=0.4)
CG_STEPS = 8


# ------------------------------------------------------------------- cases
def _case(kind, dtype, H, E, n, m, M=1, S=1, N=None, name=None):
    case = dict(kind=kind, dtype=dtype, H=H, E=E, n=n, m=m, M=M, S=S,
                N=N or min(g for g in GP_GRIDS if g >= H))
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # one gradient of a small cutout: ten launches of little work each
        _case("grad", "f32", 128, 1, 4, 16, name="grad_128x1E"),
        # the benchmark's evaluation: four energy bins, 8 x 8 patches
        _case("grad", "f32", 1024, 4, 8, 64, name="grad_1024x4E"),
        # seven telescope modules that see one sky in three energy bins
        _case("grad", "f32", 1024, 3, 10, 60, M=7, name="grad_1024x3Ex7M"),
        # float64 (what the reference enforces) on a 512 sky in its padded GP grid
        _case("grad", "f64", 512, 2, 4, 32, N=567, name="grad_512x2E_f64"),
        # a Newton step's KL and gradient over four samples of a large mosaic
        _case("kl", "f32", 2048, 4, 16, 64, S=4, name="kl_2048x4E_S4"),
        # metric products of 32 sample tangents on a small observation
        _case("metric", "f32", 256, 1, 6, 22, S=32, name="metric_256x1E_S32"),
        # conjugate-gradient steps of four sample draws
        _case("solve", "f32", 512, 1, 8, 32, S=4, name="solve_512x1E_S4"),
        # diffuse sky plus point sources with an inverse-gamma prior
        _case("points", "f32", 512, 3, 8, 32, name="points_512x3E"),
        # the PSF operator alone, forward and adjoint, at the default margin,
        # whose window length 332 has no plan of its own
        _case("psf", "f32", 1024, 1, 10, 64, name="psf_1024x1E_m64"),
        # the drop-in linpatch_convolve with full-frame kernels, float64
        _case("dropin", "f64", 512, 2, 4, 32, name="dropin_512x2E_f64"),
        # the sky alone on the padded grid of a 1024 sky, and its transpose
        _case("gp", "f32", 1024, 2, 8, 64, N=1134, name="gp_1134x2E"),
        # exposure, read-out and Poisson energy as separate calls, and back
        _case("response", "f64", 512, 3, 8, 32, M=7, name="response_512x3Ex7M_f64"),
    ]


def _cost(c):
    d = c["H"] // c["n"]
    L = 2 * d + 2 * c["m"]
    per = {"dropin": 3, "points": 2, "solve": CG_STEPS, "response": 0.1, "gp": 0.2}
    return (per.get(c["kind"], 1) * (2 if c["dtype"] == "f64" else 1) * c["S"] * c["M"] * c["E"]
            * c["n"] ** 2 * L * L)


# Window lengths 2 d + 2 m that the PSF operator takes: its own FFT lengths,
# or any length that fits one of them together with twice the window.
_LENGTHS = (16, 24, 32, 48, 64, 96, 128, 192, 224, 256, 320, 324, 384, 432, 512)


def _window_ok(w, m):
    return w + 2 * m in _LENGTHS or max(w + 2 * m, 2 * w) <= _LENGTHS[-1]


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["grad", "grad", "kl", "metric", "solve", "points", "psf", "dropin",
                           "gp", "response"])
        dtype = rng.choice(["f32", "f32", "f64"])
        H = int(round(2.0 ** rng.uniform(6, 11 if kind in ("grad", "kl", "psf") else 10)))
        n = rng.choice([2, 3, 4, 5, 6, 8, 10, 12, 16])
        if kind == "dropin":
            H += H % 2  # full-frame kernels are cut about an even frame's centre
            n = max(n, 3)
        d = H // n
        # the margin is a quarter to a half of the patch stride
        m = max(1, int(d * rng.uniform(0.25, 0.5)))
        if d < 8 or H - n * d > d // 4 or not _window_ok(2 * d, m):
            continue
        E = rng.choice([1, 1, 2, 3, 4])
        M = rng.choice([1, 1, 2, 3, 7]) if kind in ("grad", "response") else 1
        S = rng.choice([2, 4, 8, 16, 32]) if kind in ("kl", "metric", "solve") else 1
        N = rng.choice([g for g in GP_GRIDS if g >= H][:2])
        case = _case(kind, dtype, H, E, n, m, M=M, S=S, N=N)
        if _cost(case) <= most:
            return case


# ------------------------------------------------------------------ inputs
def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    return gen


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64)


def _amplitude(N):
    """Power-law amplitude field, slope -4, unit fluctuations."""
    k = torch.fft.fftfreq(N, device="cuda", dtype=torch.float64)
    amp = (k[:, None] ** 2 + k[None, :] ** 2)
    amp[0, 0] = 1.0
    amp = 1.0 / amp
    amp[0, 0] = 0.0
    return amp / torch.sqrt((amp ** 2).sum())


def _psf_windows(gen, n, E, w):
    """(n * n, E, w, w) windows: an elliptical Gaussian mixed with a Moffat
    profile, wider and more elliptical across the field and with energy."""
    P = n * n
    c = torch.arange(w, device="cuda", dtype=torch.float64) - w // 2
    t = torch.linspace(0.0, 1.0, P, device="cuda", dtype=torch.float64)[:, None]
    e = torch.arange(E, device="cuda", dtype=torch.float64)[None, :]
    sigma = ((1.0 + 3.0 * t) * (1.0 + 0.15 * e))[..., None, None]
    flat = (1.0 - 0.3 * t)[..., None, None]
    ang = math.pi * torch.rand((P, E), generator=gen, device="cuda", dtype=torch.float64)
    ca, sa = torch.cos(ang)[..., None, None], torch.sin(ang)[..., None, None]
    y, x = c[:, None], c[None, :]
    r2 = ((ca * x + sa * y) ** 2 + ((ca * y - sa * x) / flat) ** 2) / sigma ** 2
    total = lambda a: a / a.sum(dim=(-2, -1), keepdim=True)  # noqa: E731
    return total(0.5 * total(torch.exp(-0.5 * r2)) + 0.5 * total((1.0 + 0.25 * r2) ** -2.5))


def _sky64(i, xi, xa):
    """exp of the correlated field, cropped to the sky grid."""
    hartley = lambda a: (lambda f: f.real + f.imag)(torch.fft.fft2(a))  # noqa: E731
    log_s = (hartley(i["amp_ref"].double() * xi.double()) + ZERO_MODE)[None]
    if xa is not None:
        index = hartley(i["amp_alpha"].double() * xa.double()) + INDEX_MEAN
        log_s = log_s + index * i["dnu"].double()[:, None, None]
    return torch.exp(log_s)[:, :i["H"], :i["H"]].contiguous()


def _inputs(case, seed):
    """The arrays a program holds before the call, in the case's dtype."""
    gen = _generator(seed)
    dt = DTYPES[case["dtype"]]
    kind, H, E, n, m, M, S, N = (case[k] for k in ("kind", "H", "E", "n", "m", "M", "S", "N"))
    spectral = E > 1
    i = dict(case=case, H=H, w=2 * (H // n))
    i["dnu"] = torch.log(torch.linspace(1.0, 2.5, E, device="cuda", dtype=torch.float64)).to(dt)
    if kind != "response":
        amp = _amplitude(N)
        i["amp_ref"] = amp.to(dt)
        i["amp_alpha"] = (0.5 * amp).to(dt) if spectral else None
    true = _randn(gen, 2, N, N)
    near = true + 0.1 * _randn(gen, 2, N, N)
    i["xi"] = near[0].to(dt)
    i["xa"] = near[1].to(dt) if spectral else None
    if kind in ("grad", "kl", "metric", "solve", "points", "psf"):
        i["win"] = torch.stack([_psf_windows(gen, n, E, i["w"]).to(dt) for _ in range(M)])
    if kind == "dropin":
        # full frames with the PSF centre at pixel (0, 0), as the reference takes them
        full = torch.zeros((n * n, E, H, H), device="cuda", dtype=dt)
        c = (H - i["w"]) // 2
        full[..., c:c + i["w"], c:c + i["w"]] = _psf_windows(gen, n, E, i["w"]).to(dt)
        i["full"] = torch.fft.ifftshift(full, dim=(-2, -1)).contiguous()
    if kind in ("grad", "kl", "metric", "solve", "points", "response"):
        # exposure ramp in seconds, 5 % of the pixels masked, counts of the sky
        ramp = torch.linspace(5e2, 2e3, H, device="cuda", dtype=torch.float64)
        keep = torch.rand((M, E, H, H), generator=gen, device="cuda") >= 0.05
        i["expo"] = (ramp * keep).to(dt)
        if kind == "response":
            sky = torch.exp(-2.0 + 0.5 * _randn(gen, M, E, H, H))
            i["x"] = (sky * torch.exp(0.05 * _randn(gen, M, E, H, H))).to(dt)
        else:
            sky = _sky64(i, true[0], true[1] if spectral else None)[None]
        counts = torch.poisson((sky * ramp).expand(M, E, H, H).contiguous(), generator=gen)
        i["counts"] = torch.where(keep, counts, -torch.ones_like(counts)).to(torch.int32)
    if kind == "kl":
        i["dr"] = (0.1 * _randn(gen, S, N, N)).to(dt)
        i["da"] = (0.1 * _randn(gen, S, N, N)).to(dt) if spectral else None
    if kind in ("metric", "solve"):
        i["vr"] = _randn(gen, S, N, N).to(dt)
        i["va"] = _randn(gen, S, N, N).to(dt) if spectral else None
    if kind == "points":
        i["xp"] = _randn(gen, H, H).to(dt)
        i["xpa"] = _randn(gen, H, H).to(dt) if spectral else None
    if kind in ("psf", "dropin"):
        i["x"] = _sky64(i, i["xi"], i["xa"]).to(dt) if kind == "psf" else \
            torch.exp(-2.0 + _randn(gen, E, H, H)).to(dt)
        i["y"] = _randn(gen, E, H, H).to(dt)
    if kind == "gp":
        i["y"] = _randn(gen, E, H, H).to(dt)
    return i


def prepare(case, seed):
    i = _inputs(case, seed)
    dt = DTYPES[case["dtype"]]
    kind, H, E, n, m, M, S = (case[k] for k in ("kind", "H", "E", "n", "m", "M", "S"))
    st = dict(i)
    if kind in ("grad", "kl", "metric", "solve", "points", "gp"):
        st["sky"] = ja.CorrelatedFieldSky(case["N"], (H, H), i["amp_ref"], i["amp_alpha"],
                                          zm=ZERO_MODE, mu=INDEX_MEAN if E > 1 else 0.0,
                                          dnu=i["dnu"].double().cpu().numpy(), dtype=dt)
    if "win" in i:
        st["op"] = ja.LinpatchOperator((E, H, H), n, m, n_modules=M, dtype=dt)
        st["op"].set_kernel(i["win"] if M > 1 else i["win"][0], layout="window")
        del st["win"]
    if kind in ("grad", "kl", "metric", "solve", "points"):
        st["model"] = ja.XrayModel(st["sky"], st["op"], 1.0, i["expo"], i["counts"],
                                   max_samples=S)
    if kind in ("metric", "solve"):
        st["model"].nll_and_grad(i["xi"], i["xa"])  # the base point of the metric
    if kind == "solve":
        st["model"].reserve_solver()
    if kind == "points":
        st["model"].set_point_sources(POINTS["a"], POINTS["q"], POINTS["alpha_mean"],
                                      POINTS["alpha_std"])
    if kind == "dropin":
        st["domain"] = ja.Domain((E, H, H), (1.0, 1.0, 1.0))
    if kind == "response":
        keys = ["tm%d" % (k + 1) for k in range(M)]
        flags = (i["counts"] >= 0).cpu().numpy().astype(np.float64)
        st["exposure"] = ja.build_exposure_function(i["expo"])
        st["readout"] = ja.build_readout_function(flags, keys=keys)
        data = {k: c[c >= 0].to(dt) for k, c in zip(keys, i["counts"])}
        st["likelihood"] = ja.Poissonian(ja.Vector(data))
    return st


# --------------------------------------------------------------------- run
def run(st):
    kind = st["case"]["kind"]
    if kind == "grad":
        return st["model"].nll_and_grad(st["xi"], st["xa"])
    if kind == "kl":
        return ja.kl_value_and_grad(st["model"], st["xi"], st["xa"], st["dr"], st["da"])
    if kind == "metric":
        return st["model"].metric_batch(st["vr"], st["va"])
    if kind == "solve":
        return st["model"].metric_solve(st["vr"], st["va"], maxiter=CG_STEPS)[0]
    if kind == "points":
        return st["model"].nll_and_grad_points(st["xi"], st["xa"], st["xp"], st["xpa"])
    if kind == "psf":
        return st["op"].forward(st["x"]), st["op"].adjoint(st["y"])
    if kind == "dropin":
        c = st["case"]
        return ja.linpatch_convolve(st["x"], st["domain"], st["full"], c["n"], c["m"])
    if kind == "gp":
        s = st["sky"](st["xi"], st["xa"])
        return s, st["sky"].vjp(s, st["y"])
    # response: exposure, read-out, Poisson energy, and the gradient back
    lam = st["readout"](st["exposure"](st["x"]))
    energy, g = st["likelihood"].energy_and_gradient(lam)
    return energy, st["exposure"](st["readout"].transpose(g))


# -------------------------------------------------------------------- work
def work(case):
    """Inputs read once, outputs written once; FFT operations at 2.5 N log2 N
    per real 2-D transform."""
    kind, H, E, n, m, M, S, N = (case[k] for k in ("kind", "H", "E", "n", "m", "M", "S", "N"))
    es = 4 if case["dtype"] == "f32" else 8
    w = 2 * (H // n)
    L = w + 2 * m
    P, J, F = n * n, M * E, 2 if E > 1 else 1
    lat, img = N * N, H * H
    fft = lambda k: 2.5 * k * math.log2(k)  # noqa: E731
    gp = F * fft(N * N)                       # one direction of the sky
    psf = J * P * (2 * fft(L * L) + 3 * L * L)  # one direction of the PSF
    kern = J * P * w * w * es
    data = J * img * (es + 4)                 # exposure and counts
    if kind == "grad":
        return {"bytes": 3 * F * lat * es + kern + data, "flops": 2 * (gp + psf)}
    if kind == "kl":
        return {"bytes": (2 + S + 1) * F * lat * es + kern + data,
                "flops": S * 2 * (gp + psf)}
    if kind == "metric":
        # per tangent the tangent and the product; the base point's sky and rate once
        return {"bytes": (1 + 2 * S) * F * lat * es + kern + data + (E + J) * img * es,
                "flops": S * 2 * (gp + psf)}
    if kind == "solve":
        # every step applies the metric and must see its direction again
        step = 2 * S * F * lat * es + kern + data + (E + J) * img * es + F * lat * es
        return {"bytes": CG_STEPS * step, "flops": CG_STEPS * S * 2 * (gp + psf)}
    if kind == "points":
        return {"bytes": 3 * F * lat * es + 2 * F * img * es + kern + data,
                "flops": 2 * (gp + psf) + 200 * img}
    if kind == "psf":
        return {"bytes": 2 * kern + 4 * E * img * es, "flops": 2 * psf}
    if kind == "dropin":
        return {"bytes": kern + 2 * E * img * es, "flops": psf + J * P * fft(L * L)}
    if kind == "gp":
        return {"bytes": (4 * F * lat + 3 * E * img) * es, "flops": 2 * gp}
    return {"bytes": J * img * 6 * es, "flops": 10 * J * img}


# ------------------------------------------------------------------- exact
class _Psf64:
    """The linear-patching PSF in float64: windows of stride d with tent
    weights, circular convolution at the padded window length, overlap-add."""

    def __init__(self, win, H, n, m):
        self.win, self.H, self.n, self.m = win, H, n, m
        self.w = win.shape[-1]
        d = self.w // 2
        self.h = d // 2
        self.L = self.w + 2 * m
        ramp = torch.linspace(0.0, 1.0, d, device="cuda", dtype=torch.float64)
        tent = torch.cat([ramp, ramp.flip(0)])
        self.tent = tent[:, None] * tent[None, :]
        s = torch.tensor([min(k * d, H + 2 * self.h - self.w) for k in range(n)], device="cuda")
        p = torch.arange(n * n, device="cuda")
        self.px, self.py = s[p % n], s[p // n]

    def _index(self, side, width):
        a = torch.arange(side, device="cuda")
        return ((self.px[:, None, None] + a[:, None]) * width + self.py[:, None, None] + a)

    def _spectrum(self, e):
        k = torch.nn.functional.pad(self.win[:, e].double(), (self.m,) * 4)
        k = torch.fft.ifftshift(k / k.sum(dim=(-2, -1), keepdim=True), dim=(-2, -1))
        return torch.fft.rfft2(k)

    def _apply(self, z, e, conj):
        k = self._spectrum(e)
        return torch.fft.irfft2(torch.fft.rfft2(z) * (k.conj() if conj else k),
                                s=(self.L, self.L))

    def forward(self, x):
        pad, out = torch.nn.functional.pad, []
        for e in range(x.shape[0]):
            xp = pad(x[e], (self.h,) * 4)
            z = xp.reshape(-1)[self._index(self.w, xp.shape[-1])] * self.tent
            y = self._apply(pad(z, (self.m,) * 4), e, False)
            o = self.h + self.m
            side = self.H + 2 * o
            canvas = torch.zeros(side * side, device="cuda", dtype=torch.float64)
            canvas.index_add_(0, self._index(self.L, side).reshape(-1), y.reshape(-1))
            out.append(canvas.reshape(side, side)[o:o + self.H, o:o + self.H])
        return torch.stack(out)

    def adjoint(self, y):
        out = []
        for e in range(y.shape[0]):
            yp = torch.nn.functional.pad(y[e], (self.h + self.m,) * 4)
            z = self._apply(yp.reshape(-1)[self._index(self.L, yp.shape[-1])], e, True)
            z = z[:, self.m:self.m + self.w, self.m:self.m + self.w] * self.tent
            side = self.H + 2 * self.h
            canvas = torch.zeros(side * side, device="cuda", dtype=torch.float64)
            canvas.index_add_(0, self._index(self.w, side).reshape(-1), z.reshape(-1))
            out.append(canvas.reshape(side, side)[self.h:self.h + self.H,
                                                  self.h:self.h + self.H])
        return torch.stack(out)


def _hartley_back(i, u):
    """Cotangents of the latents for the cotangent u of the log sky."""
    N = i["case"]["N"]
    full = torch.zeros((u.shape[0], N, N), device="cuda", dtype=torch.float64)
    full[:, :u.shape[1], :u.shape[2]] = u
    hartley = lambda a: (lambda f: f.real + f.imag)(torch.fft.fft2(a))  # noqa: E731
    g_r = i["amp_ref"].double() * hartley(full.sum(0))
    if i["amp_alpha"] is None:
        return g_r, None
    dnu = i["dnu"].double()[:, None, None]
    return g_r, i["amp_alpha"].double() * hartley((full * dnu).sum(0))


def _response64(i, psfs, x):
    return torch.stack([p.forward(x) for p in psfs]) * i["expo"].double()


def _back64(i, psfs, cot):
    return sum(p.adjoint(c) for p, c in zip(psfs, cot * i["expo"].double()))


def _nll64(i, psfs, total):
    """NLL and the cotangent of the sky that the PSF sees."""
    lam = _response64(i, psfs, total)
    keep, d = i["counts"] >= 0, i["counts"].double()
    one = torch.ones_like(lam)
    safe = torch.where(keep, lam, one)
    nll = torch.where(keep, safe - d * torch.log(safe), 0 * one).sum()
    return float(nll), _back64(i, psfs, torch.where(keep, 1.0 - d / safe, 0 * one)), safe


def _grad64(i, psfs, xi, xa):
    s = _sky64(i, xi, xa)
    nll, xbar, _ = _nll64(i, psfs, s)
    return (nll,) + _hartley_back(i, s * xbar)


def _metric64(i, psfs):
    """v -> J^T diag(1 / lam) J v at the base point."""
    s = _sky64(i, i["xi"], i["xa"])
    keep = i["counts"] >= 0
    lam = torch.where(keep, _response64(i, psfs, s), torch.ones((), device="cuda",
                                                                dtype=torch.float64))

    def apply(vr, va):
        hartley = lambda a: (lambda f: f.real + f.imag)(torch.fft.fft2(a))  # noqa: E731
        dl = hartley(i["amp_ref"].double() * vr)[None]
        if va is not None:
            dl = dl + hartley(i["amp_alpha"].double() * va) * i["dnu"].double()[:, None, None]
        ds = s * dl[:, :i["H"], :i["H"]]
        cot = torch.where(keep, _response64(i, psfs, ds) / lam, torch.zeros_like(lam))
        return _hartley_back(i, s * _back64(i, psfs, cot))

    return apply


def _solve64(apply, br, ba):
    """CG_STEPS conjugate-gradient steps on (1 + metric) x = b from zero."""
    pack = lambda r, a: r[None] if a is None else torch.stack([r, a])  # noqa: E731
    b = pack(br, ba)
    x, r, p = torch.zeros_like(b), b, b
    rr = (r * r).sum()
    for _ in range(CG_STEPS):
        ap = p + pack(*apply(p[0], p[1] if ba is not None else None))
        alpha = rr / (p * ap).sum()
        x, r = x + alpha * p, r - alpha * ap
        new = (r * r).sum()
        p, rr = r + new / rr * p, new
    return x


def _invgamma64(xi):
    """Point-source brightness q / y with Q(a, y) = Phi(xi), and its
    logarithmic derivative; y by bisection in its logarithm."""
    a = torch.full_like(xi, POINTS["a"])
    lo, hi = torch.full_like(xi, -60.0), torch.full_like(xi, 8.0)
    phi = lambda t: 0.5 * torch.special.erfc(-t * math.sqrt(0.5))  # noqa: E731
    small, large = phi(-xi), phi(xi)
    for _ in range(64):
        t = 0.5 * (lo + hi)
        y = torch.exp(t)
        above = torch.where(xi > 0, torch.special.gammainc(a, y) > small,
                            torch.special.gammaincc(a, y) < large)
        lo, hi = torch.where(above, lo, t), torch.where(above, t, hi)
    t = 0.5 * (lo + hi)
    dlog = torch.exp(-0.5 * xi ** 2 - 0.5 * math.log(2 * math.pi) + math.lgamma(POINTS["a"])
                     - POINTS["a"] * t + torch.exp(t))
    return POINTS["q"] * torch.exp(-t), dlog


def _points64(i, psfs):
    dnu = i["dnu"].double()[:, None, None]
    s = _sky64(i, i["xi"], i["xa"])
    bright, dlog = _invgamma64(i["xp"].double())
    alpha = 0.0 if i["xpa"] is None else \
        POINTS["alpha_mean"] + POINTS["alpha_std"] * i["xpa"].double()
    p = bright[None] * torch.exp(alpha * dnu) if i["xpa"] is not None else bright[None]
    nll, xbar, _ = _nll64(i, psfs, s + p)
    g_r, g_a = _hartley_back(i, s * xbar)
    g_pa = None if i["xpa"] is None else POINTS["alpha_std"] * (p * xbar * dnu).sum(0)
    return nll, g_r, g_a, dlog * (p * xbar).sum(0), g_pa


def exact(case, seed):
    i = _inputs(case, seed)
    kind, n, m, S = case["kind"], case["n"], case["m"], case["S"]
    psfs = [_Psf64(win, i["H"], n, m) for win in i["win"]] if "win" in i else None
    if kind == "grad":
        return _grad64(i, psfs, i["xi"], i["xa"])
    if kind == "kl":
        value, g_r, g_a = 0.0, 0.0, 0.0
        for s in range(S):
            # the positions are sums in the case's dtype, as the call forms them
            xr = (i["xi"] + i["dr"][s]).double()
            xa = None if i["xa"] is None else (i["xa"] + i["da"][s]).double()
            nll, a, b = _grad64(i, psfs, xr, xa)
            prior = 0.5 * float((xr ** 2).sum() + (0.0 if xa is None else (xa ** 2).sum()))
            value += (nll + prior) / S
            g_r = g_r + (a + xr) / S
            g_a = None if xa is None else g_a + (b + xa) / S
        return value, (g_r, g_a)
    if kind == "metric":
        apply = _metric64(i, psfs)
        out = [apply(i["vr"][s].double(), None if i["va"] is None else i["va"][s].double())
               for s in range(S)]
        return (torch.stack([o[0] for o in out]),
                None if i["va"] is None else torch.stack([o[1] for o in out]))
    if kind == "solve":
        apply = _metric64(i, psfs)
        out = [_solve64(apply, i["vr"][s].double(),
                        None if i["va"] is None else i["va"][s].double()) for s in range(S)]
        return (torch.stack([o[0] for o in out]),
                None if i["va"] is None else torch.stack([o[1] for o in out]))
    if kind == "points":
        return _points64(i, psfs)
    if kind == "psf":
        return psfs[0].forward(i["x"].double()), psfs[0].adjoint(i["y"].double())
    if kind == "dropin":
        w, c = i["w"], (i["H"] - i["w"]) // 2
        win = torch.fft.fftshift(i["full"], dim=(-2, -1))[..., c:c + w, c:c + w]
        return _Psf64(win, i["H"], n, m).forward(i["x"].double())
    if kind == "gp":
        s = _sky64(i, i["xi"], i["xa"])
        return s, _hartley_back(i, s * i["y"].double())
    lam = i["x"].double() * i["expo"].double()
    keep, d = i["counts"] >= 0, i["counts"].double()
    safe = torch.where(keep, lam, torch.ones_like(lam))
    zero = torch.zeros_like(lam)
    energy = torch.where(keep, safe - d * torch.log(safe), zero).sum()
    return float(energy), torch.where(keep, 1.0 - d / safe, zero) * i["expo"].double()
