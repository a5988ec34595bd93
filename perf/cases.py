"""The work that a user of this package has it do, as cases that can be timed and compared.

``listed()`` holds the cases, ``draw(rng)`` gives more of the same ranges, ``prepare(case, seed)`` builds what a
program holds before the call (inputs, plans), ``run(state)`` is one pass through the public classes, ``work(case)``
says what a pass cannot do without and ``exact(case, seed)`` is the same result in 64 bits from plain torch.

Kinds of case:
  prop      Propagation.D (and DT of its result) of a stack of fields at each distance
  radon     Tomo.R, Tomo.RT, Tomo.fbp, or R followed by RT, on a slab of slices
  shift     Shift.coeff, S, Sadj on a stack of planes, with ``deriv`` also dS, d2S and the adjoint differential
  gradient  Rec.gradients_fused of a chunk of angles where the fused passes take the detector size, else
            Rec.gradients_cascade (the choice that Rec.gradients makes)
  bilinear  Rec.hessian_pair_fused or Rec.hessian_fused of a chunk of angles
"""
import math
from types import SimpleNamespace

import numpy as np
import torch

DEV = "cuda"

# the reference's synthetic test geometry, four focus-to-sample distances (m)
_Z1 = (5.110e-3, 5.464e-3, 6.879e-3, 9.817e-3)
_F2D = 1.217
_ENERGY = 17.1
_PIXEL = 1.4760147601476e-6 * 2


def listed():
    return [
        # one small field through one propagator: an interactive call, launch latency
        dict(name="prop_256_one", kind="prop", n=256, nz=256, batch=1, ndist=1, both=False),
        # a stack of small fields, D then DT at four distances: the operator benchmark's size
        dict(name="prop_256_b16_d4", kind="prop", n=256, nz=256, batch=16, ndist=4, both=True),
        # full-size detector fields: one distance of a 16-angle chunk
        dict(name="prop_2048_b16", kind="prop", n=2048, nz=2048, batch=16, ndist=1, both=True),
        # a binned detector that is not a power of two
        dict(name="prop_1536_b4", kind="prop", n=1536, nz=1536, batch=4, ndist=1, both=True),
        # the Radon transform of a whole volume and its adjoint: the operator benchmark's size
        dict(name="radon_R_256", kind="radon", op="R", n=256, nz=256, ntheta=384, real=False),
        dict(name="radon_RT_256", kind="radon", op="RT", n=256, nz=256, ntheta=384, real=False),
        # filtered back-projection of a real sinogram, an odd slab of slices and an odd number of angles
        dict(name="radon_fbp_512_real", kind="radon", op="fbp", n=512, nz=45, ntheta=451, real=True),
        # a request of the serving mix: R and RT of eight slices at few angles
        dict(name="radon_slab8_512", kind="radon", op="RRT", n=512, nz=8, ntheta=64, real=False),
        # prefilter, shift and adjoint shift of a stack of projections: the operator benchmark's size
        dict(name="shift_256_b384", kind="shift", n=256, nz=256, npsi=256, nzpsi=256, batch=384, real=False,
             deriv=False),
        # gradient request of the serving mix at its commonest grid
        dict(name="gradient_256_a48_d2", kind="gradient", n=256, nobj=256, ndist=2, angles=48, real=False),
        # the headline gradient: 2048^2 detector, 4 distances, 1024^2 object plane, 16 angles
        dict(name="gradient_2048_a16_d4", kind="gradient", n=2048, nobj=1024, ndist=4, angles=16, real=False),
        # the two bilinear forms of the solver's beta step at a 1024^2 detector, one chunk of angles
        dict(name="bilinear_1024_a16_d4", kind="bilinear", form="pair", n=1024, nobj=512, ndist=4, angles=16,
             real=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _even(x, lo):
    return max(lo, int(x) // 2 * 2)


def _length(rng, lo, hi):
    """An even transform length over its logarithm; real sizes have no large prime factor (at most 67 here)."""
    while True:
        x = m = _even(_log_int(rng, lo, hi), lo)
        for p in range(2, 68):
            while m % p == 0:
                m //= p
        if m == 1:
            return x


def draw(rng):
    """One more case of the listed ranges: sizes over their logarithm, even, odd and ragged ones among them."""
    kind = rng.choices(["prop", "radon", "shift", "gradient", "bilinear"], [3, 3, 2, 3, 2])[0]
    pow2 = rng.random() < 0.6
    if kind == "prop":
        if pow2:
            n = nz = rng.choice([256, 512, 1024, 2048])
        else:
            n, nz = _length(rng, 96, 2500), _length(rng, 96, 2500)
        batch = min(_log_int(rng, 1, 64), max(1, 16 * 2048 * 2048 // (n * nz)))
        if n & (n - 1) or nz & (nz - 1):  # lengths that are not powers of two cost more a point
            batch = min(batch, max(1, 4 * 1536 * 1536 // (n * nz)))
        return dict(kind=kind, n=n, nz=nz, batch=batch, ndist=rng.randint(1, 4), both=rng.random() < 0.7)
    if kind == "radon":
        n = rng.choice([128, 256, 512]) if pow2 else _length(rng, 96, 640)
        ntheta = min(_log_int(rng, 16, 720), 512 * 451 // n)
        nz = min(_log_int(rng, 1, 256), 256 ** 3 // (n * n))
        return dict(kind=kind, op=rng.choice(["R", "RT", "fbp", "RRT"]), n=n, nz=nz, ntheta=ntheta,
                    real=rng.random() < 0.4)
    if kind == "shift":
        n, nz = _log_int(rng, 128, 1024), _log_int(rng, 128, 1024)
        if pow2:
            n = nz = rng.choice([256, 512, 1024])
        npsi, nzpsi = _even(n * rng.uniform(0.6, 1.3), 96), _even(nz * rng.uniform(0.6, 1.3), 96)
        most = max(1, 384 * 256 * 256 // max(n * nz, npsi * nzpsi))
        deriv = rng.random() < 0.4
        return dict(kind=kind, n=n, nz=nz, npsi=npsi, nzpsi=nzpsi, batch=min(_log_int(rng, 2, 384), most),
                    real=rng.random() < 0.4, deriv=deriv)
    ndist = rng.randint(1, 4)
    if kind == "gradient":
        n = rng.choice([128, 256, 512, 1024, 2048])
        other = rng.random() < 0.15  # detector sizes that the fused passes do not take
        if other:
            n = rng.choice([384, 600, 768, 1000])
        nobj = rng.choice([n, n // 2, _even(n * rng.uniform(0.5, 1.0), 64)])
        most = 2 ** 22 if other else 16 * 4 * 2 ** 22
        angles = min(_log_int(rng, 1, 128), max(1, most // (ndist * n * n)))
        return dict(kind=kind, n=n, nobj=nobj, ndist=ndist, angles=angles, real=rng.random() < 0.3)
    n = rng.choice([128, 256, 512, 1024])
    nobj = rng.choice([n, n // 2, _even(n * rng.uniform(0.5, 1.0), 64)])
    angles = min(_log_int(rng, 1, 64), max(1, 16 * 4 * 2 ** 20 // (ndist * n * n)))
    return dict(kind=kind, form=rng.choice(["pair", "same", "general"]), n=n, nobj=nobj, ndist=ndist, angles=angles,
                real=rng.random() < 0.3)


# ---- inputs -------------------------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _grid(nz, n):
    y = torch.arange(nz, device=DEV, dtype=torch.float32)[:, None] / nz - 0.5
    x = torch.arange(n, device=DEV, dtype=torch.float32)[None, :] / n - 0.5
    return y, x


def _ellipses(g, nz, n, count=20):
    """Sum of random filled ellipses of amplitude U[0, 1] on a [nz, n] grid."""
    y, x = _grid(nz, n)
    p = torch.rand((count, 6), device=DEV, generator=g).tolist()
    out = torch.zeros((nz, n), device=DEV)
    for cy, cx, ay, ax, t, a in p:
        c, s = math.cos(math.pi * t), math.sin(math.pi * t)
        dy, dx = y - 0.6 * (cy - 0.5), x - 0.6 * (cx - 0.5)
        u, v = dx * c + dy * s, dy * c - dx * s
        out += a * ((u / (0.03 + 0.17 * ax)) ** 2 + (v / (0.03 + 0.17 * ay)) ** 2 <= 1)
    return out


def _phases(g, batch, nz, n):
    """[batch, nz, n] ellipse phases, shifted from plane to plane, with a little noise."""
    base = _ellipses(g, nz, n)
    out = torch.empty((batch, nz, n), device=DEV)
    for b in range(batch):
        out[b] = torch.roll(base, ((5 * b) % nz, (3 * b) % n), (0, 1))
    return out + 0.02 * torch.randn(out.shape, device=DEV, generator=g)


def _fields(g, batch, nz, n):
    ph = _phases(g, batch, nz, n)
    return torch.polar(torch.exp(-0.1 * ph), ph)


def _probe(g, ndist, nz, n):
    y, x = _grid(nz, n)
    amp = torch.exp(-(x * x + y * y) / (2 * 0.3 ** 2))
    out = torch.empty((ndist, nz, n), dtype=torch.complex64, device=DEV)
    for j in range(ndist):
        a = (2 * torch.rand((8, 2), device=DEV, generator=g) - 1).tolist()
        ph = sum(0.2 * torch.cos(2 * math.pi * (4 * p * x + 4 * q * y) + p - q) for p, q in a)
        out[j] = torch.polar(amp, ph)
    return out


def _planes(g, batch, nz, n, real, scale=1.0):
    ph = scale * _phases(g, batch, nz, n)
    return ph if real else torch.complex(ph, 0.01 * ph)


def _physics(n, ndist):
    z1 = np.array(_Z1[:ndist], dtype=np.float64)
    pixel = _PIXEL * (2048.0 / n)
    mag = _F2D / z1
    norm = mag / mag[0]
    return SimpleNamespace(z1=z1, pixel=pixel, wavelength=1.24e-09 / _ENERGY,
                           distance=(z1 * (_F2D - z1)) / _F2D * norm ** 2, voxelsize=pixel / mag[0],
                           demag=(1.0 / norm).astype(np.float32))


def _theta(ntheta):
    return np.arange(ntheta) * math.pi / ntheta


def _inputs(case, seed):
    """The case's arrays on the GPU, from the seed alone and from plain torch."""
    g, c = _gen(seed), SimpleNamespace(**case)
    if c.kind == "prop":
        return SimpleNamespace(x=_fields(g, c.batch, c.nz, c.n))
    if c.kind == "radon":
        y, x = _grid(c.n, c.n)
        obj = _planes(g, c.nz, c.n, c.n, c.real) * (x * x + y * y < 0.23)
        if c.op in ("R", "RRT"):
            return SimpleNamespace(x=obj)
        # sinograms: the smooth traces that a sum of ellipses leaves on the detector, with noise
        k = torch.arange(c.ntheta, device=DEV)[:, None] * (math.pi / c.ntheta)
        t = (torch.arange(c.n, device=DEV)[None, :] / c.n - 0.5)
        p = torch.rand((12, 4), device=DEV, generator=g).tolist()
        trace = torch.zeros((c.ntheta, c.n), device=DEV)
        for a, r, w, q in p:
            d = t - 0.35 * r * torch.cos(k + 2 * math.pi * q)
            trace += a * torch.sqrt(torch.clamp(1 - (d / (0.03 + 0.1 * w)) ** 2, min=0))
        z = 0.5 + torch.rand((c.nz,), device=DEV, generator=g)
        s = trace[:, None, :] * z[None, :, None]
        s = s + 0.01 * torch.randn(s.shape, device=DEV, generator=g)
        return SimpleNamespace(x=s.contiguous() if c.real else torch.complex(s, 0.01 * s))
    if c.kind == "shift":
        m = 1.0 + 0.9 * torch.rand((c.batch,), device=DEV, generator=g)
        if c.n == c.npsi and c.nz == c.nzpsi:
            m = torch.ones_like(m)
        two = lambda amp: amp * (2 * torch.rand((c.batch, 2), device=DEV, generator=g) - 1)  # noqa: E731
        s = SimpleNamespace(psi=_planes(g, c.batch, c.nzpsi, c.npsi, c.real), r=two(5.0), m=m,
                            g=_planes(g, c.batch, c.nz, c.n, c.real))
        if c.deriv:
            s.psi1 = _planes(g, c.batch, c.nzpsi, c.npsi, c.real, 0.1)
            s.dr = two(0.3)
        return s
    ph = _physics(c.n, c.ndist)
    s = SimpleNamespace(prb=_probe(g, c.ndist, c.n, c.n), proj=_planes(g, c.angles, c.nobj, c.nobj, c.real, 0.5))
    s.pos = 3 * (2 * torch.rand((c.angles, c.ndist, 2), device=DEV, generator=g) - 1)
    # measured amplitudes: of the true variables, which are off from the current ones, with noise
    s.data = torch.empty((c.angles, c.ndist, c.n, c.n), device=DEV)
    tpos = s.pos + 0.3 * torch.randn(s.pos.shape, device=DEV, generator=g)
    for b in range(c.angles):
        co = _coeff(1.25 * s.proj[b])
        for j in range(c.ndist):
            wy, wx = (_taps(c.n, c.nobj, float(ph.demag[j]), float(tpos[b, j, k]), 0).to(co.dtype) for k in (0, 1))
            e = torch.exp(1j * (wy @ co @ wx.T))
            x0 = _fresnel(1.1 * s.prb[j] * e, ph.wavelength, ph.voxelsize, ph.distance[j], False)
            noise = 1 + 0.01 * torch.randn((c.n, c.n), device=DEV, generator=g)
            s.data[b, j] = x0.abs() * noise
    if c.kind == "bilinear":
        for k, f in (("y", 1.0), ("z", 0.7)):
            d = dict(prb=f * 0.1 * torch.flip(s.prb, (1,)).contiguous(),
                     proj=_planes(g, c.angles, c.nobj, c.nobj, c.real, 0.05 * f),
                     pos=0.3 * f * torch.randn(s.pos.shape, device=DEV, generator=g))
            setattr(s, k, d)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s.case = c = SimpleNamespace(**case)
    if c.kind == "prop":
        from holotomocupy_amd import Propagation
        ph = _physics(c.n, c.ndist)
        s.prop = Propagation(c.n, c.nz, c.batch, c.ndist, ph.wavelength, ph.voxelsize, ph.distance)
    elif c.kind == "radon":
        from holotomocupy_amd import Tomo
        s.tomo = Tomo(c.n, c.nz, _theta(c.ntheta), 0)
    elif c.kind == "shift":
        from holotomocupy_amd import Shift
        s.shift = Shift(c.n, c.npsi, c.nz, c.nzpsi, "float32" if c.real else "complex64", c.batch)
    else:
        from holotomocupy_amd.rec import Rec
        ph = _physics(c.n, c.ndist)
        s.rec = Rec(SimpleNamespace(energy=_ENERGY, detector_pixelsize=ph.pixel, focustodetectordistance=_F2D,
                                    z1=ph.z1, ndist=c.ndist, ntheta=c.angles, nz=c.n, n=c.n, nzobj=c.nobj,
                                    nobj=c.nobj, obj_dtype="float32" if c.real else "complex64",
                                    rho=[1.0, 0.05, 0.02]))
        s.vars = dict(prb=s.prb, proj=s.proj, pos=s.pos)
        s.grads = {k: torch.zeros_like(v) for k, v in s.vars.items()}
        s.fused = s.rec.fused_available()
    return s


def run(s):
    c = s.case
    if c.kind == "prop":
        out = []
        for j in range(c.ndist):
            out.append(s.prop.D(s.x, j))
            if c.both:
                out.append(s.prop.DT(out[-1], j))
        return out
    if c.kind == "radon":
        if c.op == "R":
            return s.tomo.R(s.x)
        if c.op == "RT":
            return s.tomo.RT(s.x)
        if c.op == "fbp":
            return s.tomo.fbp(s.x)
        sino = s.tomo.R(s.x)
        return [sino, s.tomo.RT(sino)]
    if c.kind == "shift":
        co = s.shift.coeff(s.psi)
        out = [co, s.shift.S(co, s.r, s.m), s.shift.Sadj(s.g, s.r, s.m)]
        if c.deriv:
            c1 = s.shift.coeff(s.psi1)
            out.append(s.shift.dcurlySc(co, s.r, s.m, c1, s.dr))
            out.append(s.shift.d2curlySc(co, s.r, s.m, c1, s.dr, c1, s.dr))
            out += s.shift.dcurlySadjc(co, s.r, s.m, s.g)
        return out
    if c.kind == "gradient":
        s.grads["prb"].zero_()
        (s.rec.gradients_fused if s.fused else s.rec.gradients_cascade)(s.vars, s.grads, s.data)
        return s.grads
    # the forms of an FP32 computation, rounded to it as the step lengths that they give are
    if c.form == "pair":
        return s.rec.hessian_pair_fused(s.vars, s.y, s.z, s.data).float()
    return s.rec.hessian_fused(s.vars, s.y, s.y if c.form == "same" else s.z, s.data).float()


def work(case):
    c = SimpleNamespace(**case)
    fft = lambda n: 5.0 * n * math.log2(n)  # noqa: E731
    if c.kind == "prop":
        field, calls = c.n * c.nz, c.batch * c.ndist * (2 if c.both else 1)
        ops = calls * (2 * c.nz * fft(c.n) + 2 * c.n * fft(c.nz) + 28.0 * field)
        # x read once, every result written once (D's result is DT's input)
        return dict(bytes=8.0 * field * (c.batch + calls), flops=ops)
    if c.kind == "radon":
        size = 4 if c.real else 8
        vol, sino = c.nz * c.n * c.n, c.ntheta * c.nz * c.n
        ops = c.nz * (3 * c.n * fft(2 * c.n)) + c.ntheta * c.nz * fft(c.n) + 81 * 4.0 * sino
        if c.op == "RRT":
            return dict(bytes=float(size * (2 * vol + sino)), flops=2 * ops)
        return dict(bytes=float(size * (vol + sino)), flops=ops)
    if c.kind == "shift":
        size, k = (4, 1) if c.real else (8, 2)
        fo, f = c.batch * c.npsi * c.nzpsi, c.batch * c.n * c.nz
        nbytes = size * (fo + fo + f + f + fo)
        ops = k * (2 * 50.0 * fo + 2 * 40.0 * f)
        if c.deriv:
            nbytes += size * (fo + fo + f + f + fo)
            ops += k * (50.0 * fo + 2 * 4 * 32.0 * f)
        return dict(bytes=float(nbytes), flops=ops)
    size = 4 if c.real else 8
    f, fo, a, nd = c.n * c.n, c.nobj * c.nobj, c.angles, c.ndist
    line = 2 * c.n * fft(c.n)
    if c.kind == "gradient":
        # projections read and their gradient written, data read, probe read and its gradient written
        nbytes = 2 * size * a * fo + 4 * a * nd * f + 2 * 8 * nd * f
        return dict(bytes=float(nbytes), flops=a * nd * (4 * line + 250.0 * f))
    nf, np_ = {"pair": (5, 3), "general": (4, 3), "same": (3, 2)}[c.form]
    return dict(bytes=float(np_ * size * a * fo + 4 * a * nd * f + np_ * 8 * nd * f),
                flops=a * nd * nf * (2 * line + 80.0 * f))


# ---- the same results in 64 bits, from plain torch ----------------------------------------------------------------


def _fresnel(x, wavelength, voxelsize, z, adjoint):
    """crop(IFFT2(FFT2(symmetric pad x) exp(-i pi wavelength z f^2))), one axis after the other; DT conjugates."""
    for axis in (-1, -2):
        n = x.shape[axis]
        f = torch.fft.fftfreq(2 * n, d=voxelsize, dtype=torch.float64, device=x.device)
        ph = (1.0 if adjoint else -1.0) * math.pi * wavelength * z * f * f
        k = torch.polar(torch.ones_like(ph), ph).to(x.dtype)
        x = x.movedim(axis, -1)
        x = torch.fft.ifft(torch.fft.fft(torch.cat([x, x.flip(-1)], -1)) * k)[..., :n].movedim(-1, axis)
    return x


def _coeff(x):
    """Periodic cubic B-spline prefilter: the inverse of the periodic [1 4 1] filter along both axes."""
    real = not x.is_complex()
    d = [4 + 2 * torch.cos(2 * math.pi * torch.arange(n, device=x.device, dtype=torch.float64) / n)
         for n in x.shape[-2:]]
    y = torch.fft.ifft2(torch.fft.fft2(x) / (d[0][:, None] * d[1][None, :]).to(x.real.dtype))
    return y.real if real else y


def _taps(npix, npsi, m, r, order):
    """[npix, npsi] matrix of 6 beta3 (or its derivative of that order) at x = m (t - npix/2) - r + (m-1)/2 + npsi/2."""
    t = torch.arange(npix, device=DEV, dtype=torch.float64)
    x = m * (t - npix // 2) - r + (m - 1) / 2 + npsi // 2
    fx = torch.floor(x)
    d = x - fx
    u = 1 - d
    w = ((u ** 3, 4 - 6 * d * d + 3 * d ** 3, 4 - 6 * u * u + 3 * u ** 3, d ** 3),
         (-3 * u * u, -12 * d + 9 * d * d, 12 * u - 9 * u * u, 3 * d * d),
         (6 * u, -12 + 18 * d, -12 + 18 * u, 6 * d))[order]
    out = torch.zeros((npix, npsi), device=DEV, dtype=torch.float64)
    row = torch.arange(npix, device=DEV)
    for j in range(4):
        col = fx.long() + j - 1
        ok = (col >= 0) & (col < npsi)
        out[row[ok], col[ok]] = w[j][ok]
    return out


def _up(x):
    return x.to(torch.complex128 if x.is_complex() else torch.float64)


def _gridding(n, ntheta):
    """Taps of the polar samples on the 2n grid: first-tap rows and columns and the 2m + 1 weights along each."""
    mu = -math.log(1e-3) / (2.0 * n * n)
    m = math.ceil(2 * n / math.pi * math.sqrt(-mu * math.log(1e-3) + (mu * n) ** 2 / 4))
    th = torch.from_numpy(_theta(ntheta).astype(np.float32).astype(np.float64)).to(DEV)[:, None]
    t = (torch.arange(n, device=DEV, dtype=torch.float64)[None, :] - n // 2) / n
    x, y = (t * torch.cos(th)).reshape(-1), (-t * torch.sin(th)).reshape(-1)
    i = torch.arange(2 * m + 1, device=DEV)
    bx, by = (torch.floor(2 * n * v).long() - m for v in (x, y))
    wx, wy = (torch.exp(-math.pi ** 2 / mu * ((b[:, None] + i) / (2.0 * n) - v[:, None]) ** 2)
              for b, v in ((bx, x), (by, y)))
    return mu, m, (by[:, None] + i + n) % (2 * n), (bx[:, None] + i + n) % (2 * n), wy * math.pi / mu, wx


def _radon_parts(n, ntheta):
    mu, m, gy, gx, wy, wx = _gridding(n, ntheta)
    p = torch.arange(n, device=DEV, dtype=torch.float64) / n - 0.5
    phi = torch.exp(mu * n * n * (p[:, None] ** 2 + p[None, :] ** 2)) * (1 - n % 4) / (n * math.sqrt(n * ntheta))
    s = lambda k: 1.0 - 2.0 * (torch.arange(k, device=DEV) % 2).double()  # noqa: E731
    c2 = s(2 * n)[:, None] * s(2 * n)[None, :]
    return m, gy, gx, wy, wx, phi, -s(n), c2


def _radon(obj, ntheta):
    nz, n = obj.shape[0], obj.shape[-1]
    m, gy, gx, wy, wx, phi, c1, c2 = _radon_parts(n, ntheta)
    out = torch.empty((ntheta, nz, n), dtype=torch.complex128, device=DEV)
    for z0 in range(0, nz, 16):
        x = obj[z0:z0 + 16]
        emb = torch.zeros((x.shape[0], 2 * n, 2 * n), dtype=torch.complex128, device=DEV)
        emb[:, n // 2:n // 2 + n, n // 2:n // 2 + n] = x * phi
        grid = (torch.fft.fft2(emb * c2) * c2).reshape(x.shape[0], -1).T.contiguous()
        acc = torch.zeros((ntheta * n, x.shape[0]), dtype=torch.complex128, device=DEV)
        for a in range(2 * m + 1):
            for b in range(2 * m + 1):
                acc += grid[gy[:, a] * 2 * n + gx[:, b]] * (wy[:, a] * wx[:, b])[:, None]
        acc = acc.reshape(ntheta, n, -1).transpose(1, 2)
        out[:, z0:z0 + 16] = c1 * torch.fft.ifft(c1 * acc / n) / 4
    return out if obj.is_complex() else out.real.contiguous()


def _radon_adj(data, filt=None):
    ntheta, nz, n = data.shape
    m, gy, gx, wy, wx, phi, c1, c2 = _radon_parts(n, ntheta)
    if filt is not None:
        y = torch.fft.ifft(filt * torch.fft.fft(data))
        data = y if data.is_complex() else y.real
    out = torch.empty((nz, n, n), dtype=torch.complex128, device=DEV)
    for z0 in range(0, nz, 16):
        s = (c1 * torch.fft.fft(c1 * data[:, z0:z0 + 16])).transpose(1, 2).reshape(ntheta * n, -1)
        grid = torch.zeros((4 * n * n, 2 * s.shape[1]), dtype=torch.float64, device=DEV)
        s = torch.view_as_real(s.contiguous()).reshape(ntheta * n, -1)
        for a in range(2 * m + 1):
            for b in range(2 * m + 1):
                grid.index_add_(0, gy[:, a] * 2 * n + gx[:, b], s * (wy[:, a] * wx[:, b])[:, None])
        grid = torch.view_as_complex(grid.reshape(4 * n * n, -1, 2)).T.reshape(-1, 2 * n, 2 * n)
        full = torch.fft.ifft2(grid * c2) * c2
        out[z0:z0 + 16] = full[:, n // 2:n // 2 + n, n // 2:n // 2 + n] * phi
    return out if data.is_complex() else out.real.contiguous()


def _exact_shift(c, s):
    B, cplx = c.batch, not c.real
    dt = torch.complex128 if cplx else torch.float64
    co, g = _coeff(_up(s.psi)), _up(s.g)
    r, m = s.r.double().tolist(), s.m.double().tolist()
    S = torch.empty((B, c.nz, c.n), dtype=dt, device=DEV)
    Sadj = torch.empty((B, c.nzpsi, c.npsi), dtype=dt, device=DEV)
    if c.deriv:
        c1, dr = _coeff(_up(s.psi1)), s.dr.double().tolist()
        d1, d2, out2 = torch.empty_like(S), torch.empty_like(S), torch.empty((B, 2), dtype=torch.float64, device=DEV)
    for b in range(B):
        Y = [_taps(c.nz, c.nzpsi, m[b], r[b][0], k).to(dt) for k in range(3 if c.deriv else 1)]
        X = [_taps(c.n, c.npsi, m[b], r[b][1], k).to(dt) for k in range(3 if c.deriv else 1)]
        S[b] = Y[0] @ co[b] @ X[0].T
        Sadj[b] = Y[0].T @ g[b] @ X[0]
        if c.deriv:
            dy, dx = dr[b]
            cy, cx = Y[1] @ co[b] @ X[0].T, Y[0] @ co[b] @ X[1].T
            d1[b] = Y[0] @ c1[b] @ X[0].T - dx * cx - dy * cy
            first = dx * (Y[0] @ c1[b] @ X[1].T) + dy * (Y[1] @ c1[b] @ X[0].T)
            d2[b] = (dx * dx * (Y[0] @ co[b] @ X[2].T) + 2 * dx * dy * (Y[1] @ co[b] @ X[1].T)
                     + dy * dy * (Y[2] @ co[b] @ X[0].T) - 2 * first)
            for k, t in ((0, cy), (1, cx)):
                out2[b, k] = -(g[b].conj() * t).sum().real if cplx else -(g[b] * t).sum()
    return [co, S, Sadj] + ([d1, d2, Sadj, out2] if c.deriv else [])


def _exact_gradient(c, s, ph):
    rho, size = (1.0, 0.05, 0.02), c.angles * c.ndist * c.n * c.n
    prb, proj = _up(s.prb), _up(s.proj)
    gprb, gproj = torch.zeros_like(prb), torch.empty_like(proj)
    gpos = torch.empty((c.angles, c.ndist, 2), dtype=torch.float64, device=DEV)
    for b in range(c.angles):
        co = _coeff(proj[b])
        acc = torch.zeros_like(co)
        for j in range(c.ndist):
            m, r = float(ph.demag[j]), s.pos[b, j].double().tolist()
            Y, X = ([_taps(c.n, c.nobj, m, r[a], k).to(co.dtype) for k in (0, 1)] for a in (0, 1))
            e = torch.exp(1j * (Y[0] @ co @ X[0].T))
            x0 = _fresnel(prb[j] * e, ph.wavelength, ph.voxelsize, ph.distance[j], False)
            y0 = 2.0 / size * (x0 - s.data[b, j].double() * x0 / x0.abs())
            y12 = _fresnel(y0, ph.wavelength, ph.voxelsize, ph.distance[j], True)
            gprb[j] += y12 * e.conj()
            y22 = -1j * y12 * prb[j].conj() * e.conj()
            y22 = y22.real if c.real else y22
            acc += Y[0].T @ y22 @ X[0]
            for k, t in ((0, Y[1] @ co @ X[0].T), (1, Y[0] @ co @ X[1].T)):
                gpos[b, j, k] = -((y22 * t).sum() if c.real else (y22 * t.conj()).sum().real)
        gproj[b] = _coeff(acc)
    return dict(prb=gprb * rho[1] ** 2, proj=gproj * rho[0] ** 2, pos=gpos * rho[2] ** 2)


def _exact_bilinear(c, s, ph):
    size = c.angles * c.ndist * c.n * c.n
    dirs = [s.y, s.y if c.form == "same" else s.z]
    pairs = [(0, 1), (1, 1)] if c.form == "pair" else [(0, 1)]
    tot = [0.0 for _ in pairs]
    for b in range(c.angles):
        co, cd = _coeff(_up(s.proj[b])), [_coeff(_up(d["proj"][b])) for d in dirs]
        for j in range(c.ndist):
            m, r = float(ph.demag[j]), s.pos[b, j].double().tolist()
            Y, X = ([_taps(c.n, c.nobj, m, r[a], k).to(co.dtype) for k in (0, 1, 2)] for a in (0, 1))
            dr = [d["pos"][b, j].double().tolist() for d in dirs]
            sh = lambda v, p, q: Y[p] @ v @ X[q].T  # noqa: E731
            D = lambda v: _fresnel(v, ph.wavelength, ph.voxelsize, ph.distance[j], False)  # noqa: E731
            p, e = _up(s.prb[j]), torch.exp(1j * sh(co, 0, 0))
            pd = [_up(d["prb"][j]) for d in dirs]
            cx, cy = sh(co, 0, 1), sh(co, 1, 0)
            v22 = [sh(cd[k], 0, 0) - dr[k][1] * cx - dr[k][0] * cy for k in (0, 1)]
            v12 = [1j * e * v for v in v22]
            x0 = D(p * e)
            f0 = [D(pd[k] * e + p * v12[k]) for k in (0, 1)]
            a, d = x0.abs(), s.data[b, j].double()
            for i, (y, z) in enumerate(pairs):
                w22 = (dr[y][1] * dr[z][1] * sh(co, 0, 2) + dr[y][0] * dr[z][0] * sh(co, 2, 0)
                       + (dr[y][1] * dr[z][0] + dr[y][0] * dr[z][1]) * sh(co, 1, 1))
                for k in (y, z):
                    w22 = w22 - dr[k][1] * sh(cd[k], 0, 1) - dr[k][0] * sh(cd[k], 1, 0)
                w0 = D(pd[y] * v12[z] + pd[z] * v12[y] + p * e * (1j * w22 - v22[y] * v22[z]))
                re = lambda u, v: u.real * v.real + u.imag * v.imag  # noqa: E731
                t = ((1 - d / a) * (re(f0[y], f0[z]) + re(x0, w0)) + d / a ** 3 * re(x0, f0[y]) * re(x0, f0[z]))
                tot[i] += 2.0 / size * float(t.sum())
    return torch.tensor(tot, dtype=torch.float64)


def exact(case, seed):
    c, s = SimpleNamespace(**case), _inputs(case, seed)
    if c.kind == "prop":
        ph, out = _physics(c.n, c.ndist), []
        for j in range(c.ndist):
            x = torch.empty(s.x.shape, dtype=torch.complex128, device=DEV)
            y = torch.empty_like(x)
            for b in range(c.batch):
                x[b] = _fresnel(_up(s.x[b]), ph.wavelength, ph.voxelsize, ph.distance[j], False)
                y[b] = _fresnel(x[b], ph.wavelength, ph.voxelsize, ph.distance[j], True)
            out += [x, y] if c.both else [x]
        return out
    if c.kind == "radon":
        x = _up(s.x)
        if c.op == "R":
            return _radon(x, c.ntheta)
        if c.op == "RT":
            return _radon_adj(x)
        if c.op == "fbp":
            f = torch.fft.fftfreq(c.n, dtype=torch.float64, device=DEV)
            return _radon_adj(x, 4 * c.n * f.abs()) * math.sqrt(c.n / c.ntheta)
        sino = _radon(x, c.ntheta)
        return [sino, _radon_adj(sino)]
    if c.kind == "shift":
        return _exact_shift(c, s)
    ph = _physics(c.n, c.ndist)
    return _exact_gradient(c, s, ph) if c.kind == "gradient" else _exact_bilinear(c, s, ph)
