"""Workloads of the nuSHT operators: what users call, over the range of sizes they call it with.

Kinds of case (all inputs are device tensors, as in a program that keeps its fields on the GPU):

  lens      one lensed map per pass with its own deflection (simulation pipelines): pointing, binning,
            synthesis and interpolation, through the batch entry point with one job
  unlens    the adjoint of `lens` (lensing-estimator and map-making steps)
  recon     one gclm2lenmap and one lenmap2gclm at a fixed deflection (an iteration of a reconstruction or
            conjugate-gradient solve), through the transformer class
  points    nusht2d2 at arbitrary points of the sphere (catalogues, pointing timelines, ray tracing)
  gather    nusht2d1, its adjoint
  sht       synthesis and quadrature analysis on the pointing grid (filtering between lensing steps)
  pointing  deflected angles and rotation angle of a deflection field
  maps      several maps that share one deflection (T, E and B realisations behind one lens), one call
  jobs      independent lensing jobs of uneven size in one batch
"""
import ctypes
import math

import numpy as np
import torch

import cunusht_amd
from cunusht_amd import _lib
from cunusht_amd.batch import BatchJob, LensingPlan, execute

ARCMIN = math.pi / 180.0 / 60.0


def listed():
    return [
        # the smallest full-sky map anyone lenses: launches and latency
        {"name": "lens-255-s0", "kind": "lens", "lmax": 255, "spin": 0, "eps": 1e-10, "geom": "gl", "odd": True},
        # small adjoint on an uneven lmax: latency again, the other direction
        {"name": "unlens-300-s2", "kind": "unlens", "lmax": 300, "spin": 2, "eps": 1e-7, "geom": "gl", "odd": False},
        # a catalogue-sized point set on a mid-size transform (the dot-product test's configuration)
        {"name": "points-1024-20k", "kind": "points", "lmax": 1024, "spin": 0, "eps": 1e-8, "npts": 20000},
        # polarisation on a HEALPix grid, ragged rings
        {"name": "lens-1000-s2-hp", "kind": "lens", "lmax": 1000, "spin": 2, "eps": 1e-7, "geom": "healpix",
         "odd": False},
        # filtering between lensing steps, spin 2
        {"name": "sht-1500-s2", "kind": "sht", "lmax": 1500, "spin": 2, "odd": False},
        # single-precision evaluation of a full point set
        {"name": "points-2047-8m-f32", "kind": "points", "lmax": 2047, "spin": 0, "eps": 1e-5, "npts": 2048 * 4095},
        # the tight-accuracy adjoint of it
        {"name": "gather-2047-8m", "kind": "gather", "lmax": 2047, "spin": 0, "eps": 1e-10, "npts": 2048 * 4095},
        # one iteration of a lensing reconstruction at a fixed deflection
        {"name": "recon-3001-s2", "kind": "recon", "lmax": 3001, "spin": 2, "eps": 1e-7, "odd": False},
        # a queue of uneven jobs
        {"name": "jobs-8", "kind": "jobs", "njobs": 8, "lmin": 511, "lmax": 2047, "eps": 1e-7},
        # the full-size polarised map, both directions, and eight of them behind one lens
        {"name": "lens-4095-s2", "kind": "lens", "lmax": 4095, "spin": 2, "eps": 1e-7, "geom": "gl", "odd": True},
        {"name": "unlens-4095-s2", "kind": "unlens", "lmax": 4095, "spin": 2, "eps": 1e-7, "geom": "gl", "odd": True},
        {"name": "maps-8-4095-s2", "kind": "maps", "lmax": 4095, "spin": 2, "eps": 1e-7, "nmaps": 8, "odd": True},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["lens", "unlens", "recon", "points", "gather", "sht", "pointing", "maps", "jobs"])
    spin = rng.choice([0, 0, 2, 2, 1])
    eps = rng.choice([1e-5, 1e-7, 1e-7, 1e-10])
    ragged = rng.random() < 0.5

    def odd(L):  # rings of 2 lmax + 1 pixels (any factors; up to lmax 2000) or the next 2-3-5-smooth length
        return ragged and L <= 2000

    if kind in ("lens", "unlens"):
        if rng.random() < 0.25:
            return {"kind": kind, "lmax": size(64, 1100), "spin": spin, "eps": eps, "geom": "healpix", "odd": False}
        L = size(64, 4000)
        return {"kind": kind, "lmax": L, "spin": spin, "eps": eps, "geom": "gl", "odd": odd(L)}
    if kind == "recon":
        L = size(64, 3500)
        return {"kind": kind, "lmax": L, "spin": spin, "eps": eps, "odd": odd(L)}
    if kind in ("points", "gather"):
        return {"kind": kind, "lmax": size(64, 3000), "spin": spin, "eps": eps, "npts": size(100, 8000000)}
    if kind in ("sht", "pointing"):
        L = size(64, 4000)
        return {"kind": kind, "lmax": L, "spin": 1 if kind == "pointing" else spin, "odd": odd(L)}
    if kind == "maps":
        L = size(64, 3000)
        return {"kind": kind, "lmax": L, "spin": spin, "eps": eps, "nmaps": rng.randint(2, 8), "odd": odd(L)}
    return {"kind": "jobs", "njobs": rng.randint(3, 8), "lmin": size(64, 500), "lmax": size(600, 2047), "eps": eps}


# ---------------------------------------------------------------------------- inputs
def _nalm(L):
    return (L + 1) * (L + 2) // 2


_LM = {}


def _lm(L):
    """l and m of every coefficient in the m-major layout, on the GPU (the last few sizes are kept)."""
    if L not in _LM:
        if len(_LM) > 8:
            _LM.clear()
        m = torch.repeat_interleave(torch.arange(L + 1, device="cuda"),
                                    torch.arange(L + 1, 0, -1, device="cuda"))
        ofs = torch.arange(L + 1, device="cuda")
        ofs = ofs * (2 * L + 1 - ofs) // 2
        _LM[L] = (torch.arange(_nalm(L), device="cuda") - ofs[m], m)
    return _LM[L]


def _gauss_alm(L, cl, gen):
    """Gaussian coefficients of a real field with spectrum cl."""
    l, m = _lm(L)
    re = torch.randn(_nalm(L), dtype=torch.float64, device="cuda", generator=gen)
    im = torch.randn(_nalm(L), dtype=torch.float64, device="cuda", generator=gen)
    amp = torch.sqrt(cl)[l]
    zero = m == 0
    re = torch.where(zero, re * math.sqrt(2.0), re)
    im = torch.where(zero, torch.zeros_like(im), im)
    return torch.complex(re * amp * math.sqrt(0.5), im * amp * math.sqrt(0.5))


def _field(L, spin, gen, ncomp=None):
    """A red, smoothed spectrum (temperature-like for spin 0, E and weaker B otherwise)."""
    ll = torch.arange(L + 1, dtype=torch.float64, device="cuda")
    cl = torch.exp(-(ll / (0.75 * L)) ** 2) / (ll * (ll + 1)).clamp(min=1.0)
    cl[:max(2, spin)] = 0.0
    n = (1 if spin == 0 else 2) if ncomp is None else ncomp
    return torch.stack([_gauss_alm(L, cl * (1.0 if c == 0 else 0.1), gen) for c in range(n)])


def _deflection(L, gen):
    """dlm / sqrt(l (l + 1)) of a gradient deflection of 2.5 arcmin rms with C_l ~ l^-2."""
    ll = torch.arange(L + 1, dtype=torch.float64, device="cuda")
    cl = torch.zeros_like(ll)
    cl[2:] = ll[2:] ** -2.0
    cl *= (2.5 * ARCMIN) ** 2 / (torch.sum((2 * ll + 1) * cl) / (4 * math.pi))
    fl = torch.zeros_like(ll)
    fl[1:] = (ll[1:] * (ll[1:] + 1)) ** -0.5
    return (_gauss_alm(L, cl, gen) * fl[_lm(L)[0]]).contiguous()


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _geominfo(case, L):
    if case.get("geom") == "healpix":
        nside = 1 << max(4, math.ceil(math.log2((L + 1) / 2.0)))
        return ("healpix", {"nside": nside, "lmax": L})
    return ("gl", {"lmax": L, "nphi": 2 * L + 1} if case.get("odd") else {"lmax": L})


def _npix(case, L):
    g = _geominfo(case, L)
    if g[0] == "healpix":
        return 12 * g[1]["nside"] ** 2
    n = 2 * L + 1
    if "nphi" not in g[1]:
        n = cunusht_amd.geometry.good_size(n, True)
    return (L + 1) * n


def _points(n, gen):
    """Uniform on the sphere, (n, 2) rows (theta, phi)."""
    z = 2.0 * torch.rand(n, dtype=torch.float64, device="cuda", generator=gen) - 1.0
    phi = 2.0 * math.pi * torch.rand(n, dtype=torch.float64, device="cuda", generator=gen)
    return torch.stack([torch.acos(z), phi], 1).contiguous()


def _map(n, spin, gen):
    m = torch.randn((1 if spin == 0 else 2, n), dtype=torch.float64, device="cuda", generator=gen)
    return m[0].contiguous() if spin == 0 else m


def _job_list(case):
    """(lmax, spin) of each job: sizes spread over the range, spins in turn."""
    n = case["njobs"]
    r = (case["lmax"] / case["lmin"]) ** (1.0 / max(1, n // 2 - 1))
    return [(min(case["lmax"], int(round(case["lmin"] * r ** (i // 2)))), 2 if i % 2 else 0) for i in range(n)]


def _transformer(case, spin):
    L = case["lmax"]
    return cunusht_amd.get_transformer("GPU")(_geominfo(case, L), nuFFTtype=2 if "eps" in case else None,
                                              epsilon=case.get("eps"), spin=spin)


def prepare(case, seed):
    kind, L = case["kind"], case["lmax"]
    g = _gen(seed)
    if kind == "jobs":
        jobs = []
        for l, s in _job_list(case):
            plan = LensingPlan(l, s, case["eps"], max_maps=4)
            jobs.append(BatchJob("gclm2lenmap", plan, _deflection(l, g), _field(l, s, g)))
        return {"case": case, "jobs": jobs}
    spin = case["spin"]
    if kind == "lens":
        plan = LensingPlan(L, spin, case["eps"], _geominfo(case, L))
        return {"case": case, "jobs": [BatchJob("gclm2lenmap", plan, _deflection(L, g), _field(L, spin, g))]}
    if kind == "unlens":
        plan = LensingPlan(L, spin, case["eps"], _geominfo(case, L))
        return {"case": case,
                "jobs": [BatchJob("lenmap2gclm", plan, _deflection(L, g), _map(plan.npix(), spin, g))]}
    if kind == "maps":
        plan = LensingPlan(L, spin, case["eps"], _geominfo(case, L), max_maps=8)
        alm = torch.stack([_field(L, spin, g) for _ in range(case["nmaps"])]).contiguous()
        out = torch.empty((case["nmaps"], 1 if spin == 0 else 2, plan.npix()), dtype=torch.float64, device="cuda")
        return {"case": case, "plan": plan, "alm": alm, "dlm": _deflection(L, g), "out": out}
    T = _transformer(case, spin)
    st = {"case": case, "T": T}
    if kind == "recon":
        st.update(alm=_field(L, spin, g), dlm=_deflection(L, g), map=_map(T.npix(), spin, g))
    elif kind == "sht":
        st.update(alm=_field(L, spin, g), map=_map(T.npix(), spin, g))
    elif kind == "pointing":
        st.update(dlm=_deflection(L, g))
    else:
        st.update(loc=_points(case["npts"], g))
        if kind == "points":
            st.update(alm=_field(L, spin, g))
        else:
            st.update(map=_map(case["npts"], spin, g))
    return st


def run(st):
    case = st["case"]
    kind, L = case["kind"], case["lmax"]
    if kind in ("lens", "unlens", "jobs"):
        execute(st["jobs"])
        return [j.out for j in st["jobs"]]
    spin = case["spin"]
    if kind == "maps":
        p, out, alm = st["plan"], st["out"], st["alm"]
        nmap, ncmp = out.shape[0], out.shape[1]
        ptr = lambda t: ctypes.c_void_p(t.data_ptr())
        _lib.call("nusht_gclm2lenmap_batch", p.nuplan._h, p.ring._h, nmap, ptr(alm), 2 * alm[0].numel(),
                  ptr(st["dlm"]), ptr(out[0, 0]), ptr(out[0, 1]) if spin else None, ncmp * out.shape[2], 1,
                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        return out
    T = st["T"]
    if kind == "recon":
        return [T.gclm2lenmap(st["alm"], L, L, dlm_scaled=st["dlm"], spin=spin),
                T.lenmap2gclm(st["map"], st["dlm"], None, L, L, spin=spin)]
    if kind == "sht":
        return [T.synthesis(st["alm"], spin=spin), T.adjoint_synthesis(st["map"], spin=spin)]
    if kind == "pointing":
        return T.dlm2pointing(st["dlm"], gamma=True)
    if kind == "points":
        return T.nusht2d2(L, L, st["alm"], st["loc"], spin=spin)
    return T.nusht2d1(L, L, st["map"], st["loc"], spin=spin)


# ---------------------------------------------------------------------------- what a pass cannot do without
def _legendre(L, spin, rings, ncomp):
    """Flops of one ring transform: per (l, m, ring pair) the recursion and the contraction, over the part of
    the (l, m, theta) range where the functions are not negligible (m < l sin theta: 2 / pi of it)."""
    per = 6 if spin == 0 else (14 if ncomp == 1 else 22)
    return 2.0 / math.pi * _nalm(L) * ((rings + 1) // 2) * per


def _fft(n, howmany):
    return 5.0 * n * max(1.0, math.log2(n)) * howmany


def _nonuniform(L, eps, npts, spin):
    """Double-Fourier transform of (2 lmax + 2)^2 modes and a kernel of one cell per digit and axis."""
    w = max(2, math.ceil(-math.log10(eps)) + 1)
    n = 2 * L + 2
    return _fft(n, 2 * n) + npts * 4.0 * w * w


def work(case):
    kind, L = case["kind"], case["lmax"]
    if kind == "jobs":
        per = [work({"kind": "lens", "lmax": l, "spin": s, "eps": case["eps"]}) for l, s in _job_list(case)]
        return {k: sum(p[k] for p in per) for k in ("bytes", "flops")}
    spin = case["spin"]
    nc = 1 if spin == 0 else 2
    alm = 16.0 * _nalm(L)
    if kind in ("points", "gather"):
        n = case["npts"]
        return {"bytes": nc * alm + 16.0 * n + 8.0 * nc * n,
                "flops": _legendre(L, spin, L + 2, nc) + _nonuniform(L, case["eps"], n, spin)}
    npix = _npix(case, L)
    point = _legendre(L, 1, L + 1, 1) + _fft(2 * L + 1, L + 1) + 60.0 * npix
    if kind == "pointing":
        return {"bytes": alm + 24.0 * npix, "flops": point}
    if kind == "sht":
        return {"bytes": 2 * (nc * alm + 8.0 * nc * npix),
                "flops": 2 * (_legendre(L, spin, L + 1, nc) + _fft(2 * L + 1, L + 1))}
    one = _legendre(L, spin, L + 2, nc) + _nonuniform(L, case["eps"], npix, spin)
    if kind == "maps":
        return {"bytes": alm + case["nmaps"] * (nc * alm + 8.0 * nc * npix), "flops": point + case["nmaps"] * one}
    if kind == "recon":  # the pointing is kept from the first pass
        return {"bytes": 2 * (nc * alm + 8.0 * nc * npix) + alm, "flops": 2 * one}
    return {"bytes": alm + nc * alm + 8.0 * nc * npix, "flops": point + one}


# ---------------------------------------------------------------------------- the results in 64 bits
def _wigner(L, s, theta):
    """Yields (l, U, V), l = s..L: U[m] = N_l d^l_{m,-s}(theta), V[m] = N_l d^l_{m,+s}(theta) for m = 0..L (rows
    m > l zero; V is None at s = 0), N_l = sqrt((2l + 1) / 4 pi), from the three-term recursion in l with the
    closed forms at l = max(m, s).  Plain FP64 without rescaling: starting values that underflow belong to
    functions that stay negligible for l <= L up to about L = 1800."""
    dev = theta.device
    x = torch.cos(theta)
    lc, ls = torch.log(torch.cos(theta / 2)), torch.log(torch.sin(theta / 2))
    lg = math.lgamma

    def start(m, sg):  # N_l0 d^{l0}_{m, sg s}
        l0 = max(m, s)
        if m >= s:
            mu, o, sign = sg * s, m, (-1.0) ** (m - s)
            c = 0.5 * (lg(2 * o + 1) - lg(o + mu + 1) - lg(o - mu + 1))
            pc, ps = o + mu, o - mu
        else:
            c = 0.5 * (lg(2 * s + 1) - lg(s + m + 1) - lg(s - m + 1))
            pc, ps = s + sg * m, s - sg * m
            sign = 1.0 if sg > 0 else (-1.0) ** (m + s)
        c += 0.5 * math.log((2 * l0 + 1) / (4 * math.pi))
        v = torch.full_like(theta, c)
        if pc:
            v = v + pc * lc
        if ps:
            v = v + ps * ls
        return sign * torch.exp(v)

    P = theta.numel()
    chains = [(-1, +1.0)] + ([(+1, -1.0)] if s else [])
    cur = [torch.zeros((L + 1, P), dtype=torch.float64, device=dev) for _ in chains]
    prev = [torch.zeros_like(c) for c in cur]
    for m in range(s + 1):
        for c, (sg, _) in zip(cur, chains):
            if m <= L:
                c[m] = start(m, sg)
    ms = torch.arange(L + 1, dtype=torch.float64, device=dev)[:, None]
    for l in range(s, L + 1):
        yield l, cur[0], cur[1] if s else None
        if l == L:
            return
        n = l + 1  # rows m <= l step to l + 1, row l + 1 starts there
        mm = ms[:n]
        if l == 0:
            al, be, ga = torch.full_like(mm, math.sqrt(3.0)), torch.zeros_like(mm), torch.zeros_like(mm)
        else:
            d1 = torch.sqrt(((l + 1.0) ** 2 - mm * mm) * ((l + 1.0) ** 2 - s * s))
            d0 = torch.sqrt((l * l - mm * mm) * (l * l - s * s))
            f = math.sqrt((2.0 * l + 3) * (2.0 * l + 1))
            al, be = f * (l + 1) / d1, f * mm * s / (l * d1)
            ga = math.sqrt((2.0 * l + 3) / (2.0 * l - 1)) * (l + 1) * d0 / (l * d1)
        for k, (sg, b) in enumerate(chains):
            nxt = prev[k]
            nxt[:n].mul_(-ga).addcmul_(al * x + b * be, cur[k][:n])
            nxt[n] = start(n, sg)
            prev[k], cur[k] = cur[k], nxt


def _row(alm, L, l):
    """Coefficients (l, m = 0..l) of one component."""
    m = torch.arange(l + 1, device=alm.device)
    return alm[m * (2 * L + 1 - m) // 2 + l]


def _ring_coefficients(alm, L, s, theta):
    """G_m (m = 0..L) and, for s > 0, G_{-m} of the field at colatitudes theta: (L + 1, P) complex each."""
    P = theta.numel()
    acc = [torch.zeros((L + 1, P), dtype=torch.float64, device=theta.device) for _ in range(2 if s == 0 else 4)]
    for l, U, V in _wigner(L, s, theta):
        n = l + 1
        e = _row(alm[0], L, l)
        if s == 0:
            acc[0][:n].addcmul_(U[:n], e.real[:, None])
            acc[1][:n].addcmul_(U[:n], e.imag[:, None])
            continue
        b = _row(alm[1], L, l) if alm.shape[0] > 1 else torch.zeros_like(e)
        p = -((-1.0) ** s) * (e + 1j * b)
        q = -(e.conj() + 1j * b.conj())
        acc[0][:n].addcmul_(U[:n], p.real[:, None])
        acc[1][:n].addcmul_(U[:n], p.imag[:, None])
        acc[2][:n].addcmul_(V[:n], q.real[:, None])
        acc[3][:n].addcmul_(V[:n], q.imag[:, None])
    return torch.complex(acc[0], acc[1]), (torch.complex(acc[2], acc[3]) if s else None)


def _chunk(L):
    return max(256, (1 << 23) // (L + 1))


def _synth(alm, L, s, theta, phi):
    """Values at points: real (spin 0) or Q + iU."""
    out = []
    m = torch.arange(L + 1, dtype=torch.float64, device=theta.device)[:, None]
    for a in range(0, theta.numel(), _chunk(L)):
        t, p = theta[a:a + _chunk(L)], phi[a:a + _chunk(L)]
        e = torch.polar(torch.ones((L + 1, t.numel()), dtype=torch.float64, device=t.device), m * p)
        gp, gm = _ring_coefficients(alm, L, s, t)
        if s == 0:
            v = (gp * e).real
            out.append(2 * v.sum(0) - v[0])
        else:
            out.append((gp * e).sum(0) + (gm[1:] * e[1:].conj()).sum(0))
    return torch.cat(out)


def _rows_to_alm(rows, L):
    """rows[l] = coefficients (l, m = 0..l) -> m-major vector."""
    out = torch.zeros(_nalm(L), dtype=torch.complex128, device="cuda")
    for l, r in rows.items():
        m = torch.arange(l + 1, device="cuda")
        out[m * (2 * L + 1 - m) // 2 + l] = r
    return out


def _adjoint_rows(L, s, theta, pm, qm, rows):
    """Adds sum_p over these colatitudes: pm = P_m = sum v e^{-im phi} (m = 0..L), qm = conj(P_{-m})."""
    sg = (-1.0) ** s
    for l, U, V in _wigner(L, s, theta):
        n = l + 1
        X = torch.complex((U[:n] * pm[0][:n]).sum(1), (U[:n] * pm[1][:n]).sum(1))
        if s == 0:
            X[0] = X[0].real + 0j
            new = (X,)
        else:
            X = sg * X
            Y = torch.complex((V[:n] * qm[0][:n]).sum(1), (V[:n] * qm[1][:n]).sum(1))
            new = (-0.5 * (X + Y), 0.5j * (X - Y))
        for c, r in enumerate(new):
            rows[c][l] = rows[c][l] + r if l in rows[c] else r


def _gather(v, L, s, theta, phi):
    """Adjoint of _synth for values v (real, or Q + iU)."""
    rows = [{} for _ in range(1 if s == 0 else 2)]
    m = torch.arange(L + 1, dtype=torch.float64, device=theta.device)[:, None]
    for a in range(0, theta.numel(), _chunk(L)):
        sl = slice(a, a + _chunk(L))
        e = torch.polar(torch.ones((L + 1, theta[sl].numel()), dtype=torch.float64, device="cuda"), -m * phi[sl])
        pm = e * v[sl]
        qm = e * v[sl].conj() if s else pm
        _adjoint_rows(L, s, theta[sl], (pm.real.contiguous(), pm.imag.contiguous()),
                      (qm.real.contiguous(), qm.imag.contiguous()), rows)
    return torch.stack([_rows_to_alm(r, L) for r in rows])


def _to_rings(alm, L, s, theta, n):
    """Map on uniform rings of n >= 2L + 1 pixels: (rings, n) real, or Q + iU."""
    gp, gm = _ring_coefficients(alm, L, s, theta)
    spec = torch.zeros((theta.numel(), n), dtype=torch.complex128, device="cuda")
    spec[:, :L + 1] = gp.T
    if L:
        spec[:, n - L:] = (gp[1:].conj() if s == 0 else gm[1:]).flip(0).T
    f = torch.fft.ifft(spec, dim=1) * n
    return f.real if s == 0 else f


def _from_rings(f, L, s, theta, n):
    """Adjoint of _to_rings."""
    spec = torch.fft.fft(f.to(torch.complex128), dim=1)
    pm = spec[:, :L + 1].T.contiguous()
    qm = pm.clone()
    if s:
        qm[1:] = spec[:, n - L:].flip(1).T if L else qm[1:]
        qm = qm.conj()
    rows = [{} for _ in range(1 if s == 0 else 2)]
    _adjoint_rows(L, s, theta, (pm.real.contiguous(), pm.imag.contiguous()),
                  (qm.real.contiguous(), qm.imag.contiguous()), rows)
    return torch.stack([_rows_to_alm(r, L) for r in rows])


def _exact_pointing(dlm_scaled, L, theta, n):
    """theta', phi', gamma of every pixel of uniform rings, flat."""
    l = _lm(L)[0].to(torch.float64)
    d = _to_rings((dlm_scaled * torch.sqrt(l * (l + 1)))[None], L, 1, theta, n)
    dt, dp = d.real, d.imag
    th = theta[:, None]
    ph = 2 * math.pi / n * torch.arange(n, dtype=torch.float64, device="cuda")[None, :]
    a = torch.sqrt(dt * dt + dp * dp)
    sa, ca = torch.sinc(a / math.pi), torch.cos(a)
    st, ct = torch.sin(th), torch.cos(th)
    n1, n2, n3 = st * ca + ct * dt * sa, -dp * sa, ct * ca - st * dt * sa
    tp = torch.atan2(torch.sqrt(n1 * n1 + n2 * n2), n3)
    pp = ph - torch.atan2(n2, n1)
    pp = torch.where(pp >= 2 * math.pi, pp - 2 * math.pi, pp)
    gam = torch.atan2(dp, dt) - torch.atan2(dp, a * torch.sin(a) * ct / st + dt * ca)
    return tp.reshape(-1), pp.reshape(-1), gam.reshape(-1)


def _gl(case):
    L = case["lmax"]
    g = cunusht_amd.geometry.Geom
    geom = g.get_gl_geometry(L, nphi=2 * L + 1) if case.get("odd") else g.get_gl_geometry(L)
    return torch.as_tensor(geom.theta, device="cuda"), int(geom.nph[0]), torch.as_tensor(geom.weight, device="cuda")


def exact(case, seed):
    kind, L = case["kind"], case["lmax"]
    if kind in ("jobs", "maps", "recon") or case.get("geom") == "healpix" or L > 1500:
        return None
    spin = case["spin"]
    points = case["npts"] if kind in ("points", "gather") else 0 if kind in ("sht", "pointing") else _npix(case, L)
    if points * float(L + 1) ** 2 * (1 if spin == 0 else 2) > 5e10:  # beyond about 20 s
        return None
    g = _gen(seed)
    if kind == "points":
        loc, alm = _points(case["npts"], g), _field(L, spin, g)
        v = _synth(alm, L, spin, loc[:, 0], loc[:, 1])
        return v if spin == 0 else torch.stack([v.real, v.imag])
    if kind == "gather":
        loc, x = _points(case["npts"], g), _map(case["npts"], spin, g)
        v = x if spin == 0 else torch.complex(x[0], x[1])
        r = _gather(v, L, spin, loc[:, 0], loc[:, 1])
        return r[0] if spin == 0 else r
    theta, n, weight = _gl(case)
    if kind == "sht":
        alm, x = _field(L, spin, g), _map(_npix(case, L), spin, g)
        f = _to_rings(alm, L, spin, theta, n).reshape(-1)
        x = (x if spin == 0 else torch.complex(x[0], x[1])).reshape(L + 1, n) * weight[:, None]
        r = _from_rings(x, L, spin, theta, n)
        return [f if spin == 0 else torch.stack([f.real, f.imag]), r[0] if spin == 0 else r]
    dlm = _deflection(L, g)
    tp, pp, gam = _exact_pointing(dlm, L, theta, n)
    if kind == "pointing":  # phi' and gamma have branch cuts: values either side of one are both right
        return None
    rot = torch.polar(torch.ones_like(gam), spin * gam)
    if kind == "lens":
        v = _synth(_field(L, spin, g), L, spin, tp, pp)
        v = v if spin == 0 else v * rot
        return [v if spin == 0 else torch.stack([v.real, v.imag])]
    x = _map(_npix(case, L), spin, g)
    v = x if spin == 0 else torch.complex(x[0], x[1]) * rot.conj()
    return [_gather(v, L, spin, tp, pp)]
