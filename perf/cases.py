"""Timing cases of the framework's main paths on one GPU, through the Python entry points.

Kinds of case ("kind"):

  step     a run of CNAB2 steps from a given state: set_state, run, get_state
           (prec: arithmetic of transforms and products; full: radial
           components and every product, the MHD step; graph: replayed graph)
  sht      one synthesis and one analysis of a radial stack, scalar or vector
           (tangential pair)
  cnab2    build_rhs_cnab2 and solve_implicit_step of one field, the operators
           a host-driven time loop calls
  erk2     the four staged ERK2 calls of one field
  adjoint  forward run, temperature misfit and backward pass: the gradient
           with respect to the initial state
  batch    independent shells of uneven size advanced together

Sizes are those of the repository's configurations and tests (lmax 31..255,
nr 33..97, 3(L+1)/2 x 3(L+1) grids) and odd ones between.

exact() restates each path in 64 bits with dense operators and torch's FFT.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "geodynamo.jl_amd"))

E, PM, PR, RA, RRATIO, DT, THETA, BW = 1e-3, 5.0, 1.0, 500.0, 0.35, 1e-5, 0.5, 3
DEV = "cuda"
F64 = torch.float64


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # a first look at a run: one eager step of the smallest configuration, launch latency
        dict(name="step-fp64-31", kind="step", lmax=31, nlat=48, nlon=96, nr=33, prec="fp64", full=False, steps=1,
             graph=False),
        # production runs between two outputs at the headline size, mixed and FP64
        dict(name="step-mixed-127", kind="step", lmax=127, nlat=192, nlon=384, nr=65, prec="fp32", full=False,
             steps=20, graph=True),
        dict(name="step-fp64-127", kind="step", lmax=127, nlat=192, nlon=384, nr=65, prec="fp64", full=False,
             steps=10, graph=True),
        # the MHD step with radial components and every product, a restart of two steps (this
        # explicit form is not stable over many steps at these parameters)
        dict(name="step-full-mixed-127", kind="step", lmax=127, nlat=192, nlon=384, nr=65, prec="fp32", full=True,
             steps=2, graph=False),
        # post-processing and the small end of the transforms: latency
        dict(name="sht-scalar-fp64-31", kind="sht", lmax=31, mmax=31, nlat=48, nlon=96, nr=33, prec="fp64",
             vector=False),
        # transforms of large stacks: FP64 scalar, FP32 vector
        dict(name="sht-scalar-fp64-255", kind="sht", lmax=255, mmax=255, nlat=384, nlon=768, nr=97, prec="fp64",
             vector=False),
        dict(name="sht-vector-fp32-255", kind="sht", lmax=255, mmax=255, nlat=384, nlon=768, nr=97, prec="fp32",
             vector=True),
        # a truncated, odd-sized shell: nlat/2 odd, a ring length without a compiled plan
        dict(name="sht-vector-fp64-ragged", kind="sht", lmax=106, mmax=90, nlat=162, nlon=324, nr=41, prec="fp64",
             vector=True),
        # the implicit operators as a host-driven time loop calls them
        dict(name="cnab2-127", kind="cnab2", lmax=127, nr=65, bc_rows=True),
        # one field of the staged exponential integrator
        dict(name="erk2-63", kind="erk2", lmax=63, nr=65),
        # data assimilation: the gradient of a 20-step run, checkpoints every 5
        dict(name="adjoint-mixed-63", kind="adjoint", lmax=63, nlat=96, nlon=192, nr=65, prec="fp32", steps=20,
             every=5),
        # a parameter study: uneven shells in one batch
        dict(name="batch-fp64-12", kind="batch", shells=12, pick=3, prec="fp64", steps=4),
    ]


def _log_int(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def _smooth(n):
    """The next ring length 2^a 3^b >= n."""
    while True:
        k = n
        for p in (2, 3):
            while k % p == 0:
                k //= p
        if k == 1:
            return n
        n += 1


def _grid(lmax, mmax):
    nlat = (3 * (lmax + 1) + 1) // 2
    return nlat + nlat % 2, _smooth(3 * mmax + 3)


def draw(rng):
    kind = rng.choices(("step", "sht", "cnab2", "erk2", "adjoint", "batch"), (35, 33, 12, 6, 7, 7))[0]
    if kind == "step":
        full = rng.random() < 0.35
        lmax = _log_int(rng, 15, 100 if full else 127)
        nlat, nlon = _grid(lmax, lmax)
        return dict(kind=kind, lmax=lmax, nlat=nlat, nlon=nlon, nr=rng.randint(17, 65),
                    prec=rng.choice(("fp64", "fp32", "fp32", "bf16x3")), full=full,
                    steps=rng.randint(1, 2 if full else 10),
                    graph=rng.random() < 0.7)
    if kind == "sht":
        lmax = _log_int(rng, 15, 230)
        mmax = lmax if rng.random() < 0.6 else rng.randint(lmax // 2, lmax)
        nlat, nlon = _grid(lmax, mmax)
        return dict(kind=kind, lmax=lmax, mmax=mmax, nlat=nlat, nlon=nlon, nr=rng.randint(5, 90),
                    prec=rng.choice(("fp64", "fp64", "fp32", "bf16x3")), vector=rng.random() < 0.5)
    if kind == "cnab2":
        return dict(kind=kind, lmax=_log_int(rng, 15, 200), nr=rng.randint(17, 97), bc_rows=rng.random() < 0.7)
    if kind == "erk2":
        return dict(kind=kind, lmax=_log_int(rng, 15, 63), nr=rng.randint(17, 65))
    if kind == "adjoint":
        lmax = _log_int(rng, 15, 63)
        nlat, nlon = _grid(lmax, lmax)
        return dict(kind=kind, lmax=lmax, nlat=nlat, nlon=nlon, nr=rng.randint(17, 65),
                    prec=rng.choice(("fp64", "fp32")), steps=rng.randint(4, 12), every=rng.randint(2, 5))
    return dict(kind=kind, shells=rng.randint(2, 12), pick=rng.randint(10, 10000), prec="fp64", steps=rng.randint(1, 4))


# ---------------------------------------------------------------- inputs
def _lm(lmax, mmax):
    l = np.array([l for l in range(lmax + 1) for _ in range(min(l, mmax) + 1)])
    m = np.array([m for l in range(lmax + 1) for m in range(min(l, mmax) + 1)])
    return torch.from_numpy(l).to(DEV), torch.from_numpy(m).to(DEV)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _spectrum(g, lead, lmax, mmax, amp, power):
    """Normal coefficients times amp (l+1)^-power, m = 0 real: (re, im) of shape lead + (nlm,)."""
    l, m = _lm(lmax, mmax)
    w = amp * (l + 1).to(F64) ** -power
    shape = tuple(lead) + (l.numel(),)
    re = torch.randn(shape, generator=g, device=DEV, dtype=F64) * w
    im = torch.randn(shape, generator=g, device=DEV, dtype=F64) * w * (m > 0)
    return re, im


def _state(g, lmax, nr, amp=1e-3):
    """Five fields of radial sine modes (zero at both boundaries: no-slip, isothermal, insulating)."""
    x = 0.5 * (1 - torch.cos(math.pi * torch.arange(nr, device=DEV, dtype=F64) / (nr - 1)))
    k = torch.arange(1, 9, device=DEV, dtype=F64)
    modes = torch.sin(math.pi * x[:, None] * k) / k
    re, im = (torch.matmul(modes, z).contiguous() for z in _spectrum(g, (5, 8), lmax, lmax, amp, 2.0))
    for z in (re, im):
        z[:, 0] = 0.0
        z[:, -1] = 0.0
    return re, im


def _field_on_grid(g, nr, nlon, nlat):
    """A field with a broad spectrum: products of longitude and (radius, colatitude) profiles plus noise."""
    a = torch.randn((nr, 8, nlat), generator=g, device=DEV, dtype=F64)
    k = torch.arange(1, 9, device=DEV, dtype=F64)[:, None] * (2 * math.pi / nlon)
    b = torch.cos(k * torch.arange(nlon, device=DEV, dtype=F64) + 6.28 * torch.rand((8, 1), generator=g, device=DEV, dtype=F64))
    f = torch.matmul(b.t().contiguous()[None], a)
    return (f + 0.1 * torch.randn(f.shape, generator=g, device=DEV, dtype=F64)).contiguous()


def _shells(case):
    """(lmax, nr, radius ratio) of a batch's shells."""
    r = np.random.RandomState(case["pick"])
    return [(int(r.choice([31, 47, 63, 95])), int(r.choice([33, 49, 65])), float(r.uniform(0.2, 0.5)))
            for _ in range(case["shells"])]


def _sht_inputs(c, g):
    n = 2 if c["vector"] else 1
    spec = []
    for _ in range(n):
        re, im = _spectrum(g, (c["nr"],), c["lmax"], c["mmax"], 1.0, 1.5)
        if c["vector"]:
            re[:, 0] = 0.0  # the pair has no l = 0 part
            im[:, 0] = 0.0
        spec.append((re, im))
    return spec, [_field_on_grid(g, c["nr"], c["nlon"], c["nlat"]) for _ in range(n)]


def _plane_inputs(c, g, n):
    """Planes of one field: the field and n nonlinear terms of the size they have in a step."""
    u = _spectrum(g, (c["nr"],), c["lmax"], c["lmax"], 1e-3, 2.0)
    return u, [_spectrum(g, (c["nr"],), c["lmax"], c["lmax"], 1.0, 2.0) for _ in range(n)]


def _adjoint_inputs(c, g):
    re, im = _state(g, c["lmax"], c["nr"], 1e-2)
    target = 1e-2 * _field_on_grid(g, 1, c["nlon"], c["nlat"])[0]
    return re, im, target


# ---------------------------------------------------------------- prepare and run
def _new_step(lmax, nlat, nlon, nr, prec, full=False, rratio=RRATIO):
    import gdhip

    return gdhip.CNAB2Step(lmax, nlat, nlon, nr, E=E, Pm=PM, Pr=PR, Ra=RA, rratio=rratio, dt=DT, theta=THETA, bw=BW,
                           precision=prec, radials=full, full_products=full)


def prepare(case, seed):
    import gdhip

    c, g, s = case, _gen(seed), {"case": case}
    if c["kind"] == "step":
        s["step"] = _new_step(c["lmax"], c["nlat"], c["nlon"], c["nr"], c["prec"], c["full"])
        s["in"] = _state(g, c["lmax"], c["nr"], 1e-5 if c["full"] else 1e-3)
        s["out"] = [torch.empty_like(x) for x in s["in"]]
    elif c["kind"] == "sht":
        cfg = gdhip.create_shtnskit_config(c["lmax"], c["mmax"], c["nlat"], c["nlon"], precision=c["prec"])
        spec, phys = _sht_inputs(c, g)
        s["cfg"] = cfg
        s["spec"] = [gdhip.SHTnsSpectralField(cfg, c["nr"], re, im) for re, im in spec]
        s["phys"] = [gdhip.SHTnsPhysicalField(cfg, c["nr"], f) for f in phys]
        s["to_phys"] = [gdhip.SHTnsPhysicalField(cfg, c["nr"], torch.empty_like(f)) for f in phys]
        s["to_spec"] = [gdhip.SHTnsSpectralField(cfg, c["nr"], torch.empty_like(re), torch.empty_like(im))
                        for re, im in spec]
    elif c["kind"] in ("cnab2", "erk2"):
        cfg = gdhip.create_shtnskit_config(c["lmax"])
        dom = gdhip.create_radial_domain(c["nr"], RRATIO)
        u, nls = _plane_inputs(c, g, 2)

        def field(p):
            return gdhip.SHTnsSpectralField(cfg, c["nr"], p[0], p[1])

        s.update(cfg=cfg, u=field(u), nls=[field(p) for p in nls],
                 work=[field([torch.empty_like(x) for x in u]) for _ in range(2)])
        if c["kind"] == "cnab2":
            s["mats"] = gdhip.create_shtns_timestepping_matrices(cfg, dom, PM, DT, THETA, bw=BW, bc_rows=c["bc_rows"])
        else:
            s["cache"] = gdhip.create_erk2_cache(cfg, dom, 1.0, DT, bw=BW)
            s["buf"] = gdhip.ERK2FieldBuffers(s["u"], s["nls"][0], s["cache"])
    elif c["kind"] == "adjoint":
        s["step"] = _new_step(c["lmax"], c["nlat"], c["nlon"], c["nr"], c["prec"])
        re, im, target = _adjoint_inputs(c, g)
        s["in"], s["target"] = (re, im), target.cpu().numpy()
        s["out"] = [torch.empty_like(re), torch.empty_like(im)]
        s["adj"] = gdhip.CNAB2Adjoint(s["step"], c["steps"], c["every"])
    else:
        s["steps"], s["in"] = [], []
        for lmax, nr, rr in _shells(c):
            nlat, nlon = 3 * (lmax + 1) // 2, 3 * (lmax + 1)
            s["steps"].append(_new_step(lmax, nlat, nlon, nr, c["prec"], rratio=rr))
            s["in"].append(_state(g, lmax, nr))
        s["out"] = [[torch.empty_like(x) for x in p] for p in s["in"]]
        s["batch"] = gdhip.StepBatch(s["steps"])
    torch.cuda.synchronize()
    return s


def run(s):
    import gdhip

    c = s["case"]
    if c["kind"] == "step":
        s["step"].set_state(*s["in"])
        s["step"].run(c["steps"], graph=c["graph"])
        s["step"].get_state(*s["out"])
        return s["out"]
    if c["kind"] == "sht":
        if c["vector"]:
            out = gdhip.SHTnsVectorField(s["cfg"], c["nr"], [None] + s["to_phys"])
            gdhip.shtnskit_vector_synthesis(s["spec"][0], s["spec"][1], out)
            vec = gdhip.SHTnsVectorField(s["cfg"], c["nr"], [None] + s["phys"])
            gdhip.shtnskit_vector_analysis(vec, s["to_spec"][0], s["to_spec"][1])
        else:
            gdhip.shtnskit_spectral_to_physical(s["spec"][0], s["to_phys"][0])
            gdhip.shtnskit_physical_to_spectral(s["phys"][0], s["to_spec"][0])
        return {"phys": [p.data for p in s["to_phys"]], "spec": [[p.data_real, p.data_imag] for p in s["to_spec"]]}
    if c["kind"] == "cnab2":
        rhs, sol = s["work"]
        gdhip.build_rhs_cnab2(rhs, s["u"], s["nls"][0], s["nls"][1], DT, s["mats"])
        gdhip.solve_implicit_step(sol, rhs, s["mats"])
        return [rhs.data_real, rhs.data_imag, sol.data_real, sol.data_imag]
    if c["kind"] == "erk2":
        stage, new = s["work"]
        gdhip.erk2_prepare_field(s["buf"], s["u"], s["nls"][0], s["cache"], s["cfg"], DT)
        gdhip.erk2_apply_stage(s["buf"], stage)
        gdhip.erk2_store_stage_nonlinear(s["buf"], s["nls"][1])
        gdhip.erk2_finalize_field(s["buf"], new, s["cache"], s["cfg"], DT)
        return [stage.data_real, stage.data_imag, new.data_real, new.data_imag]
    if c["kind"] == "adjoint":
        s["step"].set_state(*s["in"])
        s["adj"].forward()
        J = s["adj"].misfit(s["target"], kind="T")
        s["adj"].backward(out=s["out"])
        return [J] + list(s["out"])
    for st, p in zip(s["steps"], s["in"]):
        st.set_state(*p)
    s["batch"].run(c["steps"])
    for st, p in zip(s["steps"], s["out"]):
        st.get_state(*p)
    return s["out"]


# ---------------------------------------------------------------- what a pass cannot do without
def _nlm(lmax, mmax):
    return sum(min(l, mmax) + 1 for l in range(lmax + 1))


def _step_work(lmax, nlat, nlon, nr, full):
    """One step: state and history read and written; the Legendre sums (even / odd symmetric) and the FFTs."""
    nlm = _nlm(lmax, lmax)
    fields = 5 if full else 3  # fields with a nonlinear term
    legendre = (16 + 2 + 5 + 8 + 1) if full else (4 + 2 + 4 + 1)
    rings = (15 + 5) if full else (4 + 3)
    return dict(bytes=(2 * 5 + 2 * fields) * 16.0 * nlm * nr,
                flops=2.0 * legendre * nlat * nlm * nr + 2.5 * rings * nlat * nr * nlon * math.log2(nlon)
                + 5 * 2 * 2 * 3 * (2 * BW + 1) * nlm * nr)


def work(case):
    c = case
    if c["kind"] == "step":
        w = _step_work(c["lmax"], c["nlat"], c["nlon"], c["nr"], c["full"])
        return {k: v * c["steps"] for k, v in w.items()}
    if c["kind"] == "sht":
        nlm, k = _nlm(c["lmax"], c["mmax"]), 2 if c["vector"] else 1
        return dict(bytes=2.0 * k * c["nr"] * (16 * nlm + 8 * c["nlat"] * c["nlon"]),
                    flops=2.0 * k * k * 2 * c["nlat"] * nlm * c["nr"]
                    + 2 * k * 2.5 * c["nlat"] * c["nr"] * c["nlon"] * math.log2(c["nlon"]))
    if c["kind"] == "cnab2":
        n = _nlm(c["lmax"], c["lmax"]) * c["nr"]
        return dict(bytes=16.0 * 6 * n, flops=2.0 * n * 2 * 2 * (2 * BW + 1))
    if c["kind"] == "erk2":
        nlm, nr = _nlm(c["lmax"], c["lmax"]), c["nr"]
        return dict(bytes=16.0 * 5 * nlm * nr + 8.0 * 5 * (c["lmax"] + 1) * nr * nr, flops=5 * 2.0 * 2 * nlm * nr * nr)
    if c["kind"] == "adjoint":
        w = _step_work(c["lmax"], c["nlat"], c["nlon"], c["nr"], False)
        return {k: 3 * v * c["steps"] for k, v in w.items()}
    tot = dict(bytes=0.0, flops=0.0)
    for lmax, nr, _ in _shells(c):
        w = _step_work(lmax, 3 * (lmax + 1) // 2, 3 * (lmax + 1), nr, False)
        tot = {k: tot[k] + w[k] * c["steps"] for k in tot}
    return tot


# ---------------------------------------------------------------- the same in 64 bits, densely
class _Dense:
    """Spherical-harmonic transforms with dense FP64 Legendre matrices and torch's FFT.
    Coefficients: complex (..., nr, nlm), l-major; grid values (..., nr, nlon, nlat)."""

    def __init__(self, lmax, mmax, nlat, nlon):
        self.lmax, self.mmax, self.nlat, self.nlon = lmax, mmax, nlat, nlon
        x, w = np.polynomial.legendre.leggauss(nlat)
        x, w = x[::-1].copy(), w[::-1].copy()
        s = np.sqrt(1 - x * x)
        m = np.arange(mmax + 1)[:, None]
        logs = np.zeros(mmax + 1)
        for k in range(1, mmax + 1):
            logs[k] = logs[k - 1] + 0.5 * math.log((2 * k - 1) / (2 * k))
        with np.errstate(under="ignore"):
            pmm = (-1.0) ** m * np.exp(0.5 * np.log((2 * m + 1) / (4 * math.pi)) + logs[:, None] + m * np.log(s)[None])
        P = np.zeros((mmax + 1, lmax + 1, nlat))
        for l in range(lmax + 1):
            k = min(l, mmax + 1)  # orders below l
            if l <= mmax:
                P[l, l] = pmm[l]
            if k:
                mm = m[:k]
                a = np.sqrt((4.0 * l * l - 1) / (l * l - mm * mm))
                b = np.sqrt(np.maximum((l - 1.0) ** 2 - mm * mm, 0) / (4.0 * (l - 1) ** 2 - 1))
                P[:k, l] = a * (x * P[:k, l - 1] - (b * P[:k, l - 2] if l > 1 else 0))
        l = np.arange(lmax + 1)[None, :, None]
        c = np.sqrt(np.maximum((2.0 * l + 1) * (l * l - m[:, :, None] ** 2) / np.maximum(2.0 * l - 1, 1), 0))
        D = l * x * P
        D[:, 1:] -= (c * 1.0)[:, 1:] * P[:, :-1]
        D /= s
        self.P, self.D = torch.from_numpy(P).to(DEV), torch.from_numpy(D).to(DEV)
        self.Q = torch.from_numpy(m[:, :, None] * P / s).to(DEV)
        self.w = torch.from_numpy(2 * math.pi * w / nlon).to(DEV)
        self.costh = torch.from_numpy(x).to(DEV)
        self.sinth = torch.from_numpy(s).to(DEV)
        ll, mm = _lm(lmax, mmax)
        self.l, self.m = ll, mm
        self.place = mm * (lmax + 1) + ll
        self.ll1 = (ll * (ll + 1)).to(F64)

    def _cols(self, a):
        d = torch.zeros(a.shape[:-1] + ((self.mmax + 1) * (self.lmax + 1),), dtype=a.dtype, device=a.device)
        d = d.index_copy(-1, self.place, a)
        return d.reshape(a.shape[:-1] + (self.mmax + 1, self.lmax + 1)).movedim(-2, 0)

    def _sum(self, cols, tab):
        """cols (m, ..., l) times tab (m, l, i) -> (..., m, i)"""
        flat = cols.reshape(cols.shape[0], -1, cols.shape[-1])
        o = torch.complex(torch.matmul(flat.real.contiguous(), tab), torch.matmul(flat.imag.contiguous(), tab))
        return o.reshape(cols.shape[:-1] + (tab.shape[-1],)).movedim(0, -2)

    def _ifft(self, F):
        return torch.fft.irfft(F, n=self.nlon, dim=-2, norm="forward")

    def _fft(self, f):
        return torch.fft.rfft(f, dim=-2)[..., : self.mmax + 1, :] * self.w

    def _ana(self, G, tab):
        """sum over nodes of G (..., m, i) tab (m, l, i) -> (..., nlm)"""
        g = G.movedim(-2, 0)
        flat = g.reshape(g.shape[0], -1, g.shape[-1])
        t = tab.transpose(1, 2).contiguous()
        o = torch.complex(torch.matmul(flat.real.contiguous(), t), torch.matmul(flat.imag.contiguous(), t))
        o = o.reshape(g.shape[:-1] + (tab.shape[1],)).movedim(0, -2)
        return o.reshape(o.shape[:-2] + (-1,)).index_select(-1, self.place)

    def _real0(self, a):
        return torch.complex(a.real, a.imag * (self.m > 0))

    def synth(self, a):
        return self._ifft(self._sum(self._cols(a), self.P))

    def analysis(self, f):
        return self._real0(self._ana(self._fft(f), self.P))

    def synth_vec(self, S, T):
        s, t = self._cols(S), self._cols(T)
        return (self._ifft(self._sum(s, self.D) + 1j * self._sum(t, self.Q)),
                self._ifft(1j * self._sum(s, self.Q) - self._sum(t, self.D)))

    def raw_vec(self, vt, vp):
        """(S, T) before the division by l(l+1)"""
        gt, gp = self._fft(vt), self._fft(vp)
        return (self._real0(self._ana(gt, self.D) - 1j * self._ana(gp, self.Q)),
                self._real0(-1j * self._ana(gt, self.Q) - self._ana(gp, self.D)))

    def analysis_vec(self, vt, vp):
        inv = torch.where(self.ll1 > 0, 1.0 / self.ll1.clamp(min=1.0), torch.zeros_like(self.ll1))
        S, T = self.raw_vec(vt, vp)
        return S * inv, T * inv


def _radial(nr, rratio):
    """r, dense D1, D2 on the band stencils."""
    ri = rratio / (1 - rratio)
    r = 0.5 * (1 + np.cos(math.pi * (nr - np.arange(1, nr + 1)) / (nr - 1))) + ri
    D = np.zeros((2, nr, nr))
    for n in range(nr):
        a, b = max(0, n - BW), min(nr - 1, n + BW)
        d = r[a:b + 1] - r[n]
        h = np.abs(d).max()
        V = (d[None] / h) ** np.arange(b - a + 1)[:, None]
        for k in (1, 2):
            rhs = np.zeros(b - a + 1)
            rhs[k] = math.factorial(k) / h ** k
            D[k - 1, n, a:b + 1] = np.linalg.solve(V, rhs)
    t = [torch.from_numpy(v).to(DEV) for v in (r, D[0], D[1])]
    return t[0], t[1], t[2], t[2] + (2.0 / t[0])[:, None] * t[1]


def _operators(lmax, r, lap, nu):
    """L_l, l = 0..lmax"""
    l = torch.arange(lmax + 1, device=DEV, dtype=F64)
    return nu * (lap[None] - torch.diag_embed((l * (l + 1))[:, None] / (r * r)[None]))


def _implicit(L, rows):
    """The two halves of the step's operator: E = I/dt + (1-theta) L and S = I/dt - theta L with Dirichlet rows."""
    nr = L.shape[-1]
    eye = torch.eye(nr, device=DEV, dtype=F64) / DT
    S = eye - THETA * L
    if rows:
        S[:, 0] = 0.0
        S[:, -1] = 0.0
        S[:, 0, 0] = 1.0
        S[:, -1, -1] = 1.0
    return eye + (1 - THETA) * L, S


def _per_l(M, x, lvals, lmax, solve=False):
    """M_l x or M_l^-1 x of complex planes x (nr, nlm)."""
    ncol = torch.bincount(lvals, minlength=lmax + 1)
    width, nr = int(ncol.max()), x.shape[0]
    slot = torch.cat([torch.arange(int(n), device=DEV) for n in ncol.tolist()]) + lvals * width
    z = torch.cat([x.real, x.imag], 0).reshape(2, nr, -1)
    d = torch.zeros((2, nr, (lmax + 1) * width), dtype=F64, device=DEV).index_copy(-1, slot, z)
    d = d.reshape(2, nr, lmax + 1, width).permute(2, 1, 0, 3).reshape(lmax + 1, nr, 2 * width)
    y = torch.linalg.solve(M, d) if solve else torch.matmul(M, d)
    y = y.reshape(lmax + 1, nr, 2, width).permute(2, 1, 0, 3).reshape(2, nr, -1).index_select(-1, slot)
    return torch.complex(y[0], y[1])


def _exact_steps(lmax, nlat, nlon, nr, full, steps, x, rratio=RRATIO):
    """CNAB2 steps of the state x: five complex planes (nr, nlm)."""
    T = _Dense(lmax, lmax, nlat, nlon)
    r, D1, D2, lap = _radial(nr, rratio)
    nus = (PM, PM, 1.0, 1.0, PM / PR)
    ops = {nu: _implicit(_operators(lmax, r, lap, nu), True) for nu in set(nus)}
    ro, rr = PM / E, r[:, None]
    j = torch.clamp(torch.arange(nlon, device=DEV), max=nlat - 1)
    ct, st = T.costh[j][None, :, None], T.sinth[j][None, :, None]
    inner = torch.ones(nr, 1, device=DEV, dtype=F64)
    inner[0] = inner[-1] = 0.0

    def D(M, a):
        return torch.complex(torch.matmul(M, a.real), torch.matmul(M, a.imag))

    def nonlinear(x):
        ut, up, bt, bp, tm = x
        zero = torch.zeros_like(ut)
        vt, vp = T.synth_vec(up, ut)
        gt, gp = T.synth_vec(tm / rr, zero)
        if not full:
            S, Z = T.analysis_vec(ro * ct * vp, -ro * ct * vt)
            return [Z, S, zero, zero, T.analysis(-(vt * gt + vp * gp))]
        curl = lambda p, t: (-T.ll1 / rr ** 2 * t, T.ll1 / rr ** 2 * p - D(D2, p) - 2 / rr * D(D1, p))  # noqa: E731
        rad = lambda p: T.synth(T.ll1 * p / rr ** 2)  # noqa: E731
        wp_, wt_ = curl(up, ut)
        jp_, jt_ = curl(bp, bt)
        wt, wp = T.synth_vec(wp_, wt_)
        Bt, Bp = T.synth_vec(bp, bt)
        jt, jp = T.synth_vec(jp_, jt_)
        ur, wr, Br, jr, gr = rad(up), rad(wp_), rad(bp), rad(jp_), T.synth(D(D1, tm))
        at = -ro * (vp * wr - ur * wp) + ro * ct * vp + ro * (jp * Br - jr * Bp)
        ap = -ro * (ur * wt - vt * wr) - ro * (ct * vt + st * ur) + ro * (jr * Bt - jt * Br)
        S, Z = T.analysis_vec(at, ap)
        bS, bZ = T.raw_vec(vp * Br - ur * Bp, ur * Bt - vt * Br)
        return [Z, S, bS, -bZ, T.analysis(-(ur * gr + vt * gt + vp * gp))]

    prev = None
    for _ in range(steps):
        nl = nonlinear(x)
        prev = nl if prev is None else prev
        new = []
        for f in range(5):
            Em, Sm = ops[nus[f]]
            u = x[f] * inner if f == 4 else x[f]
            rhs = (_per_l(Em, u, T.l, lmax) + 1.5 * nl[f] - 0.5 * prev[f]) * inner
            new.append(_per_l(Sm, rhs, T.l, lmax, solve=True))
        x, prev = new, nl
    return x, T, r


def _exact_state(lmax, nlat, nlon, nr, full, steps, re, im, rratio=RRATIO):
    x, _, _ = _exact_steps(lmax, nlat, nlon, nr, full, steps, list(torch.complex(re, im)), rratio)
    return [torch.stack([v.real for v in x]), torch.stack([v.imag for v in x])]


def _phi_matrices(A, h):
    """exp(hA), phi1(hA), phi2(hA) from one augmented exponential."""
    n, k = A.shape[-1], A.shape[0]
    M = torch.zeros((k, 3 * n, 3 * n), dtype=F64, device=DEV)
    M[:, :n, :n] = h * A
    eye = torch.eye(n, dtype=F64, device=DEV)
    M[:, :n, n:2 * n] = eye
    M[:, n:2 * n, 2 * n:] = eye
    X = torch.linalg.matrix_exp(M)
    return X[:, :n, :n], X[:, :n, n:2 * n], X[:, :n, 2 * n:]


def exact(case, seed):
    c, g = case, _gen(seed)
    if c["kind"] == "step":
        re, im = _state(g, c["lmax"], c["nr"], 1e-5 if c["full"] else 1e-3)
        return _exact_state(c["lmax"], c["nlat"], c["nlon"], c["nr"], c["full"], c["steps"], re, im)
    if c["kind"] == "sht":
        spec, phys = _sht_inputs(c, g)
        T = _Dense(c["lmax"], c["mmax"], c["nlat"], c["nlon"])
        a = [torch.complex(*p) for p in spec]
        if c["vector"]:
            to_phys = list(T.synth_vec(a[1], a[0]))  # the pair is (toroidal, poloidal)
            S, Z = T.analysis_vec(*phys)
            to_spec = [Z, S]
        else:
            to_phys, to_spec = [T.synth(a[0])], [T.analysis(phys[0])]
        return {"phys": to_phys, "spec": [[z.real.contiguous(), z.imag.contiguous()] for z in to_spec]}
    if c["kind"] == "cnab2":
        u, (n1, n0) = _plane_inputs(c, g, 2)
        u, n1, n0 = torch.complex(*u), torch.complex(*n1), torch.complex(*n0)
        l, _ = _lm(c["lmax"], c["lmax"])
        r, _, _, lap = _radial(c["nr"], RRATIO)
        Em, Sm = _implicit(_operators(c["lmax"], r, lap, PM), c["bc_rows"])
        rhs = _per_l(Em, u, l, c["lmax"]) + 1.5 * n1 - 0.5 * n0
        if c["bc_rows"]:
            rhs[0] = 0.0
            rhs[-1] = 0.0
        sol = _per_l(Sm, rhs, l, c["lmax"], solve=True)
        return [rhs.real.contiguous(), rhs.imag.contiguous(), sol.real.contiguous(), sol.imag.contiguous()]
    if c["kind"] == "erk2":
        u, (n0, n1) = _plane_inputs(c, g, 2)
        u, n0, n1 = torch.complex(*u), torch.complex(*n0), torch.complex(*n1)
        l, _ = _lm(c["lmax"], c["lmax"])
        r, _, _, lap = _radial(c["nr"], RRATIO)
        A = _operators(c["lmax"], r, lap, 1.0)
        Eh, p1h, _ = _phi_matrices(A, DT / 2)
        Ef, p1f, p2f = _phi_matrices(A, DT)
        dot = lambda M, x: _per_l(M, x, l, c["lmax"])  # noqa: E731
        stage = dot(Eh, u) + DT / 2 * dot(p1h, n0)
        new = dot(Ef, u) + DT * (dot(p1f, n0) + dot(p2f, n1 - n0))
        return [stage.real.contiguous(), stage.imag.contiguous(), new.real.contiguous(), new.imag.contiguous()]
    if c["kind"] == "adjoint":
        re, im, target = _adjoint_inputs(c, g)
        re.requires_grad_(True)
        im.requires_grad_(True)
        x, T, _ = _exact_steps(c["lmax"], c["nlat"], c["nlon"], c["nr"], False, c["steps"],
                               list(torch.complex(re, im).unbind(0)))
        J = 0.5 * ((T.synth(x[4][c["nr"] - 2:c["nr"] - 1])[0] - target) ** 2).sum()
        dre, dim = torch.autograd.grad(J, (re, im))
        return [float(J.detach()), dre, dim]
    return [_exact_state(lmax, 3 * (lmax + 1) // 2, 3 * (lmax + 1), nr, False, c["steps"], *_state(g, lmax, nr), rr)
            for lmax, nr, rr in _shells(c)]
