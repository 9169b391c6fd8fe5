"""What this framework is timed on: whole solves, resident marches, batched solves,
the single step operators and the learned step, through the package's entry points.

The sizes are the benchmark configurations of ``workloads.py``, the reference's
validation grids (51x51x101, 193x193x1201, 365x365x425, nT = 801), which are odd or
prime on every axis, and in ``draw`` any grid of the same ranges.  Every input is made
from the seed; ``exact`` evaluates the same path in 64 bits with plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from angularspectrum_heterogeneous_amd import SolverParams, _lib, angular_spectrum_solve, make_bowl_source_planes
from angularspectrum_heterogeneous_amd.batch import batch_solve
from angularspectrum_heterogeneous_amd.learned import LearnedStep
from angularspectrum_heterogeneous_amd.plan import MarchPlan
from angularspectrum_heterogeneous_amd.sources import skull_screen

FFT_LINES = (64, 128, 192, 256, 384)      # sizes of workloads.py
FFT_LENGTHS = (256, 512, 1024, 2048)
C, KW, NLAY = 32, 9, 4                    # the learned step's network


def _grid(kind, nX, nY, nT, steps, **opts):
    """A march case: `steps` z-steps on nX x nY x nT.  source: piston (focused, steered
    disk) or bowl (plane by plane); flux: kt, tvd, rusanov or sequential; water: lossless-like
    quadratic attenuation instead of the power law; fw, sa: frequency-weighted and
    super-absorbing boundaries; obliquity: beam-averaged nonlinear obliquity; screen:
    a skull phase and amplitude screen half way."""
    c = dict(kind=kind, nX=nX, nY=nY, nT=nT, steps=steps, source="piston", flux="kt", water=False, fw=False, sa=False,
             obliquity=False, screen=False)
    c.update(opts)
    return c


def listed():
    return [
        # the smallest validation run (validate_solver test 1): one short solve from a host
        # array, where launches, plan set-up and host work count
        dict(name="solve_51x51x101_water", **_grid("solve", 51, 51, 101, 50, flux="sequential", water=True)),
        # the small plain-method configuration, a whole solve from a host array
        dict(name="solve_64x64x256", **_grid("solve", 64, 64, 256, 65)),
        # an ordinary grid picked by spacing rather than by size: even and odd axes, TVD flux,
        # one screen, as in the transcranial workflow
        dict(name="solve_120x101x301_screen", **_grid("solve", 120, 101, 301, 24, flux="tvd", screen=True, fw=True)),
        # the headline beam (256x256x1024, all boundaries on): the resident march
        dict(name="march_256x256x1024", **_grid("march", 256, 256, 1024, 8, fw=True, sa=True)),
        # the focused-piston validation grid (193x193x1201, prime on every axis), resident
        dict(name="march_193x193x1201", **_grid("march", 193, 193, 1201, 2)),
        # nonlinear obliquity on an FFT grid
        dict(name="march_192x192x512_obliquity", **_grid("march", 192, 192, 512, 12, obliquity=True, fw=True)),
        # the bowl validation run (365x365x425, odd, plane-by-plane source, water, all boundaries)
        dict(name="solve_365x365x425_bowl", **_grid("solve", 365, 365, 425, 6, source="bowl", water=True, fw=True, sa=True)),
        # the largest: bowl through a skull screen
        dict(name="solve_384x384x1024_skull", **_grid("solve", 384, 384, 1024, 24, source="bowl", screen=True)),
        # transmit configurations of uneven size solved side by side
        dict(name="batch_8_uneven", kind="batch", count=8, most=192, steps=10),
        # every single-step operator of the ABI once (the drop-in step functions), odd nT
        dict(name="operators_128x96x801", kind="operators", nX=128, nY=96, nT=801),
        # one training step of the learned update (forward, gradients, Adam)
        dict(name="train_256x1024", kind="train", cols=256, nT=1024),
        # fused inference of the learned update over a field's columns
        dict(name="infer_16384x1024", kind="infer", cols=16384, nT=1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "march", "march", "march", "batch", "operators", "train", "infer"])
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(3, 8), most=rng.choice([128, 160, 192]), steps=rng.randint(6, 12))
    if kind == "train":
        return dict(kind=kind, cols=_log_int(rng, 16, 256), nT=rng.choice(FFT_LENGTHS))
    if kind == "infer":
        return dict(kind=kind, cols=_log_int(rng, 512, 16384), nT=rng.choice(FFT_LENGTHS))
    if rng.random() < 0.4:
        nX, nY, nT = rng.choice(FFT_LINES), rng.choice(FFT_LINES), rng.choice(FFT_LENGTHS)
    else:
        nX, nY, nT = _log_int(rng, 40, 384), _log_int(rng, 40, 384), _log_int(rng, 96, 1600)
    while nX * nY * nT > 256 * 256 * 1024:  # (the listed cases hold the largest grids)
        nX, nY, nT = max(40, nX * 3 // 4), max(40, nY * 3 // 4), nT
    if kind == "operators":
        return dict(kind=kind, nX=min(nX, 160), nY=min(nY, 160), nT=nT)
    steps = max(2, min(40, int(1.2e8 / (nX * nY * nT))))
    flux = rng.choice(["kt", "kt", "tvd", "rusanov", "sequential"])
    return _grid(kind, nX, nY, nT, steps, flux=flux, water=rng.random() < 0.3, fw=rng.random() < 0.5,
                 sa=rng.random() < 0.5 and nT <= 1024, obliquity=rng.random() < 0.2,
                 screen=kind == "solve" and rng.random() < 0.5,
                 source="bowl" if kind == "solve" and min(nX, nY) >= 160 and rng.random() < 0.5 else "piston")


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
DX, C0, RHO0, BETA, F0 = 3.08e-4, 1540.0, 1000.0, 3.5, 1e6


def _dt(nT):
    # the benchmark's 40 ns at 1024 samples; shorter windows keep the pulse inside
    return 4e-8 * max(1.0, 256.0 / nT)


def _axis(n, d):
    return (np.arange(n) - (n - 1) / 2) * d


def _piston(nX, nY, nT, rng, p0):
    """Disk with a focusing delay law and a lateral steering; float32 on the GPU."""
    x, y, t = (torch.from_numpy(a).cuda() for a in (_axis(nX, DX), _axis(nY, DX), _axis(nT, _dt(nT))))
    radius = 0.3 * min(nX, nY) * DX
    focus = radius * rng.uniform(2.5, 4.0)
    steer = rng.uniform(-0.1, 0.1) * radius
    p = p0 * rng.uniform(0.5, 1.0)
    r2 = x[:, None] ** 2 + y[None, :] ** 2
    tau = -((x[:, None] - steer) ** 2 + y[None, :] ** 2) / (2 * focus * C0) + radius ** 2 / (4 * focus * C0)
    tt = t[None, None, :] - tau[:, :, None]
    w0, cycles = 2 * np.pi * F0, 3 if nT < 512 else 5
    burst = torch.exp(-(1.05 * tt * w0 / (cycles * np.pi)) ** 4) * torch.sin(w0 * tt) * p
    return ((r2 <= radius ** 2)[:, :, None] * burst).float().contiguous()


def _field_and_params(case, seed):
    """(initial field or source slice, SolverParams keywords) of a march case."""
    rng = np.random.default_rng(seed)
    nX, nY, nT, steps = case["nX"], case["nY"], case["nT"], case["steps"]
    kw = dict(dX=DX, dY=DX, dT=_dt(nT), c0=C0, rho0=RHO0, beta=BETA, alpha0=-1.0 if case["water"] else 0.5,
              attenPow=1.1, f0=F0, propDist=(steps - 0.4) * DX, dZmin=DX, boundaryFactor=0.1,
              boundaryProfile="wendland", useSplitStep=case["flux"] != "sequential",
              fluxScheme="kt" if case["flux"] == "kt" else "rusanov", useTVD=case["flux"] == "tvd",
              useFreqWeightedBoundary=case["fw"], useSuperAbsorbing=case["sa"],
              useNonlinearityObliquity=case["obliquity"])
    if case["source"] == "bowl":
        x, y, t = _axis(nX, DX), _axis(nY, DX), _axis(nT, _dt(nT))
        radius = 0.39 * min(nX, nY) * DX
        planes, _ = make_bowl_source_planes(x, y, t, F0, C0, 4e5 * rng.uniform(0.5, 1.0), radius, 1.8 * radius, DX,
                                            ncycles=3, dur=2, inner_radius=0.4 * radius,
                                            focus=radius * rng.uniform(1.1, 1.5), n_elements=8)
        field, kw["sourcePlanes"] = planes[0][1], planes[1:]
    else:
        field = _piston(nX, nY, nT, rng, 1e6)
    if case["screen"]:
        phase, amp, _ = skull_screen(nX, nY, DX, DX, F0, seed=seed)
        kw["phaseScreens"] = [(steps // 2 * DX + 0.3 * DX, phase, amp)]
    return field, kw


def _batch_cases(case):
    rng = np.random.default_rng(case["count"] + 100 * case["steps"])  # sizes by the case, inputs by the seed
    lines = [n for n in FFT_LINES[1:] if n <= case["most"]] + [case["most"] - 28]
    return [_grid("solve", int(rng.choice(lines)), int(rng.choice(lines)), int(rng.choice([256, 512, 512, 300])),
                  case["steps"] + k % 3, fw=True) for k in range(case["count"])]


def _bursts(cols, nT, seed, lo=1e3):
    """Tone bursts of amplitude lo .. 1.5 MPa (log-uniform), random cycles, delay and phase:
    a field's columns from its edge to its beam; float32 on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def uni(a, b):
        return a + (b - a) * torch.rand((cols, 1), generator=g, device="cuda", dtype=torch.float64)

    t = torch.from_numpy(_axis(nT, 4e-8)).cuda()
    p0 = torch.exp(uni(math.log(lo), math.log(1.5e6)))
    cyc, delay, phase = uni(3.0, 6.0), uni(-0.25, 0.25) * nT * 4e-8, uni(0.0, 2 * np.pi)
    w0 = 2 * np.pi * F0 * uni(0.85, 1.15)
    tt = t[None, :] - delay
    return (torch.exp(-(1.05 * tt * w0 / (cyc * np.pi)) ** 4) * torch.sin(w0 * tt + phase) * p0).float().contiguous()


def _weights(seed):
    """Network parameters as LearnedStep lays them out: per layer W[out][in][tap], then the bias."""
    rng = np.random.default_rng(seed)
    flat = []
    for j in range(NLAY):
        W = rng.normal(0.0, math.sqrt(2.0 / (KW * (2 if j == 0 else C))), size=(C, C, KW))
        b = rng.normal(0.0, 0.02, size=C)
        if j == 0:
            W[:, 2:] = 0.0
        if j == NLAY - 1:
            W[1:], b[1:] = 0.0, 0.0
            W *= 0.1
        flat += [W.reshape(-1), b]
    return np.concatenate(flat).astype(np.float32)


BURGERS = BETA / (2 * C0 ** 3 * RHO0)
NET_C = DX * BURGERS / 4e-8
DPDT_MAX = 6e12


def _net_inputs(case, seed):
    u = _bursts(case["cols"], case["nT"], seed, 1e5 if case["kind"] == "train" else 1e3)
    if case["kind"] == "infer":
        return u, None
    return u, _kt(u.double(), BURGERS, DX, 4e-8).float()


def _operator_inputs(case, seed):
    shape = (case["nX"], case["nY"], case["nT"])
    c = _grid("operators", *shape, 1, flux="kt", fw=True, sa=True)
    field, kw = _field_and_params(c, seed)
    phase, amp, _ = skull_screen(shape[0], shape[1], DX, DX, F0, seed=seed)
    dz_cfl = 1.7 * kw["dT"] / (BURGERS * float(field.abs().max()))  # CFL 1.7: four sub-steps at target 0.5
    return field, kw, phase, amp, dz_cfl


class _State:
    def __init__(self, **kw):
        self.__dict__.update(kw)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "solve":
        field, kw = _field_and_params(case, seed)
        if isinstance(field, torch.Tensor):
            field = field.cpu().numpy()  # a solve's field comes from the host (a sparse source stays sparse)
        return _State(kind=kind, field=field, params=SolverParams(**kw))
    if kind == "march":
        field, kw = _field_and_params(case, seed)
        shape, rows = tuple(field.shape), case["steps"]
        plan = MarchPlan(shape, SolverParams(**kw))
        plan.set_dz(DX)
        outs = torch.zeros((4, rows) + shape[:2], device="cuda")
        pax = torch.zeros((rows, shape[2]), device="cuda")
        stats = torch.zeros(rows + 1, dtype=torch.int32, device="cuda")
        io = _lib.AshStepIO()
        io.max_rows, io.dz = rows, DX
        io.pnp_dev, io.ppp_dev, io.pI_dev, io.pIloss_dev = (outs[k].data_ptr() for k in range(4))
        io.pax_dev, io.stats_dev = pax.data_ptr(), stats.data_ptr()
        return _State(kind=kind, field=field, plan=plan, outs=outs, pax=pax, stats=stats, io=io, rows=rows,
                      final=torch.empty_like(field))
    if kind == "batch":
        made = [_field_and_params(c, 100 * seed + k) for k, c in enumerate(_batch_cases(case))]
        return _State(kind=kind, instances=[(f, SolverParams(**kw)) for f, kw in made])
    if kind == "operators":
        field, kw, phase, amp, dz_cfl = _operator_inputs(case, seed)
        plan = MarchPlan(tuple(field.shape), SolverParams(**kw))
        plan.set_dz(DX)
        return _State(kind=kind, field=field, plan=plan, phase=torch.from_numpy(phase).cuda(),
                      amp=torch.from_numpy(amp).cuda(), dz_cfl=dz_cfl, dT=kw["dT"])
    u, un = _net_inputs(case, seed)
    return _State(kind=kind, u=u, un=un, net=LearnedStep(case["nT"], max_cols=min(case["cols"], 256),
                                                         params=_weights(seed)))


def run(s):
    if s.kind == "solve":
        return angular_spectrum_solve(s.field, s.params, verbose=False)
    if s.kind == "march":
        s.stats.zero_()
        s.plan.load(s.field, s.stats)
        for row in range(s.rows):
            s.io.row = row
            s.plan.step(s.io)
        s.plan.store(s.final)
        return s.final, s.outs, s.pax, s.stats.view(torch.float32)
    if s.kind == "batch":
        return batch_solve(s.instances)
    if s.kind == "operators":
        p, x = s.plan, s.field
        return {
            "attenuation": p.attenuation_step(x, 0.5),
            "propagator": p.angular_spectrum_step(x, True),
            "freq_weighted": p.freq_weighted_boundary_step(x),
            "super_absorbing": p.super_absorbing_step(x),
            "screen": p.apply_phase_screen(x, s.phase, s.amp),
            "kt_adaptive": p.nonlinear_step(x, _lib.NL_KT, s.dz_cfl, 1.0, _lib.SUBCYCLE_GLOBAL),
            "kt_minmod": p.nonlinear_step(x, _lib.NL_KT_MINMOD, DX),
            "rusanov": p.nonlinear_step(x, _lib.NL_RUSANOV, DX),
            "tvd": p.nonlinear_step(x, _lib.NL_TVD, DX, 1.5),
            "march": p.march_step(x),
        }
    if s.kind == "train":
        loss, grads = s.net.loss_grad(s.u, s.un, NET_C)
        s.net.adam(grads, 1e-3)
        return loss, grads
    u = s.u.clone()  # (the update is in place; the next pass starts from the same columns)
    flags = s.net.apply(u, NET_C, DPDT_MAX, 4e-8)
    return u, flags


def work(case):
    """Bytes: the inputs once and the outputs once.  Flops: real transforms at 2.5 n log2 n and
    complex ones at 5 n log2 n per line, the flux at 60 per sample, the network's products."""
    kind = case["kind"]
    if kind in ("train", "infer"):
        n = case["cols"] * case["nT"]
        per = 2 * KW * (2 * C + 2 * C * C + C)  # products of one forward pass, per sample
        return {"bytes": n * 8, "flops": n * per * (3 if kind == "train" else 1)}
    if kind == "batch":
        parts = [work(c) for c in _batch_cases(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    nX, nY, nT = case["nX"], case["nY"], case["nT"]
    vox = nX * nY * nT
    visit = vox / 2 * 2 * 5 * math.log2(nX * nY)  # nT/2 bins, 2-D transform and its inverse
    column = vox * 2 * 2.5 * math.log2(nT)        # inverse and forward real transform
    if kind == "operators":
        return {"bytes": 10 * 8 * vox, "flops": 7 * visit + 9 * column + 12 * 60 * vox}
    visits, columns = (2, 2) if case["flux"] == "sequential" else (3, 3)
    if case["obliquity"]:
        visits, columns = visits + 1, columns + 1
    step = visits * visit + columns * column + vox * 60
    return {"bytes": 8 * vox + case["steps"] * 4 * (4 * nX * nY + nT), "flops": step * case["steps"]}


# ---------------------------------------------------------------------------
# The same paths in 64 bits
# ---------------------------------------------------------------------------
def _kt_rate(u, coef, mc):
    dm, dp = u[..., 1:-1] - u[..., :-2], u[..., 2:] - u[..., 1:-1]
    size = torch.minimum(dm.abs(), dp.abs())
    if mc:
        size = torch.minimum(2 * size, 0.5 * (dm + dp).abs())
    half = torch.zeros_like(u)
    half[..., 1:-1] = torch.where(dm * dp > 0, torch.sign(dm) * size, torch.zeros_like(dm)) / 2
    a, b = (u + half)[..., :-1], (u - half)[..., 1:]
    hi = torch.maximum(-a, -b).clamp(min=0.0)
    lo = torch.minimum(-a, -b).clamp(max=0.0)
    gap = hi - lo
    flux = (-0.5 * hi * a * a + 0.5 * lo * b * b - hi * lo * (b - a)) / torch.where(gap < 1e-14, torch.ones_like(gap), gap)
    small = 0.5 * (-0.5 * a * a - 0.5 * b * b) - 0.5 * torch.maximum(a.abs(), b.abs()) * (b - a)
    flux = torch.where(gap < 1e-14, small, flux)
    rate = torch.zeros_like(u)
    rate[..., 1:-1] = -coef * (flux[..., 1:] - flux[..., :-1])
    return rate


def _kt(u, N, dz, dT, mc=True, cfl=None):
    n = 1
    if cfl is not None:
        n = max(1, math.ceil(N * float(u.abs().max()) * dz / dT / cfl))
    for _ in range(n):
        mid = u + dz / n * _kt_rate(u, N / dT, mc)
        u = 0.5 * u + 0.5 * (mid + dz / n * _kt_rate(mid, N / dT, mc))
    return u


def _rusanov(u, cf, tvd=None):
    a, b = u[..., :-1], u[..., 1:]
    speed = torch.maximum(a.abs(), b.abs())
    if tvd is None:
        flux = -(a * a + b * b) / 2 - speed * (b - a)
        phi = 1.0
    else:
        flux = -(a * a + b * b) / 4 - 0.5 * speed * (b - a)
        dm, dp = u[..., 1:-1] - u[..., :-2], u[..., 2:] - u[..., 1:-1]
        eps = 1e-30

        def limit(p, q):
            r = p / (q + eps * torch.sign(q + eps))
            return torch.clamp(torch.minimum((tvd * r).clamp(max=1.0), r.clamp(max=tvd)), min=0.0)

        phi = 0.5 * (limit(dp, dm) + limit(dm, dp))
    out = u.clone()
    out[..., 1:-1] -= cf * phi * (flux[..., 1:] - flux[..., :-1])
    return out


class _Exact:
    """The march of SolverParams keywords `kw` on an nX x nY x nT grid in float64."""

    def __init__(self, shape, kw):
        self.shape, self.kw = shape, kw
        nX, nY, nT = shape
        dT = kw["dT"]

        def centred(n, d):
            k = np.arange(n) / (n - 1) / d * 2 * np.pi
            return np.fft.ifftshift(k - np.mean(k))

        kx, ky = centred(nX, DX), centred(nY, DX)
        self.kk = torch.from_numpy(kx ** 2).cuda()[:, None] + torch.from_numpy(ky ** 2).cuda()[None, :]
        kt = np.arange(nT) / (nT - 1) / dT * 2 * np.pi / C0
        kt = kt - np.mean(kt)
        self.lam = C0 / np.mean(np.abs(kt[kt != 0]))
        nat = np.fft.ifftshift(kt)
        m = np.arange(nT // 2 + 1)
        kept = (m >= 1) & (m <= (nT + 1) // 2 - 1)
        self.kt = np.where(kept, nat[: nT // 2 + 1], 0.0)
        f = m / (nT * dT)
        self.f = f
        self.ka = 2 * np.pi * f / C0
        db = 20 * np.log10(np.e)
        if kw["alpha0"] < 0:
            conv = 2.17e-3 / 1e12 * 1e2 / db
            self.al = conv * f ** 2
            disp = conv / (2 * np.pi) ** 2 * np.tan(np.pi) * (2 * np.pi * f - 2 * np.pi * F0)
        else:
            y = kw["attenPow"]
            conv = kw["alpha0"] / 1e6 ** y * 1e2 / db
            self.al = conv * f ** y
            disp = conv / (2 * np.pi) ** y * np.tan(np.pi * y / 2) * ((2 * np.pi * f) ** (y - 1) - (2 * np.pi * F0) ** (y - 1))
        self.disp = np.where(m > 0, 2 * np.pi * disp * f, 0.0)
        self.water = kw["alpha0"] < 0
        self.taps, self.ramps = [], []
        for n in shape:
            w = max(round(n * kw["boundaryFactor"]), 1)
            i = np.arange(n)
            s = np.where(i >= n - w, (i - (n - w - 1)) / w, np.where(i < w, (w - i - 1) / w, -1.0))
            prof = np.clip(1 - 10 * s ** 3 + 15 * s ** 4 - 6 * s ** 5, 0, 1)
            self.taps.append(torch.from_numpy(np.where(s < 0, 1.0, prof)).cuda())
            self.ramps.append(torch.from_numpy(np.maximum(s, 0.0)).cuda())
        self.f0_bin = max(F0 * nT * dT, 1.0)
        self.cache = {}

    def row(self, v):
        return torch.from_numpy(np.ascontiguousarray(v)).cuda()

    def operator(self, dz_prop, dz_att, dz):
        key = (dz_prop, dz_att, dz)
        if key in self.cache:
            return self.cache[key]
        kk = self.kk[:, :, None]
        phase, log = torch.zeros(self.kk.shape + (len(self.f),), dtype=torch.float64, device="cuda"), None
        gain = None
        if dz_prop:
            kmax = np.pi / DX
            cut = 0.05 * (1 + 0.7 * (dz / self.lam) * 5)
            hi = min(kmax * (1 - cut), kmax * 0.95)
            lo = 0.8 * hi
            k = torch.sqrt(self.kk)
            band = torch.where(k <= lo, torch.ones_like(k), 0.5 * (1 + torch.cos(np.pi * (k - lo) / (hi - lo))))
            band = torch.where(k > hi, torch.zeros_like(k), band)
            kt = self.row(self.kt)
            d2 = kt * kt - kk
            root = torch.sqrt(d2.abs())
            phase += torch.where(d2 > 0, dz_prop * (kk / (kt + root).clamp(min=1e-300)), dz_prop * kt)
            log = torch.where(d2 > 0, torch.zeros_like(d2), -dz_prop * root)
            gain = band[:, :, None] * (kt > 0)
            del d2, root
        if dz_att:
            ka = self.row(self.ka)
            z2 = ka * ka - kk
            path = torch.where(z2 > 0, ka / torch.maximum(torch.sqrt(z2.clamp(min=0.0)), ka * 1e-6).clamp(min=1e-300), torch.zeros_like(z2))
            path[..., 0] = 0.0
            del z2
            shift = -self.row(self.disp * dz_att) * path
            phase += shift
            loss = -self.row(self.al * dz_att) * path
            log = loss if log is None else log + loss
            if self.water:
                keep = (torch.cos(shift) >= 0).double()
                gain = keep if gain is None else gain * keep
            del path, shift, loss
        amp = torch.exp(log)
        if gain is not None:
            amp = amp * gain
        self.cache[key] = torch.polar(amp, phase)
        return self.cache[key]

    def forward(self, u):
        return torch.fft.rfft(u, dim=2)

    def back(self, S):
        nT = self.shape[2]
        S = S.clone()
        S[..., 0] = S[..., 0].real + 0j
        if nT % 2 == 0:
            S[..., -1] = S[..., -1].real + 0j
        return torch.fft.irfft(S, n=nT, dim=2)

    def visit(self, u, dz_prop, dz_att, dz):
        S = torch.fft.fft2(self.forward(u), dim=(0, 1))
        S *= self.operator(dz_prop, dz_att, dz)
        return self.back(torch.fft.ifft2(S, dim=(0, 1)))

    def taper(self, u, half):
        x, y, t = (torch.sqrt(v) if half else v for v in self.taps)
        return u * x[:, None, None] * y[None, :, None] * t[None, None, :]

    def oblique(self, u):
        power = torch.fft.fft2(self.forward(u), dim=(0, 1)).abs() ** 2
        ka = self.row(self.ka)
        z2 = ka * ka - self.kk[:, :, None]
        power = torch.where(z2 > 0, power, torch.zeros_like(power))
        power[..., 0] = 0.0
        path = torch.where(z2 > 0, ka / torch.maximum(torch.sqrt(z2.clamp(min=0.0)), ka * 1e-6).clamp(min=1e-300), torch.zeros_like(z2))
        return float((power * path).sum() / (power.sum() + 1e-30))

    def step(self, u, dz):
        kw = self.kw
        N = BURGERS
        if not kw["useSplitStep"]:
            u = self.taper(self.visit(u, dz, 0.0, dz), False)
            if kw["useNonlinearityObliquity"]:
                N = N * self.oblique(u)
            u = _rusanov(u, N * dz / kw["dT"])
            return self.visit(u, 0.0, dz, dz)
        u = self.taper(self.visit(u, dz / 2, dz / 2, dz), True)
        if kw["useNonlinearityObliquity"]:
            N = N * self.oblique(u)
        if kw["fluxScheme"] == "kt":
            u = _kt(u, N, dz, kw["dT"])
        else:
            tvd = max(1.0, 2.0 - 0.7 * dz / (C0 / F0) * 10) if kw["useTVD"] else None
            u = _rusanov(u, N * dz / kw["dT"], tvd)
        u = self.taper(self.visit(u, dz / 2, 0.0, dz), True)
        return self.visit(u, 0.0, dz / 2, dz)

    def weighted(self, u):
        f1 = self.f[1]
        power = self.row(np.clip(F0 / np.maximum(self.f, f1), 0.1, 10.0))
        lg = torch.log2(self.taps[0])[:, None] + torch.log2(self.taps[1])[None, :]
        return self.back(self.forward(u) * torch.exp2(power * lg[:, :, None]))

    def absorb(self, u, strength=0.8):
        S = self.forward(u)
        w = 2 * np.pi * self.f
        coef = self.row(np.where(w > 0.5 * w[1], C0 / np.where(w > 0, w, 1.0), 0.0)) * -1j
        for ax in (0, 1):
            n = self.shape[ax]
            L = S.transpose(0, ax)
            d = torch.empty_like(L)
            d[1:-1] = (L[2:] - L[:-2]) / (2 * DX)
            d[0], d[-1] = (L[1] - L[0]) / DX, (L[-1] - L[-2]) / DX
            side = torch.where(torch.arange(n, device="cuda") < n // 2, 1.0, -1.0).double()
            wt = strength * self.ramps[ax]
            S = (L - wt[:, None, None] * 0.5 * (L + side[:, None, None] * coef * d)).transpose(0, ax)
        return self.back(S)

    def screen(self, u, phase, amp):
        fs = self.row(np.arange(len(self.f)) / self.f0_bin)
        ph = self.row(phase.astype(np.float64))[:, :, None] * fs
        am = self.row(np.clip(amp.astype(np.float64), 1e-6, 1.0))[:, :, None] ** fs
        S = self.forward(u)
        return self.back(S * torch.polar(am, -ph))

    def source(self, sl):
        t, d = self.row(sl.taxis), self.row(sl.delays)
        tt = t[None, None, :] - d[:, :, None]
        w0 = 2 * np.pi * sl.f0
        burst = torch.exp(-(1.05 * tt * w0 / (sl.ncycles * np.pi)) ** (2 * sl.dur)) * torch.sin(w0 * tt) * sl.p0
        return (self.row(sl.mask.astype(np.float64))[:, :, None] * burst).float().double()

    def solve(self, field, dz_last=None, steps=None):
        """All outputs of a solve over kw's distance (or `steps` whole steps)."""
        kw = self.kw
        u = field.double() if isinstance(field, torch.Tensor) else self.source(field)
        before = (u * u).sum(2)
        z, zs, rows = 0.0, [], []
        while (z < kw["propDist"] - 1e-15) if steps is None else len(zs) < steps:
            dz = min(DX, kw["propDist"] - z) if steps is None else DX
            if dz != DX:
                self.cache.clear()
            u = self.step(u, dz)
            if kw["useFreqWeightedBoundary"]:
                u = self.weighted(u)
            if kw["useSuperAbsorbing"]:
                u = self.absorb(u)
            for zp, phase, amp in kw.get("phaseScreens") or []:
                if z < zp <= z + dz:
                    u = self.screen(u, phase, amp)
            for zp, sl in kw.get("sourcePlanes") or []:
                if z < zp <= z + dz:
                    u = u + self.source(sl)
            after = (u * u).sum(2)
            rows.append((u.amin(2), u.amax(2), after, (before - after).clamp(min=0.0),
                         u[self.shape[0] // 2, self.shape[1] // 2].clone(), u.abs().amax()))
            before = after
            zs.append(dz)
            z = sum(zs)
        maps = [torch.stack([r[k] for r in rows], 0) for k in range(4)]
        return u, maps, np.cumsum(zs), torch.stack([r[4] for r in rows], 0), [float(r[5]) for r in rows]

    def outputs(self, field):
        u, maps, zs, pax, _ = self.solve(field)
        return [u.cpu().numpy()] + [m.permute(1, 2, 0).cpu().numpy() for m in maps] + [zs, pax.t().cpu().numpy()]


def _network(u, params):
    """Output of the network for columns u (cols, nT) in float64, and the columns' amplitudes."""
    A = u.abs().amax(1, keepdim=True)
    x = u / A
    h = torch.stack([x, x * x], 1)
    nT, at = u.shape[1], 0
    for j in range(NLAY):
        W = params[at: at + C * C * KW].view(C, C, KW)
        b = params[at + C * C * KW: at + C * C * KW + C]
        at += C * C * KW + C
        if j == 0:
            W = W[:, :2]
        if j == NLAY - 1:
            W, b = W[:1], b[:1]
        pad = torch.nn.functional.pad(h, (KW // 2, KW // 2))
        out = b[None, :, None]
        for k in range(KW):
            out = out + torch.matmul(W[:, :, k].contiguous(), pad[:, :, k: k + nT].contiguous())
        h = torch.relu(out) if j < NLAY - 1 else out
    return h[:, 0], A


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve":
        field, kw = _field_and_params(case, seed)
        return _Exact((case["nX"], case["nY"], case["nT"]), kw).outputs(field)
    if kind == "batch":
        got = []
        for k, c in enumerate(_batch_cases(case)):
            field, kw = _field_and_params(c, 100 * seed + k)
            got.append(_Exact((c["nX"], c["nY"], c["nT"]), kw).outputs(field))
        return got
    if kind == "march":
        field, kw = _field_and_params(case, seed)
        e = _Exact((case["nX"], case["nY"], case["nT"]), kw)
        u, maps, _, pax, peaks = e.solve(field, steps=case["steps"])
        return u, torch.stack(maps, 0), pax, torch.tensor([float(field.abs().max())] + peaks, dtype=torch.float64)
    if kind == "operators":
        field, kw, phase, amp, dz_cfl = _operator_inputs(case, seed)
        e, u, dT = _Exact(tuple(field.shape), kw), field.double(), kw["dT"]
        return {
            "attenuation": e.visit(u, 0.0, DX / 2, DX),
            "propagator": e.taper(e.visit(u, DX / 2, 0.0, DX), True),
            "freq_weighted": e.weighted(u),
            "super_absorbing": e.absorb(u),
            "screen": e.screen(u, phase, amp),
            "kt_adaptive": _kt(u, BURGERS, dz_cfl, dT, True, 0.5),
            "kt_minmod": _kt(u, BURGERS, DX, dT, False),
            "rusanov": _rusanov(u, BURGERS * DX / dT),
            "tvd": _rusanov(u, BURGERS * DX / dT, 1.5),
            "march": e.step(u, DX),
        }
    u, un = _net_inputs(case, seed)
    params = torch.from_numpy(_weights(seed).astype(np.float64)).cuda()
    if kind == "train":
        params.requires_grad_(True)
        y, A = _network(u.double(), params)
        want = (un.double() - u.double()) / (NET_C * A * A)
        loss = ((y - want) ** 2).mean()
        loss.backward()
        return float(loss), params.grad
    out = torch.empty(u.shape, dtype=torch.float64, device="cuda")
    for at in range(0, u.shape[0], 1024):
        v = u[at: at + 1024].double()
        y, A = _network(v, params)
        steep = (v[:, 1:] - v[:, :-1]).abs().amax(1, keepdim=True) / 4e-8 > DPDT_MAX
        out[at: at + 1024] = torch.where(steep, v, v + NET_C * A * A * y)
    return out, None
