"""Performance cases of the P-SV engine: the calls that users of this
framework spend their time in, over the sizes its configurations, tests and
benchmark use.

A case is a dict of plain values.  `kind` says which path a pass takes:

  gradient  one launch of shots through Engine: set_shots, shot_gradient
            (forward with snapshots, residual, adjoint with the correlation,
            chain rule), the gradient read back -- the inner loop of an inversion
  forward   forward modelling through Engine: set_shots, forward, seismograms
  trial     one trial of an inversion's step-length search through FWI: the
            model update on the device, the model set, a forward run and its misfit
  dropin    one shot gradient through the reference's own entry points
            (DropinShot), one call per kernel and time step

exact() restates the scheme in 64 bits with plain torch operations.
"""
import math

import numpy as np
import torch

import ifos_amd
from ifos_amd import workloads
from ifos_amd.dropin import DropinShot
from ifos_amd.fwi import FWI

# Stencil coefficients: Taylor (error class 0) and Holberg at 0.1 % group
# velocity error (class 1) for FDORDER 2, 4, ... 12.
HOLBERG = {
    (0, 2): (1.0,),
    (0, 4): (9 / 8, -1 / 24),
    (0, 8): (1225 / 1024, -245 / 3072, 49 / 5120, -5 / 7168),
    (1, 2): (1.0010,),
    (1, 4): (1.1382, -0.046414),
    (1, 6): (1.1965, -0.078804, 0.0081781),
    (1, 8): (1.2257, -0.099537, 0.018063, -0.0026274),
    (1, 10): (1.2415, -0.11231, 0.026191, -0.0064682, 0.001191),
    (1, 12): (1.2508, -0.12034, 0.032131, -0.010142, 0.0029857, -0.00066667),
}
VMIN, VMAX = 1800.0, 4500.0
TAU = 0.1        # 2 / Q at Q = 20
FL = (10.0, 40.0, 80.0, 20.0, 5.0)


def case(kind, NX, NY, NT, **kw):
    c = dict(kind=kind, NX=NX, NY=NY, NT=NT, FDORDER=8, relerr=1, L=0, FW=20, DTINV=2, VELOCITY=1, FREE_SURF=1,
             BOUNDARY=0, DH=2.0, fc=20.0, npower=4.0, kmax=8.0, stype=1, nsrc=1, rec_step=5, rec_row=2, shots=1,
             snap="fp32", q="uniform", eprecond=0, autotune=False)
    unknown = set(kw) - set(c) - {"name"}
    assert not unknown, unknown
    c.update(kw)
    return c


def listed():
    return [
        # the smallest gradients: the size of the smoke test and of quick checks of a setup
        case("gradient", 64, 48, 400, name="gradient_64x48", FDORDER=4, FW=10, fc=25.0, npower=2.0, kmax=1.0,
             rec_step=3, rec_row=3),
        # forward modelling at the size of the reference's example parameter file: vertical force, 80 geophones
        case("forward", 500, 100, 2000, name="forward_500x100", FDORDER=2, relerr=0, DH=0.2, fc=31.25, stype=3),
        # the elastic toy inversion, one shot at a time
        case("gradient", 400, 200, 1000, name="gradient_400x200", FDORDER=4, DH=1.0, fc=30.0, VELOCITY=0, npower=2.0,
             kmax=1.0, rec_step=2, rec_row=5),
        # a small request of the server, odd sizes, four shots of a survey in one launch, energy preconditioned
        case("gradient", 301, 151, 600, name="gradient_301x151_4shots", FDORDER=4, L=2, FW=15, DTINV=3, shots=4,
             eprecond=1),
        # a middle-sized forward request: elastic, eighth order
        case("forward", 1200, 600, 900, name="forward_1200x600", rec_step=4),
        # wide-aperture survey, one shot at a time
        case("gradient", 1700, 350, 1500, name="gradient_1700x350", L=2, FW=30, DTINV=3, DH=8.0),
        # the same survey as it is run in bulk: as many shots per launch as the cache holds, 16-bit snapshots
        case("gradient", 1700, 350, 900, name="gradient_1700x350_5shots", L=2, FW=30, DTINV=4, DH=8.0, shots=5,
             snap="bf16"),
        # the headline benchmark's shot gradient with its launch tuning
        case("gradient", 2000, 800, 1500, name="gradient_2000x800", L=2, FW=30, DTINV=3, autotune=True),
        # the largest forward requests of the server: odd sizes, layered Q, fourth order
        case("forward", 2999, 1201, 500, name="forward_2999x1201", FDORDER=4, L=2, FW=30, q="layered"),
        # the largest gradient: three relaxation mechanisms, 16-bit snapshots
        case("gradient", 4000, 1000, 1000, name="gradient_4000x1000", L=3, FW=30, DTINV=2, fc=15.0, snap="bf16",
             autotune=True),
        # step-length search of the toy inversion: a forward run for a model of its own
        case("trial", 400, 200, 1000, name="trial_400x200", FDORDER=4, DH=1.0, fc=30.0, npower=2.0, kmax=1.0,
             rec_step=2, rec_row=5),
        # a program that keeps the reference's own call sequence
        case("dropin", 2000, 800, 300, name="dropin_2000x800", L=2, FW=30, DTINV=3),
    ]


def bytes_per_step(c):
    """Bytes a time step of one shot has to move per cell when every array is
    read once and written once by each half step."""
    L = c["L"]
    vel = 4 * (3 + 2 + 2 + 2)
    return vel + (4 * (2 + 3 + 3 * L + 6 + 3 + 3 * L) if L else 4 * (2 + 3 + 3 + 3))


def cost(c):
    runs = {"gradient": 2, "dropin": 2}.get(c["kind"], 1)
    return c["NX"] * c["NY"] * c["NT"] * c["shots"] * runs * bytes_per_step(c)


def draw(rng):
    most = max(cost(c) for c in listed()) / 4
    kind = rng.choices(["gradient", "forward", "trial", "dropin"], [10, 6, 1, 1])[0]
    NX = int(math.exp(rng.uniform(math.log(64), math.log(4000))))
    NY = int(math.exp(rng.uniform(math.log(48), math.log(1201))))
    L = rng.choice([0, 0, 2, 2, 2, 3, 1])
    order = rng.choice([2, 4, 4, 8, 8, 8, 6, 12])
    DTINV = rng.choice([1, 2, 3, 4])
    FW = min(rng.choice([8, 10, 20, 30]), NX // 2 - 6, NY // 2 - 6)
    shots = 1
    if kind in ("gradient", "forward") and NX * NY < 700000:
        shots = rng.choice([1, 1, 1, 2, 3, 4, 5])
    snap = rng.choice(["fp32", "fp32", "bf16", "fp16"])
    periodic = kind in ("gradient", "forward") and rng.random() < 0.1
    c = case(kind, NX, NY, 12, FDORDER=order, L=L, FW=FW, DTINV=DTINV, VELOCITY=rng.choice([1, 1, 0]),
             FREE_SURF=0 if kind != "dropin" and rng.random() < 0.25 else 1, BOUNDARY=int(periodic),
             DH=rng.choice([0.2, 0.5, 1.0, 2.0, 5.0, 8.0, 12.5]),
             npower=rng.choice([2.0, 4.0]), kmax=rng.choice([1.0, 8.0]),
             stype=rng.choice([1, 1, 1, 2, 3]) if kind in ("gradient", "forward") else 1,
             nsrc=rng.choice([1, 1, 2]) if kind in ("gradient", "forward") else 1,
             rec_step=rng.choice([1, 2, 3, 5, 10]), rec_row=rng.choice([1, 2, 5]), shots=shots, snap=snap,
             q=rng.choice(["uniform", "layered"]), eprecond=rng.choice([0, 0, 0, 1]) if kind == "gradient" else 0)
    if kind == "dropin":
        c["VELOCITY"] = 1
    # two wave lengths of 30 cells at the slowest speed at least
    c["fc"] = round(VMIN / 1.8 / (c["DH"] * 15.0), 2)
    per_step = cost(c) / c["NT"]
    nt = min(rng.choice([300, 600, 900, 1500]), int(most / per_step), 240 if kind == "dropin" else 1500)
    c["NT"] = max(12, nt // 12 * 12)
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def time_step(c):
    """Half the stability limit for the fastest model of the range, in 32 bits."""
    gamma = sum(abs(v) for v in HOLBERG[(c["relerr"], c["FDORDER"])])
    vmax = 1.05 * VMAX * math.sqrt(1.0 + c["L"] * 1.5 * TAU)
    return float(np.float32(0.5 * c["DH"] / (math.sqrt(2.0) * gamma * vmax)))


def config(c):
    return ifos_amd.make_config(
        NX=c["NX"], NY=c["NY"], DH=c["DH"], DT=time_step(c), NT=c["NT"], FDORDER=c["FDORDER"],
        MAXRELERROR=c["relerr"], FW=c["FW"], FREE_SURF=c["FREE_SURF"], BOUNDARY=c["BOUNDARY"], VPPML=VMAX,
        FPML=c["fc"], DTINV=c["DTINV"], VELOCITY=c["VELOCITY"], L=c["L"], FL=list(FL[:c["L"]]) or None,
        F_REF=c["fc"], npower=c["npower"], k_max_PML=c["kmax"], SOURCE_TYPE=c["stype"])


def smooth_field(rng, NX, NY):
    """A smooth random field in [-1, 1]: a few long-wavelength cosines."""
    x = np.linspace(0.0, 1.0, NX, dtype=np.float32)[None, :]
    y = np.linspace(0.0, 1.0, NY, dtype=np.float32)[:, None]
    f = np.zeros((NY, NX), np.float32)
    for _ in range(3):
        a, b = rng.uniform(1.0, 8.0, 2)
        p, q = rng.uniform(0.0, 2 * np.pi, 2)
        f += np.cos(np.float32(np.pi * a) * x + np.float32(p)) * np.cos(np.float32(np.pi * b) * y + np.float32(q))
    return f / np.float32(3.0)


def make_model(c, rng, layered):
    """A model as surveys meet it: layers whose speed grows with depth along
    undulating interfaces (the ground), or a smooth trend (an inversion's start)."""
    NX, NY = c["NX"], c["NY"]
    y = np.arange(NY, dtype=np.float32)[:, None] / np.float32(NY)
    x = np.arange(NX, dtype=np.float32)[None, :] / np.float32(NX)
    if layered:
        depth = np.sort(rng.uniform(0.08, 0.95, 9)).astype(np.float32)
        speed = np.sort(rng.uniform(VMIN, VMAX, 10)).astype(np.float32)
        level = y + np.float32(0.03) * np.cos(np.float32(np.pi * rng.uniform(1.0, 5.0)) * x +
                                              np.float32(rng.uniform(0.0, 6.0)))
        idx = np.zeros((NY, NX), np.int64)
        for d in depth:
            idx += level > d
        vp = speed[idx]
        tau = (TAU * (1.5 - np.arange(10) / 10.0)).astype(np.float32)[idx]
    else:
        vp = (VMIN + (VMAX - VMIN) * (np.float32(0.15) + np.float32(0.7) * y)).astype(np.float32) * \
            (1.0 + np.float32(0.04) * smooth_field(rng, NX, NY))
        tau = np.broadcast_to((TAU * (1.5 - y)).astype(np.float32), (NY, NX))
    vp = np.ascontiguousarray(vp, np.float32)
    m = dict(vp=vp, vs=(vp / np.float32(1.8)).astype(np.float32),
             rho=(np.float32(310.0) * np.sqrt(np.sqrt(vp))).astype(np.float32))
    if c["L"]:
        t = np.full((NY, NX), np.float32(TAU)) if c["q"] == "uniform" else np.ascontiguousarray(tau, np.float32)
        m["taus"], m["taup"] = t, t
    return m


def make_shots(c, rng):
    """Sources along a line near the surface, one line of receivers for all shots."""
    NX, NY, FW = c["NX"], c["NY"], c["FW"]
    rx = np.arange(FW + 1, NX - FW + 1, c["rec_step"], dtype=np.int32)
    rec = np.stack([rx, np.full_like(rx, c["rec_row"])], 1).astype(np.int32)
    sy = max(2, min(10, NY // 6)) + (0 if c["FREE_SURF"] else FW if NY > 3 * FW else 0)
    shots = []
    # the wavelet begins half a period early, so that short runs carry waves too
    for _ in range(c["shots"]):
        src = [workloads.source_row(int(rng.integers(FW + 3, NX - FW - 2)), sy + k, c["fc"], tshift=-0.5 / c["fc"],
                                    stype=c["stype"]) for k in range(c["nsrc"])]
        shots.append((np.stack(src), rec))
    return shots


def make_observed(c, rng, shots):
    """Traces as a survey records them: direct and reflected arrivals with the
    amplitudes of a line source, first sample zero."""
    NT, dt, dh, fc = c["NT"], time_step(c), c["DH"], c["fc"]
    t = (np.arange(1, NT + 1) * dt).astype(np.float32)[None, :]
    rho = 310.0 * 2200.0 ** 0.25
    w = 2 * math.pi * fc
    scale = 1e10 * (w ** 1.5 / (4 * rho * 2200.0 ** 3) if c["stype"] == 1 else w ** 0.5 / (4 * rho * 2200.0 ** 2))
    vx, vy = [], []
    for src, rec in shots:
        dx = (rec[:, 0] - src[0, 0]).astype(np.float64) * dh
        out = np.zeros((2, len(rec), NT), np.float32)
        for speed, h, a in ((2200.0, 3.0 * dh, 1.0), (2600.0, rng.uniform(0.3, 0.8) * c["NY"] * dh, 0.3)):
            r = np.sqrt(dx * dx + 4 * h * h)
            arg = (math.pi * fc * (t - (1.0 / fc + r / speed).astype(np.float32)[:, None])).astype(np.float32) ** 2
            pulse = (1 - 2 * arg) * np.exp(-arg) * (a * scale * np.sqrt(speed / (2 * math.pi * r)))[:, None]
            out[0] += (pulse * (dx / r)[:, None]).astype(np.float32)
            out[1] += (pulse * (2 * h / r)[:, None]).astype(np.float32)
        out[:, :, 0] = 0.0
        vx.append(out[0])
        vy.append(out[1])
    return np.concatenate(vx), np.concatenate(vy)


def inputs(c, seed):
    rng = np.random.default_rng(seed)
    model = make_model(c, rng, layered=c["kind"] in ("forward", "dropin"))
    shots = make_shots(c, rng)
    obs = make_observed(c, rng, shots) if c["kind"] != "forward" else None
    direction = None
    if c["kind"] == "trial":
        direction = [smooth_field(rng, c["NX"], c["NY"]) for _ in range(3)]
    return model, shots, obs, direction


class State:
    pass


class Dropin:
    """A drop-in shot that gives its device arrays back."""

    def __init__(self, cfg, model):
        self.shot = DropinShot(ifos_amd.lib(), cfg, model)

    def __del__(self):
        self.shot.close()


def prepare(c, seed):
    model, shots, obs, direction = inputs(c, seed)
    cfg = config(c)
    s = State()
    s.case, s.shots, s.obs = c, shots, obs
    if c["kind"] == "dropin":
        s.dropin = Dropin(cfg, model)
        nd = s.dropin.shot.nd
        s.zeros = np.zeros((cfg.NY + 2 * nd, cfg.NX + 2 * nd), np.float32)
        return s
    if c["kind"] == "trial":
        w = workloads.Workload("trial", cfg, model, model,
                               [workloads.Shot(srcpos=a, recpos=b) for a, b in shots])
        s.fwi = FWI(w, slots=1)
        s.fwi.obs = [obs]
        s.fwi.direction(direction, 1)
        return s
    s.eng = ifos_amd.Engine(cfg, slots=c["shots"])
    s.eng.set_snapshot_precision(c["snap"])
    if c["eprecond"]:
        s.eng.set_eprecond(c["eprecond"], per_shot=True)
    s.eng.set_model(**model)
    s.eng.set_shots(shots)
    if obs is not None:
        s.dev = [ifos_amd.DeviceBuffer.from_array(a) for a in obs]
    if c["autotune"]:
        s.eng.autotune()
    return s


def run(s):
    c = s.case
    if c["kind"] == "forward":
        s.eng.set_shots(s.shots)
        s.eng.forward(snapshots=False)
        vx, vy = s.eng.seismograms()
        return {"vx": vx, "vy": vy}
    if c["kind"] == "gradient":
        s.eng.set_shots(s.shots)
        misfit = s.eng.shot_gradient(*s.dev)
        g = s.eng.gradient()
        return {"misfit": misfit, "vp": g[0], "vs": g[1], "rho": g[2]}
    if c["kind"] == "trial":
        new, eps = s.fwi.trial(0.01, 1, 1)
        return {"vp": new["vp"], "vs": new["vs"], "rho": new["rho"], "misfit": float(s.fwi.test_misfit(new))}
    d = s.dropin.shot
    src, rec = s.shots[0]
    for k in ("wc", "wc_u", "wc_rho"):  # the correlation sums of the last shot
        d.lib.ifos_dev_copy_array(d.D[k], s.zeros.ctypes.data, 0)
    vx, vy = d.forward(src, rec, True)
    g = d.adjoint_gradient(rec, np.ascontiguousarray((vx - s.obs[0])[:, ::-1]),
                           np.ascontiguousarray((vy - s.obs[1])[:, ::-1]))
    return {"vx": vx, "vy": vy, "vp": g[0], "vs": g[1], "rho": g[2]}


def work(c):
    """Each time step reads and writes the wavefields and memory variables
    once and reads the materials once (for all shots of a launch); a gradient
    writes and reads five snapshot planes and updates three correlation
    planes per stored step."""
    cells, NT, S, L = c["NX"] * c["NY"], c["NT"], c["shots"], c["L"]
    state = 4 * 2 * (5 + 3 * L)
    mats = 4 * (8 if L else 5)
    runs = 2 if c["kind"] in ("gradient", "dropin") else 1
    ntr = len(range(c["FW"] + 1, c["NX"] - c["FW"] + 1, c["rec_step"])) * S
    b = runs * NT * cells * (S * state + mats) + 2 * 4 * ntr * NT * runs
    if runs == 2:
        snap = 5 * (4 if c["snap"] == "fp32" or c["kind"] == "dropin" else 2)
        b += NT // c["DTINV"] * cells * S * (2 * snap + 4 * 2 * 3)
    N = c["FDORDER"] // 2
    f = runs * NT * cells * S * (8 * 3 * N + 30 + 30 * L)
    return {"bytes": b, "flops": f}


def tolerance(c):
    """About four times what the 32-bit scheme differs from its 64-bit
    restatement by.  Seismograms: up to 8e-6 over the listed and drawn cases
    (2e-4 at one sample).  Gradients with 32-bit snapshots: up to 4e-6, with
    FP16 8e-5 and with BF16 7e-4; single cells by the source, where the mu
    correlation's terms cancel, up to 30 times that.  On fine grids the
    relaxation factors 1 - eta / 2, eta the step over the relaxation time,
    keep few digits of eta in 32 bits: up to 2e-3."""
    if c["L"] and c["DH"] < 1.0:
        return {"rel": 8e-3, "max": 0.1}
    if c["kind"] in ("forward", "trial", "dropin") or c["snap"] == "fp32":
        return {"rel": 5e-5, "max": 2e-3}
    return {"rel": 4e-3, "max": 0.1}


# ---------------------------------------------------------------------------
# the scheme in 64 bits
# ---------------------------------------------------------------------------
def profiles(c):
    """CPML profiles (K, a, b) at full and half points of both strips, 2 FW values each."""
    FW, DH, DT = c["FW"], c["DH"], time_step(c)
    thick = FW * DH
    amax = math.pi * c["fc"]
    d0 = -(c["npower"] + 1) * VMAX * math.log(0.001) / (2.0 * thick)
    out = []
    for shift in (0.0, 0.5):
        low = thick - DH * (np.arange(FW) + shift)
        high = DH * (np.arange(1, FW + 1) + shift)
        an = np.concatenate([low, high]) / thick
        d = d0 * an ** c["npower"]
        K = 1.0 + (c["kmax"] - 1.0) * an ** c["npower"]
        al = amax * (1.0 - an)
        al = np.where(al < 0, 0.0, al)
        b = np.exp(-(d / K + al) * DT)
        a = np.where(np.abs(d) >= 1.0, d * (b - 1.0) / (K * (d + K * al)), 0.0)
        out.append((K, a, b))
    return out


class Scheme:
    """All shots of a case together, fields [shot][row][column] with a margin."""

    def __init__(self, c, model, dev):
        self.c, self.dev = c, dev
        f64 = lambda a: torch.from_numpy(np.asarray(a, np.float64)).to(dev)
        self.hc = HOLBERG[(c["relerr"], c["FDORDER"])]
        self.hc = [float(np.float32(v)) for v in self.hc]
        self.N = len(self.hc)
        self.H = self.N + 1
        self.DT, self.DH = time_step(c), float(np.float32(c["DH"]))
        NX, NY, L, S = c["NX"], c["NY"], c["L"], c["shots"]
        self.NX, self.NY, self.L, self.S, self.FW = NX, NY, L, S, c["FW"]
        vp, vs, rho = f64(model["vp"]), f64(model["vs"]), f64(model["rho"])
        self.vp, self.vs, self.rho = vp, vs, rho
        dn = lambda a: torch.roll(a, -1, 0)
        rt = lambda a: torch.roll(a, -1, 1)
        self.rjp = 1.0 / (0.5 * (rho + dn(rho)))
        self.rip = 1.0 / (0.5 * (rho + rt(rho)))
        mu = rho * vs * vs
        self.muss, self.lamss = mu, rho * vp * vp - 2 * mu
        u = 4.0 / (1 / mu + 1 / rt(mu) + 1 / dn(mu) + 1 / dn(rt(mu)))
        DT = self.DT
        if L:
            ts, tp = f64(model["taus"]), f64(model["taup"])
            ti = 0.25 * (ts + rt(ts) + dn(ts) + dn(rt(ts)))
            pts = [1.0 / (2 * math.pi * FL[l]) for l in range(L)]
            ws = 2 * math.pi * float(np.float32(c["fc"]))
            total = sum((ws * p) ** 2 / (1 + (ws * p) ** 2) for p in pts)
            m, p, ui = mu / (1 + total * ts), rho * vp * vp / (1 + total * tp), u / (1 + total * ti)
            self.f, self.g, self.fi = m * DT * (1 + L * ts), p * DT * (1 + L * tp), ui * DT * (1 + L * ti)
            self.eta = [DT / v for v in pts]
            self.dm, self.em, self.di = m * ts, p * tp, ui * ti
            self.mu_r, self.pi_r, self.ts, self.tp = m, p, ts, tp
        else:
            self.f, self.g, self.fi = mu, self.lamss, u
        K = profiles(c)
        self.px = [[f64(v)[None, None, :] for v in K[h]] for h in (0, 1)]
        self.py = [[f64(v)[None, :, None] for v in K[h]] for h in (0, 1)]
        self.reset()

    def reset(self):
        z = lambda *s: torch.zeros(s, dtype=torch.float64, device=self.dev)
        S, NX, NY, H, FW = self.S, self.NX, self.NY, self.H, self.FW
        pad = lambda: z(S, NY + 2 * H, NX + 2 * H)
        self.vx, self.vy, self.sxx, self.syy, self.sxy = (pad() for _ in range(5))
        self.psi = {k: z(S, NY, 2 * FW) for k in ("sxx_x", "sxy_x", "vxx", "vyx")}
        self.psi.update({k: z(S, 2 * FW, NX) for k in ("syy_y", "sxy_y", "vyy", "vxy")})
        self.psi_s = z(S, 1, 2 * FW)
        self.r, self.p, self.q = ([z(S, NY, NX) for _ in range(self.L)] for _ in range(3))

    def at(self, a, dj=0, di=0):
        H = self.H
        return a[:, H + dj:H + dj + self.NY, H + di:H + di + self.NX]

    def diff(self, a, axis, forward):
        """Staggered difference along axis (0 y, 1 x): half a cell ahead or behind."""
        out = None
        for m, h in enumerate(self.hc, 1):
            hi, lo = (m, 1 - m) if forward else (m - 1, -m)
            A = self.at(a, hi, 0) if axis == 0 else self.at(a, 0, hi)
            B = self.at(a, lo, 0) if axis == 0 else self.at(a, 0, lo)
            out = (A - B).mul_(h) if out is None else out.add_(A - B, alpha=h)
        return out

    def strip(self, d, psi, prof, lo, hi, axis):
        K, a, b = prof
        FW = self.FW
        n = d.shape[axis]
        for on, s0, d0 in ((lo, 0, 0), (hi, FW, n - FW)):
            if not on:
                continue
            sl = lambda t, o: t.narrow(axis, o, FW)
            P, D = sl(psi, s0), sl(d, d0)
            P.mul_(sl(b, s0)).add_(sl(a, s0) * D)
            D.div_(sl(K, s0)).add_(P)

    def pml_x(self, d, name, half):
        if not self.c["BOUNDARY"] and self.FW:
            self.strip(d, self.psi[name], self.px[half], True, True, 2)

    def pml_y(self, d, name, half):
        if self.FW:
            self.strip(d, self.psi[name], self.py[half], not self.c["FREE_SURF"], True, 1)

    def wrap(self, *fields):
        if self.c["BOUNDARY"]:
            H, NX = self.H, self.NX
            for a in fields:
                a[:, H:H + self.NY, :H] = a[:, H:H + self.NY, NX:NX + H]
                a[:, H:H + self.NY, H + NX:] = a[:, H:H + self.NY, H:2 * H]

    def velocity(self):
        """Returns the accelerations; the velocities are advanced."""
        sx = self.diff(self.sxx, 1, True)
        sy = self.diff(self.sxy, 1, False)
        self.pml_x(sx, "sxx_x", 1)
        self.pml_x(sy, "sxy_x", 0)
        tx = self.diff(self.sxy, 0, False)
        ty = self.diff(self.syy, 0, True)
        self.pml_y(ty, "syy_y", 1)
        self.pml_y(tx, "sxy_y", 0)
        ax, ay = sx.add_(tx).mul_(self.rip / self.DH), sy.add_(ty).mul_(self.rjp / self.DH)
        self.at(self.vx).add_(ax, alpha=self.DT)
        self.at(self.vy).add_(ay, alpha=self.DT)
        return ax, ay

    def stress(self, amp, rates):
        """amp: explosive amplitude per (shot, row, column, value); returns the stress rates when asked."""
        c, L, DT, N, H = self.c, self.L, self.DT, self.N, self.H
        scale = 1.0 / self.DH if L else DT / self.DH
        xx, yx = self.diff(self.vx, 1, False).mul_(scale), self.diff(self.vy, 1, True).mul_(scale)
        xy, yy = self.diff(self.vx, 0, True).mul_(scale), self.diff(self.vy, 0, False).mul_(scale)
        self.pml_x(xx, "vxx", 0)
        self.pml_x(yx, "vyx", 1)
        self.pml_y(yy, "vyy", 0)
        self.pml_y(xy, "vxy", 1)
        SX, SY, SXY = self.at(self.sxx), self.at(self.syy), self.at(self.sxy)
        shear, div = yx.add_(xy), xx + yy
        out = None
        if not L:
            gd, f2 = self.g * div, 2 * self.f
            ix, iy, ixy = gd + f2 * xx, gd + f2 * yy, self.fi * shear
            if rates:
                out = [ix / DT, iy / DT, ixy / DT]
            SX += ix
            SY += iy
            SXY += ixy
        else:
            half = 0.5 * DT
            gd, f2 = self.g * div, 2 * self.f
            old = [sum(t[1:], t[0]) for t in (self.p, self.q, self.r)]
            ed, d2 = self.em * div, 2 * self.dm
            for l in range(L):
                e = self.eta[l]
                b, k = 1.0 / (1.0 + 0.5 * e), 1.0 - 0.5 * e
                self.r[l].mul_(k).sub_(self.di * shear, alpha=e).mul_(b)
                self.p[l].mul_(k).sub_(ed, alpha=e).add_(d2 * yy, alpha=e).mul_(b)
                self.q[l].mul_(k).sub_(ed, alpha=e).add_(d2 * xx, alpha=e).mul_(b)
            new = [sum(t[1:], t[0]) for t in (self.p, self.q, self.r)]
            both = [a + b for a, b in zip(old, new)]
            ix, iy, ixy = gd - f2 * yy, gd - f2 * xx, self.fi * shear
            if rates:
                out = [ix / DT + 0.5 * both[0], iy / DT + 0.5 * both[1], ixy / DT + 0.5 * both[2]]
            SX.add_(ix).add_(both[0], alpha=half)
            SY.add_(iy).add_(both[1], alpha=half)
            SXY.add_(ixy).add_(both[2], alpha=half)
        for s, j, i, v in amp:
            SX[s, j, i] += 0.5 * v
            SY[s, j, i] += 0.5 * v
        if c["FREE_SURF"]:
            self.surface(out)
        self.wrap(self.sxx, self.sxy)
        return out

    def surface(self, out):
        L, DT, N, H, NX, FW = self.L, self.DT, self.N, self.H, self.NX, self.FW
        self.syy[:, H] = 0.0
        if out:
            out[1][:, 0] = 0.0
        for m in range(1, N + 1):
            self.syy[:, H - m, H:H + NX] = -self.syy[:, H + m, H:H + NX]
            self.sxy[:, H - m, H:H + NX] = -self.sxy[:, H + m - 1, H:H + NX]
        xx = yy = 0.0
        for m, h in enumerate(self.hc, 1):
            xx = xx + h * (self.vx[:, H, H + m - 1:H + m - 1 + NX] - self.vx[:, H, H - m:H - m + NX])
            yy = yy + h * (self.vy[:, H + m - 1, H:H + NX] - self.vy[:, H - m, H:H + NX])
        xx, yy = xx / self.DH, yy / self.DH
        if FW and not self.c["BOUNDARY"]:
            d = xx[:, None, :]
            self.strip(d, self.psi_s, self.px[0], True, True, 2)
            xx = d[:, 0]
        SX = self.sxx[:, H, H:H + NX]
        if not L:
            f, g = 2 * self.f[0], self.g[0]
            SX -= DT * (g * g / (g + f) * xx + g * yy)
            if out:
                out[0][:, 0] = (2 * g * f + f * f) / (g + f) * xx
            return
        f = 2 * self.mu_r[0] * (1 + L * self.ts[0])
        g = self.pi_r[0] * (1 + L * self.tp[0])
        d, e = 2 * self.mu_r[0] * self.ts[0], self.pi_r[0] * self.tp[0]
        before = sum(p[:, 0] for p in self.p)
        change = (d - e) * (f / g - 1) * xx - (d - e) * yy
        for l in range(L):
            self.q[l][:, 0] = 0.0
            self.p[l][:, 0] += self.eta[l] / (1 + 0.5 * self.eta[l]) * change
        after = sum(p[:, 0] for p in self.p)
        step = -((g - f) ** 2 * xx / g) - (g - f) * yy
        SX += DT * step + 0.5 * DT * (after - before)
        if out:
            out[0][:, 0] += step + 0.5 * (after - before)


def signals(c, src):
    t = np.arange(1, c["NT"] + 1) * time_step(c)
    fc = np.float64(np.float32(c["fc"]))
    tau = (math.pi * (t - 1.5 / fc - np.float64(src[3])) * fc) ** 2
    return (1 - 2 * tau) * np.exp(-tau) * float(src[5])


def exact(c, seed):
    if c["kind"] == "gradient" and 5 * 8 * c["NX"] * c["NY"] * c["shots"] * (c["NT"] // c["DTINV"]) > 90e9:
        return None
    if c["NT"] * c["shots"] * max(c["NX"] * c["NY"] / 1.5e6, 0.25) > 6000:
        return None
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    model, shots, obs, direction = inputs(c, seed)
    NT, DT, DH, NX, NY = c["NT"], time_step(c), c["DH"], c["NX"], c["NY"]
    updated = None
    if c["kind"] == "trial":
        updated = {}
        for k, d in zip(("vp", "vs", "rho"), direction):  # the first PCG direction is the gradient itself
            m, d = model[k].astype(np.float64), d.astype(np.float64)
            updated[k] = m - 0.01 * m.max() / np.abs(d).max() * d
        model = dict(model, **updated)
    A = Scheme(c, model, dev)
    gradient = c["kind"] in ("gradient", "dropin")
    nsnap = NT // c["DTINV"]
    sig = [[signals(c, row) for row in src] for src, _ in shots]
    rec = [(torch.from_numpy(r[:, 1].astype(np.int64) - 1 + A.H).to(dev),
            torch.from_numpy(r[:, 0].astype(np.int64) - 1 + A.H).to(dev)) for _, r in shots]
    seis = [torch.zeros((2, len(r), NT), dtype=torch.float64, device=dev) for _, r in shots]
    snaps = torch.zeros((nsnap, 5, A.S, NY, NX), dtype=torch.float64, device=dev) if gradient else None
    energy = [0.0, 0.0]
    for n in range(NT):
        snap = gradient and n % c["DTINV"] == 0
        ax, ay = A.velocity()
        for s, (src, _) in enumerate(shots):
            for k, row in enumerate(src):
                j, i, t = int(row[1]) - 1, int(row[0]) - 1, int(row[7])
                if t == 2:
                    A.at(A.vx)[s, j, i] += DT * A.rip[j, i] * sig[s][k][n] / DH ** 2
                if t == 3:
                    A.at(A.vy)[s, j, i] += DT * A.rjp[j, i] * sig[s][k][n] / DH ** 2
        A.wrap(A.vx, A.vy)
        if c["eprecond"]:
            energy[0] = energy[0] + A.at(A.vx) ** 2 + A.at(A.vy) ** 2
        amp = []
        for s, (src, _) in enumerate(shots):
            for k, row in enumerate(src):
                if int(row[7]) == 1:
                    w = sig[s][k]
                    v = (w[n + 1] if n + 1 < NT else 0.0) - (w[n - 1] if n else 0.0)
                    amp.append((s, int(row[1]) - 1, int(row[0]) - 1, v / (2 * DH * DH)))
        rates = A.stress(amp, snap and c["VELOCITY"] == 1)
        if snap:
            F = snaps[n // c["DTINV"]]
            F[0], F[1] = ax, ay
            three = rates if c["VELOCITY"] else [A.at(A.sxx), A.at(A.syy), A.at(A.sxy)]
            for k in range(3):
                F[2 + k] = three[k]
        for s in range(A.S):
            seis[s][0, :, n] = A.vx[s][rec[s]]
            seis[s][1, :, n] = A.vy[s][rec[s]]
    syn = torch.cat([x for x in seis], 1)
    if c["kind"] == "forward":
        return {"vx": syn[0].cpu().numpy(), "vy": syn[1].cpu().numpy()}
    want = torch.from_numpy(np.stack(obs).astype(np.float64)).to(dev)
    have = syn
    if c["VELOCITY"] == 0:
        want, have = torch.cumsum(want, 2) * DT, torch.cumsum(syn, 2) * DT
    res = have - want
    misfit = [float((res ** 2).sum()), float((want ** 2).sum())]
    if c["kind"] == "trial":
        return dict({k: v for k, v in updated.items()}, misfit=misfit[0] / misfit[1])
    back = torch.flip(res, [2])
    A.reset()
    wc, wu, wr = (torch.zeros((A.S, NY, NX), dtype=torch.float64, device=dev) for _ in range(3))
    vxp, vyp = torch.zeros_like(wc), torch.zeros_like(wc)
    counts = np.cumsum([0] + [len(r) for _, r in shots])
    la, mu = A.lamss, A.muss
    for n in range(NT):
        corr = (NT - n - 1) % c["DTINV"] == 0
        if c["VELOCITY"] == 0:
            vxp.add_(A.at(A.vx), alpha=DT)
            vyp.add_(A.at(A.vy), alpha=DT)
        elif corr:
            vxp.copy_(A.at(A.vx))
            vyp.copy_(A.at(A.vy))
        A.velocity()
        for s in range(A.S):
            A.vx[s].index_put_(rec[s], back[0, counts[s]:counts[s + 1], n], accumulate=True)
            A.vy[s].index_put_(rec[s], back[1, counts[s]:counts[s + 1], n], accumulate=True)
        A.wrap(A.vx, A.vy)
        if c["eprecond"]:
            energy[1] = energy[1] + A.at(A.vx) ** 2 + A.at(A.vy) ** 2
        A.stress([], False)
        if corr:
            F = snaps[(NT - n - 1) // c["DTINV"]]
            SX, SY, SXY = A.at(A.sxx), A.at(A.syy), A.at(A.sxy)
            wr += vxp * F[0] + vyp * F[1]
            wc += (F[2] + F[3]) * (SX + SY)
            wu += F[4] * SXY / mu ** 2 + 0.25 * (F[2] + F[3] * (SX + SY)) / (la + mu) ** 2 + \
                0.25 * (F[2] - F[3] * (SX - SY)) / mu ** 2
    vp, vs, rho = A.vp, A.vs, A.rho
    wl = -DT * wc / (4 * (la + mu) ** 2)
    wm, wq = -DT * wu, -DT * wr
    g = [2 * vp * rho * wl, -4 * rho * vs * wl + 2 * rho * vs * wm,
         (vp ** 2 - 2 * vs ** 2) * wl + vs ** 2 * wm + wq]
    if c["eprecond"]:
        w = torch.sqrt(energy[0] * energy[1])
        w = w + 0.005 * w.amax((1, 2), keepdim=True)
        w = w / w.amax((1, 2), keepdim=True)
        g = [v / w for v in g]
    g = [v.sum(0).cpu().numpy() for v in g]
    if c["kind"] == "dropin":
        return {"vx": syn[0].cpu().numpy(), "vy": syn[1].cpu().numpy(), "vp": g[0], "vs": g[1], "rho": g[2]}
    return {"misfit": np.array(misfit), "vp": g[0], "vs": g[1], "rho": g[2]}

