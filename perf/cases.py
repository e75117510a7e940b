"""What this framework's users have it compute, as cases to time and to compare.

One case is one call pattern of the public entry points at one size: plane-wave images
from a plan or from host arrays, full synthetic apertures, ensembles and job queues in one
graph, the forward/adjoint pair of an inversion, a gradient step of the autofocus, and
line-by-line scans.  `listed()` holds the fixed cases, `draw()` more of the same ranges,
`prepare()` / `run()` one pass, `exact()` the same outputs in 64 bits from torch alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import f_number_amd as fa

PITCH, WIDTH, C0, FS = 0.3048e-3, 0.27e-3, 1540.0, 20.832e6  # the linear array of the benchmark
BAND, WIDE_BAND = (2.25e6, 6.75e6), (1e6, 9e6)
N_SCATTERERS = 300
DOPPLER_ANGLES = 5
# queue of independent jobs: (axial, lateral) grids and angle counts of the batching benchmark
QUEUE = ((128, 128, 1), (256, 384, 3), (512, 512, 11), (128, 128, 11), (512, 768, 1), (256, 384, 31),
         (128, 128, 3), (256, 384, 1), (128, 128, 31), (256, 384, 11))


def _case(name, kind, **kw):
    c = dict(kind=kind, n_tx=11, n_el=128, n_t=2048, n_x=256, n_z=256, band="narrow", window="tukey", parameter=0.5,
             F="angle_lb", semantics="cpu", precision="fp32", rf64=False)
    c.update(kw)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one plane wave from host arrays, the call the reference's example makes per angle:
        # plan, transfers and a small image, so latency and host work count
        _case("das_pw_host_1ang_128x96", "das_pw", n_tx=1, n_t=1024, n_x=128, n_z=96, parameter=0.2),
        # the ordinary compounded frame of a live view
        _case("pw_11ang_256x256", "pw"),
        # the headline benchmark: 75 angles, wide band, full-size image, untruncated Hann
        _case("pw_75ang_1024x512_hann", "pw", n_tx=75, n_t=3328, n_x=512, n_z=1024, band="wide", window="hann"),
        # a fixed F-number with the boxcar window, the conventional beamformer users compare with
        _case("pw_31ang_512x384_boxcar", "pw", n_tx=31, n_t=1536, n_x=384, n_z=512, window="boxcar", F="fixed"),
        # a long compounding sequence in the split 16-bit form
        _case("pw_75ang_512x512_bf16x3", "pw", n_tx=75, n_x=512, n_z=512, window="hann", precision="bf16x3"),
        # a wider probe on a ragged grid, the GPU gateway's semantics, float64 samples
        _case("pw_7ang_211x173_192el_mex", "pw", n_tx=7, n_el=192, n_x=173, n_z=211, window="triangular",
              semantics="mex", rf64=True),
        # full synthetic aperture, FP32 and a smaller ragged one in fp16
        _case("sa_128el_512x512", "sa", n_tx=128, n_t=3000, n_x=512, n_z=512),
        _case("sa_96el_201x149_fp16", "sa", n_tx=96, n_el=96, n_t=1800, n_x=149, n_z=201, window="hann",
              precision="fp16"),
        # a Doppler ensemble and a queue of mixed jobs in one graph
        _case("batch_100fr_10jobs_fp16", "batch", n_tx=100, n_t=1536, window="hann", precision="fp16"),
        # one iteration of the autofocus: new delays, image with its tangent, gradients
        _case("autofocus_step_11ang_384x384", "grad", n_x=384, n_z=384),
        # forward and adjoint of an iterative reconstruction, a small probe on a ragged grid
        _case("fwd_adj_3ang_263x191_64el", "fwd_adj", n_tx=3, n_el=64, n_t=1500, n_x=191, n_z=263, window="hann"),
        # a focused line-by-line scan
        _case("lines_128x512", "lines", n_tx=128, n_x=128, n_z=512),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    most = 0.4 * work(listed()[2])["flops"]
    while True:
        kind = rng.choice(["das_pw", "pw", "pw", "pw", "pw", "sa", "sa", "batch", "grad", "fwd_adj", "lines"])
        c = _case(None, kind, n_t=rng.randint(900, 3000), n_x=rng.randint(70, 400), n_z=rng.randint(70, 600),
                  n_el=rng.choice([32, 64, 80, 96, 128, 128, 128]), n_tx=log_int(1, 75),
                  window=rng.choice(["tukey", "tukey", "hann", "boxcar", "triangular"]),
                  parameter=rng.choice([0.2, 0.5, 1.0]), F=rng.choice(["angle_lb", "angle_lb", "angle_lb", "fixed"]),
                  band=rng.choice(["narrow", "narrow", "wide"]), semantics=rng.choice(["cpu", "cpu", "mex"]))
        if kind in ("pw", "das_pw"):
            c["precision"] = rng.choice(["fp32", "fp32", "fp32", "bf16x3", "fp16"])
            c["n_el"] = rng.choice([c["n_el"], 160, 192])
            c["rf64"] = rng.random() < 0.2
        if kind == "das_pw":
            c.update(n_tx=1, n_x=min(c["n_x"], 200), n_z=min(c["n_z"], 200))
        if kind == "sa":
            c.update(n_tx=c["n_el"], precision=rng.choice(["fp32", "fp32", "bf16x3", "fp16"]))
        if kind == "batch":
            c.update(n_tx=rng.randint(20, 100), n_el=128, n_x=256, n_z=256, n_t=rng.randint(1000, 1536), window="hann",
                     F="angle_lb", band="narrow", semantics="cpu", precision=rng.choice(["fp16", "fp32"]))
        if kind in ("grad", "fwd_adj"):
            c["n_tx"] = min(c["n_tx"], 31)
            c["n_x"], c["n_z"] = min(c["n_x"], 300), min(c["n_z"], 300)
        if kind == "lines":
            c.update(n_tx=c["n_x"])
        if c["window"] == "triangular" and c["semantics"] == "cpu":
            c["semantics"] = "mex"  # untruncated, its weights can sum to zero
        if work(c)["flops"] <= most:
            return c


# ---------------------------------------------------------------------------------------
# acquisition
# ---------------------------------------------------------------------------------------
def _band(case):
    return WIDE_BAND if case["band"] == "wide" else BAND


def _grid(n_x, n_z):
    return np.linspace(-19e-3, 19e-3, n_x), np.linspace(5e-3, 40e-3, n_z)


def _angles(case):
    if case["kind"] in ("sa", "lines"):
        return np.zeros(case["n_tx"])
    n = DOPPLER_ANGLES if case["kind"] == "batch" else case["n_tx"]
    return np.deg2rad(np.linspace(-18.5, 18.5, 75)[:n] if n == 75 else np.linspace(-10.0, 10.0, n)) if n > 1 else np.zeros(1)


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _elements(n_el, dev):
    return (torch.arange(n_el, dtype=torch.float64, device=dev) - (n_el - 1) / 2.0) * PITCH


def _plane_time(angles, n_el, x, z, dev):
    """[n_tx, ...] transmit times of plane waves at x, z"""
    a = torch.as_tensor(angles, dtype=torch.float64, device=dev).reshape(-1, *([1] * x.dim()))
    e_x, e_z = -torch.sin(a), torch.cos(a)
    x_ref = torch.sign(e_x) * (-(n_el - 1) / 2.0 * PITCH)
    return (e_x * (x - x_ref) + e_z * z) / C0


def _acquire(tau_tx, tau_rx, amp, n_t, gen, dev):
    """RF (n_tx, n_el, n_t) float32: 5 MHz Gaussian pulses of 60 % bandwidth at
    tau_tx[tx, s] + tau_rx[el, s] (leading axes of tau_rx broadcast), noise at 30 dB."""
    n_tx, n_el = tau_tx.shape[0], tau_rx.shape[-2]
    n = 1 << (n_t + 64 - 1).bit_length()
    out = torch.empty((n_tx, n_el, n_t), dtype=torch.float32, device=dev)
    f = torch.arange(n // 2 + 1, dtype=torch.float64, device=dev) * FS / n
    sigma = 0.6 * 5e6 / (2.0 * math.sqrt(2.0 * math.log(2.0)))
    pulse = torch.exp(-0.5 * ((f - 5e6) / sigma) ** 2).float()
    step = max(1, (1 << 27) // (n_el * n))
    for a in range(0, n_tx, step):
        t = tau_tx[a:a + step]
        k = t.shape[0]
        q = (t[:, None, :] + tau_rx) * FS
        i = q.floor()
        frac = (q - i).float()
        i = i.long()
        ok = (i >= 0) & (i + 1 < n_t)
        row = (torch.arange(k * n_el, device=dev) * n).reshape(k, n_el, 1)
        buf = torch.zeros(k * n_el * n, dtype=torch.float32, device=dev)
        w = torch.where(ok, amp.float().expand_as(frac), torch.zeros((), device=dev))
        at = row + i.clamp(0, n - 2)
        # scatterers one after the other: every channel gets one sample at a time, so the sums
        # come in one order and the samples do not depend on the run
        for s in range(at.shape[-1]):
            idx = at[..., s].reshape(-1)
            buf[idx] += (w[..., s] * (1 - frac[..., s])).reshape(-1)
            buf[idx + 1] += (w[..., s] * frac[..., s]).reshape(-1)
        spec = torch.fft.rfft(buf.reshape(k, n_el, n)) * pulse
        out[a:a + k] = torch.fft.irfft(spec, n=n)[..., :n_t]
    rms = out.square().mean().sqrt()
    for a in range(0, n_tx, step):
        o = out[a:a + step]
        o += rms * 10 ** (-30 / 20) * torch.randn(o.shape, generator=gen, device=dev)
    return out


def _scene(gen, dev, n=N_SCATTERERS):
    u = torch.rand((2, n), generator=gen, device=dev, dtype=torch.float64)
    amp = torch.randn(n, generator=gen, device=dev, dtype=torch.float64)
    amp[:8] = 8.0  # bright points among the speckle
    return (u[0] - 0.5) * 38e-3, 5e-3 + u[1] * 35e-3, amp


def _rf(case, seed, dev, angles=None, n_tx=None):
    """the acquisition of a case (or of one queue job of it) from its seed"""
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    xs, zs, amp = _scene(gen, dev)
    xe = _elements(case["n_el"], dev)
    rx = torch.sqrt((xe[:, None] - xs) ** 2 + zs ** 2) / C0
    if case["kind"] == "sa":
        tx = rx
    elif case["kind"] == "lines":
        px, fz = torch.as_tensor(_grid(case["n_x"], case["n_z"])[0], device=dev), 20e-3
        r = torch.sqrt((xs - px[:, None]) ** 2 + (zs - fz) ** 2)
        tx = (torch.sqrt(px * px + fz * fz)[:, None] + torch.where(zs >= fz, r, -r)) / C0
    else:
        tx = _plane_time(_angles(case) if angles is None else angles, case["n_el"], xs, zs, dev)
    return _acquire(tx, rx, amp, case["n_t"], gen, dev)


def _rf_ensemble(case, seed, dev):
    """(n_frames, n_angles, n_el, n_t): the scatterers drift down at up to 0.5 m/s, 5 kHz"""
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    xs, zs, amp = _scene(gen, dev, 120)
    v = 0.5 * torch.rand(120, generator=gen, device=dev, dtype=torch.float64)
    xe = _elements(case["n_el"], dev)
    ang = _angles(case)
    out = torch.empty((case["n_tx"], ang.size, case["n_el"], case["n_t"]), dtype=torch.float32, device=dev)
    for f0 in range(0, case["n_tx"], 25):
        k = min(25, case["n_tx"] - f0)
        z = zs + v * 2e-4 * torch.arange(f0, f0 + k, device=dev, dtype=torch.float64)[:, None]  # [frame, s]
        tx = _plane_time(ang, case["n_el"], xs.expand_as(z), z, dev).permute(1, 0, 2).reshape(k * ang.size, -1)
        rx = torch.sqrt((xe[:, None] - xs) ** 2 + z[:, None, :] ** 2) / C0  # [frame, el, s]
        rx = rx.repeat_interleave(ang.size, dim=0)
        for a in range(0, k * ang.size, 125):
            out[f0:f0 + k].reshape(-1, case["n_el"], case["n_t"])[a:a + 125] = _acquire(
                tx[a:a + 125], rx[a:a + 125], amp, case["n_t"], gen, dev)
    return out


def _delays(case, seed):
    return np.random.default_rng(seed).normal(0.0, 20e-9, case["n_el"])


def _speckle(case, seed, dev):
    gen = torch.Generator(device=dev).manual_seed(int(seed) + 1)
    y = torch.randn((case["n_x"], case["n_z"], 2), generator=gen, device=dev)
    return torch.view_as_complex(y)


def _jobs(case):
    """the queue of a batch: (n_z, n_x, angles)"""
    return [(nz, nx, np.deg2rad(np.linspace(-15.0, 15.0, na)) if na > 1 else np.zeros(1)) for nz, nx, na in QUEUE]


# ---------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------
def _window(case):
    w = case["window"]
    return fa.windows.tukey(case["parameter"]) if w == "tukey" else getattr(fa.windows, w)()


def _F(case):
    return fa.f_numbers.constant(1.5) if case["F"] == "fixed" else fa.f_numbers.grating.angle_lb(60, 1.5)


def _pw_plan(case, n_x, n_z, angles, **kw):
    x, z = _grid(n_x, n_z)
    return fa.PwPlan(x, z, case["n_t"], case["n_el"], angles, FS, WIDTH, PITCH, C0, _band(case), 0.0, window=_window(case),
                     F_number=_F(case), semantics=case["semantics"], precision=case["precision"], **kw)


def prepare(case, seed):
    dev = torch.device("cuda")
    kind, n_x, n_z = case["kind"], case["n_x"], case["n_z"]
    s = {"case": case, "kind": kind}

    def image(*lead, nx=n_x, nz=n_z):
        return torch.empty((*lead, nx, nz), dtype=torch.complex64, device=dev)

    if kind == "batch":
        s["rfs"], s["images"], plans = [_rf_ensemble(case, seed, dev)], [image(case["n_tx"])], []
        plans.append(_pw_plan(case, n_x, n_z, _angles(case), n_frames=case["n_tx"]))
        for j, (nz, nx, ang) in enumerate(_jobs(case)):
            s["rfs"].append(_rf(case, seed + 1000 * (j + 1), dev, ang))
            s["images"].append(image(nx=nx, nz=nz))
            plans.append(_pw_plan(case, nx, nz, ang))
        s["plans"], s["batch"] = plans, fa.Batch(plans)
        return s
    rf = _rf(case, seed, dev)
    if case["rf64"]:
        rf = rf.double()
    if kind == "das_pw":
        # MATLAB's [N_t, N_el] on the host
        s["rf"] = np.asfortranarray(rf[0].cpu().numpy().T)
        s["x"], s["z"] = _grid(n_x, n_z)
        s["window"], s["F"] = _window(case), _F(case)
        return s
    s["rf"], s["image"] = rf, image()
    x, z = _grid(n_x, n_z)
    if kind == "sa":
        s["plan"] = fa.SaPlan(x, z, case["n_t"], case["n_el"], FS, WIDTH, PITCH, C0, _band(case), 0.0,
                              window_tx=_window(case), F_number_tx=_F(case), semantics=case["semantics"],
                              precision=case["precision"])
    elif kind == "lines":
        s["plan"] = fa.LineScan(x, z, case["n_t"], case["n_el"], FS, WIDTH, PITCH, C0, _band(case), 20e-3,
                                window=_window(case), F_number=_F(case), semantics=case["semantics"])
    else:
        s["plan"] = _pw_plan(case, n_x, n_z, _angles(case))
    if kind == "grad":
        s["delays"], s["dimage"] = _delays(case, seed), image()
    if kind == "fwd_adj":
        s["y"] = _speckle(case, seed, dev)
        s["rf_adj"] = torch.empty_like(rf)
    return s


def run(state):
    kind = state["kind"]
    if kind == "das_pw":
        c = state["case"]
        img, weights, _ = fa.das_pw(state["x"], state["z"], state["rf"], FS, 0.0, WIDTH, PITCH, C0, _band(c), 0,
                                    state["window"], state["F"], semantics=c["semantics"], precision=c["precision"],
                                    return_weights=True)
        return {"image": img, "weights": weights}
    if kind == "batch":
        state["batch"].execute(state["rfs"], state["images"])
        return {"images": state["images"]}
    plan, rf, image = state["plan"], state["rf"], state["image"]
    if kind == "grad":
        plan.set_tof(1500.0, state["delays"])
        plan.execute_tangent(rf, image, state["dimage"])
        g = 2.0 * image
        vd, vc = plan.vjp(rf, g, state["dimage"])
        # the optimiser keeps its parameters and moments in float32
        return {"image": image, "dimage": state["dimage"], "d_delay": vd.float(), "d_c": vc.float()}
    plan.execute(rf, image)
    if kind == "fwd_adj":
        plan.adjoint(state["y"], state["rf_adj"])
        return {"image": image, "rf_adj": state["rf_adj"]}
    return {"image": image}


# ---------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------
def _dft(case, n_z):
    """(N, first bin, last bin) of the padded band-limited DFT"""
    z = _grid(2, n_z)[1]
    z0 = z[1] if case["semantics"] == "mex" and n_z > 1 else z[0]
    span = (case["n_el"] - 1) * PITCH
    n = case["n_t"] + math.ceil((math.sqrt(span * span + z0 * z0) - z0) * FS / C0)
    n = n + 1 - n % 2
    f_lb, f_ub = _band(case)
    return n, math.ceil(f_lb * n / FS), math.floor(f_ub * n / FS)


def _f_values(case, f):
    """F-numbers at the frequencies f (numpy)"""
    if case["F"] == "fixed":
        return np.full(f.shape, 1.5)
    r = PITCH * f / C0
    th = math.sin(math.radians(60.0))
    lower, upper = 1 / (1 + th), 1 / (1 / math.sqrt(1 + 9.0) + th)
    with np.errstate(divide="ignore", invalid="ignore"):
        v = np.where((r > lower) & (r < upper), np.sqrt(np.maximum(1 / (1 / r - th) ** 2 - 1, 0)) / 2, 0.0)
        v = np.where(r >= upper, 1.5, v)
        # the angular distance of 10 degrees to the grating lobe
        o, s = 1 + math.cos(math.radians(10.0)), math.sin(math.radians(10.0))
        d = np.where((r < 1 / o) & (r >= 0.5), np.sqrt(np.maximum(1 / (1 / r - 1) ** 2 - 1, 0)) / 2, 0.0)
        t = r * r
        d = np.where((r >= 1 / o) & (r < 1 / s),
                     (np.sqrt(np.maximum(2 * o * t - 1, 0)) + o * s * t) / (2 - 2 * s * s * t), d)
        d = np.where(r >= 1 / s, np.inf, d)
    return np.maximum(v, d)


def _active(case, n_x, n_z):
    """mean over voxels and bins of the receive elements with nonzero weight (sampled)"""
    N, lb, ub = _dft(case, n_z)
    f = FS * np.linspace(lb, ub, 24) / N
    x, z = (np.linspace(-19e-3, 19e-3, 24), np.linspace(5e-3, 40e-3, 24))
    if case["window"] in ("hann", "triangular") and case["semantics"] == "cpu":
        return float(case["n_el"])
    F = _f_values(case, f)[:, None]
    if case["semantics"] == "cpu" and case["kind"] != "sa":
        F = np.minimum(F, np.sqrt(f[:, None] * z / (2.88 * C0)))
    with np.errstate(divide="ignore"):
        hp = (z / (2 * F) / PITCH)[:, None, :]
    m = (case["n_el"] - 1) / 2.0
    lo = np.maximum(np.ceil(m + x[:, None] / PITCH - hp), 0)
    hi = np.minimum(np.floor(m + x[:, None] / PITCH + hp), case["n_el"] - 1)
    return float(np.maximum(hi - lo + 1, 0).mean())


def work(case):
    kind = case["kind"]

    def one(n_x, n_z, rows, rows_per_voxel=None):
        """RF read once and image written once; a complex multiply-add per voxel, bin, active
        element and transmit row"""
        N, lb, ub = _dft(case, n_z)
        act = _active(case, n_x, n_z)
        per = act if kind == "sa" else (rows_per_voxel or rows)
        size = 8 if case["rf64"] else 4
        return size * rows * case["n_el"] * case["n_t"], 8.0 * n_x * n_z, 8.0 * (ub - lb + 1) * n_x * n_z * act * per

    if kind == "batch":
        rf, img, fl = one(case["n_x"], case["n_z"], case["n_tx"] * DOPPLER_ANGLES)
        b, fl = rf + img * case["n_tx"], fl
        for nz, nx, ang in _jobs(case):
            r, i, f = one(nx, nz, ang.size)
            b, fl = b + r + i, fl + f
        return {"bytes": b, "flops": fl}
    rf, img, fl = one(case["n_x"], case["n_z"], case["n_tx"], 1 if kind == "lines" else None)
    if kind == "grad":  # image and tangent, then the contraction of the gradient
        return {"bytes": rf + 2 * img, "flops": 3 * fl}
    if kind == "fwd_adj":
        return {"bytes": 2 * (rf + img), "flops": 2 * fl}
    return {"bytes": rf + img + (img / 2 if kind == "das_pw" else 0), "flops": fl}


# ---------------------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------------------
class _Aperture:
    """normalized weights [voxel, element] per bin: snapped half-widths around each voxel,
    the window on each side, the sum over the elements"""

    def __init__(self, case, x, z, f, clamp):
        dev = x.device
        self.case, self.x, self.z, self.f, self.clamp = case, x, z, f, clamp
        self.F = _f_values(case, f)
        n_el = case["n_el"]
        self.m = (n_el - 1) / 2.0
        self.k = torch.arange(n_el, dtype=torch.float64, device=dev)
        self.d = (self.k - self.m) * PITCH - x[:, None]
        self.abs_d, self.left = self.d.abs(), self.d < 0
        self.xp, self.zp = x / PITCH, z / (2 * PITCH)

    def weights(self, b):
        """(weights [V, n_el], sums [V], valid [V])"""
        c, n_el = self.case, self.case["n_el"]
        F = torch.full_like(self.z, float(self.F[b]))
        if self.clamp:
            F = torch.minimum(F, torch.sqrt(float(self.f[b]) * self.z / (2.88 * C0)))
        hp = self.zp / F
        lb = torch.ceil(self.m + (self.xp - hp)).clamp_min(0)
        ub = torch.floor(self.m + (self.xp + hp)).clamp_max(n_el - 1)
        valid = lb <= ub
        w = c["window"]
        if w == "boxcar" and c["semantics"] == "cpu":
            a = (self.abs_d < (hp * PITCH)[:, None]).double()
        else:
            wl = self.x - ((lb - self.m) * PITCH - 0.5 * WIDTH)
            wr = ((ub - self.m) * PITCH + 0.5 * WIDTH) - self.x
            t = self.abs_d * torch.where(self.left, (1 / wl.abs())[:, None], (1 / wr.abs())[:, None])
            if w == "boxcar":
                a = torch.ones_like(t)
            elif w == "hann":
                a = 0.5 + 0.5 * torch.cos(math.pi * t)
            elif w == "triangular":
                a = 1 - t
            else:
                p = c["parameter"]
                a = 0.5 + 0.5 * torch.cos(math.pi * ((t - (1 - p)) / p).clamp_min(0))
            if c["semantics"] == "mex":
                a = a * ((self.k >= lb[:, None]) & (self.k <= ub[:, None]))
            if w != "boxcar" and (c["semantics"] == "mex" or w == "tukey"):
                a = a * (t < 1)
        return a, a.sum(1), valid


def _spectra(rf, N, lb, ub):
    """[bin, element, row] complex128 of rf (rows, elements, samples)"""
    out = torch.empty((ub - lb + 1, rf.shape[1], rf.shape[0]), dtype=torch.complex128, device=rf.device)
    for a in range(0, rf.shape[0], 16):
        out[:, :, a:a + 16] = torch.fft.rfft(rf[a:a + 16].double(), n=N)[..., lb:ub + 1].permute(2, 1, 0)
    return out


def _voxels(n_x, n_z, dev, step):
    x, z = _grid(n_x, n_z)
    X = torch.as_tensor(np.repeat(x, n_z), device=dev)
    Z = torch.as_tensor(np.tile(z, n_x), device=dev)
    for v in range(0, X.numel(), step):
        yield slice(v, min(v + step, X.numel())), X[v:v + step], Z[v:v + step]


class _Phase:
    """e^{j w_n tau} for the bins in turn: one complex multiplication per bin"""

    def __init__(self, tau, N, lb):
        w = 2 * math.pi * FS / N
        self.e = torch.polar(torch.ones_like(tau), w * lb * tau)
        self.r = torch.polar(torch.ones_like(tau), w * tau)

    def next(self):
        self.e = self.e * self.r


def _exact_pw(case, rf, n_x, n_z, angles, c_tof=C0, delays=None, y=None, grad=False, frames=1):
    """image (and, asked for, weights of the last bin, adjoint, tangent and gradients)"""
    dev = rf.device
    N, lb, ub = _dft(case, n_z)
    nf, n_el, rows = ub - lb + 1, case["n_el"], rf.shape[0]
    f = FS * np.arange(lb, ub + 1) / N
    X = _spectra(rf, N, lb, ub)
    xe = _elements(n_el, dev)
    scale = 2.0 / N
    V = n_x * n_z
    image = torch.zeros((frames, V), dtype=torch.complex128, device=dev)
    wsum = torch.zeros(V, dtype=torch.float64, device=dev)
    dimage = torch.zeros(V, dtype=torch.complex128, device=dev) if grad else None
    d_delay = torch.zeros(n_el, dtype=torch.float64, device=dev) if grad else None
    Zs = torch.zeros((nf, n_el, rows), dtype=torch.complex128, device=dev) if y is not None else None
    na = len(angles)
    for sl, x, z in _voxels(n_x, n_z, dev, 32768):
        ap = _Aperture(case, x, z, f, case["semantics"] == "cpu")
        if case["kind"] == "lines":
            px, fz = x, 20e-3  # line i is focused at its own x: r = |z - fz|
            t_tx = ((torch.sqrt(px * px + fz * fz) + (z - fz)) / c_tof)[:, None]
        else:
            t_tx = (_plane_time(angles, n_el, x, z, dev) * (C0 / c_tof)).T
        t_rx = torch.sqrt((xe - x[:, None]) ** 2 + (z * z)[:, None]) / c_tof
        d = torch.zeros(n_el, dtype=torch.float64, device=dev)
        if delays is not None:
            d = torch.as_tensor(delays, device=dev)
        E, T = _Phase(t_rx + d, N, lb), _Phase(t_tx, N, lb)
        for b in range(nf):
            a, s, valid = ap.weights(b)
            inv = torch.where(valid, 1 / s, torch.zeros_like(s))
            B = a * inv[:, None] * E.e
            if case["kind"] == "lines":
                col = torch.arange(sl.start, sl.stop, device=dev) // n_z
                P = ((B * X[b].T[col]).sum(1) * T.e[:, 0])[None]
            else:
                Y = (B @ X[b]).reshape(-1, frames, na)
                P = (Y * T.e[:, None, :]).sum(2).T
            image[:, sl] += P
            if grad:
                w = 2 * math.pi * float(f[b])
                dP = ((B * t_rx) @ X[b] * T.e).sum(1) + (Y[:, 0] * T.e * t_tx).sum(1)
                dimage[sl] += (-1j * w / c_tof) * dP
            if y is not None:
                Zs[b] += (B.conj().T @ (y.reshape(-1)[sl].to(torch.complex128)[:, None] * T.e.conj())) * scale
            if b == nf - 1:
                wsum[sl] = s
            E.next()
            T.next()
        if grad:  # dJ/d delay of J = sum |image|^2: the cotangent is 2 image
            g = 2.0 * scale * image[0, sl]
            E, T = _Phase(t_rx + d, N, lb), _Phase(t_tx, N, lb)
            for b in range(nf):
                a, s, valid = ap.weights(b)
                B = a * torch.where(valid, scale / s, torch.zeros_like(s))[:, None] * E.e
                M = B.T @ (g.conj()[:, None] * T.e)
                d_delay += (2j * math.pi * float(f[b]) * (X[b] * M).sum(1)).real
                E.next()
                T.next()
    out = {"image": scale * image, "weights": wsum}
    if y is not None:
        full = torch.zeros((rows, n_el, N), dtype=torch.complex128, device=dev)
        full[..., lb:ub + 1] = Zs.permute(2, 1, 0)
        out["rf_adj"] = (torch.fft.ifft(full, dim=-1) * N).real[..., :case["n_t"]].contiguous()
    if grad:
        out["dimage"] = scale * dimage
        out["d_delay"] = d_delay
        out["d_c"] = (2.0 * out["image"][0].conj() * out["dimage"]).real.sum().reshape(1)
    return out


def _exact_sa(case, rf):
    dev = rf.device
    n_x, n_z, n_el = case["n_x"], case["n_z"], case["n_el"]
    N, lb, ub = _dft(case, n_z)
    f = FS * np.arange(lb, ub + 1) / N
    X = _spectra(rf, N, lb, ub)
    xe = _elements(n_el, dev)
    image = torch.zeros(n_x * n_z, dtype=torch.complex128, device=dev)
    for sl, x, z in _voxels(n_x, n_z, dev, 32768):
        ap = _Aperture(case, x, z, f, False)
        E = _Phase(torch.sqrt((xe - x[:, None]) ** 2 + (z * z)[:, None]) / C0, N, lb)
        for b in range(ub - lb + 1):
            a, s, valid = ap.weights(b)
            B = a * torch.where(valid, 1 / s, torch.zeros_like(s))[:, None] * E.e
            image[sl] += ((B @ X[b]) * B).sum(1)
            E.next()
    return 2.0 / N * image


def exact(case, seed):
    dev = _device()
    kind, n_x, n_z = case["kind"], case["n_x"], case["n_z"]
    if kind == "batch":
        rf = _rf_ensemble(case, seed, dev)
        img = _exact_pw(case, rf.reshape(-1, case["n_el"], case["n_t"]), n_x, n_z, _angles(case),
                        frames=case["n_tx"])["image"].reshape(-1, n_x, n_z)
        images = [img]
        for j, (nz, nx, ang) in enumerate(_jobs(case)):
            rf = _rf(case, seed + 1000 * (j + 1), dev, ang)
            images.append(_exact_pw(case, rf, nx, nz, ang)["image"].reshape(nx, nz))
        return {"images": images}
    rf = _rf(case, seed, dev)
    if kind == "sa":
        return {"image": _exact_sa(case, rf).reshape(n_x, n_z)}
    grad = kind == "grad"
    r = _exact_pw(case, rf, n_x, n_z, _angles(case), c_tof=1500.0 if grad else C0,
                  delays=_delays(case, seed) if grad else None, grad=grad,
                  y=_speckle(case, seed, dev) if kind == "fwd_adj" else None)
    image = r["image"].reshape(n_x, n_z)
    if kind == "das_pw":
        return {"image": image.T.contiguous(), "weights": r["weights"].reshape(n_x, n_z).T.contiguous()}
    out = {"image": image}
    if kind == "fwd_adj":
        out["rf_adj"] = r["rf_adj"]
    if grad:
        out.update(dimage=r["dimage"].reshape(n_x, n_z), d_delay=r["d_delay"], d_c=r["d_c"])
    return out
