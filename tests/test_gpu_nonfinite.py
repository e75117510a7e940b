"""Samples that are not finite: a channel with one NaN or Inf sample turns the voxels whose
receive aperture holds its element to NaN and leaves every other voxel, frame and job as it is
without it.

Which voxels: those the FP64 oracle's image changes at when the channel's samples change.  The
others: relative L2 against the image of the same samples with the channel at zero, 1e-5 for the
FP32 forms (both within 5e-6 of exact), 1e-4 and 1e-2 for bf16x3 and fp16 (whose scale per bin
may differ by the channel).
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

PITCH, WIDTH, C0, FS, BAND = 0.3048e-3, 0.27e-3, 1540.0, 20.832e6, (4e6, 6e6)
N_EL, N_T, NX, NZ = 64, 600, 14, 23
TOL = {"fp32": 1e-5, "fp16x3": 1e-5, "bf16x3": 1e-4, "fp16": 1e-2}
X, Z = np.linspace(-9e-3, 9e-3, NX), np.linspace(4e-3, 22e-3, NZ)


@pytest.fixture(scope="module")
def fa():
    import f_number_amd as fa

    fa.load()
    return fa


def _window(fa, win):
    return fa.windows.tukey(0.5) if win == "tukey" else getattr(fa.windows, win)()


def _F(fa, F):
    return fa.f_numbers.constant(1.5) if F == "constant" else fa.f_numbers.grating.angle_lb(60, 1.5)


def _plan(fa, n_ang, win="tukey", F="angle_lb", precision="fp32", x=X, angles=None, **kw):
    angles = np.linspace(-0.2, 0.2, n_ang) if angles is None else angles
    return fa.PwPlan(x, Z, N_T, N_EL, angles, FS, WIDTH, PITCH, C0, BAND, 0.0, window=_window(fa, win),
                     F_number=_F(fa, F), precision=precision, output_scale="cpu", **kw)


def _oracle_F(oracle, F):
    return oracle.fnumber("constant", 1.5) if F == "constant" else oracle.fnumber("angle_lb", 60, 1.5, 10)


def _rf(n_tx, seed):
    return np.random.default_rng(seed).standard_normal((n_tx, N_EL, N_T)).astype(np.float32)


def _met(oracle, rf, chan, win, F, mode="pw", n_ang=0, x=X):
    """voxels (N_x, N_z) at which the oracle's image changes with channel (tx, element)"""
    a, b = rf.copy(), rf.copy()
    a[chan], b[chan] = 0.0, np.random.default_rng(9).standard_normal(N_T)
    param = 0.5 if win == "tukey" else 0.0
    out = []
    for r in (a, b):
        if mode == "sa":
            img, _ = oracle.das_sa(x, Z, r, FS, WIDTH, PITCH, C0, BAND, 0.0, (win, param), (win, param),
                                   _oracle_F(oracle, F), _oracle_F(oracle, F))
        else:
            img, _ = oracle.das_pw(x, Z, r, FS, np.linspace(-0.2, 0.2, n_ang), WIDTH, PITCH, C0, BAND, 0.0, (win, param),
                                   _oracle_F(oracle, F), "on")
        out.append(np.asarray(img).T)
    return out[0] != out[1]


def _check(img, clean, met, tol):
    img, clean = img.cpu().numpy(), clean.cpu().numpy()
    assert 0 < met.sum() < met.size
    assert np.all(np.isnan(img[met]))
    assert np.all(np.isfinite(img[~met]))
    assert rel_l2(img[~met], clean[~met]) <= tol


def _pair(plan, rf, chan, value, run=None):
    """images of rf with one sample of the channel at `value`, and with the channel at zero"""
    import torch

    out = []
    for v in (value, None):
        r = rf.copy()
        if v is None:
            r[chan] = 0.0
        else:
            r[chan + (N_T // 3,)] = v
        img = torch.empty((plan._keep[0].size, NZ), dtype=torch.complex64, device="cuda")
        d = torch.from_numpy(r).cuda()
        if run:
            run(d, img)
        else:
            plan.execute(d, img)
        torch.cuda.synchronize()
        out.append(img)
    return out


# 3 and 17 angles: mirrored voxels on this symmetric grid; 40: three tiles; shifted: one voxel a lane
@pytest.mark.parametrize("n_ang,shift", [(3, 0.0), (17, 0.0), (40, 0.0), (3, 1e-3)])
@pytest.mark.parametrize("precision", ["fp32", "bf16x3", "fp16"])
@pytest.mark.parametrize("win,value", [("tukey", np.nan), ("boxcar", np.inf)])
def test_plane_waves(fa, oracle, n_ang, shift, precision, win, value):
    x, rf, chan = X + shift, _rf(n_ang, 5), (n_ang // 2, 11)
    plan = _plan(fa, n_ang, win, precision=precision, x=x)
    print(f"case pw {n_ang} angles shift {shift} {precision} {win} {value}", flush=True)
    img, clean = _pair(plan, rf, chan, value)
    _check(img, clean, _met(oracle, rf, chan, win, "angle_lb", n_ang=n_ang, x=x), TOL[precision])


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
def test_synthetic_aperture(fa, oracle, precision):
    """the receive side decides (a transmitter outside its aperture has zero weight, and the
    matrix rows of a launch stay apart)"""
    rf, chan = _rf(N_EL, 6), (30, 9)
    plan = fa.SaPlan(X, Z, N_T, N_EL, FS, WIDTH, PITCH, C0, BAND, 0.0, window_tx=_window(fa, "tukey"),
                     F_number_tx=_F(fa, "angle_lb"), precision=precision, output_scale="cpu")
    print(f"case sa {precision}", flush=True)
    img, clean = _pair(plan, rf, chan, np.nan)
    # (every transmitter of the same receive element changes the image where the element is met)
    a, b = rf.copy(), rf.copy()
    b[:, chan[1]] = np.random.default_rng(9).standard_normal((N_EL, N_T))
    a[:, chan[1]] = 0.0
    o = [np.asarray(oracle.das_sa(X, Z, r, FS, WIDTH, PITCH, C0, BAND, 0.0, ("tukey", 0.5), ("tukey", 0.5),
                                  _oracle_F(oracle, "angle_lb"), _oracle_F(oracle, "angle_lb"))[0]).T for r in (a, b)]
    _check(img, clean, o[0] != o[1], TOL[precision])


def test_tangent(fa, oracle):
    import torch

    rf, chan = _rf(3, 7), (1, 50)
    for x in (X, X + 1e-3):
        plan = _plan(fa, 3, x=x)
        d = torch.empty((NX, NZ), dtype=torch.complex64, device="cuda")
        ds = []

        def run(r, img):
            plan.execute_tangent(r, img, d)
            ds.append(d.clone())

        img, clean = _pair(plan, rf, chan, np.inf, run)
        met = _met(oracle, rf, chan, "tukey", "angle_lb", n_ang=3, x=x)
        _check(img, clean, met, 1e-5)
        _check(ds[0], ds[1], met, 2e-5)


@pytest.mark.parametrize("precision", ["fp32", "fp16"])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_frames_and_jobs_stay_apart(fa, oracle, precision, value):
    """one frame of an ensemble, one job of a row stack, one plan of a persistent batch"""
    import torch

    n, n_ang, bad, chan = 5, 3, 3, (2, 11)
    rf = np.stack([_rf(n_ang, 20 + f) for f in range(n)])
    hit = rf.copy()
    hit[(bad,) + chan + (77,)] = value
    met = _met(oracle, rf[bad], chan, "tukey", "angle_lb", n_ang=n_ang)
    one = _plan(fa, n_ang, precision=precision)
    eager = []
    for f in range(n):
        r = rf[f].copy()
        if f == bad:
            r[chan] = 0.0
        img = torch.empty((NX, NZ), dtype=torch.complex64, device="cuda")
        one.execute(torch.from_numpy(r).cuda(), img)
        torch.cuda.synchronize()
        eager.append(img)
    hit_d = torch.from_numpy(hit).cuda()

    def check(imgs):
        torch.cuda.synchronize()
        for f in range(n):
            if f == bad:
                _check(imgs[f], eager[f], met, TOL[precision])
            else:
                assert rel_l2(imgs[f].cpu().numpy(), eager[f].cpu().numpy()) <= TOL[precision], f

    print(f"case apart {precision} {value}", flush=True)
    ens = _plan(fa, n_ang, precision=precision, n_frames=n)
    imgs = torch.empty((n, NX, NZ), dtype=torch.complex64, device="cuda")
    ens.execute(hit_d, imgs)
    check(imgs)
    plans = [_plan(fa, n_ang, precision=precision) for _ in range(n)]
    outs = [torch.empty((NX, NZ), dtype=torch.complex64, device="cuda") for _ in range(n)]
    rfs = [hit_d[f].contiguous() for f in range(n)]
    for kw in (dict(stacking=True), dict(stacking=False, persistent=True), dict(stacking=False)):
        batch = fa.Batch(plans, **kw)
        for _ in range(2):
            batch.execute(rfs, outs)
        check(outs)
        assert batch.info()["stacked_plans"] == (n if kw["stacking"] else 0)
        batch.close()
    # and a pass on finite samples after it
    rfs2 = [torch.from_numpy(rf[f]).cuda() for f in range(n)]
    batch = fa.Batch(plans)
    for f in range(n):
        rfs[f].copy_(rfs2[f])
    batch.execute(rfs, outs)
    torch.cuda.synchronize()
    assert all(torch.isfinite(torch.view_as_real(o)).all() for o in outs)
    batch.close()


@pytest.mark.parametrize("shift", [0.0, 1e-3])
@pytest.mark.parametrize("win,value", [("tukey", np.nan), ("boxcar", np.inf)])
def test_line_scan(fa, oracle, shift, win, value):
    """mirrored columns and columns that are not: only the bad transmit's own column, at the depths
    whose aperture holds the element"""
    import torch

    x, rf, n_z = np.linspace(-9e-3, 9e-3, 19) + shift, _rf(19, 8), 150
    z, chan = np.linspace(3e-3, 40e-3, n_z), (4, 30)
    p = fa.LineScan(x, z, N_T, N_EL, FS, WIDTH, PITCH, C0, BAND, 15e-3, window=_window(fa, win),
                    F_number=_F(fa, "angle_lb"), output_scale="cpu")
    print(f"case lines shift {shift} {win} {value}", flush=True)
    imgs = []
    for v in (value, None):
        r = rf.copy()
        if v is None:
            r[chan] = 0.0
        else:
            r[chan + (99,)] = v
        img = torch.empty((19, n_z), dtype=torch.complex64, device="cuda")
        p.execute(torch.from_numpy(r).cuda(), img)
        torch.cuda.synchronize()
        imgs.append(img)
    met = np.zeros((19, n_z), dtype=bool)
    cols = []
    for seed in (1, 2):
        r = rf[chan[0]:chan[0] + 1].copy()
        r[0, chan[1]] = np.random.default_rng(seed).standard_normal(N_T)
        col, _ = oracle.das_pw(x[chan[0]:chan[0] + 1], z, r, FS, np.zeros(1), WIDTH, PITCH, C0, BAND, 0.0,
                               (win, 0.5 if win == "tukey" else 0.0), _oracle_F(oracle, "angle_lb"), "on",
                               virtual_sources=[[x[chan[0]], 15e-3]])
        cols.append(np.asarray(col).reshape(-1))
    met[chan[0]] = cols[0] != cols[1]
    _check(imgs[0], imgs[1], met, 1e-5)


@pytest.mark.parametrize("win", ["tukey", "boxcar"])
def test_one_f_number(fa, oracle, win):
    """one F-number for every bin: the interpolated form"""
    import torch

    rf, chan, x, z = _rf(2, 10), (1, 20), np.linspace(-9e-3, 9e-3, 90), np.linspace(4e-3, 22e-3, 130)
    plan = fa.PwPlan(x, z, N_T, N_EL, np.linspace(-0.2, 0.2, 2), FS, WIDTH, PITCH, C0, BAND, 0.0, window=_window(fa, win),
                     F_number=_F(fa, "constant"), output_scale="cpu")
    imgs = []
    for v in (np.nan, None):
        r = rf.copy()
        if v is None:
            r[chan] = 0.0
        else:
            r[chan + (99,)] = v
        img = torch.empty((90, 130), dtype=torch.complex64, device="cuda")
        plan.execute(torch.from_numpy(r).cuda(), img)
        torch.cuda.synchronize()
        imgs.append(img)
    o = []
    for seed in (1, 2):
        r = rf.copy()
        r[chan] = np.random.default_rng(seed).standard_normal(N_T)
        img, _ = oracle.das_pw(x, z, r, FS, np.linspace(-0.2, 0.2, 2), WIDTH, PITCH, C0, BAND, 0.0,
                               (win, 0.5 if win == "tukey" else 0.0), _oracle_F(oracle, "constant"), "on")
        o.append(np.asarray(img).T)
    _check(imgs[0], imgs[1], o[0] != o[1], 1e-5)


@pytest.mark.parametrize("precision", ["bf16x3", "fp16"])
def test_tangent_beside_another_precision(fa, oracle, precision):
    """a tangent on FP32 products after a forward call whose samples were not finite"""
    import torch

    plan, rf = _plan(fa, 3, precision=precision), _rf(3, 12)
    img, d = (torch.empty((NX, NZ), dtype=torch.complex64, device="cuda") for _ in range(2))
    bad = rf.copy()
    bad[1, 30, 40] = np.nan
    plan.execute(torch.from_numpy(bad).cuda(), img)
    plan.execute_tangent(torch.from_numpy(rf).cuda(), img, d)
    torch.cuda.synchronize()
    ref, _ = oracle.das_pw(X, Z, rf, FS, np.linspace(-0.2, 0.2, 3), WIDTH, PITCH, C0, BAND, 0.0, ("tukey", 0.5),
                           _oracle_F(oracle, "angle_lb"), "on")
    assert torch.isfinite(torch.view_as_real(d)).all() and rel_l2(img.cpu().numpy().T, ref) <= 5e-6
