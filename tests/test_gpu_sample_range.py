"""Samples of very different size in one launch: frames of an ensemble and jobs of a row stack
do not see each other's amplitudes.

Bar (relative L2 against the same samples' own single-frame plan): both images are within the
FP32 forms' 5e-6 of the exact one, so 1e-5.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-5
PITCH, WIDTH, C0, FS, BAND = 0.3048e-3, 0.27e-3, 1540.0, 20.832e6, (2.25e6, 6.75e6)
X, Z = np.linspace(-8e-3, 8e-3, 13), np.linspace(5e-3, 30e-3, 21)
AMPLITUDES = [1.0, 1e8, 1e-8, 1e-20, 1e15]


@pytest.fixture(scope="module")
def fa():
    import f_number_amd as fa

    fa.load()
    return fa


def _plan(fa, n_el, angles, n_t, win, band=BAND, **kw):
    x, z = X, Z
    window = fa.windows.tukey(0.5) if win == "tukey" else getattr(fa.windows, win)()
    return fa.PwPlan(x, z, n_t, n_el, angles, FS, WIDTH, PITCH, C0, band, 0.0, window=window,
                     F_number=fa.f_numbers.grating.angle_lb(60, 1.5), **kw)


def _rf(n, n_ang, n_el, n_t, seed):
    import torch

    return torch.randn((n, n_ang, n_el, n_t), generator=torch.Generator().manual_seed(seed)).cuda()


def _eager(plan, rf):
    import torch

    img = torch.empty((13, 21), dtype=torch.complex64, device="cuda")
    plan.execute(rf.contiguous(), img)
    torch.cuda.synchronize()
    return img.cpu().numpy()


@pytest.mark.parametrize("n_el,n_ang,win", [(128, 3, "tukey"), (64, 5, "hann"), (33, 1, "boxcar"), (128, 17, "hann")])
def test_frames_of_an_ensemble(fa, n_el, n_ang, win):
    import torch

    n, n_t = len(AMPLITUDES), 700
    rf = _rf(n, n_ang, n_el, n_t, 3)
    rf *= torch.tensor(AMPLITUDES, device="cuda").reshape(-1, 1, 1, 1)
    angles = np.linspace(-0.2, 0.2, n_ang)
    ens, one = _plan(fa, n_el, angles, n_t, win, n_frames=n), _plan(fa, n_el, angles, n_t, win)
    imgs = torch.empty((n, 13, 21), dtype=torch.complex64, device="cuda")
    print(f"case ensemble {n_el} elements {n_ang} angles {win}", flush=True)
    ens.execute(rf, imgs)
    torch.cuda.synchronize()
    for f in range(n):
        assert rel_l2(imgs[f].cpu().numpy(), _eager(one, rf[f])) <= TOL, f


@pytest.mark.parametrize("n_el,n_ang,win", [(128, 3, "tukey"), (64, 1, "hann")])
def test_jobs_of_a_row_stack(fa, n_el, n_ang, win):
    import torch

    n, n_t = len(AMPLITUDES), 700
    rf = _rf(n, n_ang, n_el, n_t, 4)
    rf *= torch.tensor(AMPLITUDES, device="cuda").reshape(-1, 1, 1, 1)
    plans = [_plan(fa, n_el, np.linspace(-0.2, 0.2, n_ang) + 0.01 * j, n_t, win) for j in range(n)]
    imgs = [torch.empty((13, 21), dtype=torch.complex64, device="cuda") for _ in plans]
    rfs = [r.contiguous() for r in rf]
    batch = fa.Batch(plans)
    print(f"case stack {n_el} elements {n_ang} angles {win}", flush=True)
    for replay in range(2):
        for r in rfs:
            r.mul_(2.0)
        batch.execute(rfs, imgs)
        torch.cuda.synchronize()
        got = [i.cpu().numpy() for i in imgs]
        for p, r, g in zip(plans, rfs, got):
            assert rel_l2(g, _eager(p, r)) <= TOL
    assert batch.info()["stacked_plans"] == n
    batch.close()


@pytest.mark.parametrize("n_ang", [3, 40])
def test_channels_of_one_frame(fa, oracle, n_ang):
    """a channel 1e5 louder than the others of its frame (100 dB, below 2^17): the voxels that do
    not meet its element keep their bits"""
    import torch

    n_el, n_t, k = 128, 700, 5
    plan = _plan(fa, n_el, np.linspace(-0.2, 0.2, n_ang), n_t, "tukey", band=(4e6, 6e6))  # (lower bins take every element)
    rf = _rf(1, n_ang, n_el, n_t, 6)[0]
    quiet, only = rf.clone(), torch.zeros_like(rf)
    quiet[:, k] = 0
    only[:, k] = rf[:, k] * 1e5
    # (in the oracle a weight outside the aperture is an exact zero)
    ref, _ = oracle.das_pw(X, Z, only.cpu().numpy(), FS, np.linspace(-0.2, 0.2, n_ang), WIDTH, PITCH, C0, (4e6, 6e6), 0.0,
                           ("tukey", 0.5), oracle.fnumber("angle_lb", 60, 1.5, 10), "on")
    apart = np.asarray(ref).T == 0
    assert 0 < apart.sum() < apart.size
    print(f"case loud channel {n_ang} angles", flush=True)
    a, b = _eager(plan, quiet + only), _eager(plan, quiet)
    assert rel_l2(a[apart], b[apart]) <= TOL
