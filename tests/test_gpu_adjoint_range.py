"""Adjoint images of very different size or that are not finite: elements that no such voxel
meets keep their samples.

Bar (relative L2 against the adjoint of the quiet voxels alone): 1e-5, both within the FP32
forms' 5e-6 of exact.  Which elements a voxel meets: those whose samples change the forward
image there.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

PITCH, WIDTH, C0, FS, BAND = 0.3048e-3, 0.27e-3, 1540.0, 20.832e6, (4e6, 6e6)
N_T, NX, NZ = 600, 9, 70


@pytest.fixture(scope="module")
def fa():
    import f_number_amd as fa

    fa.load()
    return fa


def _plan(fa, n_el, win, shift):
    x, z = np.linspace(-0.45, 0.45, NX) * n_el * PITCH + shift, np.linspace(4e-3, 20e-3, NZ)
    window = fa.windows.tukey(0.5) if win == "tukey" else getattr(fa.windows, win)()
    return fa.PwPlan(x, z, N_T, n_el, np.linspace(-0.1, 0.1, 2), FS, WIDTH, PITCH, C0, BAND, 0.0, window=window,
                     F_number=fa.f_numbers.grating.angle_lb(60, 1.5))


def _met(plan, n_el, voxels):
    """elements whose samples change the image at one of the voxels"""
    import torch

    met = np.zeros(n_el, dtype=bool)
    img = torch.empty((NX, NZ), dtype=torch.complex64, device="cuda")
    g = torch.Generator().manual_seed(2)
    for k in range(n_el):
        rf = torch.zeros((2, n_el, N_T))
        rf[:, k] = torch.randn((2, N_T), generator=g)
        plan.execute(rf.cuda(), img)
        torch.cuda.synchronize()
        met[k] = any(abs(img[v].item()) > 0 for v in voxels)
    return met


def _y(seed):
    import torch

    return torch.randn((NX, NZ), dtype=torch.complex64, generator=torch.Generator().manual_seed(seed)).cuda()


@pytest.mark.parametrize("n_el,win,shift", [(64, "tukey", 0.0), (128, "boxcar", 0.0), (100, "tukey", 1e-4)])
@pytest.mark.parametrize("loud", [1e8, 1e20, np.inf, np.nan, 1e-20])
def test_elements_that_meet_no_loud_voxel(fa, n_el, win, shift, loud):
    import torch

    plan, y = _plan(fa, n_el, win, shift), _y(7)
    voxels = [(0, 10), (0, 33), (1, 0)]
    met = _met(plan, n_el, voxels)
    assert 0 < met.sum() < n_el
    if loud < 1:  # all others that much louder
        y *= 1.0 / loud
        quiet = y.clone()
        for v in voxels:
            y[v] *= loud
            quiet[v] = 0
    else:
        quiet = y.clone()
        for v in voxels:
            quiet[v] = 0
            y[v] = y[v] * loud if np.isfinite(loud) else complex(loud, 0.0)
    print(f"case adjoint {n_el} elements {win} {loud}", flush=True)
    a, b = plan.adjoint(y).cpu().numpy(), plan.adjoint(quiet).cpu().numpy()
    if loud < 1:
        assert rel_l2(a, b) <= 1e-5
        return
    assert rel_l2(a[:, ~met], b[:, ~met]) <= 1e-5
    if np.isfinite(loud):
        c = plan.adjoint(y - quiet).cpu().numpy()
        assert np.all(np.isfinite(a)) and rel_l2(a[:, met], c[:, met]) <= 1e-5 + 2.0 * NX * NZ / loud
    else:
        assert np.all(np.isnan(a[:, met]))


def test_sizes_that_change_along_the_depth(fa):
    """1e-15 .. 1e15 over the depths, up and down: the elements' sums are those of the pieces"""
    import torch

    plan, y = _plan(fa, 64, "tukey", 0.0), _y(8)
    amp = torch.logspace(-15, 15, NZ).cuda()
    for a in (amp, amp.flip(0)):
        whole = plan.adjoint(y * a).cpu().numpy().astype(np.float64)
        parts = np.zeros_like(whole)
        for z0 in range(0, NZ, 7):
            piece = torch.zeros_like(y)
            piece[:, z0:z0 + 7] = (y * a)[:, z0:z0 + 7]
            parts += plan.adjoint(piece).cpu().numpy()
        for k in range(64):
            assert rel_l2(whole[:, k], parts[:, k]) <= 1e-5, k
