"""Symmetric lateral grids whose aperture bounds fall on elements: the two sides of the array
round such a bound each in its own way, so a column's weights are not those of its mirror image.
(The oracle rounds these bounds by another order of operations, so the reference is the image
without the last column, a grid that is not symmetric.)

Bar (relative L2): 1e-5 for plane waves and line scans, both images within 5e-6 of the exact one
of the same bounds; weights 2e-5.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

PITCH, WIDTH, C0, FS, BAND = 0.3048e-3, 0.27e-3, 1540.0, 20.832e6, (2.25e6, 6.75e6)
N_T, F_UB = 700, 1.5


@pytest.fixture(scope="module")
def fa():
    import f_number_amd as fa

    fa.load()
    return fa


def _window(fa, win):
    return fa.windows.tukey(0.5) if win == "tukey" else getattr(fa.windows, win)()


def _grid(n_el, cols, n_z):
    """columns on elements, symmetric about the array; depths at which the half-width at F_UB is a
    whole or half number of pitches"""
    m = (n_el - 1) / 2.0
    k = np.unique(np.round(np.linspace(0, m - 0.5, (cols + 1) // 2)))
    k = np.concatenate([k, n_el - 1 - k[::-1]]) if n_el % 2 == 0 else np.unique(np.concatenate([k, n_el - 1 - k]))
    z = np.arange(12, 12 + n_z) * PITCH * F_UB
    return (k - m) * PITCH, z


def _ties(n_el, x, z):
    """voxels whose bounds at F_UB are not the mirror image of their partner's"""
    m = (n_el - 1) / 2.0
    xp, hp = x[:, None] / PITCH, (z / (2.0 * PITCH))[None, :] / F_UB
    lo = np.maximum(np.ceil(m + (xp - hp)), 0)
    hi = np.minimum(np.floor(m + (xp + hp)), n_el - 1)
    return int(np.sum(lo + hi[::-1] != n_el - 1))


def _F(fa):
    return fa.f_numbers.grating.angle_lb(60, F_UB)


@pytest.mark.parametrize("n_el,cols", [(128, 22), (64, 17), (33, 9), (192, 22)])
@pytest.mark.parametrize("win,sem", [("boxcar", "cpu"), ("tukey", "cpu"), ("triangular", "mex")])
def test_plane_waves(fa, n_el, cols, win, sem):
    import torch

    x, z = _grid(n_el, cols, 40)
    assert _ties(n_el, x, z) > 0 and np.all(np.abs(x + x[::-1]) <= 1e-12 * PITCH)
    rf = torch.randn((3, n_el, N_T), generator=torch.Generator().manual_seed(n_el)).cuda()
    angles = np.linspace(-0.2, 0.2, 3)
    print(f"case ties {n_el} elements {x.size} columns {win} {sem}", flush=True)
    out = []
    for cols_x in (x, x[:-1]):
        plan = fa.PwPlan(cols_x, z, N_T, n_el, angles, FS, WIDTH, PITCH, C0, BAND, 0.0, window=_window(fa, win),
                         F_number=_F(fa), semantics=sem, output_scale="cpu")
        img = torch.empty((cols_x.size, z.size), dtype=torch.complex64, device="cuda")
        wt = torch.empty((cols_x.size, z.size), dtype=torch.float32, device="cuda")
        plan.execute(rf, img, wt)
        res = [img.clone()]
        if n_el <= 128:
            d = torch.empty_like(img)
            plan.execute_tangent(rf, img, d)
            res += [img.clone(), d]
        torch.cuda.synchronize()
        out.append([r.cpu().numpy() for r in res] + [wt.cpu().numpy()])
    n = x.size - 1
    for a, b in zip(out[0][:-1], out[1][:-1]):
        assert rel_l2(a[:n], b) <= 1e-5
    np.testing.assert_allclose(out[0][-1][:n], out[1][-1], rtol=2e-5)
    # the call from host arrays
    img, _, _ = fa.das_pw(x, z, np.asfortranarray(rf[0].cpu().numpy().T), FS, angles[:1], WIDTH, PITCH, C0, BAND, 0,
                          _window(fa, win), _F(fa), semantics=sem, return_weights=True)
    ref, _, _ = fa.das_pw(x[:-1], z, np.asfortranarray(rf[0].cpu().numpy().T), FS, angles[:1], WIDTH, PITCH, C0, BAND, 0,
                          _window(fa, win), _F(fa), semantics=sem, return_weights=True)
    assert rel_l2(img[:, :n], ref) <= 1e-5


@pytest.mark.parametrize("n_el,cols", [(128, 22), (33, 9)])
@pytest.mark.parametrize("win", ["boxcar", "tukey"])
def test_line_scans(fa, n_el, cols, win):
    import torch

    x, z = _grid(n_el, cols, 40)
    assert _ties(n_el, x, z) > 0
    n = x.size
    rf = torch.randn((n, n_el, N_T), generator=torch.Generator().manual_seed(n_el + 1)).cuda()
    print(f"case line ties {n_el} elements {n} lines {win}", flush=True)
    out = []
    for m in (n, n - 1):
        p = fa.LineScan(x[:m], z, N_T, n_el, FS, WIDTH, PITCH, C0, BAND, 20e-3, window=_window(fa, win), F_number=_F(fa),
                        output_scale="cpu")
        img = torch.empty((m, z.size), dtype=torch.complex64, device="cuda")
        p.execute(rf[:m].contiguous(), img)
        torch.cuda.synchronize()
        out.append(img.cpu().numpy())
    assert rel_l2(out[0][:-1], out[1]) <= 1e-5
