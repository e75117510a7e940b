"""Line scans at the edges of their kernel: columns that share their weights with their mirror
image (even and odd counts) and columns that cannot, ragged element counts, one and many
depth tiles, bands shorter than a round of its waves; delay offsets that are not symmetric;
and a captured batch whose plan gets other delays.

Bars: the line scans' own (rel-L2 1e-4, peak -80 dB) against the FP64 oracle; against
single-column plans, which round differently, 2e-6 (both are within 1e-6 of exact)."""
import numpy as np
import pytest

from conftest import peak_db, rel_l2

pytestmark = pytest.mark.gpu

PITCH, WIDTH, C0, FS = 0.3048e-3, 0.27e-3, 1540.0, 20.832e6


@pytest.fixture(scope="module")
def fa():
    import f_number_amd as fa

    fa.load()
    return fa


def _window(fa, win):
    return fa.windows.tukey(0.5) if win == "tukey" else getattr(fa.windows, win)()


@pytest.mark.parametrize("n_el,n_lines,n_z,band", [(128, 16, 64, (2.25e6, 6.75e6)), (100, 17, 65, (2.25e6, 6.75e6)),
                                                   (33, 5, 130, (4.4e6, 4.6e6)), (3, 2, 3, (4.5e6, 4.55e6))])
@pytest.mark.parametrize("win,sem,shift", [("tukey", "cpu", 0.0), ("hann", "mex", 0.0), ("hann", "cpu", 1e-3),
                                           ("boxcar", "cpu", 0.0), ("triangular", "mex", 1e-3)])
def test_columns_match_oracle(fa, oracle, n_el, n_lines, n_z, band, win, sem, shift):
    import torch

    half = 0.4 * n_el * PITCH
    x, z = np.linspace(-half, half, n_lines) + shift, np.linspace(5e-3, 35e-3, n_z)
    n_t = 1000
    rf = np.random.default_rng(n_el + n_z).standard_normal((n_lines, n_el, n_t)).astype(np.float32)
    p = fa.LineScan(x, z, n_t, n_el, FS, WIDTH, PITCH, C0, band, 20e-3, window=_window(fa, win),
                    F_number=fa.f_numbers.grating.angle_lb(60, 1.5), semantics=sem, output_scale="cpu")
    img = torch.full((n_lines, n_z), float("nan"), dtype=torch.complex64, device="cuda")
    wt = torch.full((n_lines, n_z), float("nan"), dtype=torch.float32, device="cuda")
    print(f"case lines {n_el} elements {n_lines} x {n_z} {win} {sem} shift {shift}", flush=True)
    p.execute(torch.from_numpy(rf).cuda(), img, weights=wt)
    torch.cuda.synchronize()
    img = img.cpu().numpy()
    assert np.all(np.isfinite(img)) and torch.isfinite(wt).all()
    F_o = oracle.fnumber("angle_lb", 60, 1.5, 10)
    ref = np.empty((n_lines, n_z), dtype=np.complex128)
    for i in range(n_lines):
        col, _ = oracle.das_pw(x[i:i + 1], z, rf[i:i + 1], FS, np.zeros(1), WIDTH, PITCH, C0, band, 0.0,
                               (win, 0.5 if win == "tukey" else 0.0), F_o, "on", semantics=sem,
                               virtual_sources=[[x[i], 20e-3]])
        ref[i] = np.asarray(col).reshape(-1)
    assert rel_l2(img, ref) <= 1e-4 and peak_db(img, ref) <= -80.0


@pytest.mark.parametrize("even", [True, False])
def test_delays_match_single_columns(fa, even):
    import torch

    n_el, n_lines, n_z, n_t, band = 64, 6, 70, 900, (2.25e6, 6.75e6)
    x, z = np.linspace(-6e-3, 6e-3, n_lines), np.linspace(5e-3, 30e-3, n_z)
    d = np.linspace(-25e-9, 40e-9, n_el)
    if even:
        d = np.abs(np.arange(n_el) - (n_el - 1) / 2) * 1e-9
    rf = torch.randn((n_lines, n_el, n_t), generator=torch.Generator().manual_seed(5)).cuda()
    kw = dict(window=fa.windows.tukey(0.5), F_number=fa.f_numbers.grating.angle_lb(60, 1.5), output_scale="cpu")
    p = fa.LineScan(x, z, n_t, n_el, FS, WIDTH, PITCH, C0, band, 20e-3, **kw)
    img = torch.empty((n_lines, n_z), dtype=torch.complex64, device="cuda")
    # a graph captured with no delays, then replayed with them
    batch = fa.Batch([p.plan])
    batch.execute([rf], [img])
    p.plan.set_tof(1500.0, d)
    batch.execute([rf], [img])
    torch.cuda.synchronize()
    got = img.clone()
    p.execute(rf, img)
    assert torch.equal(torch.view_as_real(got), torch.view_as_real(img))
    ref = torch.empty_like(img)
    for i in range(n_lines):
        q = fa.PwPlan(x[i:i + 1], z, n_t, n_el, np.zeros(1), FS, WIDTH, PITCH, C0, band, 0.0,
                      virtual_sources=np.array([[x[i], 20e-3]]), **kw)
        q.set_tof(1500.0, d)
        q.execute(rf[i:i + 1], ref[i:i + 1])
        torch.cuda.synchronize()
    assert rel_l2(got.cpu().numpy(), ref.cpu().numpy()) <= 2e-6
    batch.close()


def test_captured_mirrored_plan_gets_other_delays(fa):
    """a plane-wave plan of mirrored voxels in a captured batch: delays that are not symmetric"""
    import torch

    n_el, n_t = 64, 900
    x, z = np.linspace(-6e-3, 6e-3, 24), np.linspace(5e-3, 30e-3, 31)
    p = fa.PwPlan(x, z, n_t, n_el, np.linspace(-0.2, 0.2, 3), FS, WIDTH, PITCH, C0, (2.25e6, 6.75e6), 0.0,
                  window=fa.windows.tukey(0.5), F_number=fa.f_numbers.grating.angle_lb(60, 1.5))
    rf = torch.randn((3, n_el, n_t), generator=torch.Generator().manual_seed(6)).cuda()
    img = torch.empty((24, 31), dtype=torch.complex64, device="cuda")
    batch = fa.Batch([p])
    for d in (None, np.linspace(-25e-9, 40e-9, n_el), None):
        p.set_tof(0.0, d)
        batch.execute([rf], [img])
        torch.cuda.synchronize()
        got = img.clone()
        p.execute(rf, img)
        torch.cuda.synchronize()
        assert rel_l2(got.cpu().numpy(), img.cpu().numpy()) <= 1e-6
    batch.close()
