"""FP32 plane-wave images of one F-number for every bin (interpolated channel samples)
against the FP64 oracle, at the edges of the path: one angle, a full group of angles and one
more, ragged element counts, odd bin counts and DFT orders, a grid that is no multiple of a
tile, voxels beside the array, clamped leading depths, delay offsets, and the call that
falls back to the sum over the bins.

Bar (relative L2): 5e-6, as for the other FP32 forms: the interpolation adds 1e-7 (3.4e-8
RMS over the band, 8.3e-8 at its edges) to the phases' 7.5e-7, the window's and the sine's
1e-6 and the spectra's and sums' 1e-6.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = 5e-6


@pytest.fixture(scope="module")
def fa():
    import f_number_amd as fa

    fa.load()
    return fa


def _run(fa, oracle, n_el, n_ang, win, sem, norm, F=1.5, n_x=61, n_z=83, band=(2.25e6, 6.75e6), z0=5e-3, vs=False,
         n_t=1000, x_max=19e-3, delays=None):
    import torch

    from f_number_amd import synth

    w = synth.scaled(synth.cpwc_small(), n_x, n_z, n_angles=min(n_ang, 11), n_samples=n_t, n_speckle=600,
                     n_elements=n_el)
    w.angles_deg = np.linspace(-12.0, 12.0, n_ang) if n_ang > 1 else np.zeros(1)
    w.positions_x, w.positions_z = np.linspace(-x_max, x_max, n_x), np.linspace(z0, 38e-3, n_z)
    w.f_bounds, w.seed = band, 8800 + n_el + n_ang
    sources = np.stack([np.linspace(-5e-3, 5e-3, n_ang), np.full(n_ang, -12e-3)], axis=1) if vs else None
    w.virtual_sources = sources
    rf = w.rf_host()
    window = {"boxcar": fa.windows.boxcar(), "hann": fa.windows.hann(), "tukey": fa.windows.tukey(0.5),
              "triangular": fa.windows.triangular()}[win]
    plan = fa.PwPlan(w.positions_x, w.positions_z, n_t, n_el, w.angles, w.f_s, w.width, w.pitch, w.c_0, band, 0.0,
                     window=window, F_number=fa.f_numbers.constant(F), normalization=getattr(fa.normalizations, norm)(),
                     semantics=sem, output_scale="cpu", virtual_sources=sources)
    if delays is not None:
        plan.set_tof(0.0, delays)
    img = torch.empty((n_x, n_z), dtype=torch.complex64, device="cuda")
    wt = torch.empty((n_x, n_z), dtype=torch.float32, device="cuda")
    print(f"case interp {n_el} elements {n_ang} angles {win} {sem} {norm} F={F}", flush=True)
    plan.execute(torch.from_numpy(rf).cuda(), img, wt)
    torch.cuda.synchronize()
    return plan, w, rf, img.cpu().numpy().T, wt.cpu().numpy().T, sources


@pytest.mark.parametrize("n_el,n_ang", [(128, 1), (128, 32), (128, 33), (100, 5), (31, 3), (192, 7)])
@pytest.mark.parametrize("win,sem,norm", [("boxcar", "cpu", "on"), ("hann", "cpu", "off"), ("tukey", "mex", "on"),
                                          ("triangular", "mex", "on")])
def test_matches_oracle(fa, oracle, n_el, n_ang, win, sem, norm):
    plan, w, rf, img, wt, vs = _run(fa, oracle, n_el, n_ang, win, sem, norm)
    ref, _ = oracle.das_pw(w.positions_x, w.positions_z, rf, w.f_s, w.angles, w.width, w.pitch, w.c_0, w.f_bounds, 0,
                           (win, 0.5 if win == "tukey" else 0.0), oracle.fnumber("constant", 1.5), norm, semantics=sem)
    assert np.all(np.isfinite(img))
    assert rel_l2(img, ref) <= TOL


def test_clamped_depths_and_empty_apertures(fa, oracle):
    """1 MHz upwards from 3 mm: F = 1.5 is clamped above 10 mm, where the sum over the bins runs;
    voxels beside the array; diverging waves"""
    for win in ("boxcar", "tukey"):
        plan, w, rf, img, wt, vs = _run(fa, oracle, 128, 7, win, "cpu", "on", band=(1e6, 9e6), z0=3e-3, vs=True,
                                        x_max=26e-3, n_x=60)
        ref, _ = oracle.das_pw(w.positions_x, w.positions_z, rf, w.f_s, w.angles, w.width, w.pitch, w.c_0, w.f_bounds,
                               0, (win, 0.5 if win == "tukey" else 0.0), oracle.fnumber("constant", 1.5), "on",
                               virtual_sources=vs)
        assert np.all(np.isfinite(img)) and np.all(np.isfinite(wt))
        assert rel_l2(img, ref) <= TOL
        top = w.positions_z < 10e-3
        assert rel_l2(img[top], ref[top]) <= TOL


def test_delays_agree_with_the_sum_over_bins(fa, oracle):
    """delay offsets: against the fp16x3 plan (the same operands' sum over the bins), each within
    the bar of the exact image"""
    import torch

    d = np.linspace(-25e-9, 40e-9, 128)
    plan, w, rf, img, wt, vs = _run(fa, oracle, 128, 5, "tukey", "cpu", "on", delays=d)
    p2 = fa.PwPlan(w.positions_x, w.positions_z, w.n_samples, 128, w.angles, w.f_s, w.width, w.pitch, w.c_0, w.f_bounds,
                   0.0, window=fa.windows.tukey(0.5), F_number=fa.f_numbers.constant(1.5), output_scale="cpu",
                   precision="fp16x3")
    p2.set_tof(0.0, d)
    a = torch.empty((61, 83), dtype=torch.complex64, device="cuda")
    b = torch.empty((61, 83), dtype=torch.float32, device="cuda")
    p2.execute(torch.from_numpy(rf).cuda(), a, b)
    torch.cuda.synchronize()
    assert rel_l2(img, a.cpu().numpy().T) <= 2 * TOL
    np.testing.assert_allclose(wt, b.cpu().numpy().T, rtol=2e-5)


def test_graph_replays(fa, oracle):
    """two interpolated plans and one that is not in a captured batch: every replay, on other
    samples, equals the eager image bit for bit"""
    import torch

    parts = [_run(fa, oracle, 128, 5, "boxcar", "cpu", "on"),
             _run(fa, oracle, 64, 3, "tukey", "cpu", "on", band=(1e6, 9e6), z0=3e-3),
             _run(fa, oracle, 64, 3, "tukey", "cpu", "on", n_x=6, n_z=5)]
    plans = [p[0] for p in parts]
    rfs = [torch.from_numpy(p[2]).cuda() for p in parts]
    outs = [torch.empty((p[1].positions_x.size, p[1].positions_z.size), dtype=torch.complex64, device="cuda") for p in parts]
    batch = fa.Batch(plans)
    for replay in range(3):
        for r in rfs:
            r.mul_(1.5)
        eager = []
        for p, r, o in zip(plans, rfs, outs):
            p.execute(r, o)
            eager.append(o.clone())
            o.fill_(float("nan"))
        batch.execute(rfs, outs)
        torch.cuda.synchronize()
        for o, e in zip(outs, eager):
            assert torch.equal(torch.view_as_real(o), torch.view_as_real(e))
    batch.close()
