"""FP32 plans on the fp16 hi + lo contraction: against the FP64 oracle at the edges of its
tiles, skips and scales, and the calls that keep the FP32 kernels.

Bar of the image (relative L2): 5e-6.  The parts, each at its largest and all of one sign:
operands of 22 bits (2^-22 for the spectra and for the weights, 4.8e-7), the two phases cut
at 2^-23 revolutions about their mean (2 pi 2^-24 each, 7.5e-7), a window and a sine of the
hardware at 1e-6, the DFT of 1000 samples at 5e-7, the reciprocal and the sums at 5e-7.
"""
import ctypes as C

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


def _window(fa, name):
    return {"boxcar": fa.windows.boxcar(), "hann": fa.windows.hann(), "tukey": fa.windows.tukey(0.5),
            "triangular": fa.windows.triangular()}[name]


def _workload(n_el, n_ang, n_x=11, n_z=9):
    from f_number_amd import synth

    w = synth.scaled(synth.cpwc_small(), n_x, n_z, n_angles=min(n_ang, 11), n_samples=1000, n_speckle=800,
                     n_elements=n_el)
    if n_ang > 11:
        w.angles_deg = np.linspace(-15.0, 15.0, n_ang)
    w.seed = 7100 + n_el + n_ang
    return w


def _image(fa, w, rf, win, semantics, norm="on", precision="fp32"):
    import torch

    plan = fa.PwPlan(w.positions_x, w.positions_z, w.n_samples, w.n_elements, w.angles, w.f_s, w.width, w.pitch,
                     w.c_0, w.f_bounds, 0.0, window=_window(fa, win), F_number=fa.f_numbers.grating.angle_lb(60, 1.5),
                     normalization=getattr(fa.normalizations, norm)(), semantics=semantics, precision=precision,
                     output_scale="cpu")
    img = torch.empty((w.positions_x.size, w.positions_z.size), dtype=torch.complex64, device="cuda")
    plan.execute(torch.from_numpy(rf).cuda(), img)
    torch.cuda.synchronize()
    return img.cpu().numpy().T


# element counts: full and ragged 8-, 16-, 32- and 48-step arrays; angle counts: one row, a
# full tile and one row more, three tiles, a last group of fewer tiles
@pytest.mark.parametrize("n_el,n_ang", [(128, 1), (128, 16), (128, 17), (128, 48), (128, 81), (100, 3), (33, 11),
                                        (31, 5), (130, 7), (192, 33)])
@pytest.mark.parametrize("win,semantics,norm", [("tukey", "cpu", "on"), ("hann", "cpu", "off"), ("boxcar", "cpu", "on"),
                                                ("triangular", "mex", "off"), ("triangular", "cpu", "off")])
def test_fp32_matches_oracle(fa, oracle, n_el, n_ang, win, semantics, norm):
    w = _workload(n_el, n_ang)
    rf = w.rf_host()
    print(f"case fp32 {n_el} elements {n_ang} angles {win} {semantics} {norm}", flush=True)
    img = _image(fa, w, rf, win, semantics, norm)
    ref, _ = oracle.das_pw(w.positions_x, w.positions_z, rf, w.f_s, w.angles, w.width, w.pitch, w.c_0, w.f_bounds, 0,
                           (win, 0.5 if win == "tukey" else 0.0), oracle.fnumber("angle_lb", 60, 1.5, 10), norm,
                           semantics=semantics)
    e = rel_l2(img, ref)
    print(f"  rel_l2={e:.2e}", flush=True)
    assert e <= TOL


@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** 90])
def test_scale_of_the_samples(fa, scale):
    """samples times a power of two: the image times it, and nothing under- or overflows"""
    w = _workload(64, 3)
    rf = w.rf_host()
    a, b = _image(fa, w, rf, "tukey", "cpu"), _image(fa, w, (rf * np.float32(scale)), "tukey", "cpu")
    assert rel_l2(b.astype(np.complex128) / scale, a) <= 1e-6


def test_noalloc_without_room_for_the_planes(fa):
    """spectra of 3 tiles x 128 elements x 542 bins fit the scratch, their planes beside them do
    not: the call still runs, and agrees with a plan (which has room) within twice the bar"""
    import torch

    from f_number_amd import _lib
    from f_number_amd.das import pw_params

    w = _workload(128, 40)
    w.n_samples = 2048
    rf = torch.from_numpy(w.rf_host()).cuda()
    P, keep, info = pw_params(w.positions_x, w.positions_z, w.n_samples, w.n_elements, w.angles, w.f_s, w.width,
                              w.pitch, w.c_0, w.f_bounds, 0.0, _window(fa, "tukey"),
                              fa.f_numbers.grating.angle_lb(60, 1.5), fa.normalizations.on(), 0, "cpu", "fp32", "cpu")
    nf = info["n_ub"] - info["n_lb"] + 1
    assert nf * 3 * 32 * 512 < (32 << 20) < 2 * nf * 3 * 32 * 512
    img = torch.empty((w.positions_x.size, w.positions_z.size), dtype=torch.complex64, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    _lib.check(_lib.load().fn_das_pw_noalloc(C.byref(P), C.c_void_p(rf.data_ptr()), _lib.DTYPE["float32"],
                                             C.c_void_p(img.data_ptr()), None, C.c_void_p(s)), "gpu_bf_das_pw_rf")
    torch.cuda.synchronize()
    ref = _image(fa, w, rf.cpu().numpy(), "tukey", "cpu")
    assert rel_l2(img.cpu().numpy().T, ref) <= 2 * TOL


@pytest.mark.parametrize("n_el,n_ang", [(128, 3), (128, 17), (100, 31), (192, 5)])
@pytest.mark.parametrize("win", ["tukey", "hann", "boxcar"])
def test_mirrored_voxels(fa, n_el, n_ang, win):
    """a lateral grid symmetric about the array (one lane for two voxels) against its columns
    on a grid that is not, with an odd and an even column count, and with delay offsets that
    are not symmetric; each side within the bar of the same exact image"""
    import torch

    w = _workload(n_el, n_ang)
    rf = torch.from_numpy(w.rf_host()).cuda()
    d = np.linspace(-30e-9, 50e-9, n_el) ** 2 * 1e7
    for n_x in (11, 12):
        x = np.linspace(-15e-3, 15e-3, n_x)

        def image(cols, delays):
            plan = fa.PwPlan(cols, w.positions_z, w.n_samples, n_el, w.angles, w.f_s, w.width, w.pitch, w.c_0,
                             w.f_bounds, 0.0, window=_window(fa, win),
                             F_number=fa.f_numbers.grating.angle_lb(60, 1.5))
            plan.set_tof(1500.0, delays)
            img = torch.empty((cols.size, w.positions_z.size), dtype=torch.complex64, device="cuda")
            wt = torch.empty((cols.size, w.positions_z.size), dtype=torch.float32, device="cuda")
            plan.execute(rf, img, wt)
            torch.cuda.synchronize()
            return img.cpu().numpy(), wt.cpu().numpy()

        print(f"case mirror {n_el} elements {n_ang} angles {win} n_x={n_x}", flush=True)
        for delays in (None, d):
            (a, wa), (b, wb) = image(x, delays), image(x[:-1], delays)
            assert rel_l2(a[:-1], b) <= 2 * TOL
            np.testing.assert_allclose(wa[:-1], wb, rtol=2e-5)
