"""fn_das_pw_noalloc: calls whose spectra and 16-bit planes fill its 32 MiB are accepted.

Without a GPU the refusal of a call that does not fit comes first ("Unsupported"); a call that fits
goes on to the device and fails there.  On a GPU the largest accepted calls agree with a plan
(relative L2 1e-5: both within 5e-6 of exact).
"""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_l2

PITCH, WIDTH, C0, FS = 0.3048e-3, 0.27e-3, 1540.0, 20.832e6
SCRATCH = 32 << 20


def _params(n_ang, n_bins, precision, n_el=128):
    """a call of `n_bins` bins (or one or two fewer)"""
    import f_number_amd as fa
    from f_number_amd.das import pw_params

    x, z, n_t = np.linspace(-5e-3, 5e-3, 6) + 1e-4, np.linspace(20e-3, 30e-3, 5), 1500
    f_lo = 1.5e6

    def make(f_hi):
        return pw_params(x, z, n_t, n_el, np.linspace(-0.3, 0.3, n_ang), FS, WIDTH, PITCH, C0, (f_lo, f_hi), 0.0,
                         fa.windows.tukey(0.5), fa.f_numbers.grating.angle_lb(60, 1.5), fa.normalizations.on(), 0, "cpu",
                         precision, "cpu"), (x, z, n_t, n_el, np.linspace(-0.3, 0.3, n_ang), FS, WIDTH, PITCH, C0,
                                             (f_lo, f_hi))

    (P, keep, info), args = make(f_lo + 1e6)
    step = FS / info["N_dft"]
    (P, keep, info), args = make(f_lo + (n_bins - 1) * step)
    n = info["n_ub"] - info["n_lb"] + 1
    assert n_bins - 2 <= n <= n_bins
    return P, keep, args


def _call(P, rf, img):
    from f_number_amd import _lib

    L = _lib.load()
    st = L.fn_das_pw_noalloc(C.byref(P), rf, _lib.DTYPE["float32"], img, None, None)
    return L.fn_status_id(st).decode() if st else ""


# spectra and planes per bin: 16 KiB per tile of 16 angles each
FULL = [(75, SCRATCH // (10 * 16384) - 2, "bf16x3"), (32, SCRATCH // (4 * 16384) - 3, "bf16x3"),
        (100, SCRATCH // (14 * 16384) - 2, "fp16x3"), (75, SCRATCH // (15 * 8192) - 2, "fp16")]


@pytest.mark.parametrize("n_ang,n_bins,precision", FULL)
def test_calls_that_fit_are_not_refused(n_ang, n_bins, precision):
    import torch

    if torch.cuda.is_available():
        pytest.skip("the call would run: see test_calls_that_fit_match_a_plan")
    P, keep, _ = _params(n_ang, n_bins, precision)
    buf = (C.c_float * 16)()  # never reached: there is no device
    p = C.cast(buf, C.c_void_p)
    status = _call(P, p, p)
    assert status not in ("", "Unsupported")


@pytest.mark.gpu
@pytest.mark.parametrize("n_ang,n_bins,precision", FULL + [(75, SCRATCH // (10 * 16384) - 2, "fp32"),
                                                           (100, SCRATCH // (7 * 16384) - 3, "fp32")])
def test_calls_that_fit_match_a_plan(n_ang, n_bins, precision):
    import torch

    import f_number_amd as fa

    P, keep, args = _params(n_ang, n_bins, precision)
    rf = torch.randn((n_ang, 128, 1500), generator=torch.Generator().manual_seed(n_ang)).cuda()
    img = torch.empty((6, 5), dtype=torch.complex64, device="cuda")
    print(f"case noalloc {n_ang} angles {n_bins} bins {precision}", flush=True)
    torch.cuda.synchronize()
    assert _call(P, C.c_void_p(rf.data_ptr()), C.c_void_p(img.data_ptr())) == ""
    torch.cuda.synchronize()
    plan = fa.PwPlan(*args, 0.0, window=fa.windows.tukey(0.5), F_number=fa.f_numbers.grating.angle_lb(60, 1.5),
                     precision=precision, output_scale="cpu")
    ref = torch.empty_like(img)
    plan.execute(rf, ref)
    torch.cuda.synchronize()
    assert rel_l2(img.cpu().numpy(), ref.cpu().numpy()) <= 1e-5
