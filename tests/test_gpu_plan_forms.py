"""Which form of the beamformer a call takes, from its report, on both sides of each rule; and the
workspaces that are laid out on demand.

Images (relative L2): 1e-5 between two forms or tilings, each within 5e-6 of exact.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

PITCH, WIDTH, C0, FS = 0.3048e-3, 0.27e-3, 1540.0, 20.832e6


@pytest.fixture(scope="module")
def fa():
    import f_number_amd as fa

    fa.load()
    return fa


def _report(fa, x, z, n_el=64, n_ang=3, win="boxcar", F=None, band=(2.25e6, 6.75e6), n_t=700, precision="fp32"):
    from f_number_amd import _lib

    window = fa.windows.tukey(0.5) if win == "tukey" else getattr(fa.windows, win)()
    rf = np.random.default_rng(1).standard_normal((n_t, n_el, n_ang)).astype(np.float32)
    fa.das_pw(x, z, np.asfortranarray(rf), FS, np.linspace(-0.2, 0.2, n_ang), WIDTH, PITCH, C0, band, 0, window,
              F if F is not None else fa.f_numbers.grating.angle_lb(60, 1.5), precision=precision, verbosity=1)
    return _lib.load().fn_last_report().decode()


def _line(report, what):
    return [l for l in report.splitlines() if what in l][0]


SYM, OFF = np.linspace(-8e-3, 8e-3, 80), np.linspace(-8e-3, 8e-3, 80) + 1e-3
DEPTHS = np.linspace(5e-3, 30e-3, 90)


def test_one_f_number_is_interpolated_where_it_pays(fa):
    F = fa.f_numbers.constant(1.5)
    r = _report(fa, SYM, DEPTHS, F=F)
    assert "fp32, interpolated" in _line(r, "contraction") and " 0 of 90" in _line(r, "samples per channel")
    # 1 MHz upwards from 3 mm: the clamp is at work above 10 mm
    r = _report(fa, SYM, np.linspace(3e-3, 30e-3, 90), F=F, band=(1e6, 6e6))
    assert "fp32, interpolated" in _line(r, "contraction") and " 0 of 90" not in _line(r, "samples per channel")
    # few voxels; another precision; an F-number per bin
    for kw in (dict(x=SYM[:5], z=DEPTHS[:4], F=F), dict(x=SYM, z=DEPTHS, F=F, precision="fp16x3"), dict(x=SYM, z=DEPTHS)):
        assert "interpolated" not in _line(_report(fa, **kw), "contraction")


def test_symmetric_grids_are_mirrored(fa):
    for n_ang, mirrored in ((1, True), (16, True), (32, True), (33, False)):
        r = _report(fa, SYM, DEPTHS, n_ang=n_ang, win="tukey")
        assert ("fp32, mirrored voxels" in _line(r, "contraction")) == mirrored, n_ang
    assert "mirrored" not in _line(_report(fa, OFF, DEPTHS, win="tukey"), "contraction")
    assert "mirrored" not in _line(_report(fa, SYM, DEPTHS, win="tukey", precision="fp16"), "contraction")


def _plan(fa, n_ang, x=OFF, n_el=128, F=None, **kw):
    return fa.PwPlan(x, DEPTHS, 700, n_el, np.linspace(-0.2, 0.2, n_ang), FS, WIDTH, PITCH, C0, (4e6, 6e6), 0.0,
                     window=fa.windows.tukey(0.5), F_number=F if F is not None else fa.f_numbers.grating.angle_lb(60, 1.5),
                     **kw)


@pytest.mark.parametrize("n_ang,precision", [(75, "fp32"), (75, "bf16x3"), (40, "fp16"), (100, "fp32")])
def test_tilings_beyond_the_default_one(fa, n_ang, precision):
    """planes for a tiling that a plan was not created with are laid out on demand, and the memory
    of a plan says so"""
    import torch

    plan = _plan(fa, n_ang, precision=precision)
    rf = torch.randn((n_ang, 128, 700), generator=torch.Generator().manual_seed(3)).cuda()
    ref = torch.empty((80, 90), dtype=torch.complex64, device="cuda")
    plan.execute(rf, ref)
    info = plan.info()
    tiles = -(-n_ang // 16)
    bins = info["n_f"]
    planes = {"fp32": 16384, "bf16x3": 16384, "fp16": 8192}[precision] * bins
    assert info["workspace_bytes"] <= tiles * 16384 * bins + (tiles + 1) * planes
    img = torch.empty_like(ref)
    batch = fa.Batch([plan])
    batch.execute([rf], [img])  # captured with the first planes
    for mt in range(1, min(tiles, 5) + 1):
        plan.set_tiling(mt, 3)
        plan.execute(rf, img)
        torch.cuda.synchronize()
        print(f"case tiling {n_ang} angles {precision} {mt}", flush=True)
        assert rel_l2(img.cpu().numpy(), ref.cpu().numpy()) <= (1e-3 if precision == "fp16" else 1e-5)
    batch.execute([rf], [img])
    torch.cuda.synchronize()
    assert rel_l2(img.cpu().numpy(), ref.cpu().numpy()) <= (1e-3 if precision == "fp16" else 1e-5)
    batch.close()


@pytest.mark.parametrize("n_ang", [3, 20, 70])
def test_interpolated_plans_tangent_and_autotune(fa, n_ang):
    """an interpolated plan holds no planes until its tangent asks; its tiling changes nothing"""
    import torch

    F = fa.f_numbers.constant(1.5)
    plan, other = _plan(fa, n_ang, F=F), _plan(fa, n_ang, F=F, precision="fp16x3")
    rf = torch.randn((n_ang, 128, 700), generator=torch.Generator().manual_seed(5)).cuda()
    ref, img, d = (torch.empty((80, 90), dtype=torch.complex64, device="cuda") for _ in range(3))
    other.execute(rf, ref)
    r = plan.autotune(rf, img, repetitions=2)
    assert r["n_candidates"] == 1
    plan.execute(rf, img)
    before = plan.info()["workspace_bytes"]
    plan.execute_tangent(rf, img, d)
    torch.cuda.synchronize()
    assert plan.info()["workspace_bytes"] > before
    assert rel_l2(img.cpu().numpy(), ref.cpu().numpy()) <= 1e-5
    plan.execute(rf, img)
    torch.cuda.synchronize()
    assert rel_l2(img.cpu().numpy(), ref.cpu().numpy()) <= 1e-5


@pytest.mark.parametrize("n,n_ang,nx,nz,stacked", [(16, 1, 64, 64, 16), (4, 1, 64, 64, 4), (8, 3, 160, 180, 0),
                                                   (2, 1, 128, 128, 0)])
def test_interpolated_plans_in_a_batch(fa, n, n_ang, nx, nz, stacked):
    """plans of one F-number share one sum over the bins where that is the faster; either way each
    image is its own plan's"""
    import torch

    x, z = np.linspace(-19e-3, 19e-3, nx), np.linspace(5e-3, 40e-3, nz)
    plans = [fa.PwPlan(x, z, 1536, 128, np.linspace(-0.2, 0.2, n_ang) + 0.01 * i, FS, WIDTH, PITCH, C0, (2.25e6, 6.75e6),
                       0.0, window=fa.windows.tukey(0.5), F_number=fa.f_numbers.constant(1.5)) for i in range(n)]
    rfs = [torch.randn((n_ang, 128, 1536), generator=torch.Generator().manual_seed(i)).cuda() for i in range(n)]
    imgs = [torch.empty((nx, nz), dtype=torch.complex64, device="cuda") for _ in range(n)]
    batch = fa.Batch(plans)
    for _ in range(2):
        batch.execute(rfs, imgs)
    torch.cuda.synchronize()
    assert batch.info()["stacked_plans"] == stacked
    ref = torch.empty_like(imgs[0])
    for p, r, g in zip(plans, rfs, imgs):
        p.execute(r, ref)
        torch.cuda.synchronize()
        assert rel_l2(g.cpu().numpy(), ref.cpu().numpy()) <= 1e-5
    batch.close()


@pytest.mark.parametrize("n_ang,stacking", [(11, False), (40, True)])
def test_batches_follow_a_new_tiling(fa, n_ang, stacking):
    """partial images grow with the bin split, in a buffer of their own: a graph that holds the old
    one is captured again"""
    import torch

    plan, other = _plan(fa, n_ang), _plan(fa, n_ang)
    rf = [torch.randn((n_ang, 128, 700), generator=torch.Generator().manual_seed(k)).cuda() for k in (7, 8)]
    img = [torch.empty((80, 90), dtype=torch.complex64, device="cuda") for _ in range(2)]
    ref = torch.empty_like(img[0])
    batch = fa.Batch([plan, other], stacking=stacking)
    for k, (mt, split) in enumerate([(1, 1), (1, 24), (1, 48), (1, 2)]):
        plan.set_tiling(mt, split)
        plan.execute(rf[0], ref)
        for _ in range(3):
            img[0].zero_()
            batch.execute(rf, img)
            torch.cuda.synchronize()
            assert rel_l2(img[0].cpu().numpy(), ref.cpu().numpy()) <= 1e-5
        assert batch.info()["captures"] == k + 1
    batch.close()


def test_a_tiling_without_memory_leaves_the_old_one(fa):
    """planes (476 MB) or partial images that the device has no room for (256 MiB left) refuse the
    tiling, and the plan goes on with the one it has, bit for bit"""
    import torch

    n_ang, n_t = 96, 8192
    x, z = np.linspace(-8e-3, 8e-3, 192) + 1e-3, np.linspace(5e-3, 30e-3, 256)
    plan = fa.PwPlan(x, z, n_t, 128, np.linspace(-0.2, 0.2, n_ang), FS, WIDTH, PITCH, C0, (1e6, 8e6), 0.0,
                     window=fa.windows.tukey(0.5), F_number=fa.f_numbers.grating.angle_lb(60, 1.5))
    rf = torch.randn((n_ang, 128, n_t), generator=torch.Generator(device="cuda").manual_seed(9), device="cuda")
    ref, img = (torch.empty((192, 256), dtype=torch.complex64, device="cuda") for _ in range(2))
    plan.execute(rf, ref)
    torch.cuda.synchronize()
    before, bins = plan.info(), plan.info()["n_f"]
    assert bins * 16384 * 10 > 400e6 and 8 * 192 * 256 * bins > 512e6
    filler = []
    while (room := torch.cuda.mem_get_info()[0] - (256 << 20)) > (2 << 20):
        filler.append(torch.empty(min(room, 16 << 30) // (2 << 20) * (2 << 20), dtype=torch.uint8, device="cuda"))
    for mt, split in ((5, 2), (plan.info()["m_tiles"], bins)):
        print(f"case no memory {mt} {split}", flush=True)
        with pytest.raises(Exception, match="memory"):
            plan.set_tiling(mt, split)
        assert plan.info() == before
        plan.execute(rf, img)
        torch.cuda.synchronize()
        assert torch.equal(img, ref)
    del filler
    torch.cuda.empty_cache()
    plan.set_tiling(5, 2)
    plan.execute(rf, img)
    torch.cuda.synchronize()
    assert rel_l2(img.cpu().numpy(), ref.cpu().numpy()) <= 1e-5
