"""GPU parity of fan-beam FBP (MFMA filter + pixel-driven backprojection)
against the oracle, the reference's golden images and the FP64 oracle."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2, rel_max
from oracle.oracle import Geom

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _ops():
    from virtualct_amd import ops
    return ops


def _geom(N=512, pix=0.1, V=800):
    from virtualct_amd import default_geometry
    return default_geometry(recon_size=N, pixel_cm=pix, n_views=V)


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _exact_plan(geom):
    """A plan whose single-sinogram backprojection adds each pixel's views in
    the reference's order (not the quarter-turn orbits)."""
    from virtualct_amd import _lib
    plan = _ops().Plan(geom)
    plan.set_option(_lib.OPT_EXACT_BACKPROJECT, 1)
    return plan


@pytest.mark.parametrize("filt", [2, 1])
def test_filter_matches_oracle(gpu, golden, oracle, filt):
    ops = _ops()
    p = golden.kat_f_input()
    plan = ops.plan_for(_geom())
    fl = ops.filter_sinogram(plan, _t(p, gpu), filt)[0].cpu().numpy()
    ref = oracle.filter_ref(Geom(), p, filt)
    f64 = oracle.filter_f64(Geom(), p, filt)
    assert rel_max(fl, ref) < TOL
    assert rel_max(fl, f64) < TOL
    assert rel_l2(fl, f64) < TOL


def test_filter_in_mode_threshold(gpu, golden, oracle):
    ops = _ops()
    p = golden.kat_f_input()
    plan = ops.plan_for(_geom())
    fl = ops.filter_sinogram(plan, _t(p, gpu), 2, in_mode=True)[0].cpu().numpy()
    ref = oracle.filter_ref(Geom(), p, 2, in_mode=True)
    plain = oracle.filter_ref(Geom(), p, 2)
    # outside the thresholds both are exactly zero; elsewhere they agree
    near = (np.abs(plain - 1000.0) < 1.0) | (np.abs(plain - 300000.0) < 10.0)
    assert np.array_equal(fl[~near] == 0, ref[~near] == 0)
    both = (fl != 0) & (ref != 0)
    assert rel_max(fl[both], ref[both]) < TOL


def test_backprojection_matches_oracle(gpu, golden, oracle):
    """Same filtered input: the exact-order BP reproduces the reference's FP64
    geometry and float accumulation order (atan from the device math library)."""
    ops = _ops()
    fl = oracle.filter_ref(Geom(), golden.kat_f_input(), 2)
    plan = _exact_plan(_geom())
    img = ops.backproject(plan, _t(fl, gpu))[0].cpu().numpy()
    ref = oracle.backproject_ref(Geom(), fl)
    assert rel_max(img, ref) < 1e-6
    assert np.count_nonzero(img != ref) < 0.01 * img.size
    mask = oracle.mask(512).astype(bool)
    assert np.all(img[~mask] == 0)
    plan.close()


@pytest.mark.parametrize("N,pix,V", [(512, 0.1, 800), (128, 0.6, 160), (64, 0.7, 2100), (96, 0.5, 84)])
def test_quarter_turn_backprojection_matches_oracle(gpu, golden, oracle, N, pix, V):
    """The default single-sinogram BP shares each pixel-view geometry over the
    4 pixels of a quarter-turn orbit (views a multiple of 4, N even): within
    1e-5 of the reference-order image and of FP64 (512^2 on the KAT-F input;
    a wide field with the library atan; 2100 views; 84 views, 96^2), zero
    outside the mask, and within 1e-5 of the exact-order kernel (the float
    sums run in another order: measured 1.2e-6 at 800 views, 2.2e-6 at 2100)."""
    ops = _ops()
    g = Geom(N=N, pix=pix, V=V)
    if (N, V) == (512, 800):
        fl = oracle.filter_ref(Geom(), golden.kat_f_input(), 2)
    else:
        fl = np.random.default_rng(N + V).normal(size=(V, 609)).astype(np.float32) * 1e3
    img = ops.backproject(ops.plan_for(_geom(N, pix, V)), _t(fl, gpu))[0].cpu().numpy()
    ref = oracle.backproject_ref(g, fl)
    f64 = oracle.backproject_f64(g, fl.astype(np.float64))
    assert rel_max(img, ref) < TOL
    assert rel_max(img, f64) < TOL
    assert rel_l2(img, f64) < 1e-6
    mask = oracle.mask(N).astype(bool)
    assert np.all(img[~mask] == 0)
    plan = _exact_plan(_geom(N, pix, V))
    exact = ops.backproject(plan, _t(fl, gpu))[0].cpu().numpy()
    assert rel_max(img, exact) < TOL
    plan.close()


def test_kat_f_end_to_end(gpu, golden, oracle):
    ops = _ops()
    p = golden.kat_f_input()
    plan = ops.plan_for(_geom())
    img = ops.fbp(plan, _t(p, gpu), 2)[0].cpu().numpy()
    ref = oracle.fbp_ref(Geom(), p, 2)  # bit-identical to the shipped KAT-F image
    f64 = oracle.fbp_f64(Geom(), p, 2)
    assert rel_max(img, ref) < TOL
    assert rel_l2(img, ref) < TOL
    assert rel_max(img, f64) < TOL


@pytest.mark.parametrize("case,N,pix,V", [("n64", 64, 0.7, 80), ("n128", 128, 0.35, 160)])
def test_small_fbp_matches_reference(gpu, golden, case, N, pix, V):
    ops = _ops()
    t = golden.npz("ref_small.npz")
    raw = t[case + "_raw"]
    norm = (raw / raw.max()).astype(np.float32)
    plan = ops.plan_for(_geom(N, pix, V))
    fl = ops.filter_sinogram(plan, _t(norm, gpu), 2)[0].cpu().numpy()
    assert rel_max(fl, t[case + "_fltd"]) < TOL
    img = ops.backproject(plan, _t(fl, gpu))[0].cpu().numpy()
    assert rel_max(img, t[case + "_img"]) < TOL


def test_batched_fbp_equals_single(gpu, golden):
    import torch
    ops = _ops()
    p = golden.kat_f_input()
    plan = _exact_plan(_geom())
    stack = torch.stack([_t(p, gpu), _t(p * np.float32(0.9), gpu), _t(np.sqrt(p), gpu)])
    many = ops.fbp(plan, stack, 2)
    for i in range(3):
        one = ops.fbp(plan, stack[i], 2)[0]
        assert torch.equal(many[i], one)


@pytest.mark.parametrize("W,V,S", [(609, 800, 3), (100, 90, 3), (1000, 64, 2), (64, 33, 1)])
@pytest.mark.parametrize("filt", [2, 1])
def test_filter_shapes_match_oracle(gpu, oracle, W, V, S, filt):
    """The split-K MFMA filter over stacked sinograms whose row count is not a
    multiple of 32, for channel counts where the edge-renormalised rows fall
    in different column tiles (Toeplitz tiles read the generator from LDS,
    edge tiles the packed matrix), against the reference-order filter and FP64."""
    from virtualct_amd import default_geometry
    ops = _ops()
    geom = default_geometry(recon_size=128, pixel_cm=0.35, n_views=V, n_channels=W, iso_channel=(W - 1) / 2.0)
    plan = ops.plan_for(geom)
    rng = np.random.default_rng(W + V + S)
    p = rng.uniform(0.02, 1.0, size=(S, V, W)).astype(np.float32)
    fl = ops.filter_sinogram(plan, _t(p, gpu), filt).cpu().numpy()
    g = Geom(N=128, pix=0.35, V=V, W=W, iso_channel=(W - 1) / 2.0)
    for s in range(S):
        assert rel_max(fl[s], oracle.filter_ref(g, p[s], filt)) < TOL, s
        assert rel_max(fl[s], oracle.filter_f64(g, p[s], filt)) < TOL, s
    # the same with a caller-owned workspace
    work = ops.filter_workspace(plan, S)
    fl2 = ops.filter_sinogram(plan, _t(p, gpu), filt, work=work).cpu().numpy()
    assert np.array_equal(fl, fl2)


def test_filter_scratch_growth_keeps_captured_graph_valid(gpu):
    """A captured forward + FBP run owns its filter workspace, and the context
    scratch only grows (a larger eager call retires the old buffer instead of
    freeing it): replays after a larger eager FBP still equal the eager run."""
    import torch
    from virtualct_amd import batch, phantoms
    ops = _ops()
    att = torch.tensor([[[0.2, 0.1]] * 6], device=gpu)
    pdf = torch.tensor([[0.6, 0.4]], device=gpu)
    N, pix = 64, 0.7
    ph = torch.from_numpy(phantoms.body_phantom(41, N=N, pix_cm=pix))[None].to(gpu)
    run = batch.BatchForwardFBP([(_geom(N, pix, 160), ph)], att, pdf, sigma=0.0, blocked=False)
    _, imgs = run.run()
    eager = [i.clone() for i in imgs]
    run.capture()
    plan = ops.plan_for(_geom())
    big = torch.rand((24, 800, 609), device=gpu) * 0.5 + 0.25
    many = ops.filter_sinogram(plan, big, 2)  # 24 sinograms: the context scratch grows
    for _ in range(2):
        _, i2 = run.replay()
        torch.cuda.synchronize()
        for a, b in zip(i2, eager):
            assert torch.equal(a, b)
    assert torch.equal(many[5], ops.filter_sinogram(plan, big[5], 2)[0])


@pytest.mark.parametrize("N,pix,V,S", [(512, 0.1, 800, 16), (512, 0.1, 800, 48),
                                        (512, 0.1, 800, 5), (512, 0.1, 200, 2), (512, 0.1, 200, 3),
                                        (512, 0.1, 200, 10), (512, 0.1, 200, 17), (512, 0.1, 200, 35),
                                        (512, 0.15, 200, 6),
                                        (128, 0.6, 160, 6), (64, 0.7, 90, 3)])
def test_multi_sinogram_backprojection_equals_single(gpu, oracle, N, pix, V, S):
    """S sinograms of one geometry share each lane's pixel-view geometry (up to
    16 per lane, in even slices: 16 -> one slice of 16, 48 -> 3 x 16, 17 -> 9 + 8,
    35 -> 12 + 12 + 11); every
    image equals the single-sinogram backprojection
    bit for bit.  512 x 0.15 cm and 128 x 0.6 cm are wide fields (library atan
    fallback); at 128^2 and 64^2 the launch keeps 2^18 lanes by running one
    sinogram per lane."""
    import torch
    ops = _ops()
    rng = np.random.default_rng(40 + S)
    fl = rng.normal(size=(S, V, 609)).astype(np.float32) * 1e3
    plan = _exact_plan(_geom(N, pix, V))
    many = ops.backproject(plan, _t(fl, gpu))
    for i in range(S):
        one = ops.backproject(plan, _t(fl[i], gpu))[0]
        assert torch.equal(many[i], one), i
    if N <= 128:
        ref = oracle.backproject_ref(Geom(N=N, pix=pix, V=V), fl[S - 1])
        assert rel_max(many[S - 1].cpu().numpy(), ref) < 1e-5
    plan.close()


def test_mbfpa_then_fbp_recovers_mu_map(gpu, golden):
    """The pipeline MBFPA -> FBP gives a mu map in 1/cm in the same
    orientation as the phantom (correlation with sum rho_m mu_m(60 keV))."""
    ops = _ops()
    from virtualct_amd import spectra
    att, pdf, e = spectra.attenuation(golden.path("spectrum_120kV.txt"), 6)
    plan = ops.plan_for(_geom())
    ph = golden.icru110()
    sino = ops.mbfpa_forward(plan, _t(ph, gpu), _t(att, gpu), _t(pdf, gpu))
    img = ops.fbp(plan, sino, 2)[0].cpu().numpy()
    i60 = int(np.argmin(np.abs(e - 0.06)))
    mu = (ph.astype(np.float64) / 1000 * att[:, i60, None, None]).sum(0)
    r = np.corrcoef(img.ravel(), mu.ravel())[0, 1]
    assert r > 0.95


@pytest.mark.parametrize("alpha,beta", [(0.01, 2.0), (0.01, 3.7)])
def test_beam_hardening_kernel_and_fused_filter(gpu, golden, oracle, alpha, beta):
    ops = _ops()
    p = golden.sigma0_120kv()
    ref, _, _ = oracle.beam_hardening(p, alpha, beta)  # bit-identical to the reference tool
    got = ops.beam_hardening(_t(p, gpu), alpha, beta).cpu().numpy()
    assert rel_max(got, ref) < 1e-6
    assert np.count_nonzero(got != ref) < 0.01 * got.size
    plan = ops.plan_for(_geom())
    fused = ops.filter_sinogram_bhc(plan, _t(p, gpu), alpha, beta)[0].cpu().numpy()
    two_step = oracle.filter_ref(Geom(), ref, 2)
    assert rel_max(fused, two_step) < 1e-5
    mx, mn = ops.minmax(_t(p, gpu))
    assert mx == p.max() and mn == p.min()


def test_bhc_driver(gpu, golden, oracle, tmp_path):
    import subprocess
    from conftest import ROOT
    import os
    p = golden.sigma0_120kv()
    p.tofile(tmp_path / "reprojection_float.raw")
    r = subprocess.run([os.path.join(ROOT, "virtualct_amd", "bin", "mvct_bhc"), "0.01", "2.0"], cwd=tmp_path,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    out = np.fromfile(tmp_path / "reprojection_float_cor.raw", np.float32).reshape(800, 609)
    ref, mn0, mn1 = oracle.beam_hardening(p, 0.01, 2.0)
    assert rel_max(out, ref) < 1e-6
    assert r.stdout.strip() == f"{mn0:f} {mn1:f}"


def test_wide_field_backprojection_takes_library_atan(gpu, oracle):
    """A 76.8 cm field (N=128, 0.6 cm) puts masked pixels at |tan(gamma)| up to
    0.53, beyond the polynomial: the kernel variant with the library atan
    fallback, against the oracle."""
    ops = _ops()
    N, pix, V = 128, 0.6, 160
    g = Geom(N=N, pix=pix, V=V)
    r = (N - 1) / 2.0 * pix
    assert r / np.sqrt(85.0 ** 2 - r ** 2) > 0.5
    rng = np.random.default_rng(31)
    fl = rng.normal(size=(V, 609)).astype(np.float32) * 1e3
    plan = ops.plan_for(_geom(N, pix, V))
    img = ops.backproject(plan, _t(fl, gpu))[0].cpu().numpy()
    ref = oracle.backproject_ref(g, fl)
    f64 = oracle.backproject_f64(g, fl.astype(np.float64))
    assert rel_max(img, ref) < 1e-5
    assert rel_max(img, f64) < 1e-5
    mask = oracle.mask(N).astype(bool)
    assert np.all(img[~mask] == 0)


def test_backprojection_more_views_than_one_trig_block(gpu, oracle):
    """2100 views: a view loop longer than 2048 views (exact-order kernel)."""
    ops = _ops()
    N, pix, V = 64, 0.7, 2100
    g = Geom(N=N, pix=pix, V=V)
    fl = np.random.default_rng(32).normal(size=(V, 609)).astype(np.float32)
    plan = _exact_plan(_geom(N, pix, V))
    img = ops.backproject(plan, _t(fl, gpu))[0].cpu().numpy()
    ref = oracle.backproject_ref(g, fl)
    assert rel_max(img, ref) < 1e-5
    assert np.count_nonzero(img != ref) < 0.05 * img.size


@pytest.mark.parametrize("N,pix,V,S", [(512, 0.1, 800, 16), (512, 0.1, 800, 5), (128, 0.6, 160, 6),
                                        (64, 0.7, 90, 3), (96, 0.5, 801, 2)])
def test_multi_sinogram_float_weights_match_exact_terms(gpu, oracle, N, pix, V, S):
    """By default several sinograms per call apply the interpolation and
    distance weights in float: within 1e-6 of the exact FP64 terms (same view
    order) and 1e-5 of the reference, and each image does not depend on how
    the call is split (one call of S, or S/2 + S/2)."""
    import torch
    ops = _ops()
    rng = np.random.default_rng(70 + S)
    fl = _t(rng.normal(size=(S, V, 609)).astype(np.float32) * 1e3, gpu)
    plan = ops.Plan(_geom(N, pix, V))
    fast = ops.backproject(plan, fl)
    exact_plan = _exact_plan(_geom(N, pix, V))
    exact = ops.backproject(exact_plan, fl)
    assert rel_max(fast.cpu().numpy(), exact.cpu().numpy()) < 1e-6
    ref = oracle.backproject_ref(Geom(N=N, pix=pix, V=V), fl[S - 1].cpu().numpy())
    assert rel_max(fast[S - 1].cpu().numpy(), ref) < 1e-5
    h = S // 2
    if h >= 2:
        halves = torch.cat([ops.backproject(plan, fl[:h].contiguous()), ops.backproject(plan, fl[h:].contiguous())])
        assert torch.equal(halves, fast)
    plan.close()
    exact_plan.close()


@pytest.mark.parametrize("N,pix,V", [(65, 0.7, 84), (65, 0.7, 90), (64, 0.7, 90), (65, 0.7, 81), (64, 0.7, 83),
                                      (127, 0.6, 90), (127, 0.6, 160), (8, 3.0, 6), (7, 3.0, 4), (9, 3.0, 2),
                                      (17, 2.0, 3)])
def test_single_sinogram_off_the_quarter_turn_grid(gpu, oracle, N, pix, V):
    """One sinogram on odd grids and at view counts that are no multiple of
    four (orbits of four, two or one pixels, the centre and the middle row of
    odd grids, more waves than views): FP64 terms and sums, so the image is
    the FP64 one rounded to float (half an ulp, 6e-8) but for the FP64
    roundings of another operation order (below 1e-11 each); 0.6 cm pixels
    take the library atan."""
    ops = _ops()
    g = Geom(N=N, pix=pix, V=V)
    fl = np.random.default_rng(N * V).normal(size=(V, 609)).astype(np.float32) * 1e3
    plan = ops.Plan(_geom(N, pix, V))
    img = ops.backproject(plan, _t(fl, gpu))[0].cpu().numpy()
    f64 = oracle.backproject_f64(g, fl.astype(np.float64))
    scale = np.abs(f64).max()
    assert np.all(np.abs(img - f64) <= 6.0e-8 * np.abs(f64) + 1.0e-9 * scale)
    assert np.all(img[~oracle.mask(N).astype(bool)] == 0)
    plan.close()


@pytest.mark.parametrize("N,pix,V,S", [(512, 0.1, 90, 2), (512, 0.1, 90, 3), (300, 0.16, 91, 5), (200, 0.25, 90, 7),
                                        (511, 0.1, 33, 9), (512, 0.1, 90, 12), (512, 0.1, 33, 13), (65, 0.7, 90, 23),
                                        (300, 0.16, 33, 51), (128, 0.6, 160, 6), (16, 3.0, 2, 97), (16, 3.0, 1, 4)])
def test_interleaved_slices_equal_plain_sinograms(gpu, N, pix, V, S):
    """Several sinograms through interleaved slices (every width, padded last
    slices, more than one pass of 48, the library atan) give the images of
    the call without a workspace bit for bit."""
    import torch
    from virtualct_amd import _lib
    ops = _ops()
    plan = ops.Plan(_geom(N, pix, V))
    fl = _t(np.random.default_rng(N + S).normal(size=(S, V, 609)).astype(np.float32) * 1e3, gpu)
    for cap in (0, 2, 5, 16):
        plan.set_option(_lib.OPT_BP_SINOS_PER_LANE, cap)
        ref = torch.full((S, N, N), float("nan"), device=gpu)
        torch.cuda.synchronize()
        _lib.call("vct_backproject", plan.handle, fl.data_ptr(), S, ref.data_ptr(), None)
        torch.cuda.synchronize()
        assert torch.equal(ops.backproject(plan, fl), ref), cap
    plan.close()


@pytest.mark.parametrize("W,V,S", [(609, 800, 5), (609, 400, 8), (100, 800, 21), (300, 801, 9), (33, 800, 45)])
def test_tall_filter_products_equal_single_sinograms(gpu, W, V, S):
    """Strips of column tiles (last strips of one to four tiles, edge tiles
    within a strip, rows that are no multiple of 32) sum each output in the
    order of a single sinogram's product: the same bits."""
    from virtualct_amd import default_geometry
    ops = _ops()
    plan = ops.plan_for(default_geometry(recon_size=64, pixel_cm=0.7, n_views=V, n_channels=W, iso_channel=W / 2.0))
    p = _t(np.random.default_rng(W + S).uniform(0.02, 1.0, (S, V, W)).astype(np.float32), gpu)
    many = ops.filter_sinogram(plan, p, 2).cpu().numpy()
    for i in (0, S // 2, S - 1):
        assert np.array_equal(many[i], ops.filter_sinogram(plan, p[i], 2)[0].cpu().numpy()), i


@pytest.mark.parametrize("N,pix,V,S", [(512, 0.4, 8, 1), (512, 0.4, 6, 1), (512, 0.4, 5, 1), (512, 0.4, 8, 3),
                                        (512, 0.4, 5, 13), (173, 1.0, 8, 1), (173, 1.0, 6, 1), (173, 1.0, 7, 2)])
def test_pixels_level_with_the_source(gpu, N, pix, V, S):
    """A field that holds the source's circle, with a line of pixels exactly at
    the source's distance in view 0 (row 43 of 512 x 0.4 cm, row 1 of 173 x 1
    cm: sid - Y = 0, and X = 0 too in the middle of the odd grid): they are off
    the detector, as in the exact option.  Each term has five float roundings
    and each image at most 8 adds, 13 * 2^-24 < 1e-6 of the summed magnitudes:
    values up to 1.5 with weights up to 1.9 and 0.9, below 5 times a unit
    sinogram's sum."""
    import torch
    from virtualct_amd import _lib
    ops = _ops()
    assert -(43 - 255.5) * 0.4 == 85.0 and -(1 - 86.0) * 1.0 == 85.0
    plan, exact_plan = ops.Plan(_geom(N, pix, V)), _exact_plan(_geom(N, pix, V))
    fl = _t(np.random.default_rng(N + V).uniform(0.5, 1.5, (S, V, 609)).astype(np.float32), gpu)
    exact = ops.backproject(exact_plan, fl)
    bound = 1e-6 * ops.backproject(exact_plan, torch.full_like(fl[:1], 5.0))
    assert torch.isfinite(exact).all() and exact.count_nonzero() > 0
    imgs = [ops.backproject(plan, fl)]
    if S > 1:
        imgs.append(torch.empty_like(imgs[0]))  # (the call without a workspace)
        _lib.call("vct_backproject", plan.handle, fl.data_ptr(), S, imgs[1].data_ptr(),
                  torch.cuda.current_stream().cuda_stream)
    for img in imgs:
        assert torch.isfinite(img).all()
        assert torch.all((img - exact).abs() <= bound)
    plan.close()
    exact_plan.close()


@pytest.mark.parametrize("S", [1, 2])
def test_degenerate_channel_pitch(gpu, S):
    """A channel pitch of zero puts every pixel off the detector, the middle
    column (0 / 0) included, as in the exact option."""
    import torch
    from virtualct_amd import _lib, default_geometry
    ops = _ops()
    fl = torch.ones((S, 8, 609), device=gpu)
    for exact in (0, 1):
        plan = ops.Plan(default_geometry(recon_size=65, pixel_cm=0.7, n_views=8, max_beta=0.0))
        plan.set_option(_lib.OPT_EXACT_BACKPROJECT, exact)
        assert not ops.backproject(plan, fl).any()
        plan.close()


@pytest.mark.parametrize("S", [1, 4])
def test_float_weights_near_a_channel(gpu, oracle, S):
    """Every third channel of one view is 1, so a pixel's value is one
    interpolation weight over L^2.  Both weights keep 24 bits where they are
    small: at most seven roundings of 2^-24 (L^2, its reciprocal (two), the view
    step, their product, the weight and its product) and 2e-10 channels of the
    arc tangent over the weight, together below 6e-7 for weights from 2e-3 on.
    (A float 1 - w made from a float w is off by 1.5e-5 there.)"""
    ops = _ops()
    N, pix, V, view = 256, 0.2, 16, 3
    plan = ops.Plan(_geom(N, pix, V))
    fl = np.zeros((V, 609), np.float32)
    fl[view, ::3] = 1.0
    ones = np.zeros((V, 609))
    ones[view] = 1.0
    g = Geom(N=N, pix=pix, V=V)
    f64 = oracle.backproject_f64(g, fl.astype(np.float64))
    whole = oracle.backproject_f64(g, ones)
    img = ops.backproject(plan, _t(np.repeat(fl[None], S, 0), gpu)).cpu().numpy().astype(np.float64)
    weight = np.divide(f64, whole, out=np.zeros_like(f64), where=whole != 0)
    use = weight >= 2e-3
    assert np.count_nonzero(use & (weight < 2e-2)) > 100
    for k in range(S):
        assert np.all(np.abs(img[k] - f64)[use] <= 6e-7 * np.abs(f64[use]))
    plan.close()


def test_backprojection_workspace_serves_smaller_calls(gpu):
    """A workspace sized for a count of sinograms serves every smaller count
    and every VCT_OPT_BP_SINOS_PER_LANE: the size grows with the count and does
    not depend on the option, and no call writes past it."""
    import torch
    from virtualct_amd import _lib
    ops = _ops()
    N, pix, V = 512, 0.1, 64
    plan = ops.Plan(_geom(N, pix, V))
    size = lambda n: int(_lib.lib().vct_backproject_workspace_bytes(plan.handle, n))
    sizes = []
    for cap in (0, 2, 3, 4, 6, 8, 11, 16):
        plan.set_option(_lib.OPT_BP_SINOS_PER_LANE, cap)
        sizes.append([size(n) for n in range(1, 70)])
    assert all(s == sizes[0] for s in sizes)
    assert sizes[0] == sorted(sizes[0]) and sizes[0][0] == 0 and sizes[0][1] > 0
    slot = V * 609
    fl = torch.randn((50, V, 609), device=gpu)
    for most in (3, 13, 25, 50):
        words = size(most) // 4
        buf = torch.full((48 * slot + words,), 7.0, device=gpu)  # (more than any call can use)
        for n in sorted({2, most - 2, most - 1, most, most * 24 // 25} - {1}):
            for cap in (0, 4, 8):
                plan.set_option(_lib.OPT_BP_SINOS_PER_LANE, cap)
                img = torch.empty((n, N, N), device=gpu)
                _lib.call("vct_backproject_ws", plan.handle, fl.data_ptr(), n, img.data_ptr(), buf.data_ptr(),
                          torch.cuda.current_stream().cuda_stream)
                assert torch.all(buf[words:] == 7.0), (most, n, cap)
    plan.close()
