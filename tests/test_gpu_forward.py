"""GPU parity of the MBFPA forward path (tracer, polyenergetic sum,
normalisation, detector noise) against the oracle and the reference's golden
vectors.  Every call goes through the C ABI of libvct.so."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2, rel_max
from oracle.oracle import Geom

pytestmark = pytest.mark.gpu

TOL = 1e-5  # relative parity bar for FP32 sinograms (max|d| / max|ref|)


def _ops():
    from virtualct_amd import ops
    return ops


def _geom(N=512, pix=0.1, V=800):
    from virtualct_amd import default_geometry
    return default_geometry(recon_size=N, pixel_cm=pix, n_views=V)


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _lnrel(a, b, floor=1e-6):
    """max relative error in the -ln domain over rays with b > floor"""
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    m = b > floor
    la, lb = -np.log(np.maximum(a[m], 1e-300)), -np.log(b[m])
    return float(np.abs(la - lb).max() / max(np.abs(lb).max(), 1e-12))


def test_segment_counts_match_reference(gpu, golden, oracle):
    ops = _ops()
    plan = ops.plan_for(_geom())
    pk, dt = ops.pack_densities(plan, _t(golden.icru110(), gpu))
    L, cnt = ops.trace_paths(plan, pk, dt, 6, counts=True)
    cnt = cnt.cpu().numpy()
    ref_cnt, total = oracle.segment_counts(Geom())
    assert int(cnt.astype(np.int64).sum()) == 282_824_404 == total
    np.testing.assert_array_equal(cnt, ref_cnt)


def test_path_integrals_match_fp64_oracle(gpu, golden, oracle):
    ops = _ops()
    ph = golden.icru110()
    plan = ops.plan_for(_geom())
    pk, dt = ops.pack_densities(plan, _t(ph, gpu))
    L = ops.trace_paths(plan, pk, dt, 6).cpu().numpy()[..., :6]
    dens = ph.astype(np.float32) / np.float32(1000)
    att = np.zeros((6, 1), np.float32)
    _, Lo = oracle.forward_f64(Geom(), dens, att, np.ones(1, np.float32), want_L=True)
    assert rel_max(L, Lo) < 1e-6
    # float densities give the same integrals
    pkf, dtf = ops.pack_densities(plan, _t(dens, gpu))
    Lf = ops.trace_paths(plan, pkf, dtf, 6).cpu().numpy()[..., :6]
    assert rel_max(Lf, Lo) < 1e-6


@pytest.mark.parametrize("case,N,pix,V", [("n64", 64, 0.7, 80), ("n128", 128, 0.35, 160)])
def test_small_geometry_matches_reference(gpu, golden, case, N, pix, V):
    ops = _ops()
    t = golden.npz("ref_small.npz")
    plan = ops.plan_for(_geom(N, pix, V))
    pk, dt = ops.pack_densities(plan, _t(t[case + "_phantom"], gpu))
    L, cnt = ops.trace_paths(plan, pk, dt, 6, counts=True)
    np.testing.assert_array_equal(cnt.cpu().numpy(), t[case + "_counts"])
    raw, stats, _ = ops.spectral_sum(plan, L, 6, _t(t["att"], gpu), _t(t["pdf"], gpu))
    raw = raw[0].cpu().numpy()
    ref = t[case + "_raw"]
    assert rel_max(raw, ref) < TOL
    assert _lnrel(raw, ref) < TOL
    mx, mn = ops.stats_values(stats)[0].tolist()
    assert mx == raw.max() and mn == raw.min()


def test_icru110_120kV_noise_free_matches_reference(gpu, golden, oracle):
    ops = _ops()
    from virtualct_amd import spectra
    att, pdf, _ = spectra.attenuation(golden.path("spectrum_120kV.txt"), 6)
    plan = ops.plan_for(_geom())
    sino = ops.mbfpa_forward(plan, _t(golden.icru110(), gpu), _t(att, gpu), _t(pdf, gpu), sigma=0.0)
    sino = sino[0].cpu().numpy()
    ref = golden.sigma0_120kv()
    assert rel_max(sino, ref) < TOL
    assert rel_l2(sino, ref) < TOL
    assert _lnrel(sino, ref) < TOL
    # against the FP64 oracle
    f64 = oracle.forward_f64(Geom(), golden.icru110().astype(np.float32) / np.float32(1000), att, pdf)
    assert rel_max(sino, f64 / f64.max()) < TOL
    # rays that miss the image are exactly air after normalisation
    assert np.all(sino[ref == ref.max()] == sino.max())


def test_shipped_6MV_650_bins(gpu, golden, oracle):
    ops = _ops()
    from virtualct_amd import spectra
    att, pdf, _ = spectra.attenuation(golden.path("spectrum_6MV.txt"), 6)
    assert att.shape == (6, 650)
    plan = ops.plan_for(_geom())
    sino = ops.mbfpa_forward(plan, _t(golden.icru110(), gpu), _t(att, gpu), _t(pdf, gpu))[0].cpu().numpy()
    f64 = oracle.forward_f64(Geom(), golden.icru110().astype(np.float32) / np.float32(1000), att, pdf)
    assert rel_max(sino, f64 / f64.max()) < TOL
    assert _lnrel(sino, f64 / f64.max()) < TOL


def test_dual_spectrum_synthetic_body_phantom(gpu, golden, oracle, tmp_path):
    """120 kV and 6 MV synthetic spectra from one trace (n_spectra = 2)."""
    ops = _ops()
    from virtualct_amd import phantoms, spectra
    ph = phantoms.body_phantom(1000)
    tabs = [spectra.attenuation(spectra.synthetic_spectrum_file(n, str(tmp_path)), 6) for n in ("120kV", "6MV")]
    NE = max(a.shape[1] for a, _, _ in tabs)
    att = np.zeros((2, 6, NE), np.float32)
    pdf = np.zeros((2, NE), np.float32)
    for s, (a, p, _) in enumerate(tabs):
        att[s, :, : a.shape[1]] = a
        pdf[s, : p.shape[0]] = p
    plan = ops.plan_for(_geom())
    sino = ops.mbfpa_forward(plan, _t(ph, gpu), _t(att, gpu), _t(pdf, gpu)).cpu().numpy()
    dens = phantoms.densities_f32(ph)
    for s, (a, p, _) in enumerate(tabs):
        f64 = oracle.forward_f64(Geom(), dens, a, p)
        assert rel_max(sino[s], f64 / f64.max()) < TOL, s
        assert _lnrel(sino[s], f64 / f64.max()) < TOL, s


def test_eight_element_calibration_phantom(gpu, oracle, tmp_path):
    ops = _ops()
    from virtualct_amd import phantoms, spectra
    ph = phantoms.calibration_phantom(2000)
    att, pdf, _ = spectra.attenuation(spectra.synthetic_spectrum_file("120kV", str(tmp_path)), 8)
    plan = ops.plan_for(_geom())
    sino = ops.mbfpa_forward(plan, _t(ph, gpu), _t(att, gpu), _t(pdf, gpu))[0].cpu().numpy()
    f64 = oracle.forward_f64(Geom(), phantoms.densities_f32(ph), att, pdf)
    assert rel_max(sino, f64 / f64.max()) < TOL
    assert _lnrel(sino, f64 / f64.max()) < TOL


def test_noise_matches_philox_box_muller(gpu, golden, oracle):
    """Noise of element r is sigma * sqrt(-2 ln U1) sin(2 pi U2) with U from
    Philox4x32-10(ctr = (r, stream, 0, 0), key = seed)."""
    import torch
    ops = _ops()
    plan = ops.plan_for(_geom())
    clean = golden.sigma0_120kv()
    raw = _t(clean[None], gpu)
    mx = np.float32(1.0)
    stats = torch.tensor([[np.float32(mx).view(np.int32), np.float32(clean.min()).view(np.int32)]],
                         dtype=torch.int32, device=gpu)
    sigma, seed, sid = 5.37e-5, 0x1234_5678_9ABC, 7
    noisy = ops.detector(plan, raw, stats, sigma, seed, sid)[0].cpu().numpy().reshape(-1)
    flat = clean.reshape(-1)
    idx = np.random.default_rng(0).choice(flat.size, 2000, replace=False)
    for r in idx:
        u = oracle.philox([r, sid, 0, 0], [seed & 0xFFFFFFFF, seed >> 32])
        u1 = (float(u[0]) + 1.0) / 4294967297.0
        u2 = (float(u[1]) + 1.0) / 4294967297.0
        z = np.sqrt(-2.0 * np.log(u1)) * np.sin(2.0 * np.pi * u2)
        x = float(flat[r]) + sigma * z
        exp = np.float32(x)
        if x < 0:
            exp = np.float32(float(np.float32(clean.min() / mx)) / 10)
        if x > 1.0:
            exp = np.float32(1.0)
        assert abs(float(noisy[r]) - float(exp)) <= 2 * np.spacing(np.float32(exp)), r


def test_noise_statistics_per_bin(gpu, golden):
    """K independent streams: per-bin mean is the clean value, variance sigma^2,
    and bins at 1.0 are clamped half of the time."""
    import torch
    ops = _ops()
    plan = ops.plan_for(_geom())
    clean = golden.sigma0_120kv()
    K, sigma = 200, 5.37e-5
    raw = _t(clean, gpu).unsqueeze(0).expand(K, -1, -1).contiguous()
    st = torch.tensor([[np.float32(1.0).view(np.int32), np.float32(clean.min()).view(np.int32)]] * K,
                      dtype=torch.int32, device=gpu)
    noisy = ops.detector(plan, raw, st, sigma, 0x5EED, 0).double()
    c = torch.from_numpy(clean).to(gpu).double()
    mean = noisy.mean(0)
    var = noisy.var(0)
    ok = (c > 6 * sigma) & (c < 1 - 6 * sigma)
    z = ((mean - c) / (sigma / K ** 0.5))[ok]
    assert abs(z.mean().item()) < 0.02
    assert abs(z.std().item() - 1.0) < 0.02
    assert z.abs().max().item() < 6.5
    ratio = (var / sigma ** 2)[ok]
    assert abs(ratio.mean().item() - 1.0) < 0.005
    assert abs(ratio.std().item() - (2.0 / (K - 1)) ** 0.5) < 0.01
    air = c == 1.0
    frac = (noisy[:, air] == 1.0).double().mean().item()
    assert abs(frac - 0.5) < 0.01
    assert noisy.max().item() <= 1.0 and noisy.min().item() >= 0.0
    # same seed and stream -> identical draw; another stream -> different
    a = ops.detector(plan, raw[:1], st[:1], sigma, 99, 3)
    b = ops.detector(plan, raw[:1], st[:1], sigma, 99, 3)
    d = ops.detector(plan, raw[:1], st[:1], sigma, 99, 4)
    assert torch.equal(a, b) and not torch.equal(a, d)


def test_sigma_zero_is_plain_normalisation(gpu, golden):
    import torch
    ops = _ops()
    plan = ops.plan_for(_geom())
    clean = golden.sigma0_120kv() * np.float32(0.731)
    raw = _t(clean[None], gpu)
    st = torch.tensor([[np.float32(clean.max()).view(np.int32), np.float32(clean.min()).view(np.int32)]],
                      dtype=torch.int32, device=gpu)
    out = ops.detector(plan, raw, st, 0.0)[0].cpu().numpy()
    np.testing.assert_array_equal(out, clean / clean.max())


def test_argument_errors_raise(gpu):
    ops = _ops()
    import torch
    from virtualct_amd import VctError
    plan = ops.plan_for(_geom())
    with pytest.raises(ValueError):
        ops.pack_densities(plan, torch.zeros((6, 256, 256), dtype=torch.int16, device=gpu))
    pk, dt = ops.pack_densities(plan, torch.zeros((6, 512, 512), dtype=torch.int16, device=gpu))
    L = ops.trace_paths(plan, pk, dt, 6)
    with pytest.raises(VctError):
        ops.spectral_sum(plan, L, 6, torch.zeros((6, 2000), device=gpu), torch.zeros(2000, device=gpu))
    with pytest.raises(VctError):
        ops.detector(plan, torch.zeros((1, 800, 609), device=gpu), torch.zeros((1, 2), dtype=torch.int32,
                                                                                  device=gpu), -1.0)


def test_fast_march_equals_exact_march(gpu, golden):
    """The guarded reciprocal march gives the exact march's segments on every
    ray of the full geometry and of a 768^2 / 0.0651 cm geometry."""
    import ctypes
    ops = _ops()
    from virtualct_amd import _lib, phantoms
    for N, pix, ph in ((512, 0.1, golden.icru110()),
                       (768, 50.0 / 768, phantoms.body_phantom(9, N=768, pix_cm=50.0 / 768))):
        plan = ops.Plan(_geom(N, pix))
        pk, dt = ops.pack_densities(plan, _t(ph, gpu))
        L_fast, c_fast = ops.trace_paths(plan, pk, dt, 6, counts=True)
        _lib.call("vct_plan_set_option", plan.handle, 1, 1)
        L_exact, c_exact = ops.trace_paths(plan, pk, dt, 6, counts=True)
        assert np.array_equal(c_fast.cpu().numpy(), c_exact.cpu().numpy())
        assert rel_max(L_fast.cpu().numpy(), L_exact.cpu().numpy()) < 1e-6
        plan.close()


@pytest.mark.parametrize("M", [3, 5])
def test_odd_material_count_u16(gpu, golden, M):
    """Odd M: integer densities give the float densities' path integrals, and
    the unused high half of the last packed word is never read."""
    import torch
    ops = _ops()
    plan = ops.plan_for(_geom(128, 0.35, 160))
    ph = golden.npz("ref_small.npz")["n128_phantom"][:M]
    pk, dt = ops.pack_densities(plan, _t(ph, gpu))
    L = ops.trace_paths(plan, pk, dt, M)
    pkf, dtf = ops.pack_densities(plan, _t(ph.astype(np.float32) / np.float32(1000), gpu))
    Lf = ops.trace_paths(plan, pkf, dtf, M)
    assert rel_max(L[..., :M].cpu().numpy(), Lf[..., :M].cpu().numpy()) < 1e-6
    dirty = pk.clone()
    dirty[..., M] = 12345  # the high half of word M // 2
    L2 = ops.trace_paths(plan, dirty, dt, M)
    assert torch.equal(L2, L)


def test_step_bound_overflow_is_reported(gpu, golden):
    """A plan whose marching step bound is below what its rays need: the
    tracer and the atomic adjoint give up on those rays and exit normally,
    the device flag makes the call raise VCT_ERR_INTERNAL, and the flag is
    clear afterwards."""
    import torch
    ops = _ops()
    from virtualct_amd import VctError, _lib
    plan = ops.Plan(_geom(128, 0.35, 160))  # own plan: the option is per plan
    ph = golden.npz("ref_small.npz")["n128_phantom"]
    pk, dt = ops.pack_densities(plan, _t(ph, gpu))
    good = ops.trace_paths(plan, pk, dt, 6)
    plan.set_option(_lib.OPT_MAX_STEPS, 8)
    with pytest.raises(VctError) as e:
        ops.trace_paths(plan, pk, dt, 6)
    assert e.value.status == _lib.ERR_INTERNAL
    with pytest.raises(VctError) as e:
        ops.mbfpa_forward(plan, None, torch.ones((6, 2), device=gpu), torch.ones(2, device=gpu) / 2,
                          packed=(pk, dt))
    assert e.value.status == _lib.ERR_INTERNAL
    w = torch.ones((160, 609, 8), device=gpu)
    with pytest.raises(VctError) as e:
        ops.trace_adjoint(plan, w, 6)
    assert e.value.status == _lib.ERR_INTERNAL
    ops.check_errors()  # cleared by the raising check
    plan.set_option(_lib.OPT_MAX_STEPS, 0)
    assert torch.equal(ops.trace_paths(plan, pk, dt, 6), good)
    plan.close()


@pytest.mark.parametrize("N,pix,V", [(512, 0.1, 800), (768, 50.0 / 768, 800), (128, 0.35, 162),
                                     (100, 0.5, 400), (16, 0.5, 40)])
def test_orbit_trace_equals_single_ray_march(gpu, golden, N, pix, V):
    """The default tracer marches the ray of view v once for the rays of views
    v + kV/4 (V a multiple of 4; 162 views take half turns): its segment
    counters equal marching every ray by itself on every ray, and the path
    integrals agree to a float ulp (the orbit shares the base ray's lengths), for
    integer and float densities.  The orbit tracer gathers from a transposed
    copy of the densities for rays along x (N = 100 leaves partial 32 x 32
    tiles in the transpose; at N = 16 the padded u16 copies are larger than
    the 32-byte transposed one), and on random densities in every voxel."""
    import torch
    ops = _ops()
    from virtualct_amd import _lib, phantoms
    ph = phantoms.body_phantom(17, N=N, pix_cm=pix)
    # every voxel nonzero, the image border included: a turned ray's index -1
    # (truncated to voxel 0) and N - 1 read real densities
    rnd = np.random.default_rng(N).integers(1, 2000, size=ph.shape, dtype=np.int16)
    cases = (("u16", _t(ph, gpu)), ("f32", _t(phantoms.densities_f32(ph), gpu)), ("u16 random", _t(rnd, gpu)))
    out = {}
    for orbit in (4, 2, 1):
        plan = ops.Plan(_geom(N, pix, V))
        plan.set_option(_lib.OPT_TRACE_ORBIT, orbit)
        for name, d in cases:
            pk, dt = ops.pack_densities(plan, d)
            L, cnt = ops.trace_paths(plan, pk, dt, 6, counts=True)
            out[(orbit, name)] = (L.cpu().numpy(), cnt.cpu().numpy())
        plan.close()
    for name, _ in cases:
        L1, c1 = out[(1, name)]
        assert c1.sum() > 0
        for orbit in (4, 2):
            L, c = out[(orbit, name)]
            np.testing.assert_array_equal(c, c1, err_msg=f"orbit {orbit} {name}")
            # float32 outputs of FP64 sums that differ in the last bits: at
            # most one float ulp apart (1.2e-7 of the largest value)
            assert rel_max(L, L1) < 2.5e-7, (orbit, name)


@pytest.mark.parametrize("N,fov,V,W,M,f32", [
    (6, 2.0, 4, 22, 1, False), (7, 2.0, 5, 23, 3, True), (64, 50.0, 80, 609, 6, False), (64, 51.2, 80, 609, 6, False),
    (128, 51.2, 48, 609, 6, True), (130, 50.0, 12, 333, 8, True), (130, 50.0, 14, 64, 8, False),
    (301, 50.0, 9, 65, 2, True), (256, 50.0, 20, 609, 5, False), (96, 30.0, 36, 80, 7, False), (33, 20.0, 6, 47, 4, True)])
def test_segment_tracer_equals_exact_march(gpu, N, fov, V, W, M, f32):
    """The segment-by-segment tracer (orbits of 4, 2 and 1 rays, partial tiles
    of 16 channels x 4 views, an odd count's last view, odd N; at 128 voxels
    on 51.2 cm the step-by-step form that such grids keep) against the
    exact-division march of every ray: the same segment counters, and path
    integrals within two float roundings, since both sum the same segments in
    FP64 with lengths equal to ~1e-11.  Some densities are negative and NaN,
    which contribute nothing."""
    from virtualct_amd import _lib, default_geometry
    ops = _ops()
    geom = default_geometry(recon_size=N, pixel_cm=fov / N, n_views=V, n_channels=W, iso_channel=W / 2.0 + 0.13)
    rng = np.random.default_rng(N + V)
    if f32:
        d = rng.uniform(0.0, 2.0, (M, N, N)).astype(np.float32)
        d[:, 0, 0] = -1.0
        d[:, N // 2, 1] = np.nan
    else:
        d = rng.integers(0, 2000, (M, N, N)).astype(np.int16)
        d[:, 0, 0] = -5
    out = []
    for exact in (0, 1):
        plan = ops.Plan(geom)
        plan.set_option(_lib.OPT_EXACT_TRACE, exact)
        pk, dt = ops.pack_densities(plan, _t(d, gpu))
        L, cnt = ops.trace_paths(plan, pk, dt, M, counts=True)
        out.append((L.cpu().numpy(), cnt.cpu().numpy()))
        plan.close()
    (L, c), (Le, ce) = out
    np.testing.assert_array_equal(c, ce)
    assert np.isfinite(L).all() and not np.any(L[..., M:])
    assert np.all(np.abs(L - Le) <= 2.0 ** -22 * np.abs(Le) + 1e-9)


@pytest.mark.parametrize("N,V,orbit", [(129, 80, 4), (128, 81, 4), (130, 22, 1)])
def test_infinite_corner_voxel_reaches_its_own_rays_only(gpu, N, V, orbit):
    """Float densities with +inf in voxel (0, 0), rays marched one by one by
    segments (odd grid, odd view count, the orbit option): the rays past that
    voxel are infinite, and all others keep their values, which the
    exact-division march gives within two float roundings."""
    from virtualct_amd import _lib, default_geometry
    ops = _ops()
    geom = default_geometry(recon_size=N, pixel_cm=49.3 / N, n_views=V, n_channels=333, iso_channel=166.4)
    d = np.random.default_rng(N).uniform(0.1, 2.0, (3, N, N)).astype(np.float32)
    d[:, 0, 0] = np.inf
    out = []
    for exact in (0, 1):
        plan = ops.Plan(geom)
        plan.set_option(_lib.OPT_EXACT_TRACE, exact)
        plan.set_option(_lib.OPT_TRACE_ORBIT, orbit)
        pk, dt = ops.pack_densities(plan, _t(d, gpu))
        out.append(ops.trace_paths(plan, pk, dt, 3).cpu().numpy())
        plan.close()
    L, Le = out
    far = np.isfinite(Le)
    assert 0 < np.count_nonzero(~far) < Le.size // 4
    np.testing.assert_array_equal(L[~far], Le[~far])
    assert np.isfinite(L[far]).all()
    assert np.all(np.abs(L[far] - Le[far]) <= 2.0 ** -22 * np.abs(Le[far]) + 1e-9)


@pytest.mark.parametrize("N,fov,V,W,M,f32", [
    (128, 51.2, 48, 333, 6, False), (128, 51.2, 48, 333, 5, False), (128, 51.2, 50, 333, 8, False),
    (384, 51.2, 12, 609, 8, False), (384, 51.2, 14, 333, 6, True), (300, 48.0, 12, 333, 8, True),
    (384, 51.2, 13, 333, 6, False), (65, 26.0, 20, 333, 8, True)])
def test_stepwise_tracers_equal_exact_march(gpu, N, fov, V, W, M, f32):
    """Grids whose plane middles meet grid lines keep the marches that go step
    by step (orbits of 4 and 2 rays, odd view counts and odd grids ray by ray):
    the same counters as the exact-division march, path integrals within two
    float roundings, and the same bits for every workgroup size."""
    from virtualct_amd import _lib, default_geometry
    ops = _ops()
    D = fov / N
    middles = np.arange(int(N // 2 * D) + 3) / D + 0.5
    assert np.abs(middles - np.rint(middles)).min() < 1e-6
    geom = default_geometry(recon_size=N, pixel_cm=D, n_views=V, n_channels=W, iso_channel=W / 2.0 + 0.13)
    rng = np.random.default_rng(N + V)
    if f32:
        d = rng.uniform(0.0, 2.0, (M, N, N)).astype(np.float32)
        d[:, N // 2, 1] = -1.0
    else:
        d = rng.integers(0, 2000, (M, N, N)).astype(np.int16)
    out = []
    for exact, block in ((1, 0), (0, 64), (0, 128), (0, 256)):
        plan = ops.Plan(geom)
        plan.set_option(_lib.OPT_EXACT_TRACE, exact)
        plan.set_option(_lib.OPT_TRACE_BLOCK, block)
        pk, dt = ops.pack_densities(plan, _t(d, gpu))
        L, cnt = ops.trace_paths(plan, pk, dt, M, counts=True)
        out.append((L.cpu().numpy(), cnt.cpu().numpy()))
        plan.close()
    (Le, ce), (L, c) = out[0], out[1]
    assert ce.sum() > 0
    np.testing.assert_array_equal(c, ce)
    assert np.all(np.abs(L - Le) <= 2.0 ** -22 * np.abs(Le) + 1e-9)
    for Lb, cb in out[2:]:
        assert np.array_equal(Lb, L) and np.array_equal(cb, c)


@pytest.mark.parametrize("N,V,M,f32,orbit", [(129, 20, 6, False, 4), (129, 22, 8, True, 4), (128, 21, 6, False, 4),
                                              (128, 23, 3, True, 4), (130, 20, 8, False, 1), (130, 20, 7, True, 1)])
def test_lone_ray_segments_equal_exact_march(gpu, N, V, M, f32, orbit):
    """One ray per march by segments (odd grids and view counts, the orbit
    option), on grids without plane middles on grid lines: counters and path
    integrals as above."""
    from virtualct_amd import _lib, default_geometry
    ops = _ops()
    geom = default_geometry(recon_size=N, pixel_cm=49.3 / N, n_views=V, n_channels=333, iso_channel=166.63)
    rng = np.random.default_rng(N + V)
    d = rng.uniform(0.0, 2.0, (M, N, N)).astype(np.float32) if f32 else \
        rng.integers(0, 2000, (M, N, N)).astype(np.int16)
    out = []
    for exact in (0, 1):
        plan = ops.Plan(geom)
        plan.set_option(_lib.OPT_EXACT_TRACE, exact)
        plan.set_option(_lib.OPT_TRACE_ORBIT, orbit)
        pk, dt = ops.pack_densities(plan, _t(d, gpu))
        L, cnt = ops.trace_paths(plan, pk, dt, M, counts=True)
        out.append((L.cpu().numpy(), cnt.cpu().numpy()))
        plan.close()
    (L, c), (Le, ce) = out
    assert ce.sum() > 0
    np.testing.assert_array_equal(c, ce)
    assert np.all(np.abs(L - Le) <= 2.0 ** -22 * np.abs(Le) + 1e-9)


@pytest.mark.parametrize("V,M,f32", [(12, 6, False), (80, 8, True), (80, 1, False), (200, 8, False), (14, 2, True),
                                      (50, 6, False), (162, 6, True), (5, 8, False), (15, 6, True), (61, 3, False)])
def test_segment_workgroup_sizes_equal_exact_march(gpu, V, M, f32):
    """Workgroups of 16, 32 and 64 orbits (few to many views) of 4, 2 and 1
    rays, with last tiles that are not full and a channel whose ray passes
    through the isocentre along the grid lines, which is left to the second
    kernel in some views: the counters of the exact-division march and its path
    integrals within two float roundings."""
    from virtualct_amd import _lib, default_geometry
    ops = _ops()
    N, W = 130, 334
    geom = default_geometry(recon_size=N, pixel_cm=49.3 / N, n_views=V, n_channels=W, iso_channel=W / 2.0)
    rng = np.random.default_rng(V + M)
    d = rng.uniform(0.0, 2.0, (M, N, N)).astype(np.float32) if f32 else \
        rng.integers(0, 2000, (M, N, N)).astype(np.int16)
    out = []
    for exact in (0, 1):
        plan = ops.Plan(geom)
        plan.set_option(_lib.OPT_EXACT_TRACE, exact)
        pk, dt = ops.pack_densities(plan, _t(d, gpu))
        L, cnt = ops.trace_paths(plan, pk, dt, M, counts=True)
        out.append((L.cpu().numpy(), cnt.cpu().numpy()))
        plan.close()
    (L, c), (Le, ce) = out
    assert ce[:, W // 2].max() > 0
    np.testing.assert_array_equal(c, ce)
    assert np.all(np.abs(L - Le) <= 2.0 ** -22 * np.abs(Le) + 1e-9) and not np.any(L[..., M:])
