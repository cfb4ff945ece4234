"""Batched execution over cached system matrices against the plain
single-phantom path (which the other GPU tests pin to the reference)."""
from __future__ import annotations

import tempfile

import numpy as np
import pytest

from conftest import rel_l2, rel_max

pytestmark = pytest.mark.gpu


def _mods():
    from virtualct_amd import batch, decompose, ops
    return ops, batch, decompose


def _geom(N=512, pix=0.1, V=800):
    from virtualct_amd import default_geometry
    return default_geometry(recon_size=N, pixel_cm=pix, n_views=V)


def _spectra(dev, names=("120kV", "6MV"), M=6):
    import torch
    from virtualct_amd import spectra
    with tempfile.TemporaryDirectory() as d:
        tabs = [spectra.attenuation(spectra.synthetic_spectrum_file(n, d), M) for n in names]
    NE = max(a.shape[1] for a, _, _ in tabs)
    att = torch.zeros((len(tabs), M, NE))
    pdf = torch.zeros((len(tabs), NE))
    for s, (a, p, _) in enumerate(tabs):
        att[s, :, : a.shape[1]] = torch.from_numpy(a)
        pdf[s, : p.shape[0]] = torch.from_numpy(p)
    return att.to(dev), pdf.to(dev)


def _phantoms(B, N, pix, dev, seed=3000):
    import torch
    from virtualct_amd import phantoms
    return torch.stack([torch.from_numpy(phantoms.densities_f32(phantoms.body_phantom(seed + b, N=N, pix_cm=pix)))
                        for b in range(B)]).to(dev)


@pytest.fixture(scope="module")
def small_setup(gpu):
    ops, batch, _ = _mods()
    plan = ops.plan_for(_geom(128, 0.35, 160))
    sm = batch.SystemMatrix(plan, transpose=True)
    return plan, sm


def test_csr_replay_equals_tracer(gpu, small_setup):
    ops, batch, _ = _mods()
    plan, sm = small_setup
    import torch
    x = _phantoms(3, 128, 0.35, gpu)
    L = torch.empty((plan.V * plan.W, 3, 8), device=gpu)
    batch.batch_paths([(sm, batch.interleave(x), L, 3)], 6)
    Ln = batch.from_planes(L)
    for b in range(3):
        pk, dt = ops.pack_densities(plan, x[b].contiguous())
        ref = ops.trace_paths(plan, pk, dt, 6).reshape(-1, 8)
        assert rel_max(Ln[:, b].cpu().numpy(), ref.cpu().numpy()) < 2e-6


def test_csc_adjoint_equals_atomic_adjoint(gpu, small_setup):
    import torch
    ops, batch, _ = _mods()
    plan, sm = small_setup
    g = torch.Generator(device=gpu).manual_seed(5)
    wn = torch.zeros((plan.V * plan.W, 2, 8), device=gpu)
    wn[..., :6] = torch.randn((plan.V * plan.W, 2, 6), generator=g, device=gpu)
    w = batch.to_planes(wn)
    out = torch.empty((128 * 128, 2, 8), device=gpu)
    batch.batch_adjoint([(sm, w, out, 2)], 6)
    outn = batch.from_planes(out)
    for b in range(2):
        ref = ops.trace_adjoint(plan, wn[:, b].contiguous().view(plan.V, plan.W, 8), 6).reshape(-1, 8)
        assert rel_l2(outn[:, b].cpu().numpy(), ref.cpu().numpy()) < 1e-5
    # deterministic: a second launch gives identical bits
    out2 = torch.empty_like(out)
    batch.batch_adjoint([(sm, w, out2, 2)], 6)
    assert torch.equal(out, out2)


def test_batch_loss_matches_plain_ops(gpu, small_setup):
    import torch
    ops, batch, decompose = _mods()
    plan, sm = small_setup
    att, pdf = _spectra(gpu)
    x = _phantoms(2, 128, 0.35, gpu)
    tgt = torch.stack([ops.mbfpa_forward(plan, (x[b] * 0.97).contiguous(), att, pdf) for b in range(2)])
    L = torch.empty((plan.V * plan.W, 2, 8), device=gpu)
    batch.batch_paths([(sm, batch.interleave(x), L, 2)], 6)
    w, loss = batch.batch_loss(plan, L, 6, att, pdf, tgt)
    Ln, wn = batch.from_planes(L), batch.from_planes(w)
    for b in range(2):
        Lb = Ln[:, b].contiguous().view(plan.V, plan.W, 8)
        raw, stats, dIdL = ops.spectral_sum(plan, Lb, 6, att, pdf, want_dIdL=True)
        imax = pdf.sum(1).view(-1, 1, 1)
        r, dI = decompose.log_residual(raw, imax, tgt[b])
        assert loss[b].item() == pytest.approx(r.square().sum().item(), rel=1e-4)
        wref = (dIdL * dI.unsqueeze(-1)).sum(0).reshape(-1, 8)
        assert rel_l2(wn[:, b].cpu().numpy(), wref.cpu().numpy()) < 1e-4


def test_batched_solver_matches_plain_loop_and_graph(gpu, small_setup):
    import torch
    ops, batch, decompose = _mods()
    plan, sm = small_setup
    att, pdf = _spectra(gpu)
    truth = _phantoms(2, 128, 0.35, gpu, seed=3100)
    tgt = torch.stack([ops.mbfpa_forward(plan, truth[b].contiguous(), att, pdf, sigma=5.37e-5, stream_id=9 * b)
                       for b in range(2)])
    init = truth * 0.9
    plain = decompose.PlainLoop(plan, tgt, att, pdf, init)
    solver = batch.BatchedSolver(sm, tgt, att, pdf, init)
    for it in range(3):
        lp = plain.step()
        lb = solver.step().clone()
        assert rel_max(lb.cpu().numpy(), lp.cpu().numpy()) < 1e-3, it
    assert rel_l2(solver.densities().cpu().numpy(), plain.x.cpu().numpy()) < 1e-3
    # graph: replays interleaved with eager work must equal the eager solver
    eager = batch.BatchedSolver(sm, tgt, att, pdf, init)
    graphed = batch.BatchedSolver(sm, tgt, att, pdf, init)
    eager.step()
    graphed.capture()  # performs the first step itself
    for it in range(4):
        le = eager.step().clone()
        lg = graphed.step().clone()
        torch.cuda.synchronize()
        _ = (truth * 2).sum().item()  # unrelated eager work between replays
        assert torch.allclose(lg, le, rtol=1e-5, atol=0), it
        assert rel_l2(graphed.x.cpu().numpy(), eager.x.cpu().numpy()) < 1e-5, it
    # the loss falls
    assert graphed.loss.sum().item() < lp.sum().item() * 5


def test_batch_spectral_zero_tail_bins(gpu, small_setup):
    """Spectra of unequal length share one zero-padded table; the kernels stop
    at each spectrum's last nonzero probability.  The padded 3-spectrum sum
    equals each spectrum's own unpadded sum bit for bit (an interior zero bin
    and a zeroed tail included), and the loss and its weights do not change
    when the table is padded further.  700 bins take the per-spectrum form of
    the sum (tables beyond 64 KB of LDS) with the same bits."""
    import torch
    ops, batch, _ = _mods()
    plan, sm = small_setup
    att, pdf = _spectra(gpu, ("80kV", "120kV", "6MV"))
    pdf[2, 7] = 0.0          # interior zero bin: summed, contributes +0
    pdf[2, -3:] = 0.0        # tail zeros with nonzero attenuation
    x = _phantoms(3, 128, 0.35, gpu)
    L = torch.empty((plan.V * plan.W, 3, 8), device=gpu)
    batch.batch_paths([(sm, batch.interleave(x), L, 3)], 6)
    raw, stats = batch.batch_spectral(plan, L, 6, att, pdf)
    for s in range(3):
        ne = int(torch.nonzero(pdf[s]).max().item()) + 1
        a1 = att[s:s + 1, :, :ne].contiguous()
        p1 = pdf[s:s + 1, :ne].contiguous()
        r1, s1 = batch.batch_spectral(plan, L, 6, a1, p1)
        assert torch.equal(raw[:, s], r1[:, 0]), s
        assert torch.equal(stats[:, s], s1[:, 0]), s
    # padded to 700 bins the tables exceed 64 KB of LDS and the sum takes one
    # (phantom, spectrum) per block: the same bits
    NE = att.shape[2]
    attw = torch.zeros((3, 6, 700), device=gpu)
    pdfw = torch.zeros((3, 700), device=gpu)
    attw[:, :, :NE], pdfw[:, :NE] = att, pdf
    rw, sw = batch.batch_spectral(plan, L, 6, attw, pdfw)
    assert torch.equal(raw, rw) and torch.equal(stats, sw)
    tgt = (raw * 0.97 + 1e-3).contiguous()
    w0, l0 = batch.batch_loss(plan, L, 6, att, pdf, tgt)
    att2 = torch.zeros((3, 6, NE + 37), device=gpu)
    pdf2 = torch.zeros((3, NE + 37), device=gpu)
    att2[:, :, :NE], pdf2[:, :NE] = att, pdf
    w1, l1 = batch.batch_loss(plan, L, 6, att2, pdf2, tgt)
    assert torch.equal(w0, w1)
    assert torch.allclose(l0, l1, rtol=1e-6)  # float atomics: order may differ


def test_batch_forward_fbp_uneven_sizes(gpu):
    import torch
    ops, batch, _ = _mods()
    att, pdf = _spectra(gpu, ("80kV", "120kV", "6MV"))
    sizes = [(64, 50.0 / 64), (96, 50.0 / 96)]
    groups = []
    for k, (N, pix) in enumerate(sizes):
        from virtualct_amd import phantoms
        ph = torch.stack([torch.from_numpy(phantoms.body_phantom(4000 + 10 * k + b, N=N, pix_cm=pix))
                          for b in range(2)]).to(gpu)
        groups.append((_geom(N, pix, 160), ph))
    # noise-free: sinograms and images against the plain calls
    run = batch.BatchForwardFBP(groups, att, pdf, sigma=0.0)
    sinos, imgs = run.run()
    for k, (geom, ph) in enumerate(groups):
        plan = ops.plan_for(geom)
        for b in range(2):
            ref = ops.mbfpa_forward(plan, ph[b].contiguous(), att, pdf)
            assert rel_max(sinos[k][3 * b: 3 * b + 3].cpu().numpy(), ref.cpu().numpy()) < 1e-5
            img = ops.fbp(plan, ref)
            assert rel_max(imgs[k][3 * b: 3 * b + 3].cpu().numpy(), img.cpu().numpy()) < 1e-5
    # noisy: the same Philox streams as the plain calls
    run = batch.BatchForwardFBP(groups, att, pdf, sigma=5.37e-5, seed=77)
    sinos, imgs = run.run()
    sid = 0
    for k, (geom, ph) in enumerate(groups):
        plan = ops.plan_for(geom)
        for b in range(2):
            ref = ops.mbfpa_forward(plan, ph[b].contiguous(), att, pdf, sigma=5.37e-5, seed=77, stream_id=sid)
            sid += 3
            assert rel_max(sinos[k][3 * b: 3 * b + 3].cpu().numpy(), ref.cpu().numpy()) < 1e-5
    # graph replays reproduce the eager run
    eager_imgs = [i.clone() for i in imgs]
    run.capture()
    for _ in range(3):
        s2, i2 = run.replay()
        torch.cuda.synchronize()
        _ = sum(float(i.sum()) for i in eager_imgs)  # eager work between replays
        for a, b in zip(i2, eager_imgs):
            assert torch.allclose(a, b, rtol=1e-5, atol=1e-7)


def test_single_phantom_split_gather_equals_lane_gather(gpu, small_setup):
    """lanes_per_row 1 (rows split over 16 lanes) gives the FP64 sums of the
    one-lane-per-phantom gather, forward and adjoint."""
    import torch
    ops, batch, _ = _mods()
    plan, sm = small_setup
    x = batch.interleave(_phantoms(1, 128, 0.35, gpu))
    L1 = torch.empty((plan.V * plan.W, 1, 8), device=gpu)
    L8 = torch.empty_like(L1)
    batch.batch_paths([(sm, x, L1, 1)], 6, 1)
    batch.batch_paths([(sm, x, L8, 1)], 6, 8)
    assert rel_max(L1.cpu().numpy(), L8.cpu().numpy()) < 1e-6
    g = torch.Generator(device=gpu).manual_seed(8)
    w = torch.zeros((plan.V * plan.W, 1, 8), device=gpu)
    w[..., :6] = torch.randn((plan.V * plan.W, 1, 6), generator=g, device=gpu)
    o1 = torch.empty((128 * 128, 1, 8), device=gpu)
    o8 = torch.empty_like(o1)
    batch.batch_adjoint([(sm, w, o1, 1)], 6, 1)
    batch.batch_adjoint([(sm, w, o8, 1)], 6, 8)
    assert rel_l2(o1.cpu().numpy(), o8.cpu().numpy()) < 1e-6
    assert torch.all(o1[..., 6:] == 0)
    with pytest.raises(RuntimeError):
        batch.batch_paths([(sm, batch.interleave(_phantoms(2, 128, 0.35, gpu)),
                            torch.empty((plan.V * plan.W, 2, 8), device=gpu), 2)], 6, 1)


def test_gather_applies_xfactor(gpu):
    """The gathers return path sums in the tracer's units (divided by xfactor)."""
    import torch
    ops, batch, _ = _mods()
    g = _geom(64, 0.7, 80)
    g.xfactor = 4.0
    plan = ops.Plan(g)
    sm = batch.SystemMatrix(plan)
    x = _phantoms(1, 64, 0.7, gpu)
    L = torch.empty((plan.V * plan.W, 1, 8), device=gpu)
    batch.batch_paths([(sm, batch.interleave(x), L, 1)], 6)
    pk, dt = ops.pack_densities(plan, x[0].contiguous())
    ref = ops.trace_paths(plan, pk, dt, 6).reshape(-1, 8)
    assert rel_max(L[:, 0].cpu().numpy(), ref.cpu().numpy()) < 2e-6


@pytest.fixture(scope="module")
def blocked_setup(gpu, small_setup):
    ops, batch, _ = _mods()
    plan, sm = small_setup
    smb = batch.SystemMatrix(plan, transpose=True, blocked=True)
    return plan, sm, smb


def _random_weights(rays, B, dev, seed):
    import torch
    from virtualct_amd import batch
    g = torch.Generator(device=dev).manual_seed(seed)
    w = torch.zeros((rays, B, 8), device=dev)
    w[..., :6] = torch.randn((rays, B, 6), generator=g, device=dev)
    return batch.to_planes(w)


@pytest.mark.parametrize("B", [1, 3, 16])
def test_blocked_gathers_equal_direct(gpu, blocked_setup, B):
    """The blocked two-stage gathers (64x64 image tiles; 50-view blocks x
    tiles for the adjoint; float partial sums) give the direct gathers' sums
    in both directions, with identical bits from launch to launch."""
    import torch
    ops, batch, _ = _mods()
    plan, sm, smb = blocked_setup
    assert smb.segments == sm.segments and smb.bytes > sm.bytes
    rays = plan.V * plan.W
    x = batch.interleave(_phantoms(B, 128, 0.35, gpu, seed=3300))
    Ld, Lb, Lb2 = (torch.empty((rays, B, 8), device=gpu) for _ in range(3))
    batch.batch_paths([(sm, x, Ld, B)], 6)
    batch.batch_paths([(smb, x, Lb, B)], 6)
    batch.batch_paths([(smb, x, Lb2, B)], 6)
    assert rel_max(Lb.cpu().numpy(), Ld.cpu().numpy()) < 1e-6
    assert torch.equal(Lb, Lb2)
    w = _random_weights(rays, B, gpu, 11)
    od, ob, ob2 = (torch.empty((128 * 128, B, 8), device=gpu) for _ in range(3))
    batch.batch_adjoint([(sm, w, od, B)], 6)
    batch.batch_adjoint([(smb, w, ob, B)], 6)
    batch.batch_adjoint([(smb, w, ob2, B)], 6)
    assert rel_l2(ob.cpu().numpy(), od.cpu().numpy()) < 1e-6
    assert torch.equal(ob, ob2)
    assert torch.all(batch.from_planes(ob)[..., 6:] == 0)


def test_blocked_gathers_mixed_groups(gpu, blocked_setup):
    """One launch holding two blocked groups on the same matrix (separate
    workspaces), a blocked group of another size and a direct group."""
    import torch
    ops, batch, _ = _mods()
    plan, sm, smb = blocked_setup
    plan2 = ops.plan_for(_geom(96, 0.45, 160))
    sm2 = batch.SystemMatrix(plan2, transpose=True, blocked=True)
    sm2d = batch.SystemMatrix(plan2, transpose=True)
    rays = plan.V * plan.W
    xa = batch.interleave(_phantoms(2, 128, 0.35, gpu, seed=3400))
    xb = batch.interleave(_phantoms(2, 128, 0.35, gpu, seed=3500))
    xc = batch.interleave(_phantoms(3, 96, 0.45, gpu, seed=3600))
    outs = [torch.empty((rays, 2, 8), device=gpu), torch.empty((rays, 2, 8), device=gpu),
            torch.empty((plan2.V * plan2.W, 3, 8), device=gpu), torch.empty((rays, 2, 8), device=gpu)]
    batch.batch_paths([(smb, xa, outs[0], 2), (smb, xb, outs[1], 2), (sm2, xc, outs[2], 3), (sm, xb, outs[3], 2)], 6)
    for (m, x, B), o in zip([(sm, xa, 2), (sm, xb, 2), (sm2d, xc, 3), (sm, xb, 2)], outs):
        ref = torch.empty_like(o)
        batch.batch_paths([(m, x, ref, B)], 6)
        assert rel_max(o.cpu().numpy(), ref.cpu().numpy()) < 1e-6
    wa, wc = _random_weights(rays, 2, gpu, 12), _random_weights(plan2.V * plan2.W, 3, gpu, 13)
    ga, gc = torch.empty((128 * 128, 2, 8), device=gpu), torch.empty((96 * 96, 3, 8), device=gpu)
    batch.batch_adjoint([(smb, wa, ga, 2), (sm2, wc, gc, 3)], 6)
    ra, rc = torch.empty_like(ga), torch.empty_like(gc)
    batch.batch_adjoint([(sm, wa, ra, 2)], 6)
    batch.batch_adjoint([(sm2d, wc, rc, 3)], 6)
    assert rel_l2(ga.cpu().numpy(), ra.cpu().numpy()) < 1e-6
    assert rel_l2(gc.cpu().numpy(), rc.cpu().numpy()) < 1e-6


def test_blocked_gathers_full_geometry(gpu):
    """512^2, 800 views x 609 channels (8x8 tiles, 16 view blocks)."""
    import torch
    ops, batch, _ = _mods()
    plan = ops.plan_for(_geom())
    sm = plan.system_matrix()
    smb = batch.SystemMatrix(plan, transpose=True, blocked=True)
    rays, B = plan.V * plan.W, 2
    x = batch.interleave(_phantoms(B, 512, 0.1, gpu, seed=3700))
    Ld, Lb = torch.empty((rays, B, 8), device=gpu), torch.empty((rays, B, 8), device=gpu)
    batch.batch_paths([(sm, x, Ld, B)], 6)
    batch.batch_paths([(smb, x, Lb, B)], 6)
    assert rel_max(Lb.cpu().numpy(), Ld.cpu().numpy()) < 1e-6
    w = _random_weights(rays, B, gpu, 14)
    od, ob = torch.empty((512 * 512, B, 8), device=gpu), torch.empty((512 * 512, B, 8), device=gpu)
    batch.batch_adjoint([(sm, w, od, B)], 6)
    batch.batch_adjoint([(smb, w, ob, B)], 6)
    assert rel_l2(ob.cpu().numpy(), od.cpu().numpy()) < 1e-6
    smb.close()


def test_blocked_solver_graph_replay(gpu, blocked_setup):
    """The solver on the blocked matrix follows the direct one, and its graph
    replays (workspace inside the graph) equal its eager steps."""
    import torch
    ops, batch, _ = _mods()
    plan, sm, smb = blocked_setup
    att, pdf = _spectra(gpu)
    truth = _phantoms(2, 128, 0.35, gpu, seed=3800)
    tgt = torch.stack([ops.mbfpa_forward(plan, truth[b].contiguous(), att, pdf, sigma=5.37e-5, stream_id=5 * b)
                       for b in range(2)])
    init = truth * 0.9
    direct = batch.BatchedSolver(sm, tgt, att, pdf, init)
    eager = batch.BatchedSolver(smb, tgt, att, pdf, init)
    graphed = batch.BatchedSolver(smb, tgt, att, pdf, init)
    direct.step()
    eager.step()
    graphed.capture()
    for it in range(4):
        ld = direct.step().clone()
        le = eager.step().clone()
        lg = graphed.step().clone()
        torch.cuda.synchronize()
        _ = (truth * 2).sum().item()  # unrelated eager work between replays
        # the loss is summed with atomics: equal to rounding, not in bits
        assert torch.allclose(lg, le, rtol=1e-6, atol=0), it
        assert rel_l2(graphed.x.cpu().numpy(), eager.x.cpu().numpy()) < 1e-6, it
        assert rel_max(le.cpu().numpy(), ld.cpu().numpy()) < 1e-4, it


@pytest.mark.parametrize("lanes", [8, 16, 32, 64])
def test_gather_every_lane_width(gpu, blocked_setup, lanes):
    """Every lanes-per-row variant (entry broadcast by permute for 8 and 32,
    DPP row broadcast for 16, lane read for 64) gives the same FP64 sums as
    another lane width, bit for bit, in both directions; the blocked form
    agrees to float rounding of its partial sums."""
    import torch
    ops, batch, _ = _mods()
    plan, sm, smb = blocked_setup
    # fewer phantoms than lanes (idle lanes still take part in the
    # broadcasts), checked against another lane width
    B, ref_lanes = {8: (5, 16), 16: (11, 32), 32: (19, 64), 64: (19, 32)}[lanes]
    rays = plan.V * plan.W
    x = batch.interleave(_phantoms(B, 128, 0.35, gpu, seed=3900))
    w = _random_weights(rays, B, gpu, 15)
    ref_L, ref_g = torch.empty((rays, B, 8), device=gpu), torch.empty((128 * 128, B, 8), device=gpu)
    batch.batch_paths([(sm, x, ref_L, B)], 6, ref_lanes)
    batch.batch_adjoint([(sm, w, ref_g, B)], 6, ref_lanes)
    L, g = torch.empty_like(ref_L), torch.empty_like(ref_g)
    batch.batch_paths([(sm, x, L, B)], 6, lanes)
    batch.batch_adjoint([(sm, w, g, B)], 6, lanes)
    assert torch.equal(L, ref_L) and torch.equal(g, ref_g)
    batch.batch_paths([(smb, x, L, B)], 6, lanes)
    batch.batch_adjoint([(smb, w, g, B)], 6, lanes)
    assert rel_max(L.cpu().numpy(), ref_L.cpu().numpy()) < 1e-6
    assert rel_l2(g.cpu().numpy(), ref_g.cpu().numpy()) < 1e-6


@pytest.mark.parametrize("B", [1, 3, 16])
def test_bb_step_matches_fp64_formula(gpu, B):
    """vct_batch_bb_step: the step length from FP64 sums of s.y and s.s
    (s = x - x_prev, y = g - g_prev, differences in float), then the
    projected update with that step; the first step keeps alpha."""
    import ctypes as C
    import torch
    from virtualct_amd import _lib
    from virtualct_amd._lib import call
    from virtualct_amd import batch
    n = 4099
    gen = torch.Generator(device=gpu).manual_seed(40 + B)
    nat = [torch.zeros((n, B, 8), device=gpu) for _ in range(4)]
    for t in nat:
        t[..., :6] = torch.rand((n, B, 6), generator=gen, device=gpu) - 0.3
    nat[0].clamp_(min=0)
    nat[1].clamp_(min=0)
    x, xp, g, gp = (batch.to_planes(t) for t in nat)
    alpha = torch.linspace(1e-3, 2e-3, B, device=gpu)
    work = torch.empty(int(_lib.lib().vct_batch_bb_workspace(B)) // 8, dtype=torch.float64, device=gpu)
    P = lambda t: C.c_void_p(t.data_ptr())
    s_ = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for first in (1, 0):
        x2, xp2, gp2, al2 = x.clone(), xp.clone(), gp.clone(), alpha.clone()
        call("vct_batch_bb_step", P(x2), P(xp2), P(gp2), P(g), P(al2), n, B, first, P(work), s_)
        torch.cuda.synchronize()
        if first:
            assert torch.equal(al2, alpha)
        else:
            s = (nat[0] - nat[1]).double()
            y = (nat[2] - nat[3]).double()
            sy, ss = (s * y).sum(dim=(0, 2)), (s * s).sum(dim=(0, 2))
            bb = torch.where(sy > 0, ss / sy.clamp_min(1e-30), alpha.double() * 2)
            a_ref = bb.clamp(1e-8, 1e2).float()
            assert torch.allclose(al2, a_ref, rtol=2e-7, atol=0)
        assert torch.equal(xp2, x) and torch.equal(gp2, g)
        ref = (nat[0] - al2.view(1, -1, 1) * nat[2]).clamp_min(0.0)
        assert torch.equal(batch.from_planes(x2), ref)


@pytest.mark.parametrize("N,pix,B,M", [(128, 0.35, 3, 6), (96, 0.45, 16, 5), (160, 0.28, 2, 8), (128, 0.35, 1, 3),
                                     (64, 0.7, 64, 2), (65, 0.69, 5, 1)])
def test_tile_stage1_equals_blocked_stage1(gpu, N, pix, B, M):
    """The forward stage 1 over the tile-resident form (the tile of each
    phantom in LDS, runs sorted by length in 64-run slices; one tile at 64^2,
    partial edge tiles at 65^2, 96^2 and 160^2) gives the bits of the blocked
    stage 1 read through L2, for 1..64 phantoms and 1..8 materials."""
    import torch
    ops, batch, _ = _mods()
    plan = ops.plan_for(_geom(N, pix, 160))
    smt = batch.SystemMatrix(plan, transpose=True, blocked=True)
    smn = batch.SystemMatrix(plan, transpose=True, blocked=True, tiles=False)
    assert smt.bytes > smn.bytes
    rays = plan.V * plan.W
    dens = _phantoms(B, N, pix, gpu, seed=4000 + N)
    if M > 6:
        dens = torch.cat([dens, dens[:, : M - 6] * 0.5], dim=1)
    x = batch.interleave(dens[:, :M].contiguous())
    Lt, Ln = torch.empty((rays, B, 8), device=gpu), torch.empty((rays, B, 8), device=gpu)
    smt.workspace(B, 0).zero_()
    smn.workspace(B, 0).zero_()
    batch.batch_paths([(smt, x, Lt, B)], M)
    batch.batch_paths([(smn, x, Ln, B)], M)
    assert torch.equal(Lt, Ln)
    n = smn.workspace(B, 0).numel()  # the partial sums (the LDS forms' workspace adds a weight copy)
    assert torch.equal(smt.workspace(B, 0)[:n], smn.workspace(B, 0))
    smt.close()
    smn.close()


@pytest.mark.parametrize("N,pix,B,M,built", [(128, 0.1, 3, 6, True), (96, 0.2, 16, 5, True), (160, 0.1, 2, 8, True),
                                           (65, 0.15, 5, 1, True), (64, 0.1, 64, 2, True), (128, 0.35, 4, 6, False)])
def test_adjoint_lds_stage1_equals_blocked_stage1(gpu, N, pix, B, M, built):
    """The adjoint stage 1 over its LDS-resident form (blocks of 50 views x
    one part of a 64x64 tile, the weights of the rays that cross the part in
    LDS, runs sorted by length in 64-run slices) gives the bits of the
    blocked stage 1 read through L2, for 2..64 phantoms and 1..8 materials,
    partial edge tiles at 65^2 and 160^2, tiles split in 1..16 parts (96^2 x
    0.2 cm).  At 128^2 x 0.35 cm a 16x16 cell sees more than 3328 rays of a
    view block, so the form is not built and the L2 path runs."""
    import torch
    ops, batch, _ = _mods()
    plan = ops.plan_for(_geom(N, pix, 160))
    smt = batch.SystemMatrix(plan, transpose=True, blocked=True)
    smn = batch.SystemMatrix(plan, transpose=True, blocked=True, tiles=False)
    smf = batch.SystemMatrix(plan, transpose=False, blocked=True)
    smfn = batch.SystemMatrix(plan, transpose=False, blocked=True, tiles=False)
    # the adjoint form adds to the bytes of the forward one when built
    assert (smt.bytes - smn.bytes > smf.bytes - smfn.bytes) == built
    smf.close()
    smfn.close()
    rays = plan.V * plan.W
    g = torch.Generator(device=gpu).manual_seed(4100 + N)
    w = torch.zeros((rays, B, 8), device=gpu)
    w[..., :M] = torch.randn((rays, B, M), generator=g, device=gpu)
    w = batch.to_planes(w)
    gt, gn = torch.empty((N * N, B, 8), device=gpu), torch.empty((N * N, B, 8), device=gpu)
    smt.workspace(B, 0).zero_()
    smn.workspace(B, 0).zero_()
    batch.batch_adjoint([(smt, w, gt, B)], M)
    batch.batch_adjoint([(smn, w, gn, B)], M)
    assert torch.equal(gt, gn)
    n = smn.workspace(B, 0).numel()  # the partial sums (then the phantom-major weight copy)
    assert torch.equal(smt.workspace(B, 0)[:n], smn.workspace(B, 0))
    smt.close()
    smn.close()


def test_sysmat_rows_equal_reference_segment_lists(gpu, golden):
    """The cached rows of the 56 rays whose segment caches the reference
    dumped at the full 512^2 / 800 x 609 geometry (tests/golden/ref_segments.npz:
    reprojection_vnum / reprojection_systemMatrixfloat per segment counter,
    zero where a counter's segment is outside the image): the voxel sequence
    bit for bit and every length within one float ulp."""
    ops, batch, _ = _mods()
    plan = ops.plan_for(_geom())
    sm = batch.SystemMatrix(plan, transpose=False)
    s = golden.npz("ref_segments.npz")
    total = 0
    for i, ray in enumerate(s["rays"]):
        n = int(s["count"][i])
        vox, ln = s["vox"][i, :n], s["length"][i, :n]
        keep = (vox != 0) | (ln != 0)
        gv, gl = sm.row(int(ray))
        np.testing.assert_array_equal(gv.astype(np.int64), vox[keep].astype(np.int64), err_msg=f"ray {ray}")
        ulp = np.spacing(np.abs(ln[keep]))
        assert np.all(np.abs(gl.astype(np.float64) - ln[keep]) <= ulp), f"ray {ray}"
        total += gv.size
    assert total > 10000
    sm.close()


@pytest.mark.parametrize("exact,wide", [(False, False), (True, False), (False, True)])
def test_interleaved_grouped_backprojection_equals_plain(gpu, exact, wide):
    """Sinograms interleaved in slices of k (4, 8, 12, 16; the last slice
    zero-padded) give the grouped backprojection's images bit for bit, with
    float-weight and exact terms, at 256^2 and 768^2 over 50/N cm plus an odd
    size, and with a 128^2 x 0.6 cm group whose fan needs the wide-angle
    arctangent (which the whole launch then takes); the interleaved array is
    the permuted stack."""
    import torch
    ops, batch, _ = _mods()
    from virtualct_amd import _lib, default_geometry
    gen = torch.Generator(device=gpu).manual_seed(13)
    sizes, Ss = (256, 768, 97), (5, 9, 3)
    pixs = [50.0 / N for N in sizes]
    if wide:
        sizes, Ss, pixs = sizes + (128,), Ss + (4,), pixs + [0.6]
    plans = [ops.plan_for(default_geometry(recon_size=N, pixel_cm=pix, n_views=120)) for N, pix in zip(sizes, pixs)]
    if exact:
        for p in plans:
            p.set_option(_lib.OPT_EXACT_BACKPROJECT, 1)
    try:
        fls = [torch.randn((S, p.V, p.W), generator=gen, device=gpu) * 100 for p, S in zip(plans, Ss)]
        for k in batch.IL_WIDTHS:
            ils = [batch.interleave_sinograms(p, f, k) for p, f in zip(plans, fls)]
            for p, f, il in zip(plans, fls, ils):
                n = il.shape[0] * k
                ref = torch.zeros((n, p.V, p.W), device=gpu)
                ref[: f.shape[0]] = f
                assert torch.equal(il, ref.view(il.shape[0], k, p.V, p.W).permute(0, 2, 3, 1)), (p.N, k)
            imgs = [torch.full((f.shape[0], p.N, p.N), float("nan"), device=gpu) for p, f in zip(plans, fls)]
            batch.backproject_groups_il([(p, il, f.shape[0], im) for p, f, il, im in zip(plans, fls, ils, imgs)], k)
            ref = [torch.full_like(im, float("nan")) for im in imgs]
            batch.backproject_groups(list(zip(plans, fls, ref)), k)
            for p, im, r in zip(plans, imgs, ref):
                assert torch.equal(im, r), (p.N, k, exact)
    finally:
        if exact:
            for p in plans:
                p.set_option(_lib.OPT_EXACT_BACKPROJECT, 0)


def test_grouped_spectral_and_backprojection_equal_per_group_calls(gpu):
    """One launch over several size groups (spectral sums of all groups, then
    the backprojections of all groups) gives each group exactly what its own
    calls give, bit for bit, for several sinograms per lane."""
    import torch
    ops, batch, _ = _mods()
    from virtualct_amd import default_geometry
    gen = torch.Generator(device=gpu).manual_seed(12)
    sizes, Bs = (64, 96, 130), (2, 3, 1)
    plans = [ops.plan_for(default_geometry(recon_size=N, pixel_cm=50.0 / N, n_views=160)) for N in sizes]
    S, M, NE = 2, 6, 7
    att = torch.rand((S, M, NE), generator=gen, device=gpu) * 0.3
    pdf = torch.rand((S, NE), generator=gen, device=gpu)
    Ls = [torch.rand((p.V * p.W, B, 8), generator=gen, device=gpu) * 3 for p, B in zip(plans, Bs)]
    raw, stats = batch.batch_spectral_groups(plans[0], Ls, Bs, M, att, pdf)
    off = 0
    for p, L, B in zip(plans, Ls, Bs):
        r1, s1 = batch.batch_spectral(p, L, M, att, pdf)
        assert torch.equal(raw[off:off + B], r1) and torch.equal(stats[off:off + B], s1)
        off += B
    fls = [torch.randn((B * S, p.V, p.W), generator=gen, device=gpu) * 100 for p, B in zip(plans, Bs)]
    for k in (2, 5, 16):
        imgs = [torch.full((f.shape[0], p.N, p.N), float("nan"), device=gpu) for p, f in zip(plans, fls)]
        batch.backproject_groups(list(zip(plans, fls, imgs)), k)
        for p, f, im in zip(plans, fls, imgs):
            assert torch.equal(im, ops.backproject(p, f)), (p.N, k)


@pytest.mark.parametrize("V,B,S,NE,M", [(2, 1, 7, 40, 6), (8, 37, 7, 17, 8), (3, 150, 2, 33, 3), (81, 1, 5, 120, 1)])
def test_batch_spectral_shared_spectra_equal_single_calls(gpu, V, B, S, NE, M):
    """Few rays: the spectra of a phantom are shared by several workgroups (all
    of them, an uneven part), each summed as in a call of one phantom, so the
    values and the statistics are the same bits."""
    import torch
    ops, batch, _ = _mods()
    from virtualct_amd import default_geometry
    plan = ops.plan_for(default_geometry(recon_size=64, pixel_cm=0.7, n_views=V))
    g = torch.Generator(device=gpu).manual_seed(V + B)
    L = torch.rand((V * 609, B, 8), generator=g, device=gpu) * 10
    L[..., M:] = 0
    att = torch.rand((S, M, NE), generator=g, device=gpu) * 0.2
    pdf = torch.rand((S, NE), generator=g, device=gpu) / NE
    raw, stats = batch.batch_spectral(plan, batch.to_planes(L), M, att, pdf)
    for b in {0, B // 2, B - 1}:
        r1, s1, _ = ops.spectral_sum(plan, L[:, b].contiguous().view(V, 609, 8), M, att, pdf)
        assert torch.equal(raw[b], r1) and torch.equal(stats[b], s1)
