"""Learned range surrogate on the GPU, checked against the float64 oracle
(oracle/surrogate.py): the matrix-core GEMM, features, loss and gradient,
the Adam step, training, and checked inference against the exact marcher."""
import math

import numpy as np
import pytest

import range_libc_amd as rl
from oracle import oracle as O
from oracle import surrogate as S
from range_libc_amd import workloads as W
from tests.conftest import assert_bits_equal

pytestmark = pytest.mark.gpu


def _torch():
    import torch

    assert torch.cuda.is_available(), "GPU test needs a device"
    return torch


def _rand_bf16(rng, shape, scale=2.0):
    return S.bf16_bits(rng.uniform(-scale, scale, shape).astype(np.float32))


@pytest.mark.parametrize("mnk", [(16, 16, 16), (64, 64, 32), (100, 70, 50), (1, 1, 1), (300, 257, 1000),
                                 (64, 256, 4096), (2, 256, 3000)])
def test_gemm_bf16_matches_cpu(ctx, mnk):
    M, N, K = mnk
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    a, b = _rand_bf16(rng, (M, K)), _rand_bf16(rng, (K, N))
    c = rl._lib.debug_gemm_bf16(ctx, a, b)
    A, B = S.bf16_to_f64(a), S.bf16_to_f64(b)
    ref = A @ B
    bound = (K * 2.0 ** -23 + 1e-7) * (np.abs(A) @ np.abs(B)) + 1e-30
    err = np.abs(c - ref)
    assert np.all(err <= bound), f"max err {err.max()} at {np.unravel_index(np.argmax(err / bound), err.shape)}"


@pytest.mark.parametrize("mnk", [(128, 128, 32), (300, 256, 64), (1000, 256, 256), (1, 128, 32), (257, 384, 96),
                                 (64, 2, 256), (100, 130, 40)])
def test_gemm_bf16_nt_matches_cpu(ctx, mnk):
    """The forward-layer layout: the 128 x 128 tile kernel (K % 32 == 0, N % 128 == 0)
    and the general kernel for the other shapes."""
    M, N, K = mnk
    rng = np.random.default_rng(M + 11 * N + 7 * K)
    a, bt = _rand_bf16(rng, (M, K)), _rand_bf16(rng, (N, K))
    c = rl._lib.debug_gemm_bf16_nt(ctx, a, bt)
    A, Bt = S.bf16_to_f64(a), S.bf16_to_f64(bt)
    ref = A @ Bt.T
    bound = (K * 2.0 ** -23 + 1e-7) * (np.abs(A) @ np.abs(Bt).T) + 1e-30
    err = np.abs(c - ref)
    assert np.all(err <= bound), f"max err {err.max()} at {np.unravel_index(np.argmax(err / bound), err.shape)}"


def _map_and_rays(n, seed=0, size=256):
    img = W.rect_disk_map(size, seed=seed)
    g = W.grid_poses(img, n, seed=seed + 1)
    h = g[:, 2]
    rays = np.stack([g[:, 0], g[:, 1], np.sin(h), np.cos(h)], axis=1).astype(np.float32)
    return img, g, rays


def _targets_for_both_regimes(p, x, R, seed):
    """Targets around the network's current prediction so the batch exercises
    both Huber regimes and both sides of the pinball loss."""
    _, o = S.forward(p, x, emulate_bf16=True)
    rng = np.random.default_rng(seed)
    return (R * o[:, 0] + rng.choice([-9.0, -0.4, 0.3, 2.0, 15.0], o.shape[0])).astype(np.float32)


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def _cos(a, b):
    return float(a @ b / max(np.linalg.norm(a) * np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("n", [3000, 64, 777])
def test_features_loss_gradient_vs_cpu(ctx, n):
    R = 120.0
    img, g, rays = _map_and_rays(n)
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    sg = rl.Surrogate(dm, seed=3)
    p, freq = sg.params()
    p = p.copy()
    p[S.B4 + 1] = 1.0  # bound e^1 cells: both sides of the pinball loss occur
    sg.set_params(p)
    # features: bf16 of the float64 features, up to fp32 phase rounding
    _, _, feat = sg.gradient(R, rays, np.zeros(n, np.float32))
    x = S.bf16_to_f64(feat)
    want = S.features(rays, freq, img.shape[1], img.shape[0])
    assert np.max(np.abs(x - want)) <= 2.0 ** -8 + 1e-4
    t = _targets_for_both_regimes(p, x, R, n)
    loss, grad, feat2 = sg.gradient(R, rays, t)
    assert np.array_equal(feat, feat2)
    l16, g16, _ = S.loss_and_grad(p, x, t, R, emulate_bf16=True)
    l64, g64, _ = S.loss_and_grad(p, x, t, R)
    assert abs(loss - l16) <= 1e-4 * abs(l16)
    report = []
    for k, (w, b, o, i) in enumerate(S.LAYERS):
        for name, sl in ((f"W{k + 1}", slice(w, w + o * i)), (f"b{k + 1}", slice(b, b + o))):
            r16, c16 = _rel(grad[sl], g16[sl]), _cos(grad[sl], g16[sl])
            r64, c64 = _rel(grad[sl], g64[sl]), _cos(grad[sl], g64[sl])
            report.append(f"{name}: rel {r16:.2e} cos {c16:.6f} | fp64 rel {r64:.2e} cos {c64:.5f}")
            assert r16 <= 1e-2 and c16 >= 0.9999, report[-1]
            assert c64 >= 0.99, report[-1]
    print("\n".join(report))


def test_fused_bf16_conversion_exhaustive(ctx):
    """The fused kernel's hardware bf16 conversion equals the per-layer
    kernels' software rounding on every float bit pattern."""
    assert rl._lib.debug_bf16_check(ctx) == 0


@pytest.mark.parametrize("n", [1, 63, 64, 777, 3000])
def test_fused_forward_equals_layers_and_cpu(ctx, n):
    """forward() (one fused kernel: features, hidden layers and heads with the
    activations in LDS) is bitwise the per-layer kernels' output, including
    ragged last tiles, and matches the float64 network on the same features."""
    img, g, rays = _map_and_rays(n, seed=5)
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    sg = rl.Surrogate(dm, seed=9)
    p, _ = sg.params()
    p = p.copy()
    rng = np.random.default_rng(n)
    p[S.B4:S.B4 + 2] = rng.uniform(-1.0, 1.0, 2)  # non-zero head biases
    sg.set_params(p)
    fused = sg.forward(rays)
    layers = sg.forward_layers(rays)
    assert_bits_equal(fused, layers, "fused vs per-layer forward")
    _, _, feat = sg.gradient(100.0, rays, np.zeros(n, np.float32))
    _, want = S.forward(p, S.bf16_to_f64(feat), emulate_bf16=True)
    for k in range(2):
        assert _rel(fused[:, k].astype(np.float64), want[:, k]) <= 1e-2, k


def test_adam_steps_vs_cpu(ctx):
    R = 120.0
    n = 2048
    img, g, rays = _map_and_rays(n, seed=5)
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    sg = rl.Surrogate(dm, seed=4)
    p0, freq = sg.params()
    want = O.Oracle(img, R, "rm").calc_range_many(g).astype(np.float32)
    p = p0.astype(np.float64)
    m1 = np.zeros_like(p)
    m2 = np.zeros_like(p)
    for t in (1, 2, 3):
        _, grad, feat = sg.gradient(R, rays, want)
        sg.step(1e-3)
        got, _ = sg.params()
        p, m1, m2 = S.adam_step(p, m1, m2, grad.astype(np.float64), t, 1e-3)
        assert np.allclose(got, p, rtol=1e-5, atol=2e-7), f"step {t}: max {np.max(np.abs(got - p))}"
        p = got.astype(np.float64)  # follow the device's fp32 parameters
    # the forward pass uses the updated bf16 weights
    out = sg.forward(rays)
    _, o = S.forward(p, S.bf16_to_f64(feat), emulate_bf16=True)
    assert np.max(np.abs(out - o)) <= 1e-3 * max(1.0, np.max(np.abs(o)))


@pytest.fixture(scope="module")
def trained(ctx):
    img = W.rect_disk_map(256, seed=7)
    R = 120.0
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    sg = rl.Surrogate(dm, seed=1)
    curve = sg.train(R, n_pairs=16384 * 256, batch=16384, lr=1e-3, seed=2)
    return img, dm, sg, R, curve


def test_training_reduces_loss(trained):
    img, dm, sg, R, curve = trained
    assert curve.shape == (256,) and np.all(np.isfinite(curve))
    first, last = float(np.mean(curve[:4])), float(np.mean(curve[-16:]))
    print(f"loss {first:.3f} -> {last:.3f}")
    assert last < 0.5 * first


def _exact_and_checked(trained, bound_max, n_part=500, n_beams=60, seed=9):
    torch = _torch()
    img, dm, sg, R, _ = trained
    ins = W.world_poses(img, n_part, seed=seed)
    ang = W.beam_angles(n_beams)
    d_ins = torch.from_numpy(ins).cuda()
    d_ang = torch.from_numpy(ang).cuda()
    exact = torch.empty(n_part * n_beams, dtype=torch.float32, device="cuda")
    got = torch.full((n_part * n_beams,), -1.0, dtype=torch.float32, device="cuda")
    dm.numpy_calc_range_angles_dev(rl.RL_METHOD_RM, R, d_ins.data_ptr(), d_ang.data_ptr(), exact.data_ptr(),
                                   n_part, n_beams)
    st = sg.calc_range_angles_dev(R, d_ins.data_ptr(), d_ang.data_ptr(), got.data_ptr(), n_part, n_beams,
                                  bound_max=bound_max)
    cnt = torch.empty(n_part * n_beams, dtype=torch.int32, device="cuda")
    dm.count_steps_dev(rl.RL_METHOD_RM, rl.RL_FRAME_ANGLES, R, d_ins.data_ptr(), d_ang.data_ptr(),
                       cnt.data_ptr(), n_part, n_beams)
    torch.cuda.synchronize()
    return exact.cpu().numpy(), got.cpu().numpy(), st, int(cnt.sum().item())


def test_checked_inference_fallback_is_exact(trained):
    exact, got, st, reads = _exact_and_checked(trained, bound_max=-1.0)
    n = exact.size
    assert st["fallback_bound"] == n and st["fallback_check"] == 0 and st["from_start"] == 0
    assert_bits_equal(got, exact, "all rays marched from the origin")
    assert st["reads"] == reads


@pytest.mark.parametrize("bound_max", [0.5, 8.0])
def test_checked_inference_error_and_reads(trained, bound_max):
    """Every ray against the exact march: the fallback rays bit for bit, the
    rays finished from the start point within the stated error (p99 <= 0.5
    cell), with the error distribution and reads printed."""
    exact, got, st, reads = _exact_and_checked(trained, bound_max=bound_max)
    n = exact.size
    assert st["fallback_bound"] + st["fallback_check"] + st["from_start"] == n
    err = np.abs(got.astype(np.float64) - exact)
    q = np.quantile(err, [0.5, 0.9, 0.99])
    print(f"from start {st['from_start'] / n:.3f}, fallback bound {st['fallback_bound'] / n:.3f}, "
          f"check {st['fallback_check'] / n:.3f}; err p50 {q[0]:.3g} p90 {q[1]:.3g} p99 {q[2]:.3g} "
          f"max {err.max():.3g}; reads/ray {st['reads'] / n:.2f} vs exact {reads / n:.2f}; "
          f"dependent rounds/ray {st['rounds'] / n:.2f}")
    # a hit cell's centre distance may exceed max_range by up to sqrt(2) cells
    assert np.all(np.isfinite(got)) and np.all(got >= 0.0) and np.all(got <= 120.0 + 1.5)
    assert np.quantile(err, 0.99) <= 0.5


def _constant_prediction(sg, frac, log_bound):
    """Network outputs forced to (frac, log_bound) for every ray."""
    p, f = sg.params()
    w4 = 256 * 64 + 256 + 2 * (256 * 256 + 256)
    p[w4:w4 + 2 * 256] = 0.0
    p[w4 + 2 * 256] = frac
    p[w4 + 2 * 256 + 1] = log_bound
    sg.set_params(p, f)


def test_checked_inference_never_tunnels(ctx):
    """A confident network that predicts 0.8 max_range for every ray: rays whose
    exact march hits well before that start point must not finish from it (the
    certificate over [0, t0] sees the wall) and come out exact; accepted rays
    end, but for a few where the exact march's sample phase skips a corner the
    probes hit, in the same cell or a neighbouring one."""
    torch = _torch()
    img = W.corridor_map(512, seed=5)
    R = 200.0
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    sg = rl.Surrogate(dm, seed=3)
    _constant_prediction(sg, 0.8, math.log(0.25))
    n_part, n_beams = 400, 60
    ins = W.world_poses(img, n_part, seed=4)
    ang = W.beam_angles(n_beams)
    d_ins = torch.from_numpy(ins).cuda()
    d_ang = torch.from_numpy(ang).cuda()
    got = torch.full((n_part * n_beams,), -1.0, dtype=torch.float32, device="cuda")
    st = sg.calc_range_angles_dev(R, d_ins.data_ptr(), d_ang.data_ptr(), got.data_ptr(), n_part, n_beams,
                                  bound_max=0.5)
    g = got.cpu().numpy()
    want = O.Oracle(img, R, "rm").numpy_calc_range_angles(ins, ang)
    before = want < 0.8 * R - 0.25 - 1.0 - 2.0  # a hit at least two cells before the start point
    assert before.sum() > 1000 and st["fallback_bound"] == 0
    assert_bits_equal(g[before], want[before], "rays with a wall before the start point")
    err = np.abs(g.astype(np.float64) - want)
    print(f"from start {st['from_start']}, check failed {st['fallback_check']}, max err {err.max():.3g}")
    assert st["from_start"] > 0 and np.quantile(err, 0.999) <= 1.5


def _step_rays(img, ins, ang, R):
    """Grid-frame rays (x0, y0, sin h, cos h) of numpy_calc_range_angles and the
    exact ranges (the oracle)."""
    rot = np.float32(-0.0 - 3 * math.pi / 2)
    th = (-ins[:, 2] + rot).astype(np.float32)
    hs = (th[:, None] - ang[None, :]).astype(np.float32).ravel()
    m = ang.size
    rays = np.stack([np.repeat(ins[:, 1], m), np.repeat(ins[:, 0], m), O.libc_sinf(hs), O.libc_cosf(hs)],
                    1).astype(np.float32)
    return rays, O.Oracle(img, R, "rm").numpy_calc_range_angles(ins, ang).astype(np.float64)


def test_trained_surrogate_gains_over_untrained(ctx):
    """What training gains: on a room with two columns (max_range 40), the
    trained network's range error is a fraction of the untrained one's and its
    error bound covers about 95% of the rays (the pinball quantile); through
    the checked path every ray still matches the exact march to p99 <= 0.5
    cell.  Reads and dependent rounds per ray are printed beside the exact
    march's (short rays like these are cheap to march, so the path does not
    save reads here)."""
    torch = _torch()
    img = np.zeros((128, 128), np.uint8)
    img[:3, :] = img[-3:, :] = 1
    img[:, :3] = img[:, -3:] = 1
    img[40:48, 40:48] = img[80:88, 70:78] = 1
    R = 40.0
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    ins = W.world_poses(img, 500, seed=8)
    ang = W.beam_angles(60)
    rays, exact = _step_rays(img, ins, ang, R)
    sg = rl.Surrogate(dm, seed=5)
    rng = np.random.default_rng(0)
    f = np.empty((32, 4), np.float32)
    f[:, :2] = rng.normal(0, 4.0, (32, 2))
    f[:, 2:] = rng.normal(0, 1.0, (32, 2))
    sg.set_params(freq=f)
    e0 = np.abs(R * sg.forward(rays)[:, 0].astype(np.float64) - exact)
    for i, lr in enumerate((1e-3, 3e-4, 1e-4)):
        sg.train(R, n_pairs=4096 * 3000, batch=4096, lr=lr, seed=20 + i, curve=False)
    out = sg.forward(rays)
    e1 = np.abs(R * out[:, 0].astype(np.float64) - exact)
    covered = float(np.mean(e1 <= np.exp(np.clip(out[:, 1], -20, 20))))
    d_ins = torch.from_numpy(ins).cuda()
    d_ang = torch.from_numpy(ang).cuda()
    got = torch.full((exact.size,), -1.0, dtype=torch.float32, device="cuda")
    cnt = torch.empty(exact.size, dtype=torch.int32, device="cuda")
    dm.count_steps_dev(rl.RL_METHOD_RM, rl.RL_FRAME_ANGLES, R, d_ins.data_ptr(), d_ang.data_ptr(), cnt.data_ptr(),
                       500, 60)
    n = exact.size
    for bmax in (0.5, 2.0):
        st = sg.calc_range_angles_dev(R, d_ins.data_ptr(), d_ang.data_ptr(), got.data_ptr(), 500, 60, bound_max=bmax)
        err = np.abs(got.cpu().numpy().astype(np.float64) - exact)
        print(f"bound <= {bmax}: from start {st['from_start'] / n:.4f}, check failed {st['fallback_check'] / n:.4f}; "
              f"reads/ray {st['reads'] / n:.2f}, rounds/ray {st['rounds'] / n:.2f} vs exact "
              f"{int(cnt.sum().item()) / n:.2f}; err p99 {np.quantile(err, 0.99):.3g} max {err.max():.3g}")
        assert np.quantile(err, 0.99) <= 0.5
    print(f"network error p50 {np.median(e0):.2f} -> {np.median(e1):.2f} cells, bound covers {covered:.3f}")
    assert np.median(e1) < 0.25 * np.median(e0)
    assert 0.9 <= covered <= 0.99


def test_surrogate_full_size_corridor(ctx):
    """The learned form at its configured size: a network trained on 50 M rays
    marched on the GPU over the 2048^2 corridor map (max_range 500), then the
    4000-particle x 60-beam step through the checked path at the 0.5-cell
    bound and at 8 cells.  Every ray is compared with the oracle: the rays not
    finished from a start point are exact, so at least that many match bit for
    bit, and the p99 error over all rays is at most 0.5 cell.  The share of
    rays that qualify is printed (on this map the trained bound stays above a
    few cells, so at 0.5 none do)."""
    torch = _torch()
    img = W.corridor_map(2048, 1)
    R = 500.0
    ins = W.world_poses(img, 4000, 2)
    ang = W.beam_angles(60)
    want = O.Oracle(img, R, "rm").numpy_calc_range_angles(ins, ang)
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    sg = rl.Surrogate(dm, seed=0)
    for i, (lr, pairs) in enumerate(((1e-3, 25_000_000), (3e-4, 15_000_000), (1e-4, 10_000_000))):
        sg.train(R, n_pairs=pairs, batch=16384, lr=lr, seed=10 + i, curve=False)
    d_ins = torch.from_numpy(ins).cuda()
    d_ang = torch.from_numpy(ang).cuda()
    got = torch.full((want.size,), -1.0, dtype=torch.float32, device="cuda")
    n = want.size
    for bmax in (0.5, 8.0):
        st = sg.calc_range_angles_dev(R, d_ins.data_ptr(), d_ang.data_ptr(), got.data_ptr(), 4000, 60, bound_max=bmax)
        g = got.cpu().numpy()
        err = np.abs(g.astype(np.float64) - want)
        q = np.quantile(err, [0.5, 0.99, 0.999])
        print(f"bound <= {bmax}: from start {st['from_start'] / n:.4f}, check failed {st['fallback_check'] / n:.4f}, "
              f"bound too large {st['fallback_bound'] / n:.4f}; err p50 {q[0]:.3g} p99 {q[1]:.3g} p99.9 {q[2]:.3g} "
              f"max {err.max():.3g}; reads/ray {st['reads'] / n:.2f}, rounds/ray {st['rounds'] / n:.2f}")
        assert st["fallback_bound"] + st["fallback_check"] + st["from_start"] == n
        assert np.sum(g.view(np.uint32) == want.view(np.uint32)) >= n - st["from_start"]
        assert q[1] <= 0.5


def test_checked_inference_untrained_any_bound(ctx):
    """An untrained network with an unlimited bound: every ray is a candidate;
    results stay within [0, max_range] and the counters add up."""
    torch = _torch()
    img = W.corridor_map(300, seed=3)
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    sg = rl.Surrogate(dm, seed=11)
    ins = torch.from_numpy(W.world_poses(img, 37, seed=1)).cuda()
    ang = torch.from_numpy(W.beam_angles(13)).cuda()
    out = torch.full((37 * 13,), -1.0, dtype=torch.float32, device="cuda")
    st = sg.calc_range_angles_dev(80.0, ins.data_ptr(), ang.data_ptr(), out.data_ptr(), 37, 13, bound_max=1e30)
    o = out.cpu().numpy()
    assert st["fallback_bound"] + st["fallback_check"] + st["from_start"] == 37 * 13
    assert np.all(np.isfinite(o)) and np.all((o >= 0) & (o <= 80.0 + 1.5))


def test_surrogate_rejects_bad_arguments(ctx):
    img = W.rect_disk_map(64, seed=1)
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    sg = rl.Surrogate(dm, seed=0)
    with pytest.raises(rl.RangeLibError):
        sg.train(10.0, n_pairs=100, batch=16)  # batch below 64
    with pytest.raises(ValueError):
        sg.set_params(np.zeros(5, np.float32))


@pytest.mark.parametrize("n", [1, 65, 1056, 70001])
def test_gradient_row_cuts_vs_cpu(ctx, n):
    """Gradients where the rows' cuts end unevenly: one ray, a workgroup of one
    ray, two slices of 544 rows (not a multiple of the 64-row stage), and 64
    slices with bias chunks that start off the 8-row loads."""
    R = 120.0
    img, g, rays = _map_and_rays(n)
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    sg = rl.Surrogate(dm, seed=3)
    p, _ = sg.params()
    _, _, feat = sg.gradient(R, rays, np.zeros(n, np.float32))
    x = S.bf16_to_f64(feat)
    t = _targets_for_both_regimes(p, x, R, n)
    loss, grad, _ = sg.gradient(R, rays, t)
    l16, g16, _ = S.loss_and_grad(p, x, t, R, emulate_bf16=True)
    assert abs(loss - l16) <= 1e-4 * abs(l16)
    for w, b, o, i in S.LAYERS:
        for sl in (slice(w, w + o * i), slice(b, b + o)):
            assert _rel(grad[sl], g16[sl]) <= 1e-2 and _cos(grad[sl], g16[sl]) >= 0.9999


@pytest.mark.parametrize("layer", [0, 1, 2])
@pytest.mark.parametrize("what,bits", [("bias", 0xffc00000), ("bias", 0x7fc00000), ("bias", 0xff800001), ("bias", 0xff800000),
                                       ("bias", 0x7f800000), ("weight", 0xffc00000), ("weight", 0xff800000)])
def test_fused_forward_of_nan_and_infinite_parameters(ctx, layer, what, bits):
    """NaNs of both signs and infinities among a hidden layer's parameters: the fused
    forward is NaN exactly where the per-layer one is, and the checked cast of a
    network that says NaN is the exact march."""
    R, n = 100.0, 100
    img, g, rays = _map_and_rays(n, seed=5)
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    sg = rl.Surrogate(dm, seed=9)
    p = sg.params()[0].copy()
    w, b, o, i = S.LAYERS[layer]
    p.view(np.uint32)[b + 3 if what == "bias" else w + 3 * i + 5] = bits
    sg.set_params(p)
    with np.errstate(invalid="ignore"):
        fused, layers = sg.forward(rays), sg.forward_layers(rays)
    assert np.array_equal(np.isnan(fused), np.isnan(layers))
    finite = ~np.isnan(layers)
    assert_bits_equal(fused[finite], layers[finite], "fused vs per-layer forward")
    if np.isnan(p).any():
        assert np.isnan(fused).all()
        torch = _torch()
        ins, ang = torch.from_numpy(W.world_poses(img, n, seed=2)).cuda(), torch.from_numpy(W.beam_angles(7)).cuda()
        got, want = (torch.zeros(7 * n, dtype=torch.float32, device="cuda") for _ in range(2))
        sg.calc_range_angles_dev(R, ins.data_ptr(), ang.data_ptr(), got.data_ptr(), n, 7, bound_max=1e9)
        dm.numpy_calc_range_angles_dev(rl.RL_METHOD_RM, R, ins.data_ptr(), ang.data_ptr(), want.data_ptr(), n, 7)
        ctx.sync()
        assert_bits_equal(got.cpu().numpy(), want.cpu().numpy(), "checked cast")


@pytest.mark.parametrize("n", [1, 63, 64, 65, 777])
def test_training_forward_equals_layers(ctx, n):
    """The training pass's hidden activations are bitwise the per-layer kernels', whose
    outputs the fused inference has: what is trained is what infers."""
    img, g, rays = _map_and_rays(n, seed=7)
    dm = rl.DeviceMap(ctx, O.xmajor(img))
    sg = rl.Surrogate(dm, seed=4)
    p = sg.params()[0].copy()
    rng = np.random.default_rng(n)
    for w, b, o, i in S.LAYERS:
        p[b:b + o] = rng.uniform(-0.5, 0.5, o)
    sg.set_params(p)
    assert np.array_equal(sg.hidden(rays, training=True), sg.hidden(rays, training=False))
    assert_bits_equal(sg.forward(rays), sg.forward_layers(rays), "fused vs per-layer forward")
