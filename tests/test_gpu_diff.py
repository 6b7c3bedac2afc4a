"""Differentiable renderer (needs a GPU).

The HIP forward must reproduce the oracle's f32 relaxation (visible slice
per pixel exactly, colours bit for bit), the adjoint must match the
oracle's vjp within 1e-5 of the gradient's scale, and both must agree
with central finite differences of the loss.
"""
import numpy as np
import pytest

from futspace_amd import View, scene, sky_color
from oracle import fs_oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from futspace_amd.diff import DiffRenderer, fit, planes_of  # noqa: E402

SUN_H, SUN_A = 0.1, 0.1


def _setup(ctx, seed=11, size=128, bits=8, sun=(SUN_H, SUN_A)):
    if bits == 8:
        col, hts = scene.scene_maps(seed, size)
    else:
        hts = scene.heightmap(seed, size, 0.6, 600)
        col = scene.colormap(seed, hts, 600)
    m = ctx.map(col, hts, height_bits=bits, shade_size=size, sun_height=sun[0], sun_ang=sun[1])
    r = DiffRenderer(ctx, m)
    alt = (np.asarray(hts, dtype=np.int32) & ((1 << bits) - 1)).astype(np.int32)
    counts = O.shadow_counts(alt, O.sun(*sun), size)
    sf = O.shade_factor(counts)
    return r, col, alt, sf


VIEWS = [
    View(x=64.3, y=100.7, height=260.0, angle=0.4, horizon=60.0, distance=300.0, fov=1.2,
         h=96, w=128, d=0.01, z0=0.5),
    View(x=64.0, y=64.0, height=200.0, angle=0.0, horizon=50.0, distance=200.0, fov=1.2,
         h=64, w=80, d=0.01, z0=0.5),                       # yaw 0: integral x, transparent
    View(x=10.5, y=3.25, height=300.0, angle=1.5707964, horizon=90.0, distance=400.0, fov=0.8,
         h=100, w=77, d=0.005, z0=1.0, scale=120.0),
    View(x=33.3, y=77.7, height=250.0, angle=5.0, horizon=300.0, distance=700.0, fov=1.2,
         h=257, w=129, d=0.003, z0=0.4, scale=64.0, n_slices=3000),
]


def test_shade_factor_matches_oracle(ctx):
    for sun in [(SUN_H, SUN_A), (0.6, 2.0), (-0.3, 0.7)]:
        r, _, _, sf = _setup(ctx, sun=sun)
        torch.cuda.synchronize()
        assert np.array_equal(r.sf.cpu().numpy().view(np.uint32), sf.view(np.uint32)), sun


@pytest.mark.parametrize("vi", range(len(VIEWS)))
def test_forward_matches_oracle(ctx, vi):
    r, col, alt, sf = _setup(ctx)
    v = VIEWS[vi]
    planes = planes_of(col)
    img, src = r.forward_raw(torch.from_numpy(planes).cuda(), 0.37, v)
    torch.cuda.synchronize()
    want_img, want_src = O.render_f32(v, planes, sf, alt, 0.37)
    got_src = src.cpu().numpy()
    cols = np.arange(v.w, dtype=np.int32)[None, :]
    got_src_o = np.where(got_src < 0, -1, got_src * v.w + cols)
    assert np.array_equal(got_src_o, want_src), f"{np.count_nonzero(got_src_o != want_src)} pixels"
    got = img.cpu().numpy()
    bad = np.count_nonzero(got.view(np.uint32) != want_img.view(np.uint32))
    assert bad == 0, f"{bad} channel values differ, max abs {np.abs(got - want_img).max()}"


def test_forward_sixteen_bit_heights(ctx):
    r, col, alt, sf = _setup(ctx, seed=13, bits=16)
    v = View(x=50.0, y=90.0, height=700.0, angle=1.0, horizon=120.0, distance=1000.0, fov=1.2,
             h=144, w=160, d=0.002, z0=0.5)
    planes = planes_of(col)
    img, src = r.forward_raw(torch.from_numpy(planes).cuda(), 0.1, v)
    want_img, want_src = O.render_f32(v, planes, sf, alt, 0.1)
    got_src = src.cpu().numpy()
    cols = np.arange(v.w, dtype=np.int32)[None, :]
    assert np.array_equal(np.where(got_src < 0, -1, got_src * v.w + cols), want_src)
    assert np.array_equal(img.cpu().numpy(), want_img)


@pytest.mark.parametrize("h,w", [(4320, 20), (9000, 7)])
def test_forward_tall_frame(ctx, h, w):
    """An 8K-tall (4320-row) frame takes 4-column slice-mode tiles, a
    9000-row one the column kernel: both bit-exact, and the fused step of
    the 9000-row one (its gradient cleared in a launch of its own) gives
    the separate calls' result."""
    r, col, alt, sf = _setup(ctx)
    v = View(x=64.3, y=100.7, height=260.0, angle=0.4, horizon=h * 0.4, distance=300.0, fov=1.2,
             h=h, w=w, d=0.01, z0=0.5, scale=h / 3.0)
    planes = planes_of(col)
    img, src = r.forward_raw(torch.from_numpy(planes).cuda(), 0.37, v)
    want_img, want_src = O.render_f32(v, planes, sf, alt, 0.37)
    got_src = src.cpu().numpy()
    cols = np.arange(v.w, dtype=np.int32)[None, :]
    assert np.array_equal(np.where(got_src < 0, -1, got_src * v.w + cols), want_src)
    assert np.array_equal(img.cpu().numpy().view(np.uint32), want_img.view(np.uint32))
    if h > 7680:
        tp = torch.from_numpy(planes).cuda()
        target = torch.from_numpy(np.random.default_rng(h).random((3, h, w), dtype=np.float32)).cuda()
        gimg, loss = r.l2_loss_grad(img, target)
        gp, gs = r.vjp_raw(tp, src, gimg, v)
        gp2 = torch.full_like(tp, 9.0)
        _, src2, gp2, gs2, loss2 = r.l2_step(tp, 0.37, v, target, gplanes=gp2)
        torch.cuda.synchronize()
        assert torch.equal(src2, src)
        assert abs(float(loss2[0]) - float(loss[0])) <= 1e-5 * float(loss[0])
        assert _rel_err(gp2.cpu().numpy(), gp.cpu().numpy()) <= 1e-5


def _rel_err(got, want):
    scale = max(float(np.abs(want).max()), 1e-30)
    return float(np.abs(got.astype(np.float64) - want.astype(np.float64)).max()) / scale


@pytest.mark.parametrize("vi", range(len(VIEWS)))
def test_vjp_matches_oracle(ctx, vi):
    """Colour-plane gradients within 1e-5 of the largest gradient; the sky
    gradient within 1e-5 of the L1 mass of its terms (f32 atomics sum it
    in no fixed order)."""
    r, col, alt, sf = _setup(ctx)
    v = VIEWS[vi]
    planes = planes_of(col)
    rng = np.random.default_rng(100 + vi)
    gimg = rng.standard_normal((3, v.h, v.w)).astype(np.float32)
    tp = torch.from_numpy(planes).cuda()
    _, src = r.forward_raw(tp, 0.37, v)
    gp, gs = r.vjp_raw(tp, src, torch.from_numpy(gimg).cuda(), v)
    torch.cuda.synchronize()
    _, want_src = O.render_f32(v, planes, sf, alt, 0.37)
    want_gp, want_gs = O.render_f32_vjp(v, planes, sf, want_src, gimg)
    assert _rel_err(gp.cpu().numpy(), want_gp) <= 1e-5
    sky_terms = np.abs(gimg[:, want_src < 0]).sum(axis=1) @ np.array([144, 144, 224]) / 255.0
    assert abs(float(gs.cpu()[0]) - want_gs) <= 1e-5 * max(sky_terms, 1e-3)


def test_vjp_accumulates(ctx):
    r, col, _, _ = _setup(ctx)
    tp = torch.from_numpy(planes_of(col)).cuda()
    g = torch.zeros_like(tp)
    gs = torch.zeros(1, device="cuda")
    total = torch.zeros_like(tp)
    for i, v in enumerate(VIEWS[:3]):
        _, src = r.forward_raw(tp, 0.2, v)
        gimg = torch.ones((3, v.h, v.w), device="cuda")
        one, _ = r.vjp_raw(tp, src, gimg, v)
        total += one
        r.vjp_raw(tp, src, gimg, v, g, gs, accumulate=i > 0)
    torch.cuda.synchronize()
    assert torch.allclose(g, total, rtol=1e-5, atol=1e-6)


def _loss64(r, planes, v, target, sky):
    img, _ = r.forward_raw(planes, sky, v)
    d = (img - target).double()
    return float((d * d).sum())


def test_autograd_function_and_finite_differences(ctx):
    """dL/dplanes through torch.autograd equals the adjoint, and agrees with
    central differences (h = 1e-2) on 64 texels, mostly visible ones."""
    r, col, alt, sf = _setup(ctx, seed=21, size=256)
    v = View(x=128.3, y=40.7, height=230.0, angle=2.7, horizon=110.0, distance=500.0, fov=1.2,
             h=180, w=240, d=0.002, z0=0.5, n_slices=1200)
    rng = np.random.default_rng(9)
    planes0 = planes_of(col)
    target = np.clip(planes0 + rng.normal(0.0, 8.0 / 255.0, planes0.shape), 0.0, 1.0)
    tgt_img, _ = r.forward_raw(torch.from_numpy(target.astype(np.float32)).cuda(), SUN_H, v)
    planes = torch.from_numpy(planes0).cuda().requires_grad_(True)
    shading = torch.tensor([0.15, SUN_A], dtype=torch.float32, requires_grad=True)
    img = r.render(planes, shading, v)
    loss = ((img - tgt_img) ** 2).sum()
    loss.backward()
    g = planes.grad.detach().clone()
    # the adjoint called directly
    _, src = r.forward_raw(planes.detach(), 0.15, v)
    g2, gs2 = r.vjp_raw(planes.detach(), src, 2.0 * (img.detach() - tgt_img), v)
    assert float((g - g2).abs().max()) <= 1e-5 * float(g2.abs().max())
    assert abs(float(shading.grad[0]) - float(gs2.cpu()[0])) <= 1e-4 * abs(float(gs2.cpu()[0]))
    assert float(shading.grad[1]) == 0.0
    # central differences
    # texels whose value stays positive under +-h (the channel mix is even
    # in each texel value, so FD across 0 would not be a derivative)
    h = 1e-2
    gh = g.cpu().numpy()
    ok = planes0 > 5 * h
    nz = np.argwhere((np.abs(gh) > 1e-3 * np.abs(gh).max()) & ok)
    pick = nz[rng.choice(len(nz), 48, replace=False)]
    allok = np.argwhere(ok)
    rand = allok[rng.choice(len(allok), 16, replace=False)]
    base = planes.detach().clone()
    for ch, y, x in list(map(tuple, pick)) + list(map(tuple, rand)):
        p = base.clone()
        p[ch, y, x] += h
        lp = _loss64(r, p, v, tgt_img, 0.15)
        p[ch, y, x] -= 2 * h
        lm = _loss64(r, p, v, tgt_img, 0.15)
        fd = (lp - lm) / (2 * h)
        an = float(gh[ch, y, x])
        assert abs(fd - an) <= 2e-2 * max(abs(an), abs(fd)) + 1e-3, (ch, y, x, fd, an)
    # sun_height through the sky pixels
    def loss_sky(s):
        return _loss64(r, base, v, tgt_img, s)
    fd = (loss_sky(0.15 + h) - loss_sky(0.15 - h)) / (2 * h)
    an = float(shading.grad[0])
    assert abs(fd - an) <= 1e-3 * max(abs(an), 1.0), (fd, an)


def test_fit_reduces_loss(ctx):
    r, col, _, _ = _setup(ctx, seed=31, size=128)
    rng = np.random.default_rng(8)
    planes0 = planes_of(col)
    target_planes = np.clip(planes0 + rng.normal(0.0, 8.0 / 255.0, planes0.shape), 0, 1)
    views = VIEWS[:3]
    tp = torch.from_numpy(target_planes.astype(np.float32)).cuda()
    targets = [r.forward_raw(tp, SUN_H, v)[0].clone() for v in views]
    planes = torch.from_numpy(planes0).cuda()
    losses = fit(r, planes, views, targets, SUN_H, steps=20, lr=2.0).cpu().numpy()
    assert np.all(np.isfinite(losses))
    assert losses[-1] < 0.5 * losses[0], losses
    p = planes.cpu().numpy()
    assert p.min() >= 0.0 and p.max() <= 1.0


def test_fit_at_the_workload_rate_does_not_diverge(ctx):
    """Adam at the fitting workload's lr 0.5 (one half u8 channel step):
    the loss falls over the first steps instead of blowing up, and the
    planes stay inside [0, 1]."""
    r, col, _, _ = _setup(ctx, seed=31, size=128)
    rng = np.random.default_rng(8)
    planes0 = planes_of(col)
    target_planes = np.clip(planes0 + rng.normal(0.0, 8.0 / 255.0, planes0.shape), 0, 1)
    views = VIEWS[:3]
    tp = torch.from_numpy(target_planes.astype(np.float32)).cuda()
    targets = [r.forward_raw(tp, SUN_H, v)[0].clone() for v in views]
    planes = torch.from_numpy(planes0).cuda()
    losses = fit(r, planes, views, targets, SUN_H, steps=12, lr=0.5).cpu().numpy()
    assert np.all(np.isfinite(losses))
    assert np.all(np.diff(losses) <= 1e-6 * losses[0]), losses
    assert losses[-1] < losses[0], losses
    p = planes.cpu().numpy()
    assert p.min() >= 0.0 and p.max() <= 1.0


def test_fused_l2_loss(ctx):
    r, _, _, _ = _setup(ctx)
    gen = torch.Generator(device="cuda").manual_seed(3)
    for n in (4, 7, 3 * 97 * 131, 3 * 720 * 1280):
        a = torch.rand(n, device="cuda", generator=gen)
        b = torch.rand(n, device="cuda", generator=gen)
        g, loss = r.l2_loss_grad(a, b)
        g2, loss2 = r.l2_loss_grad(a, b, loss=loss.clone(), accumulate=True)
        torch.cuda.synchronize()
        want = ((a.double() - b.double()) ** 2).sum()
        assert torch.equal(g, 2.0 * (a - b))
        assert abs(float(loss[0]) - float(want)) <= 1e-5 * float(want)
        assert abs(float(loss2[0]) - 2 * float(want)) <= 2e-5 * float(want)


@pytest.mark.parametrize("vi", range(len(VIEWS)))
def test_fused_step_matches_separate_calls(ctx, vi):
    """fsx_render_f32_l2_step = fsx_render_f32, fsx_l2_loss and
    fsx_render_f32_vjp: img, src and the loss gradient bit-exact, the loss
    within f32 summation order, the gradients within 1e-5 (f32 atomics);
    and against the oracle's adjoint of the same loss gradient."""
    r, col, alt, sf = _setup(ctx)
    v = VIEWS[vi]
    planes = planes_of(col)
    tp = torch.from_numpy(planes).cuda()
    rng = np.random.default_rng(200 + vi)
    target = torch.from_numpy(rng.random((3, v.h, v.w), dtype=np.float32)).cuda()
    img, src = r.forward_raw(tp, 0.37, v)
    gimg, loss = r.l2_loss_grad(img, target)
    gp, gs = r.vjp_raw(tp, src, gimg, v)
    # stale values in the outputs: the step must overwrite them
    f_img = torch.full_like(img, 7.0)
    f_src = torch.full_like(src, 5)
    f_gimg = torch.full_like(img, 3.0)
    f_gp = torch.full_like(tp, 9.0)
    f_gs = torch.full((1,), 4.0, device="cuda")
    f_loss = torch.full((1,), 2.0, device="cuda")
    r.l2_step(tp, 0.37, v, target, f_img, f_src, f_gimg, f_gp, f_gs, f_loss)
    torch.cuda.synchronize()
    assert torch.equal(f_img, img) and torch.equal(f_src, src) and torch.equal(f_gimg, gimg)
    assert abs(float(f_loss[0]) - float(loss[0])) <= 1e-5 * float(loss[0])
    assert _rel_err(f_gp.cpu().numpy(), gp.cpu().numpy()) <= 1e-5
    _, want_src = O.render_f32(v, planes, sf, alt, 0.37)
    g_np = gimg.cpu().numpy()
    want_gp, want_gs = O.render_f32_vjp(v, planes, sf, want_src, g_np)
    assert _rel_err(f_gp.cpu().numpy(), want_gp) <= 1e-5
    sky_terms = np.abs(g_np[:, want_src < 0]).sum(axis=1) @ np.array([144, 144, 224]) / 255.0
    assert abs(float(f_gs.cpu()[0]) - want_gs) <= 1e-5 * max(sky_terms, 1e-3)


@pytest.mark.parametrize("vi", [0, 3])
def test_fused_step_without_image_outputs(ctx, vi):
    """outputs=False (NULL img and dL/dimg) leaves those buffers untouched
    and gives the same src and loss bit for bit, the same gradients within
    the f32-atomic order, as the step that writes them."""
    r, col, _, _ = _setup(ctx)
    v = VIEWS[vi]
    tp = torch.from_numpy(planes_of(col)).cuda()
    rng = np.random.default_rng(300 + vi)
    target = torch.from_numpy(rng.random((3, v.h, v.w), dtype=np.float32)).cuda()
    img, src, gp, gs, loss = r.l2_step(tp, 0.37, v, target)
    src2 = torch.full_like(src, 5)
    gp2 = torch.full_like(tp, 9.0)
    gs2 = torch.full((1,), 4.0, device="cuda")
    loss2 = torch.full((1,), 2.0, device="cuda")
    out = r.l2_step(tp, 0.37, v, target, None, src2, None, gp2, gs2, loss2, outputs=False)
    torch.cuda.synchronize()
    assert out[0] is None
    assert torch.equal(src2, src)
    assert float(loss2[0]) == float(loss[0])
    assert _rel_err(gp2.cpu().numpy(), gp.cpu().numpy()) <= 1e-5
    assert abs(float(gs2[0]) - float(gs[0])) <= 1e-5 * max(abs(float(gs[0])), 1.0)


def test_fused_step_accumulates(ctx):
    """accumulate adds the loss and both gradients to the given values."""
    r, col, _, _ = _setup(ctx)
    tp = torch.from_numpy(planes_of(col)).cuda()
    rng = np.random.default_rng(7)
    g = torch.empty_like(tp)
    gs = torch.empty(1, device="cuda")
    loss = torch.empty(1, device="cuda")
    tot_g = torch.zeros_like(tp)
    tot_gs = torch.zeros(1, device="cuda")
    tot_loss = 0.0
    for i, v in enumerate(VIEWS[:3]):
        target = torch.from_numpy(rng.random((3, v.h, v.w), dtype=np.float32)).cuda()
        _, _, g1, gs1, l1 = r.l2_step(tp, 0.2, v, target)
        tot_g += g1
        tot_gs += gs1
        tot_loss += float(l1[0])
        r.l2_step(tp, 0.2, v, target, None, None, None, g, gs, loss, accumulate=i > 0)
    torch.cuda.synchronize()
    assert torch.allclose(g, tot_g, rtol=1e-5, atol=1e-6)
    assert abs(float(gs[0]) - float(tot_gs[0])) <= 1e-5 * max(abs(float(tot_gs[0])), 1.0)
    assert abs(float(loss[0]) - tot_loss) <= 1e-5 * tot_loss


@pytest.mark.parametrize("size", [99, 100])
def test_fused_step_odd_plane_sizes(ctx, size):
    """Planes that are not powers of two (floor-mod wrap), and 3*99*99
    values (not a multiple of 4: the gradient clear takes its own launch);
    a view wide enough to wrap around the map."""
    col, hts = scene.scene_maps(17, 128)
    col = np.ascontiguousarray(col[:size, :size])
    hts = np.ascontiguousarray(hts[:size, :size])
    m = ctx.map(col, hts, shade_size=size, sun_height=SUN_H, sun_ang=SUN_A)
    r = DiffRenderer(ctx, m)
    alt = np.asarray(hts, dtype=np.int32) & 255
    sf = O.shade_factor(O.shadow_counts(alt, O.sun(SUN_H, SUN_A), size))
    v = View(x=50.5, y=20.25, height=240.0, angle=2.0, horizon=80.0, distance=400.0, fov=1.4,
             h=72, w=150, d=0.004, z0=0.6, scale=90.0)
    planes = planes_of(col)
    tp = torch.from_numpy(planes).cuda()
    target = torch.from_numpy(np.random.default_rng(size).random((3, v.h, v.w),
                                                                 dtype=np.float32)).cuda()
    gp = torch.full_like(tp, 9.0)
    img, src, gp, gs, loss = r.l2_step(tp, 0.2, v, target, gplanes=gp,
                                       gsky=torch.zeros(1, device="cuda"),
                                       loss=torch.zeros(1, device="cuda"))
    torch.cuda.synchronize()
    want_img, want_src = O.render_f32(v, planes, sf, alt, 0.2)
    assert np.array_equal(img.cpu().numpy(), want_img)
    d = (want_img.astype(np.float64) - target.cpu().numpy())
    assert abs(float(loss[0]) - float((d * d).sum())) <= 1e-5 * float((d * d).sum())
    g_np = (2.0 * (img - target)).cpu().numpy()
    want_gp, _ = O.render_f32_vjp(v, planes, sf, want_src, g_np)
    assert _rel_err(gp.cpu().numpy(), want_gp) <= 1e-5


def test_forward_tall_frame(ctx):
    """The differentiable forward on a frame tall enough for 4-column
    slice-mode tiles."""
    r, col, alt, sf = _setup(ctx)
    v = View(x=64.3, y=100.7, height=260.0, angle=0.4, horizon=900.0, distance=300.0, fov=1.2,
             h=2200, w=40, d=0.01, z0=0.5, scale=700.0)
    planes = planes_of(col)
    img, src = r.forward_raw(torch.from_numpy(planes).cuda(), 0.37, v)
    torch.cuda.synchronize()
    want_img, want_src = O.render_f32(v, planes, sf, alt, 0.37)
    got_src = src.cpu().numpy()
    cols = np.arange(v.w, dtype=np.int32)[None, :]
    assert np.array_equal(np.where(got_src < 0, -1, got_src * v.w + cols), want_src)
    assert np.array_equal(img.cpu().numpy(), want_img)


@pytest.mark.parametrize("w", [128, 1600])
def test_fused_step_gradient_clear(ctx, w):
    """The fused step clears stale gradient planes either in spare
    workgroups of the slice render (a narrow view leaves most CUs idle) or
    in a launch of its own (a 1600-column view leaves too few): both give
    the separate calls' result."""
    r, col, _, _ = _setup(ctx)
    v = View(x=64.3, y=100.7, height=260.0, angle=0.4, horizon=0.0, distance=300.0, fov=1.2,
             h=40, w=w, d=0.01, z0=0.5, scale=64.0)
    tp = torch.from_numpy(planes_of(col)).cuda()
    target = torch.from_numpy(np.random.default_rng(w).random((3, v.h, v.w),
                                                              dtype=np.float32)).cuda()
    img, src = r.forward_raw(tp, 0.3, v)
    gimg, loss = r.l2_loss_grad(img, target)
    gp, gs = r.vjp_raw(tp, src, gimg, v)
    assert float(gp.abs().sum()) > 0
    for _ in range(2):
        f_gp = torch.full_like(tp, 9.0)
        out = r.l2_step(tp, 0.3, v, target, gplanes=f_gp, gsky=torch.full((1,), 4.0, device="cuda"),
                        loss=torch.full((1,), 2.0, device="cuda"))
        torch.cuda.synchronize()
        assert torch.equal(out[0], img) and torch.equal(out[1], src)
        assert _rel_err(f_gp.cpu().numpy(), gp.cpu().numpy()) <= 1e-5
        assert abs(float(out[3][0]) - float(gs[0])) <= 1e-5 * max(abs(float(gs[0])), 1e-3)
        assert abs(float(out[4][0]) - float(loss[0])) <= 1e-5 * float(loss[0])


def test_fused_step_of_a_4096x2160_frame(ctx):
    """A 4096 x 2160 frame (2^22 pixels or more: the adjoint's blocks are 64
    x 32 pixels, 4352 of them): the fused step still equals the three
    separate calls (image, src and loss gradient bit for bit, loss within
    f32 summation order, gradients within 1e-5)."""
    r, col, _, _ = _setup(ctx, seed=11, size=256)
    v = View(x=120.3, y=77.7, height=280.0, angle=0.9, horizon=700.0, distance=400.0, fov=1.2,
             h=2160, w=4096, d=0.001, z0=0.4, n_slices=900)
    planes = torch.from_numpy(planes_of(col)).cuda()
    rng = np.random.default_rng(41)
    target = torch.from_numpy(rng.random((3, v.h, v.w), dtype=np.float32)).cuda()
    img, src = r.forward_raw(planes, 0.37, v)
    gimg, loss = r.l2_loss_grad(img, target)
    gp, gs = r.vjp_raw(planes, src, gimg, v)
    f_gimg = torch.empty_like(gimg)
    f_img, f_src, f_gp, f_gs, f_loss = r.l2_step(planes, 0.37, v, target, gimg=f_gimg)
    torch.cuda.synchronize()
    assert torch.equal(f_img, img) and torch.equal(f_src, src) and torch.equal(f_gimg, gimg)
    assert abs(float(f_loss[0]) - float(loss[0])) <= 1e-5 * float(loss[0])
    assert _rel_err(f_gp.cpu().numpy(), gp.cpu().numpy()) <= 1e-5
    assert abs(float(f_gs[0]) - float(gs[0])) <= 1e-5 * max(abs(float(gs[0])), 1.0)


def test_fused_step_refuses_frames_beyond_its_partials(ctx):
    """8192 x 4128 needs 16512 loss partials (blocks of 64 x 32 pixels, more
    than 16384): the step is refused with a message naming the limit,
    before anything is enqueued (the outputs keep their contents)."""
    from futspace_amd.renderer import FutspaceError
    r, col, _, _ = _setup(ctx, seed=11, size=128)
    v = View(x=64.3, y=100.7, height=260.0, angle=0.4, horizon=60.0, distance=300.0, fov=1.2,
             h=4128, w=8192, d=0.01, z0=0.5)
    planes = torch.from_numpy(planes_of(col)).cuda()
    target = torch.zeros((3, v.h, v.w), dtype=torch.float32, device="cuda")
    img = torch.full_like(target, 7.0)
    gimg = torch.full_like(target, 3.0)
    src = torch.full((v.h, v.w), 5, dtype=torch.int32, device="cuda")
    gp = torch.full_like(planes, 9.0)
    gs = torch.full((1,), 4.0, device="cuda")
    loss = torch.full((1,), 2.0, device="cuda")
    with pytest.raises(FutspaceError, match="16384"):
        r.l2_step(planes, 0.37, v, target, img, src, gimg, gp, gs, loss)
    torch.cuda.synchronize()
    assert bool((img == 7.0).all()) and bool((gimg == 3.0).all()) and bool((src == 5).all())
    assert bool((gp == 9.0).all()) and float(gs[0]) == 4.0 and float(loss[0]) == 2.0


def test_adam_step_matches_torch_adam(ctx):
    """fsx_adam_step: three steps equal torch's Adam (default betas and
    eps, no weight decay) within the hardware sqrt / reciprocal's few ulps,
    then the clamp to [lo, hi]; a length that is not a multiple of 4 takes
    the scalar tail."""
    r, _, _, _ = _setup(ctx)
    rng = np.random.default_rng(31)
    for n in (4096, 1003):
        p0 = torch.from_numpy(rng.random(n, dtype=np.float32)).cuda()
        grads = [torch.from_numpy(rng.standard_normal(n).astype(np.float32)).cuda()
                 for _ in range(3)]
        p, m, v = p0.clone(), torch.zeros_like(p0), torch.zeros_like(p0)
        q = p0.clone().requires_grad_(True)
        opt = torch.optim.Adam([q], lr=0.01, foreach=False)
        for t, g in enumerate(grads):
            r.adam_step(p, g, m, v, 0.01, t + 1, lo=-10.0, hi=10.0)
            q.grad = g.clone()
            opt.step()
        torch.cuda.synchronize()
        assert float((p - q.detach()).abs().max()) <= 1e-6
        st = opt.state[q]
        assert torch.allclose(m, st["exp_avg"], rtol=1e-6, atol=1e-7)
        assert torch.allclose(v, st["exp_avg_sq"], rtol=1e-6, atol=1e-7)
        r.adam_step(p, grads[0] * 1e4, m, v, 1.0, 4, lo=0.25, hi=0.75)
        torch.cuda.synchronize()
        assert float(p.min()) >= 0.25 and float(p.max()) <= 0.75


@pytest.mark.parametrize("h,w,size,zoom", [
    (7, 1, 128, 1.0), (8, 64, 128, 1.0), (9, 65, 96, 1.0),       # edges of the workgroups
    (200, 300, 128, 0.02),                                       # every pixel on a few texels
    (200, 300, 512, 40.0),                                       # every sample on its own texels
])
def test_adjoint_table_and_blocks(ctx, h, w, size, zoom):
    """Gradients of both adjoints against the oracle where a workgroup's
    texel table holds a few texels, and where it overflows."""
    col, hts = scene.scene_maps(29, 128)
    m = ctx.map(col, hts, shade_size=size)
    r = DiffRenderer(ctx, m)
    alt = np.asarray(hts, np.int32) & 255
    sf = O.shade_factor(O.shadow_counts(alt, O.sun(0.1, 0.1), size))
    rng = np.random.default_rng(h + w + size)
    planes = rng.random((3, size, size), dtype=np.float32)
    d, z0 = scene.depth_for(300, 100.0 * zoom)
    v = View(x=50.3, y=20.7, height=290.0, angle=0.9, horizon=0.1 * h, distance=100.0 * zoom,
             fov=1.2, h=h, w=w, d=d, z0=z0, scale=h * zoom * 0.3, n_slices=300)
    tp = torch.from_numpy(planes).cuda()
    target = torch.from_numpy(rng.random((3, h, w), dtype=np.float32)).cuda()
    img, src, gp, gs, loss = r.l2_step(tp, 0.4, v, target)
    gimg = torch.from_numpy(rng.standard_normal((3, h, w)).astype(np.float32)).cuda()
    gp2, gs2 = r.vjp_raw(tp, src, gimg, v)
    torch.cuda.synchronize()
    want_img, want_src = O.render_f32(v, planes, sf, alt, 0.4)
    assert (want_src >= 0).sum() > h * w // 20
    assert np.array_equal(img.cpu().numpy().view(np.uint32), want_img.view(np.uint32))
    g = 2.0 * (want_img - target.cpu().numpy())
    for got, sky, gi in ((gp, gs, g.astype(np.float32)), (gp2, gs2, gimg.cpu().numpy())):
        want, want_sky = O.render_f32_vjp(v, planes, sf, want_src, gi)
        assert _rel_err(got.cpu().numpy(), want) <= 1e-5
        mass = np.abs(gi[:, want_src < 0]).sum() + 1e-3
        assert abs(float(sky[0]) - float(want_sky)) <= 1e-5 * mass
    want_loss = float(((want_img.astype(np.float64) - target.cpu().numpy()) ** 2).sum())
    assert abs(float(loss[0]) - want_loss) <= 1e-5 * want_loss


@pytest.mark.parametrize("accumulate", [False, True])
def test_step_with_given_visibility(ctx, accumulate):
    """l2_step(visible=True) over the src of a forward call: the loss bit for
    bit and the gradients of the step that renders it, src left alone."""
    r, col, _, _ = _setup(ctx)
    tp = torch.from_numpy(planes_of(col)).cuda()
    for v in VIEWS:
        rng = np.random.default_rng(v.h)
        target = torch.from_numpy(rng.random((3, v.h, v.w), dtype=np.float32)).cuda()
        outs = []
        for visible in (False, True):
            src = r.forward_raw(tp, 0.3, v)[1]
            before = src.clone()
            gp, gs, loss = torch.full_like(tp, 2.0), torch.full((1,), 3.0, device="cuda"), \
                torch.full((1,), 4.0, device="cuda")
            torch.cuda.synchronize()
            img, _, gp, gs, loss = r.l2_step(tp, 0.3, v, target, src=src, gplanes=gp, gsky=gs,
                                             loss=loss, accumulate=accumulate, visible=visible)
            torch.cuda.synchronize()
            assert torch.equal(src, before)
            outs.append((img, gp, gs, loss))
        (img, gp, gs, loss), (img2, gp2, gs2, loss2) = outs
        assert torch.equal(img, img2) and torch.equal(loss, loss2) and torch.equal(gs, gs2)
        assert _rel_err(gp2.cpu().numpy(), gp.cpu().numpy()) <= 1e-5
    with pytest.raises(ValueError):
        r.l2_step(tp, 0.3, VIEWS[0], target, visible=True)


@pytest.mark.parametrize("share", [0.125, 0.0])
def test_fit_follows_changed_views(ctx, share, monkeypatch):
    """fit() renders a view's visibility again when its camera or size
    changes between steps, and where no visibility is kept."""
    import dataclasses

    from futspace_amd import diff
    monkeypatch.setattr(diff, "FIT_VISIBLE_SHARE", share)
    r, col, _, _ = _setup(ctx)
    start = torch.from_numpy(planes_of(col)).cuda()
    views = [dataclasses.replace(VIEWS[0]), dataclasses.replace(VIEWS[1])]
    moved = dataclasses.replace(VIEWS[0], x=VIEWS[0].x + 7.3, angle=1.9)
    other = dataclasses.replace(VIEWS[1], h=VIEWS[1].h + 3)
    goal = (start * 0.5).contiguous()
    targets = [r.forward_raw(goal, 0.3, v)[0] for v in views]
    torch.cuda.synchronize()

    def swap(it):
        if it == 1:
            views[0].x, views[0].angle = moved.x, moved.angle
            views[1] = other
            for i, v in enumerate(views):
                targets[i] = r.forward_raw(goal, 0.3, v)[0]

    planes = start.clone()
    losses = fit(r, planes, views, targets, 0.3, steps=4, on_step=swap).cpu().numpy()
    # the same steps one by one through l2_step, which always renders
    p, g, m, s = start.clone(), torch.zeros_like(start), torch.zeros_like(start), \
        torch.zeros_like(start)
    for it in range(4):
        vs = [VIEWS[0], VIEWS[1]] if it < 2 else [moved, other]
        gs, loss = torch.zeros(1, device="cuda"), torch.zeros(1, device="cuda")
        for i, v in enumerate(vs):
            t = r.forward_raw(goal, 0.3, v)[0]
            r.l2_step(p, 0.3, v, t, gplanes=g, gsky=gs, loss=loss, accumulate=i > 0)
        r.adam_step(p, g, m, s, 0.5 / 255.0, it + 1)
        torch.cuda.synchronize()
        assert abs(float(loss[0]) - losses[it]) <= 1e-5 * abs(float(loss[0]))


@pytest.mark.parametrize("h,w,size", [(1537, 2049, 256), (1535, 2049, 256), (1537, 2049, 200)])
def test_adjoint_rows_per_thread(ctx, h, w, size):
    """Both adjoints against the oracle on either side of 3 * 2^20 pixels,
    where a thread takes four rows instead of two, with ragged last blocks
    (an odd row, one column)."""
    col, hts = scene.scene_maps(31, 256)
    r = DiffRenderer(ctx, ctx.map(col, hts, shade_size=size))
    sf = O.shade_factor(O.shadow_counts(np.asarray(hts, np.int32) & 255, O.sun(0.1, 0.1), size))
    rng = np.random.default_rng(h + size)
    planes = rng.random((3, size, size), dtype=np.float32)
    d, z0 = scene.depth_for(700, 500.0)
    v = View(x=50.3, y=20.7, height=290.0, angle=0.9, horizon=0.1 * h, distance=500.0, fov=1.2,
             h=h, w=w, d=d, z0=z0, n_slices=700)
    tp = torch.from_numpy(planes).cuda()
    target = torch.from_numpy(rng.random((3, h, w), dtype=np.float32)).cuda()
    img, src, gp, gs, loss = r.l2_step(tp, 0.4, v, target)
    gimg = torch.from_numpy(rng.standard_normal((3, h, w)).astype(np.float32)).cuda()
    gp2, gs2 = r.vjp_raw(tp, src, gimg, v)
    torch.cuda.synchronize()
    want_img, want_src = O.render_f32(v, planes, sf, np.asarray(hts, np.int32) & 255, 0.4)
    assert np.array_equal(img.cpu().numpy().view(np.uint32), want_img.view(np.uint32))
    g = 2.0 * (want_img - target.cpu().numpy())
    for got, sky, gi in ((gp, gs, g.astype(np.float32)), (gp2, gs2, gimg.cpu().numpy())):
        want, want_sky = O.render_f32_vjp(v, planes, sf, want_src, gi)
        assert _rel_err(got.cpu().numpy(), want) <= 1e-5
        mass = np.abs(gi[:, want_src < 0]).sum() + 1e-3
        assert abs(float(sky[0]) - float(want_sky)) <= 1e-5 * mass
    want_loss = float(((want_img.astype(np.float64) - target.cpu().numpy()) ** 2).sum())
    assert abs(float(loss[0]) - want_loss) <= 1e-5 * want_loss


@pytest.mark.parametrize("size", [128, 100])
def test_adjoint_of_slices_past_the_views_last(ctx, size):
    """vjp over a src that names slices past the view's own count (the same
    depths, more of them): the gradient is that of the longer view."""
    import dataclasses
    r, col, _, _ = _setup(ctx, size=128)
    r = DiffRenderer(ctx, ctx.map(*scene.scene_maps(11, 128), shade_size=size))
    long = dataclasses.replace(VIEWS[0], n_slices=200)
    short = dataclasses.replace(long, n_slices=20)
    planes = torch.from_numpy(np.ascontiguousarray(planes_of(col)[:, :size, :size])).cuda()
    src = r.forward_raw(planes, 0.3, long)[1]
    rng = np.random.default_rng(5)
    gimg = torch.from_numpy(rng.standard_normal((3, long.h, long.w)).astype(np.float32)).cuda()
    want = r.vjp_raw(planes, src, gimg, long)[0]
    got = r.vjp_raw(planes, src, gimg, short)[0]
    torch.cuda.synchronize()
    assert int(src.max()) >= 20
    assert _rel_err(got.cpu().numpy(), want.cpu().numpy()) <= 1e-5


@pytest.mark.parametrize("n", [1, 3, 4, 1027, 4096 * 1024 + 5])
def test_adam_first_step_takes_the_moments_as_zero(ctx, n):
    """adam_step(first=True) over moments of any content: bit for bit the
    first step from zero moments (vector part and scalar tail)."""
    r, _, _, _ = _setup(ctx)
    rng = np.random.default_rng(n)
    p = torch.from_numpy(rng.random(n, dtype=np.float32)).cuda()
    g = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).cuda()
    g[0] = -0.0
    q, zeros = p.clone(), [torch.zeros_like(p) for _ in range(2)]
    junk = [torch.full_like(p, float("nan")) for _ in range(2)]
    r.adam_step(p, g, *zeros, 0.01, 1)
    r.adam_step(q, g, *junk, 0.01, 1, first=True)
    torch.cuda.synchronize()
    for a, b in zip([p] + zeros, [q] + junk):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    with pytest.raises(ValueError):
        r.adam_step(p, g, *zeros, 0.01, 2, first=True)


class _Recorder(DiffRenderer):
    """A renderer that notes, per l2_step, whether src was given as known and
    where it lies."""

    def __init__(self, *args):
        super().__init__(*args)
        self.known, self.at = [], []

    def l2_step(self, planes, sky, view, target, img=None, src=None, *args, visible=False, **kw):
        self.known.append(visible)
        self.at.append(src.data_ptr())
        return super().l2_step(planes, sky, view, target, img, src, *args, visible=visible, **kw)


def _fit_setup(ctx, views):
    _, col, _, _ = _setup(ctx)
    r = _Recorder(ctx, ctx.map(*scene.scene_maps(11, 128), shade_size=128))
    planes = torch.from_numpy(planes_of(col)).cuda()
    goal = (planes * 0.5).contiguous()
    targets = [r.forward_raw(goal, 0.3, v)[0] for v in views]
    torch.cuda.synchronize()
    return r, planes, goal, targets


def test_fit_follows_a_camera_moved_in_place(ctx):
    """A view whose fields are arrays that on_step changes in place is
    rendered anew: what counts are the values handed to the renderer, not the
    objects that hold them."""
    import dataclasses
    view = dataclasses.replace(VIEWS[0], x=np.array(VIEWS[0].x))
    r, planes, goal, targets = _fit_setup(ctx, [view])
    moved = dataclasses.replace(VIEWS[0], x=float(view.x) + 7.25)

    def move(it):
        if it == 0:
            view.x += 7.25
            targets[0] = r.forward_raw(goal, 0.3, moved)[0]

    fit(r, planes, [view], targets, 0.3, steps=3, on_step=move)
    assert r.known == [False, False, True]


def test_fit_takes_any_view_that_gives_its_c_form(ctx):
    """A camera needs h, w and to_c, and no more."""
    from types import SimpleNamespace
    view = SimpleNamespace(h=VIEWS[0].h, w=VIEWS[0].w, to_c=VIEWS[0].to_c)
    r, planes, _, targets = _fit_setup(ctx, [VIEWS[0]])
    other = planes.clone()
    losses = fit(r, planes, [view], targets, 0.3, steps=2).cpu().numpy()
    want = fit(r, other, [VIEWS[0]], targets, 0.3, steps=2).cpu().numpy()
    assert np.allclose(losses, want, rtol=1e-5, atol=0.0)
    assert r.known == [False, True, False, True]


def test_fit_refuses_a_map_closed_meanwhile(ctx):
    r, planes, _, targets = _fit_setup(ctx, [VIEWS[0]])
    with pytest.raises(Exception, match="fsx_render_f32_l2_step"):
        fit(r, planes, [VIEWS[0]], targets, 0.3, steps=2, on_step=lambda it: r.map.close())


def _no_memory_free(monkeypatch):
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda *a: (0, 1 << 38))
    monkeypatch.setattr(torch.cuda, "memory_reserved", lambda *a: 1 << 20)
    monkeypatch.setattr(torch.cuda, "memory_allocated", lambda *a: 1 << 20)


@pytest.mark.parametrize("steps,full", [(1, False), (3, True)])
def test_fit_shares_one_buffer_where_it_keeps_none(ctx, steps, full, monkeypatch):
    """With no memory free, or one step only, views of one size share a
    buffer of visible slices."""
    import dataclasses
    views = [dataclasses.replace(VIEWS[0], angle=a) for a in (0.4, 1.4, 2.4)]
    r, planes, _, targets = _fit_setup(ctx, views)
    if full:
        _no_memory_free(monkeypatch)
    fit(r, planes, views, targets, 0.3, steps=steps)
    assert len(set(r.at)) == 1 and not any(r.known)


def test_fit_counts_the_memory_torch_holds_unused(ctx, monkeypatch):
    r, planes, _, targets = _fit_setup(ctx, [VIEWS[0]])
    _no_memory_free(monkeypatch)
    monkeypatch.setattr(torch.cuda, "memory_reserved", lambda *a: 1 << 30)
    fit(r, planes, [VIEWS[0]], targets, 0.3, steps=2)
    assert r.known == [False, True]


def test_fit_gives_up_what_it_holds_where_memory_runs_out(ctx, monkeypatch):
    """An allocation that fails while views' visible slices are held is
    repeated without them, and the fit goes on to the same result."""
    import dataclasses

    from futspace_amd import diff
    views = [dataclasses.replace(VIEWS[0], angle=a) for a in (0.4, 1.4, 2.4)]
    r, planes, _, targets = _fit_setup(ctx, views)
    want = fit(r, planes.clone(), views, targets, 0.3, steps=3).cpu().numpy()
    empty, made = torch.empty, []

    def short(*args, **kw):
        if kw.get("dtype") == torch.int32:
            made.append(args[0])
            if len(made) == 3:
                raise torch.cuda.OutOfMemoryError("no room for a third buffer")
        return empty(*args, **kw)

    monkeypatch.setattr(diff.torch, "empty", short)
    got = fit(r, planes.clone(), views, targets, 0.3, steps=3).cpu().numpy()
    assert len(made) > 3 and np.allclose(got, want, rtol=1e-5, atol=0.0)


def test_given_visibility_is_a_dense_int32_image_on_the_device(ctx):
    """With visible=True src is read: what is not laid out as the kernel reads
    it is refused before anything is queued."""
    r, col, _, _ = _setup(ctx)
    tp, v = torch.from_numpy(planes_of(col)).cuda(), VIEWS[0]
    _, src = r.forward_raw(tp, 0.3, v)
    target = torch.zeros((3, v.h, v.w), device="cuda")
    torch.cuda.synchronize()
    wide = torch.zeros((v.h, 2 * v.w), dtype=torch.int32, device="cuda")
    row = torch.zeros((1, v.w), dtype=torch.int32, device="cuda")
    for bad in (src.long(), src.short(), src.float(), src.cpu(), wide[:, ::2], wide[:, :v.w],
                row.expand(v.h, v.w), src.t().contiguous().t()):
        assert tuple(bad.shape) == (v.h, v.w)
        with pytest.raises(ValueError):
            r.l2_step(tp, 0.3, v, target, src=bad, visible=True)
    r.l2_step(tp, 0.3, v, target, src=src, visible=True)
    torch.cuda.synchronize()


@pytest.mark.parametrize("h,w", [(33, 70), (9, 1), (1537, 2049), (1543, 2050)])
@pytest.mark.parametrize("which", ["img", "gimg", "both", "none"])
def test_step_writes_the_images_it_is_given(ctx, h, w, which):
    """img and dL/dimg, each, both or neither, at both rows per thread and
    with partial blocks at either edge: bit-equal to the separate calls, in
    every pixel and in none beyond the frame, and the same loss and gradients
    whatever is written."""
    import ctypes

    from futspace_amd.diff import _ptr
    r, col, _, _ = _setup(ctx)
    tp = torch.from_numpy(planes_of(col)).cuda()
    v = View(x=64.3, y=100.7, height=260.0, angle=0.4, horizon=h * 0.6, distance=300.0, fov=1.2,
             h=h, w=w, d=0.01, z0=0.5, scale=h / 2.0)
    target = torch.rand((3, h, w), device="cuda",
                        generator=torch.Generator(device="cuda").manual_seed(h))
    img, src = r.forward_raw(tp, 0.37, v)
    gimg, loss = r.l2_loss_grad(img, target)
    gp, gs = r.vjp_raw(tp, src, gimg, v)
    n = 3 * h * w
    out = {k: torch.full((n + 64,), 7.0, device="cuda") for k in ("img", "gimg")}
    given = {k: _ptr(b) if which in (k, "both") else None for k, b in out.items()}
    f_gp, f_src = torch.full_like(tp, 9.0), torch.full_like(src, 5)
    f_gs, f_loss = torch.ones(1, device="cuda"), torch.ones(1, device="cuda")
    torch.cuda.synchronize()
    cv = v.to_c()
    ctx.check(ctx.lib.fsx_render_f32_l2_step(
        ctx.ptr, r.map.ptr, ctypes.byref(cv), _ptr(tp), _ptr(r.sf), r.hc, r.wc,
        ctypes.c_float(0.37), _ptr(target), 0, given["img"], _ptr(f_src), given["gimg"],
        _ptr(f_gp), _ptr(f_gs), _ptr(f_loss)), "fsx_render_f32_l2_step")
    ctx.sync()
    for k, want in (("img", img), ("gimg", gimg)):
        if given[k]:
            assert torch.equal(out[k][:n], want.reshape(-1)) and bool((out[k][n:] == 7.0).all())
        else:
            assert bool((out[k] == 7.0).all())
    assert torch.equal(f_src, src)
    assert abs(float(f_loss[0]) - float(loss[0])) <= 1e-5 * float(loss[0])
    assert _rel_err(f_gp.cpu().numpy(), gp.cpu().numpy()) <= 1e-5
    sky = float(gimg[:, src < 0].abs().sum())
    assert abs(float(f_gs[0]) - float(gs[0])) <= 1e-5 * max(sky, 1e-3)
