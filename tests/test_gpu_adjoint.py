"""Path-replay adjoint on the GPU.

Checks: (1) equality with the oracle's replay of the same fp32 paths (only the
fp64 summation order differs); (2) central finite differences (h = 1e-3, common
random numbers) of the GPU forward renders: without Russian roulette to 1e-3
(relative L2 of the whole gradient vector), and at the full 512x512 64-sample
configuration within 1% on every seed; with roulette, the mean over 40 seeds within
1% (tests/adjoint_fd.py);
(3) first-order gradients (no roulette curvature term) against the oracle's fp64
paths at 4x the samples, the loss adjoint taken from 256-sample images
(statistical tolerance 10%);
(4) the torch.autograd harness returns the adjoint's gradients.
"""
import numpy as np
import pytest

import cudart_amd as ca
import oracle as O
from cudart_amd import workloads as W

pytestmark = pytest.mark.gpu


def _setup(w, h, spp, seed=1, max_depth=None, rr_start=3, render_seed=W.SEED):
    # Scene, renderer and a target from perturbed parameters (another seed).
    wl = W.cornell100k(w, h)
    if max_depth is not None:
        wl.max_depth = max_depth
    scene = ca.Scene(wl.mesh)
    mats = wl.mesh.materials
    kd0 = np.array([list(m.kd) for m in mats], np.float32)
    em0 = np.array([m.ka[0] for m in mats], np.float32)
    rng = np.random.default_rng(seed)
    kdT = np.clip(kd0 + rng.uniform(-0.1, 0.1, kd0.shape), 0.05, 0.95).astype(np.float32)
    emT = (em0 + np.where(em0 > 0, rng.uniform(-0.1, 0.1, len(mats)), 0)).astype(np.float32)
    r = ca.ParallelRenderer(scene, w, h, spp, camera=wl.camera, max_depth=wl.max_depth, rr_start=rr_start,
                            seed=render_seed, integrator=ca.INTEGRATOR_WAVEFRONT)

    def render(kd, em):
        for i in range(len(mats)):
            scene.set_material_params(i, kd[i], float(em[i]))
        r.reset()
        r.render(spp)
        return r.radiance()

    # The target comes from other random numbers than the image (as a photograph
    # would): a target correlated with the image's own roulette decisions would bias
    # the comparison of the boundary terms of those decisions.
    rt = ca.ParallelRenderer(scene, w, h, spp, camera=wl.camera, max_depth=wl.max_depth, rr_start=rr_start,
                             seed=render_seed ^ 0x7A5C3E1, integrator=ca.INTEGRATOR_WAVEFRONT)
    for i in range(len(mats)):
        scene.set_material_params(i, kdT[i], float(emT[i]))
    rt.render(spp)
    target = rt.radiance()
    rt.close()
    image = render(kd0, em0)
    return wl, scene, r, render, kd0, em0, target, image


# 64x64 at 4 spp: 64 whole 8x8 tiles, each replayed by 4 workgroups of one sample;
# 60x44 at 3 spp: partial tiles at the right and bottom edges, whose pixel-samples
# split unevenly over 3 workgroups.
@pytest.mark.parametrize("w,h,spp", [(64, 64, 4), (60, 44, 3)])
def test_adjoint_equals_oracle_replay(gpu, w, h, spp):
    wl, scene, r, render, kd0, em0, target, image = _setup(w, h, spp)
    d_alb, d_em, loss = r.adjoint(target, spp, image=image)
    orc = O.OracleScene(wl.mesh.desc())
    oa, oe = orc.adjoint(wl.camera, w, h, spp, O.cfg(max_depth=wl.max_depth, seed=W.SEED), image, target)
    g = np.concatenate([d_alb.ravel(), d_em]).astype(np.float64)
    og = np.concatenate([oa.ravel(), oe])
    scale = np.abs(og).max()
    assert scale > 0
    np.testing.assert_allclose(g, og, rtol=1e-5, atol=1e-7 * scale)
    assert loss == pytest.approx(float(np.mean((image.astype(np.float64) - target) ** 2)), rel=1e-6)


def _fd_gradient(render, kd0, em0, loss, h=1e-3):
    M = len(em0)
    fd_alb = np.zeros((M, 3))
    fd_em = np.zeros(M)
    for m in range(M):
        for c in range(3):
            kp, km = kd0.copy(), kd0.copy()
            kp[m, c] += h
            km[m, c] -= h
            fd_alb[m, c] = (loss(render(kp, em0)) - loss(render(km, em0))) / (2 * h)
        ep, en = em0.copy(), em0.copy()
        ep[m] += h
        en[m] -= h
        fd_em[m] = (loss(render(kd0, ep)) - loss(render(kd0, en))) / (2 * h)
    return np.concatenate([fd_alb.ravel(), fd_em])


def test_adjoint_matches_central_differences_without_roulette(gpu):
    # Without Russian roulette (rr_start beyond max_depth) the estimator is a smooth
    # function of albedo and emission for fixed random numbers, so central differences
    # of the same renders must reproduce the adjoint closely.
    spp = 16
    wl, scene, r, render, kd0, em0, target, image = _setup(128, 128, spp, max_depth=4, rr_start=8)
    d_alb, d_em, _ = r.adjoint(target, spp, image=image)
    loss = lambda img: float(np.mean((img.astype(np.float64) - target) ** 2))  # noqa: E731
    fd = _fd_gradient(render, kd0, em0, loss)
    g = np.concatenate([d_alb.ravel(), d_em]).astype(np.float64)
    rel = np.linalg.norm(g - fd) / np.linalg.norm(fd)
    print(f"no roulette: relative L2 error vs central FD {rel:.2e}")
    assert rel <= 1e-3
    big = np.abs(fd) >= 0.1 * np.abs(fd).max()
    np.testing.assert_allclose(g[big], fd[big], rtol=5e-3)


def test_adjoint_matches_central_differences_c4_without_roulette(gpu):
    # The differentiable-render configuration at full size (512x512, 64 samples,
    # depth 6) without Russian roulette: for fixed random numbers the image is a
    # polynomial in the albedos and emissions, so central differences (h = 1e-3) of
    # the same renders must give the adjoint's gradient on every seed, within 1%.
    from tests.adjoint_fd import compare, seed_list
    errs, g, fd, g1, each = compare(seed_list(2), rr_start=64, target_spp=128)
    print(f"C4 without roulette: relative L2 error per seed {each}")
    assert max(each) <= 0.01


def test_adjoint_matches_central_differences_c4(gpu):
    # 512x512, 64 samples, depth 6 with Russian roulette from bounce 3: the mean over
    # 40 seeds of the adjoint against the mean of central differences (h = 1e-3),
    # within 1%. The roulette flips inside +-h make each seed's differences noisy
    # (2-5% relative L2 per seed); the mean over 40 seeds brings that noise near
    # 0.5%. Without the roulette curvature term the adjoint is biased by about 6%,
    # which this test must resolve. About 2.6 s per seed on an MI355X.
    from tests.adjoint_fd import compare, seed_list
    errs, g, fd, g1, each = compare(seed_list(40))
    first_order = np.linalg.norm(g1 - fd) / np.linalg.norm(fd)
    print(f"C4: relative L2 error of the mean over 40 seeds {errs[-1]:.4f} (first-order {first_order:.4f}; "
          f"per seed {min(each):.4f}..{max(each):.4f})")
    assert errs[-1] <= 0.01
    assert first_order >= 2 * errs[-1]
    big = np.abs(fd) >= 0.2 * np.abs(fd).max()
    np.testing.assert_allclose(g[big], fd[big], rtol=0.03)


def test_adjoint_close_to_high_spp_fp64_reference(gpu):
    # Loss adjoint from nearly noise-free images (256 spp), so both sides estimate the
    # same quantity sum_p dLoss/dI_p * E[dI_p/dtheta]: the GPU with 64 samples of the
    # derivative, the oracle with 256 samples on fp64 paths.
    # First-order estimates (hess = 0) of the gradient of the loss of the expected image.
    wl, scene, r, render, kd0, em0, target, image = _setup(48, 48, 256)
    spp = 64
    grad = (2.0 / image.size) * (image.astype(np.float64) - target)
    d_alb, d_em = r.adjoint_grad(grad.astype(np.float32), spp, hess=0.0)
    orc = O.OracleScene(wl.mesh.desc())
    oa, oe = orc.adjoint(wl.camera, 48, 48, 256, O.cfg(max_depth=wl.max_depth, seed=W.SEED), image, target,
                         fp64=True, hess=0.0)
    g = np.concatenate([d_alb.ravel(), d_em]).astype(np.float64)
    og = np.concatenate([oa.ravel(), oe])
    rel = np.linalg.norm(g - og) / np.linalg.norm(og)
    print(f"relative L2 difference vs 256-spp fp64 reference: {rel:.4f}")
    assert rel < 0.10  # Monte Carlo noise of the two estimates (about 0.05 expected)
    big = np.abs(og) >= 0.2 * np.abs(og).max()
    assert (np.sign(g[big]) == np.sign(og[big])).all()


def test_torch_autograd_harness(gpu):
    torch = pytest.importorskip("torch")
    from cudart_amd.torch_render import render as trender
    spp = 4
    wl, scene, r, render, kd0, em0, target, image = _setup(48, 40, spp)
    albedo = torch.tensor(kd0, requires_grad=True)
    emission = torch.tensor(em0, requires_grad=True)
    img = trender(albedo, emission, r, spp, 2.0 / image.size)
    assert np.array_equal(img.detach().numpy(), image)
    loss = ((img - torch.from_numpy(target)) ** 2).mean()
    loss.backward()
    d_alb, d_em, _ = r.adjoint(target, spp, image=image)
    np.testing.assert_allclose(albedo.grad.numpy(), d_alb, rtol=1e-4, atol=1e-7)
    np.testing.assert_allclose(emission.grad.numpy(), d_em, rtol=1e-4, atol=1e-7)


def test_torch_backward_uses_its_own_forward_parameters(gpu):
    # Two forward calls (other albedos the second time) before the first node's
    # backward: each node's gradient is the one at the parameters its own forward
    # rendered with, whatever the scene holds when backward runs.
    torch = pytest.importorskip("torch")
    from cudart_amd.torch_render import render as trender
    spp = 4
    wl, scene, r, render, kd0, em0, target, image = _setup(48, 40, spp)
    hess = 2.0 / image.size
    kd1 = np.clip(kd0 * 0.7 + 0.05, 0.05, 0.95).astype(np.float32)
    a0, e0 = torch.tensor(kd0, requires_grad=True), torch.tensor(em0, requires_grad=True)
    a1, e1 = torch.tensor(kd1, requires_grad=True), torch.tensor(em0, requires_grad=True)
    img0 = trender(a0, e0, r, spp, hess)
    img1 = trender(a1, e1, r, spp, hess)
    tt = torch.from_numpy(target)
    ((img0 - tt) ** 2).mean().backward()
    ((img1 - tt) ** 2).mean().backward()
    for kd, a, e, img in ((kd0, a0, e0, img0), (kd1, a1, e1, img1)):
        for m in range(len(em0)):
            scene.set_material_params(m, kd[m], float(em0[m]))
        d_alb, d_em, _ = r.adjoint(target, spp, image=img.detach().numpy())
        np.testing.assert_allclose(a.grad.numpy(), d_alb, rtol=1e-4, atol=1e-7)
        np.testing.assert_allclose(e.grad.numpy(), d_em, rtol=1e-4, atol=1e-7)
    assert not np.allclose(a0.grad.numpy(), a1.grad.numpy())
    # images and gradient images of another shape are refused before the C call
    with pytest.raises(ValueError):
        r.adjoint_grad(np.zeros((40, 48), np.float32), spp)
    with pytest.raises(ValueError):
        r.adjoint(np.zeros((48, 40, 3), np.float32), spp)
    with pytest.raises(ValueError):
        scene.set_material_params(0, [0.5, 0.5], 1.0)


@pytest.mark.parametrize("integrator", ["megakernel", "wavefront"])
def test_adjoint_with_kept_samples_equals_recomputed(gpu, integrator):
    # keep_samples: the forward pass stores each sample's radiance and the adjoint only
    # replays; the radiance is bit-identical to the primal trace, so are the gradients.
    wl = W.cornell100k(96, 80)
    scene = ca.Scene(wl.mesh)
    integ = ca.INTEGRATOR_WAVEFRONT if integrator == "wavefront" else ca.INTEGRATOR_MEGAKERNEL
    kw = dict(camera=wl.camera, max_depth=wl.max_depth, seed=W.SEED, integrator=integ)
    rk = ca.ParallelRenderer(scene, 96, 80, 8, keep_samples=1, **kw)
    rk.render(8)
    image = rk.radiance()
    target = np.clip(image * 0.9 + 0.01, 0, None).astype(np.float32)
    a_kept, e_kept, _ = rk.adjoint(target, 8, image=image)
    rp = ca.ParallelRenderer(scene, 96, 80, 8, **kw)
    rp.render(8)
    assert np.array_equal(rp.radiance(), image)
    a_rec, e_rec, _ = rp.adjoint(target, 8, image=image)
    np.testing.assert_array_equal(a_kept, a_rec)
    np.testing.assert_array_equal(e_kept, e_rec)
    # a material change after the forward pass invalidates the kept samples
    kd = np.array(wl.mesh.materials[0].kd, np.float32)
    scene.set_material_params(0, kd, float(wl.mesh.materials[0].ka[0]))
    a2, e2, _ = rk.adjoint(target, 8, image=image)
    np.testing.assert_array_equal(a2, a_rec)


def test_adjoint_primal_in_replay_equals_kept(gpu, monkeypatch):
    """The fallback for when the per-sample buffer does not fit: each lane traces its
    sample's primal path inside the replay kernel. Same radiance, same schedule,
    so the gradients equal the kept-radiance ones bit for bit."""
    wl = W.cornell100k(96, 80)
    scene = ca.Scene(wl.mesh)
    kw = dict(camera=wl.camera, max_depth=wl.max_depth, seed=W.SEED)
    rk = ca.ParallelRenderer(scene, 96, 80, 8, keep_samples=1, **kw)
    rk.render(8)
    image = rk.radiance()
    target = np.clip(image * 0.9 + 0.01, 0, None).astype(np.float32)
    a_kept, e_kept, _ = rk.adjoint(target, 8, image=image)
    rp = ca.ParallelRenderer(scene, 96, 80, 8, **kw)
    monkeypatch.setenv("PRT_ADJOINT_PRIMAL_IN_REPLAY", "1")
    a_in, e_in, _ = rp.adjoint(target, 8, image=image)
    np.testing.assert_array_equal(a_kept, a_in)
    np.testing.assert_array_equal(e_kept, e_in)


# The replay from kept path vertices against the replay that traces every ray: one pixel and
# ragged tiles, one sample to more than a wave's, the shortest and the longest paths,
# roulette from the first vertex and never, textured albedos, many materials. The same fp32 paths give the same fp64 terms, summed in another
# order: the results differ by a rounding to fp32 at most (2^-23), and by about 1e-16 of the
# summed terms where those cancel.
@pytest.mark.parametrize("kind,w,h,spp,depth,rr_start", [
    ("box", 1, 1, 1, 1, 3), ("box", 17, 9, 5, 16, 0), ("box", 9, 23, 70, 6, 3), ("box", 16, 8, 64, 2, 99),
    ("terrain", 33, 12, 8, 8, 3), ("materials", 25, 14, 16, 7, 2)])
def test_replay_from_vertices_equals_traced_replay(gpu, monkeypatch, kind, w, h, spp, depth, rr_start):
    mesh = {"box": lambda: W.cornell100k(w, h).mesh,
            "terrain": lambda: W.large(w, h, params="grid=60;instances=20;textures=4;texsize=32;materials=12").mesh,
            "materials": lambda: ca.Mesh.generate("spheres", f"instances=60;level=2;materials=125;width={w};height={h}",
                                                  3)}[kind]()
    scene = ca.Scene(mesh)
    rng = np.random.default_rng(5)
    grad = rng.standard_normal((h, w, 3)).astype(np.float32)
    kw = dict(camera=mesh.camera, max_depth=depth, rr_start=rr_start, seed=11, integrator=ca.INTEGRATOR_WAVEFRONT)
    kept = ca.ParallelRenderer(scene, w, h, spp, keep_samples=1, **kw)
    kept.render(spp)
    plain = ca.ParallelRenderer(scene, w, h, spp, **kw)
    from_kept = kept.adjoint_grad(grad, spp, hess=0.25)
    from_own = plain.adjoint_grad(grad, spp, hess=0.25)
    monkeypatch.setenv("PRT_ADJOINT_PRIMAL_IN_REPLAY", "1")
    traced = plain.adjoint_grad(grad, spp, hess=0.25)
    for a, b, c in zip(from_kept, from_own, traced):
        np.testing.assert_array_equal(a, b)
        np.testing.assert_allclose(a, c, rtol=2.0 ** -22, atol=1e-9 * np.abs(c).max())


# Vertices kept by either integrator's render, and those of the adjoint's own forward pass (by
# the megakernel up to 2^20 paths, by the wavefront above): the same paths, so the same bits.
# One pixel, ragged blocks, lanes sharing a pixel and not, both sides of the line.
@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (17, 9, 5), (125, 93, 8), (128, 128, 64), (128, 128, 65)])
def test_vertices_of_both_integrators_are_the_same(gpu, w, h, spp):
    mesh = W.cornell100k(w, h).mesh
    scene = ca.Scene(mesh)
    grad = np.random.default_rng(6).standard_normal((h, w, 3)).astype(np.float32)
    kw = dict(camera=mesh.camera, max_depth=7, rr_start=2, seed=12)
    results = []
    for integrator in (ca.INTEGRATOR_MEGAKERNEL, ca.INTEGRATOR_WAVEFRONT):
        r = ca.ParallelRenderer(scene, w, h, spp, keep_samples=1, integrator=integrator, **kw)
        r.render(spp)
        results.append(r.adjoint_grad(grad, spp, hess=0.25))
        r.close()
    r = ca.ParallelRenderer(scene, w, h, spp, **kw)
    results.append(r.adjoint_grad(grad, spp, hess=0.25))
    r.close()
    for other in results[1:]:
        for a, b in zip(results[0], other):
            np.testing.assert_array_equal(a, b)


def _deep_scene(w, h):
    from tests.helpers import OwnedDesc, nested_quads
    p, n, m, mats = nested_quads()
    cam = ca.camera_look_at((0, 0, 2), (0, 0, 0), (0, 1, 0), 40, w, h)
    od = OwnedDesc(p, n, m, mats, cam)
    return ca.Scene(od.desc), cam, 1


def _box_scene(w, h):
    mesh = W.cornell100k(w, h).mesh
    return ca.Scene(mesh), mesh.camera, next(i for i, m in enumerate(mesh.materials) if m.ka[0] > 0)


# The replay from vertices that a forward pass left and the one that finds them by tracing add
# the same terms in the same order: equal bits, also where the sum cancels to its rounding.
# Ragged tiles, a tile's samples in one and in several workgroups, and stacks beyond 32 entries.
@pytest.mark.parametrize("kind,w,h,spp,depth,rr_start", [
    ("box", 17, 9, 5, 16, 0), ("box", 9, 23, 70, 6, 3), ("box", 96, 80, 8, 6, 3), ("deep", 33, 18, 1, 3, 3),
    ("deep", 40, 31, 12, 4, 1)])
def test_traced_replay_adds_in_the_order_of_the_stored_one(gpu, monkeypatch, kind, w, h, spp, depth, rr_start):
    from tests.helpers import cancelling_grad
    scene, cam, light = {"box": _box_scene, "deep": _deep_scene}[kind](w, h)
    kw = dict(camera=cam, max_depth=depth, rr_start=rr_start, seed=11)
    r = ca.ParallelRenderer(scene, w, h, spp, **kw)
    kept = ca.ParallelRenderer(scene, w, h, spp, keep_samples=1, integrator=ca.INTEGRATOR_WAVEFRONT, **kw)
    kept.render(spp)
    cancel = cancelling_grad(lambda g: r.adjoint_grad(g, spp, hess=0.0)[1].astype(np.float64), w, h, light)
    noisy = np.random.default_rng(5).standard_normal((h, w, 3)).astype(np.float32)
    for grad, hess in ((cancel, 0.0), (noisy, 0.25)):
        stored = r.adjoint_grad(grad, spp, hess=hess)
        from_kept = kept.adjoint_grad(grad, spp, hess=hess)
        with monkeypatch.context() as m:
            m.setenv("PRT_ADJOINT_PRIMAL_IN_REPLAY", "1")
            traced = r.adjoint_grad(grad, spp, hess=hess)
        for a, b, c in zip(stored, from_kept, traced):
            np.testing.assert_array_equal(a, b)
            np.testing.assert_array_equal(a, c)


# The split of the sums depends on the call alone: not on the sample count that the renderer
# was made for, nor on what earlier calls made it allocate.
def test_repeated_gradients_have_the_same_bits(gpu):
    from tests.helpers import cancelling_grad
    w, h, spp = 96, 80, 16
    scene, cam, light = _box_scene(w, h)
    kw = dict(camera=cam, max_depth=6, seed=11)
    made_for = ca.ParallelRenderer(scene, w, h, spp, **kw)
    grad = cancelling_grad(lambda g: made_for.adjoint_grad(g, spp, hess=0.0)[1].astype(np.float64), w, h, light)
    want = made_for.adjoint_grad(grad, spp, hess=0.0)
    for integrator in (ca.INTEGRATOR_MEGAKERNEL, ca.INTEGRATOR_WAVEFRONT):
        r = ca.ParallelRenderer(scene, w, h, 1, integrator=integrator, **kw)
        for call in range(3):
            if call == 2:
                r.render(64)
            for a, b in zip(r.adjoint_grad(grad, spp, hess=0.0), want):
                np.testing.assert_array_equal(a, b)


# The memory of a gradient call is one block for all renderers, not one each.
def test_gradients_of_several_renderers_share_their_memory(gpu):
    from tests.helpers import device_free_bytes
    w, h, spp = 512, 256, 64
    scene, cam, _ = _box_scene(w, h)
    grad = np.random.default_rng(9).standard_normal((h, w, 3)).astype(np.float32)
    block = w * h * spp * (16 + 4 * 6)  # radiance and vertices
    left, renderers, results = [], [], []
    for seed in (1, 2, 3, 1):
        renderers.append(ca.ParallelRenderer(scene, w, h, spp, camera=cam, max_depth=6, seed=seed))
        results.append(renderers[-1].adjoint_grad(grad, spp, hess=0.25))
        left.append(device_free_bytes())
    assert left[0] - left[-1] < block, left
    for a, b in zip(results[0], results[-1]):
        np.testing.assert_array_equal(a, b)
    for r in renderers:
        r.close()
    scene.close()


# Run by itself below: the driver clears the pages of a process that has used most of the memory.
_FULL_DEVICE = """
import ctypes as C
import numpy as np
import cudart_amd as ca
from cudart_amd import workloads as W
from tests.helpers import device_free_bytes

w = h = 512
scene = ca.Scene(W.cornell100k(w, h).mesh)
cam = W.cornell100k(w, h).camera
kw = dict(camera=cam, max_depth=16, keep_samples=1, integrator=ca.INTEGRATOR_WAVEFRONT)
grad = np.random.default_rng(9).standard_normal((h, w, 3)).astype(np.float32)
before = device_free_bytes()
first = ca.ParallelRenderer(scene, w, h, 128, seed=1, **kw)
kept = 128 * w * h * (16 + 4 * 16)
assert before - device_free_bytes() >= kept, (before, device_free_bytes())
first.render(8)
want = first.adjoint_grad(grad, 8, hess=0.25)
hip = C.CDLL(next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64.so" in l))
filler = C.c_void_p()
left = device_free_bytes()
samples = 192 * w * h * 16  # of the second renderer: more than is left free, less than with the vertices
assert hip.hipMalloc(C.byref(filler), C.c_size_t(left - samples // 2)) == 0
print("filled", flush=True)
second = ca.ParallelRenderer(scene, w, h, 192, seed=1, **kw)
hip.hipFree(filler)
for r in (first, second):
    r.reset()
    r.render(8)
    for a, b in zip(r.adjoint_grad(grad, 8, hess=0.25), want):
        assert np.array_equal(a, b)
    r.close()
print("ok")
"""


def test_kept_vertices_give_way_to_a_renderer_that_needs_the_room(gpu):
    import os
    import subprocess
    import sys
    from pathlib import Path
    root = Path(__file__).resolve().parent.parent
    out = subprocess.run([sys.executable, "-u", "-c", _FULL_DEVICE], cwd=root, capture_output=True, text=True,
                         timeout=100, env={**os.environ, "PYTHONPATH": str(root)})
    assert out.returncode == 0 and out.stdout.split()[-1] == "ok", out.stdout + out.stderr
