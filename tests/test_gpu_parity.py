"""HIP path vs the CPU oracle on the same seeded inputs.

Bar: first-hit triangle ids, material ids and t are bit-exact; radiance is
compared with a per-pixel relative tolerance of 1e-5 (absolute 1e-6) and, in
practice, every pixel is bit-identical because both sides evaluate the same
IEEE-754 operations in the same order. Ray counters (primary, extension,
shadow) must be equal, since both sides trace exactly the same paths.
"""
import numpy as np
import pytest

import cudart_amd as ca
import oracle as O
from cudart_amd import workloads as W

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-5, 1e-6


def _pair(wl, **cfg):
    scene = ca.Scene(wl.mesh)
    r = ca.ParallelRenderer(scene, wl.width, wl.height, wl.spp, camera=wl.camera, max_depth=wl.max_depth,
                            rr_start=wl.rr_start, seed=W.SEED, device=0, **cfg)
    orc = O.OracleScene(wl.mesh.desc())
    c = O.cfg(max_depth=wl.max_depth, rr_start=wl.rr_start, seed=W.SEED)
    return scene, r, orc, c


@pytest.mark.parametrize("sample", [0, 1, 7])
def test_first_hit_cornell_bitexact(gpu, sample):
    wl = W.cornell(256, 256)
    _, r, orc, c = _pair(wl)
    tri, mat, t = r.first_hit(sample)
    otri, omat, ot = orc.first_hit(wl.camera, wl.width, wl.height, sample, c)
    assert np.array_equal(tri, otri)
    assert np.array_equal(mat, omat)
    assert np.array_equal(t.view(np.uint32), ot.view(np.uint32))


def test_first_hit_spheres_bitexact(gpu):
    wl = W.spheres1m(320, 180, spp=1, instances=24)
    _, r, orc, c = _pair(wl)
    tri, mat, t = r.first_hit(3)
    otri, omat, ot = orc.first_hit(wl.camera, wl.width, wl.height, 3, c)
    assert (tri >= 0).mean() > 0.3
    assert np.array_equal(tri, otri)
    assert np.array_equal(mat, omat)
    assert np.array_equal(t.view(np.uint32), ot.view(np.uint32))


def _axis_camera(eye, d, up):
    """A camera whose every primary ray is exactly d: with fov = 0 the pixel offsets
    (right * fov * aspect * ni, up * fov * nj) vanish."""
    cam = ca.Camera()
    cam.eye[:] = [float(x) for x in eye]
    cam.dir[:] = [float(x) for x in d]
    cam.up[:] = [float(x) for x in up]
    cam.right[:] = [float(x) for x in np.cross(d, up)]
    cam.fov = 0.0
    cam.aspect = 1.0
    cam.aperture_width = 0.0
    cam.focus_distance = 1.0
    cam.xpixels = cam.ypixels = 1
    return cam


def test_first_hit_axis_aligned_rays_bitexact(gpu):
    """Rays with exactly zero direction components (1/0 = inf in the slab test).
    Regression: with p * inf - o * inf the slab parameter was NaN, and a box the ray
    runs inside could be culled (or the ray walked most of the tree)."""
    wl = W.spheres1m(8, 8, spp=1, instances=24)
    scene = ca.Scene(wl.mesh)
    orc = O.OracleScene(wl.mesh.desc())
    c = O.cfg(max_depth=wl.max_depth, rr_start=wl.rr_start, seed=W.SEED)
    grid = np.linspace(-11.0, 11.0, 7)
    views = []
    for a in grid:
        for b in grid:
            views.append(((a, 40.0, b), (0.0, -1.0, 0.0), (0.0, 0.0, -1.0)))   # down onto spheres and ground
            views.append(((-60.0, 11.0 + a / 2, b), (1.0, 0.0, 0.0), (0.0, 1.0, 0.0)))  # along +x
            views.append(((a, 11.0 + b / 2, 60.0), (0.0, 0.0, -1.0), (0.0, 1.0, 0.0)))  # along -z
    hits = 0
    for eye, d, up in views:
        cam = _axis_camera(eye, d, up)
        r = ca.ParallelRenderer(scene, 1, 1, 1, camera=cam, max_depth=wl.max_depth, rr_start=wl.rr_start,
                                seed=W.SEED, device=0)
        tri, mat, t = r.first_hit(0)
        r.close()
        otri, omat, ot = orc.first_hit(cam, 1, 1, 0, c)
        btri, _, bt = orc.first_hit(cam, 1, 1, 0, c, brute=True)  # O(N) scan, no boxes
        assert np.array_equal(otri, btri) and np.array_equal(ot.view(np.uint32), bt.view(np.uint32))
        assert np.array_equal(tri, otri), (eye, d, tri, otri)
        assert np.array_equal(mat, omat)
        assert np.array_equal(t.view(np.uint32), ot.view(np.uint32))
        hits += int(tri[0, 0] >= 0)
    assert hits > len(views) // 3


def test_radiance_cornell_matches_oracle(gpu):
    wl = W.cornell(256, 256, spp=16, max_depth=5)
    _, r, orc, c = _pair(wl, count_rays=1)
    r.render(wl.spp)
    img = r.radiance()
    acc, cnt = orc.render(wl.camera, wl.width, wl.height, 0, wl.spp, c)
    oimg = acc / np.float32(wl.spp)
    assert np.isfinite(img).all()
    np.testing.assert_allclose(img, oimg, rtol=RTOL, atol=ATOL)
    st = r.stats()
    assert (st.primary_rays, st.extension_rays, st.shadow_rays) == tuple(int(x) for x in cnt)
    exact = np.mean(img.view(np.uint32) == oimg.view(np.uint32))
    print(f"bit-identical pixels: {exact:.6f}")


def test_radiance_spheres_matches_oracle(gpu):
    wl = W.spheres1m(192, 108, spp=4, max_depth=8, instances=40)
    _, r, orc, c = _pair(wl, count_rays=1)
    r.render(wl.spp)
    img = r.radiance()
    acc, cnt = orc.render(wl.camera, wl.width, wl.height, 0, wl.spp, c)
    oimg = acc / np.float32(wl.spp)
    np.testing.assert_allclose(img, oimg, rtol=RTOL, atol=ATOL)
    st = r.stats()
    assert (st.primary_rays, st.extension_rays, st.shadow_rays) == tuple(int(x) for x in cnt)


def test_samples_per_launch_and_determinism(gpu):
    wl = W.cornell(96, 64, spp=6, max_depth=6)
    scene = ca.Scene(wl.mesh)
    cam = ca.camera_look_at((2.2, 0.548, 0.0), (0.0, 0.548, 0.0), (0, 1, 0), 39.3, 96, 64)
    imgs = []
    for per in (1, 4, 6, 1):
        r = ca.ParallelRenderer(scene, 96, 64, 6, camera=cam, seed=9, spp_per_launch=per)
        r.render(6)
        imgs.append(r.radiance())
        r.close()
    for im in imgs[1:]:
        assert np.array_equal(im.view(np.uint32), imgs[0].view(np.uint32))


def test_progressive_equals_batch(gpu):
    """renderOneSamplePerPixel x n accumulates exactly like one n-sample call."""
    wl = W.cornell(64, 64, spp=5)
    scene = ca.Scene(wl.mesh)
    a = ca.ParallelRenderer(scene, 64, 64, 5, camera=wl.camera)
    for _ in range(5):
        a.renderOneSamplePerPixel()
    b = ca.ParallelRenderer(scene, 64, 64, 5, camera=wl.camera)
    b.render(5)
    assert a.getSamplesRendered() == 5
    assert np.array_equal(a.radiance(), b.radiance())


def test_image_bytes_match_oracle_tonemap(gpu):
    wl = W.cornell(64, 48, spp=3)
    cam = ca.camera_look_at((2.2, 0.548, 0.0), (0.0, 0.548, 0.0), (0, 1, 0), 39.3, 64, 48)
    scene = ca.Scene(wl.mesh)
    r = ca.ParallelRenderer(scene, 64, 48, 3, camera=cam)
    r.render(3)
    rgba = r.copyImageBytes()
    ref = O.tonemap(r.radiance()).reshape(48, 64, 4)
    assert np.array_equal(rgba, ref)


def test_radiance_textured_terrain_matches_oracle(gpu):
    # Small version of the large scene: fBm terrain + icospheres with UV-mapped RGBA8
    # textures (software bilinear with wrap on both sides).
    wl = W.large(160, 90, 4, params="grid=120;instances=40;textures=4;texsize=64;materials=12")
    assert any(m.tex_kd >= 0 for m in wl.mesh.materials)
    _, r, orc, c = _pair(wl, count_rays=1)
    r.render(wl.spp)
    img = r.radiance()
    acc, cnt = orc.render(wl.camera, wl.width, wl.height, 0, wl.spp, c)
    oimg = acc / np.float32(wl.spp)
    np.testing.assert_allclose(img, oimg, rtol=RTOL, atol=ATOL)
    st = r.stats()
    assert (st.primary_rays, st.extension_rays, st.shadow_rays) == tuple(int(x) for x in cnt)
    tri, mat, _ = r.first_hit(0)
    textured = [i for i, m in enumerate(wl.mesh.materials) if m.tex_kd >= 0]
    assert np.isin(mat, textured).mean() > 0.05


# The megakernel with 1 to 64 lanes to a pixel: every pixel block shape on images that it does
# not divide, launches of several rounds, several launches, and more launches than there are
# ticket sets, against one sample per pixel and launch.
@pytest.mark.parametrize("w,h,spp,per", [(1, 1, 64, 0), (37, 21, 2, 0), (37, 21, 4, 0), (37, 21, 13, 0), (21, 37, 48, 48),
                                         (19, 23, 127, 0), (19, 23, 96, 96), (33, 17, 40, 1), (300, 200, 32, 0)])
def test_lanes_sharing_pixels_equal_one_per_pixel(gpu, w, h, spp, per):
    scene = ca.Scene(W.spheres1m(w, h, instances=12).mesh)
    cam = ca.camera_look_at((4.0, 12.0, 35.0), (0.0, 8.0, 0.0), (0.0, 1.0, 0.0), 45.0, w, h)
    imgs = []
    for single in (True, False):
        r = ca.ParallelRenderer(scene, w, h, spp, camera=cam, max_depth=5, seed=3, count_rays=1,
                                spp_per_launch=1 if single else per)
        r.render(spp)
        st = r.stats()
        imgs.append((r.radiance().view(np.uint32), st.primary_rays, st.extension_rays, st.shadow_rays))
        r.close()
    assert np.array_equal(imgs[0][0], imgs[1][0])
    assert imgs[0][1:] == imgs[1][1:]


# Traversal stacks beyond every kernel's LDS entries (test_bvh.py walks the scene): first hits,
# one lane to a pixel and several, launches of more samples than the renderer was made for, and a
# renderer of the other integrator, whose stack area is made when it is first needed.
@pytest.mark.parametrize("w,h", [(40, 31), (300, 200)])
def test_deep_stacks_on_every_path(gpu, w, h):
    from tests.helpers import OwnedDesc, nested_quads
    p, n, m, mats = nested_quads()
    cam = ca.camera_look_at((0, 0, 2), (0, 0, 0), (0, 1, 0), 40, w, h)
    od = OwnedDesc(p, n, m, mats, cam)
    scene = ca.Scene(od.desc)
    orc, cfg = O.OracleScene(od.desc), O.cfg(max_depth=3, seed=5)
    want = orc.first_hit(cam, w, h, 0, cfg)
    acc, _ = orc.render(cam, w, h, 0, 8, cfg)
    kw = dict(camera=cam, max_depth=3, seed=5)
    for integrator in (ca.INTEGRATOR_MEGAKERNEL, ca.INTEGRATOR_WAVEFRONT):
        r = ca.ParallelRenderer(scene, w, h, 1, integrator=integrator, **kw)
        for _ in range(2):
            for a, b in zip(r.first_hit(0), want):
                assert np.array_equal(a, b)
            r.reset()
            r.render(8)
            np.testing.assert_allclose(r.radiance(), acc / np.float32(8), rtol=1e-5, atol=1e-6)
        r.close()
