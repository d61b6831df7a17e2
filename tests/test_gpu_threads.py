"""Renderers driven from several host threads at once. Each wavefront render captures
its chunk's launches into a HIP graph on the renderer's own stream; a legacy-stream
copy or fill issued by another thread during that capture makes HIP fail the
capture, so the library keeps every copy and fill on a renderer's stream. Two
threads rendering on two renderers at the same time must give exactly the images
that the same calls give one after the other."""
import threading

import numpy as np
import pytest

import cudart_amd as ca
import oracle as O
from cudart_amd import workloads as W

pytestmark = pytest.mark.gpu

CALLS, SPP = 24, 1


def _renderers(scene, wl):
    kw = dict(camera=wl.camera, max_depth=6, integrator=ca.INTEGRATOR_WAVEFRONT)
    return [ca.ParallelRenderer(scene, wl.width, wl.height, CALLS * SPP, seed=W.SEED + k, **kw) for k in range(2)]


def _work(r, errors):
    """Renders, reading the image back after each call (a readback's temporary
    device buffer is allocated and freed while the other thread may be capturing)."""
    try:
        for _ in range(CALLS):
            r.render(SPP)
            r.radiance()
    except Exception as e:  # reported by the main thread
        errors.append(e)


def test_two_threads_render_as_one_after_the_other(gpu):
    wl = W.cornell(96, 64, spp=CALLS * SPP, max_depth=6)
    scene = ca.Scene(wl.mesh)
    seq = _renderers(scene, wl)
    for r in seq:
        _work(r, [])
    want = [r.radiance() for r in seq]
    for r in seq:
        r.close()
    con = _renderers(scene, wl)
    errors = []
    threads = [threading.Thread(target=_work, args=(r, errors)) for r in con]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    got = [r.radiance() for r in con]
    for r in con:
        r.close()
    for a, b in zip(want, got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert not np.array_equal(want[0], want[1])  # the two views differ (seeds)


def test_two_threads_batch_as_one_after_the_other(gpu):
    """Two prt_render_batch calls at once (each on a stream of its own, each
    capturing its chunk's launches) give the images of the same calls made alone."""
    a = W.cornell(40, 30)
    b = W.spheres1m(50, 34, instances=12)
    sa, sb = ca.Scene(a.mesh), ca.Scene(b.mesh)
    batches = [[ca.BatchJob(sa, a.camera, 3, view_id=1), ca.BatchJob(sb, b.camera, 2, view_id=2)],
               [ca.BatchJob(sb, b.camera, 3, view_id=3), ca.BatchJob(sa, a.camera, 2, view_id=4)]]
    want = [ca.render_batch(jobs, max_depth=6)[0] for jobs in batches]
    got, errors = [None, None], []

    def run(k):
        try:
            for _ in range(8):
                got[k] = ca.render_batch(batches[k], max_depth=6)[0]
        except Exception as e:  # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for w, g in zip(want, got):
        for x, y in zip(w, g):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32))


# Results larger and smaller than the staging block's segments, whole and partial segments,
# several destinations to a segment, from several threads at once (each takes its own block).
@pytest.mark.parametrize("w,h", [(300, 200), (512, 342), (600, 437), (1100, 960)])
def test_results_of_any_size_from_several_threads(gpu, w, h):
    scene = ca.Scene(W.cornell().mesh)
    cam = ca.camera_look_at((2.2, 0.548, 0.1), (0.0, 0.548, 0.0), (0.0, 1.0, 0.0), 39.3, w, h)

    def results(seed, out):
        r = ca.ParallelRenderer(scene, w, h, 1, camera=cam, max_depth=2, seed=seed)
        r.render(1)
        out[seed] = [r.radiance(), r.copyImageBytes(), *r.first_hit(0)]
        r.close()

    alone, together = {}, {}
    for seed in (1, 2, 3, 4):
        results(seed, alone)
    threads = [threading.Thread(target=results, args=(seed, together)) for seed in (1, 2, 3, 4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for seed in alone:
        for a, b in zip(alone[seed], together[seed]):
            assert np.array_equal(a, b)
        orc, cfg = O.OracleScene(scene._src.desc()), O.cfg(max_depth=2, seed=seed)
        acc, _ = orc.render(cam, w, h, 0, 1, cfg)
        np.testing.assert_allclose(alone[seed][0], acc, rtol=1e-5, atol=1e-6)
        for a, b in zip(alone[seed][2:], orc.first_hit(cam, w, h, 0, cfg)):
            assert np.array_equal(a, b)


# A batch call leaves its queues for the next: calls of other sizes and scenes, calls from two
# threads at once, and calls after every scene on the device has gone.
def test_batch_calls_share_no_results(gpu):
    def images(side, spp, seed):
        scene = ca.Scene(W.cornell().mesh)
        cam = ca.camera_look_at((2.2, 0.548, 0.1), (0.0, 0.548, 0.0), (0.0, 1.0, 0.0), 39.3, side, side)
        out, _ = ca.render_batch([ca.BatchJob(scene, cam, spp, v) for v in (1, 2)], max_depth=4, seed=seed)
        scene.close()
        return out

    sizes = [(40, 3, 1), (90, 9, 2), (17, 1, 3), (40, 3, 1)]
    first = [images(*s) for s in sizes]
    assert np.array_equal(first[0], first[3])
    got = {}
    threads = [threading.Thread(target=lambda k: got.update({k: images(*sizes[k])}), args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(4):
        assert np.array_equal(first[k], got[k])


# Gradients from more threads than scratch blocks are kept, of sizes that share blocks in any
# order: each call has its block to itself.
def test_gradients_from_several_threads(gpu):
    scene = ca.Scene(W.cornell100k(64, 48).mesh)
    cam = W.cornell100k(64, 48).camera

    def gradients(seed, out):
        w, h, spp = 64, 48, 1 + 7 * seed
        r = ca.ParallelRenderer(scene, w, h, spp, camera=cam, max_depth=5, seed=seed)
        grad = np.random.default_rng(seed).standard_normal((h, w, 3)).astype(np.float32)
        out[seed] = [r.adjoint_grad(grad, spp, hess=0.25) for _ in range(4)]
        r.close()

    alone, together = {}, {}
    for seed in range(6):
        gradients(seed, alone)
    threads = [threading.Thread(target=gradients, args=(seed, together)) for seed in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for seed in range(6):
        for one, other in zip(alone[seed], together[seed]):
            for a, b, c in zip(one, other, alone[seed][0]):
                np.testing.assert_array_equal(a, b)
                np.testing.assert_array_equal(a, c)
