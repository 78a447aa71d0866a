"""The wavefront integrator's iterations and their end: both sets of queue
counters, single-launch finishing of the last paths (from the first iteration
for small images, after many regenerations with small pools), captured
iterations. The mega-kernel, which has none of these, gives the image."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _settings(approach, term, rng):
    from path_amd.renderer import Settings
    s = Settings()
    s.kernel_approach = approach
    s.rng = rng
    s.term_prob = term
    s.n_iters = 5
    s.constant_prob = 0.2
    return s


# 12 x 9 x 7: one ragged block, finished after one iteration; 128 x 96 x 1 and
# 2: at and above the finishing limit; 301 x 97 x 30: three pipelines, finished
# after several iterations; pool: fewer slots than samples
@pytest.mark.parametrize("x,y,spp,pool,pipes", [
    (1, 1, 1, 0, 0), (12, 9, 7, 0, 0), (128, 96, 1, 0, 0), (128, 96, 2, 0, 0),
    (301, 97, 30, 0, 0), (64, 48, 9, 300, 1), (64, 48, 9, 5000, 4)])
@pytest.mark.parametrize("which,term,rng", [
    ("cornell", "Constant", "Uniform"), ("cornell_sphere", "Constant", "Sobel"),
    ("cornell_sphere", "NIters", "Uniform")])
def test_streaming_equals_megakernel(renderer, request, which, term, rng, x, y, spp, pool, pipes):
    from path_amd.datagen import set_launch_params, set_pipelines
    scene, ftw = request.getfixturevalue(which)
    mega, _ = renderer.render(scene, ftw, x, y, spp, _settings("MegaKernel", term, rng))
    rays = renderer.last_stats().rays
    s = _settings("Streaming", term, rng)
    if pool:
        s.max_num_samples_per_launch = pool
    try:
        if pipes:
            set_pipelines(renderer, pipes)
        for iters, graphs in ((1, False), (3, False), (1, True), (3, True)):
            set_launch_params(renderer, 0, iters, graphs)
            img, _ = renderer.render(scene, ftw, x, y, spp, s)
            assert np.array_equal(img.view(np.uint32), mega.view(np.uint32)), (iters, graphs)
            assert renderer.last_stats().rays == rays, (iters, graphs)
            auto = min(3, max(1, x * y * spp >> 18))
            assert renderer.last_stats().pipelines == (pipes or auto)
    finally:
        set_launch_params(renderer, 0, 1, False)
        if pipes:
            set_pipelines(renderer, 0)


# 1 and 3 samples: finished after the first iteration; 40: after several.
# forced 1 sample per thread and 512 samples: several sample blocks per pixel
# (two reduction passes); the others are reduced in one launch
@pytest.mark.parametrize("spp,forced", [(1, 0), (3, 0), (40, 0), (512, 1)])
def test_batch_equals_single_renders(renderer, spp, forced):
    from path_amd.datagen import datagen_settings, generate_scene, render_batch
    gens = [g for g in map(generate_scene, range(40)) if g.resolution <= 64][:3]
    assert len({g.resolution for g in gens}) > 1
    s = datagen_settings()
    s.term_prob = "Constant"
    s.constant_prob = 0.3
    if forced:
        s.render_work_division.force_target_samples = 1
        s.render_work_division.forced_target_samples_per_thread = forced
    images, gbufs, _ = render_batch(renderer, gens, spp, s)
    s.kernel_approach = "MegaKernel"
    for g, img, gb in zip(gens, images, gbufs):
        mega, _ = renderer.render(g.scene, g.film_to_world, g.resolution, g.resolution, spp, s)
        assert np.array_equal(np.asarray(img).reshape(mega.shape).view(np.uint32),
                              mega.view(np.uint32))
        assert np.isfinite(gb).all() and np.abs(gb).sum() > 0


# either side of the sizes at which MegaKernel images run on the wavefront's
# kernels: samples, depth; roulette from 4.2 M samples; ragged images
@pytest.mark.parametrize("x,y,spp,term,iters,handed_over", [
    (261, 211, 29, "NIters", 3, True), (256, 256, 24, "NIters", 2, False),
    (256, 255, 24, "NIters", 4, False), (256, 256, 64, "Constant", 0, True),
    (256, 255, 64, "Constant", 0, False)])
def test_megakernel_images_on_the_wavefront(renderer, benchmark_scene, x, y, spp, term, iters,
                                            handed_over):
    scene, ftw = benchmark_scene
    small = _settings("Streaming", "NIters", "Sobel")
    renderer.render(scene, ftw, 20, 15, 4, small)
    resummed = renderer.last_render_fp64(20, 15)
    s = _settings("MegaKernel", term, "Sobel")
    s.n_iters = iters
    s.max_num_samples_per_launch = 100  # the Streaming integrator's, not this call's
    try:
        renderer.set_megakernel_split(False)
        ref, _ = renderer.render(scene, ftw, x, y, spp, s)
        assert renderer.last_stats().mega_launches > 0
        rays = renderer.last_stats().rays
    finally:
        renderer.set_megakernel_split(True)
    img, _ = renderer.render(scene, ftw, x, y, spp, s)
    assert (renderer.last_stats().mega_launches == 0) == handed_over
    assert renderer.last_stats().rays == rays
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
    # the last Streaming render can still be summed in FP64
    assert np.array_equal(renderer.last_render_fp64(20, 15), resummed)
