"""Host side of the renders (which kernels a call takes, what memory it holds,
what an error return leaves behind) on the CPU: the library's host sources
linked with a HIP runtime that runs nothing (native/fake_hip.cpp)."""
import concurrent.futures as cf
import ctypes as C
import gc
import subprocess
from pathlib import Path

import numpy as np
import pytest

from path_amd import _lib as L
from path_amd import build

FAKE = Path(__file__).resolve().parent / "native" / "fake_hip.cpp"


@pytest.fixture(scope="module")
def host_library(tmp_path_factory):
    d = tmp_path_factory.mktemp("host")
    srcs = [build.CSRC / s for s in build.SOURCES if s.endswith(".cpp")] + [FAKE]

    def compiled(src):
        obj = d / (src.name + ".o")
        subprocess.run([build.HIPCC, "-x", "hip", "--cuda-host-only", "-O1", "-std=c++20", "-fPIC",
                        "-ffp-contract=off", "-march=x86-64-v3", f"--offload-arch={build.ARCH}",
                        "-c", str(src), "-o", str(obj)], check=True, capture_output=True)
        return str(obj)
    with cf.ThreadPoolExecutor(8) as ex:
        objs = list(ex.map(compiled, srcs))
    so = d / "libhost.so"
    subprocess.run(["g++", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-pthread", "-o", str(so), *objs],
                   check=True)
    lib = C.CDLL(str(so))
    for name, (res, args) in L.SIGNATURES.items():
        if hasattr(lib, name):
            getattr(lib, name).restype, getattr(lib, name).argtypes = res, args
    for name in ("live", "largest", "launches", "pool", "blocks", "in_flight"):
        getattr(lib, "fake_" + name).restype = C.c_uint64
    lib.fake_limit.argtypes = [C.c_uint64]
    return lib


@pytest.fixture
def fake(host_library, monkeypatch):
    """The package on that library; every object of the test is gone before
    the real one is back."""
    monkeypatch.setattr(L, "_lib", host_library)
    host_library.fake_reset()
    yield host_library
    gc.collect()


def _settings(**kw):
    from path_amd.renderer import Settings
    s = Settings()
    s.kernel_approach, s.rng = "MegaKernel", "Uniform"
    s.term_prob, s.n_iters = "NIters", 5
    for k, v in kw.items():
        setattr(s, k, v)
    return s


def _scene(n_tris, walls=6, albedo=0.7):
    """Small triangles in a box with so many of its walls; the camera is at the
    origin."""
    from path_amd.renderer import Scene, material
    rng = np.random.default_rng(1)
    v = [rng.uniform(-1, 1, (n_tris, 1, 3)) + rng.uniform(-0.05, 0.05, (n_tris, 3, 3))]
    for w in range(walls):
        axis, side = w % 3, 1.5 if w >= 3 else -1.5  # the first three meet at a corner
        q = np.array([(side, a, b) for a, b in ((-1.5, -1.5), (1.5, -1.5), (1.5, 1.5), (-1.5, 1.5))])
        q = np.roll(q, axis, 1)
        v += [q[[0, 1, 2]][None], q[[0, 2, 3]][None]]
    v = np.concatenate(v)
    s = Scene()
    mats = np.zeros(len(v), np.uint32)
    mats[0] = 1
    s.add_mesh(v.reshape(-1, 9).astype(np.float32), mats,
               [material("Diffuse", diffuse=(albedo,) * 3),
                material("Diffuse", diffuse=(albedo,) * 3, emission=(1, 1, 1))])
    return s


FTW = np.eye(3, 4, dtype=np.float32).ravel()


def _rays(n, seed=0):
    return np.random.default_rng(seed).uniform(-1, 1, (n, 6)).astype(np.float32)


# what a call above the hand-over's sizes runs on
@pytest.mark.parametrize("control,wavefront", [
    (lambda r: None, True),
    (lambda r: r.set_megakernel_split(False), False),
    (lambda r: r.set_profiling(True), False)])
def test_controls_of_the_hand_over(fake, control, wavefront):
    from path_amd.renderer import Renderer
    r, scene = Renderer(0), _scene(1100)
    control(r)
    r.render(scene, FTW, 256, 256, 24, _settings())
    assert (fake.fake_launches(b"mega") == 0) == wavefront
    r.render_rays_batch([(scene, _rays(4096), None)], 64, 0, _settings())
    assert (fake.fake_launches(b"mega_batch") == 0) == wavefront
    assert (fake.fake_launches(b"wf_trace") > 0) == wavefront


# 6,291,456 samples each; the traversal's grid is 3 blocks per CU for an image
# and 6 for a batch. 3 x 256 paths per block of the limit; an image's pool of
# fewer than 2^20 is not worth it
@pytest.mark.parametrize("limit,image_paths,rays_paths", [
    (0, 1 << 22, 1 << 22), (1 << 20, 1 << 22, 1 << 22), (5462, 1 << 22, 1 << 22),
    (4096, 3145728, 3145728), (1536, 1179648, 1179648), (1535, 1178880, 0), (1366, 1049088, 0),
    (1365, 0, 0), (767, 0, 0), (1, 0, 0)])
def test_hand_over_honours_the_launch_limit(fake, limit, image_paths, rays_paths):
    from path_amd.renderer import Renderer
    r, scene = Renderer(0), _scene(1100)
    s = _settings(max_blocks_per_launch_gpu=limit)

    def check(call, mega, paths):
        fake.fake_reset()
        call()
        assert (fake.fake_launches(mega) == 0) == (paths > 0)
        assert fake.fake_pool() == paths
        if paths and limit:
            assert fake.fake_blocks() <= limit
    check(lambda: r.render(scene, FTW, 512, 256, 48, s), b"mega", image_paths)
    check(lambda: r.render_rays_batch([(scene, _rays(32768), None)], 192, 0, s), b"mega_batch",
          rays_paths)


# images above the hand-over's sizes whose paths go on, or end at once: rays
# that miss, dark surfaces and likely termination with roulette
@pytest.mark.parametrize("tris,walls,albedo,spp,settings,wavefront", [
    (1100, 6, 0.7, 24, {}, True), (1100, 6, 0.1, 24, {}, True),
    (1100, 0, 0.7, 24, {}, False), (1100, 0, 0.7, 500, {}, False), (1100, 1, 0.7, 24, {}, False),
    (4200, 6, 0.7, 64, dict(term_prob="Constant", constant_prob=0.3), True),
    (4200, 6, 0.7, 64, dict(term_prob="Constant", constant_prob=0.9), False),
    (4200, 6, 0.7, 64, dict(term_prob="MultiplierFunc"), True),
    (4200, 6, 0.05, 64, dict(term_prob="MultiplierFunc"), False)])
def test_images_of_short_paths_stay_on_the_megakernel(fake, tris, walls, albedo, spp, settings,
                                                      wavefront):
    from path_amd.renderer import Renderer
    r, scene = Renderer(0), _scene(tris, walls, albedo)
    r.render(scene, FTW, 256, 256, spp, _settings(**settings))
    assert (fake.fake_launches(b"mega") == 0) == wavefront


# items whose rays have several sample blocks are reduced one by one: 16,384
# samples for each such image, or the mega-kernel
@pytest.mark.parametrize("items,rays,spp,steps,wavefront", [
    (200, 10, 256, 6, False), (1, 2000, 256, 6, True), (31, 4, 3000, 3, False), (7, 4, 20000, 3, True),
    (200, 200, 16, 6, True)])
def test_ray_batches_of_many_reductions(fake, items, rays, spp, steps, wavefront):
    from path_amd.renderer import Renderer
    r, scene = Renderer(0), _scene(20)
    s = _settings()
    s.render_work_division.max_samples_per_thread = 8
    out = r.render_rays_batch([(scene, _rays(rays), None)] * items, spp, steps, s)
    assert len(out) == items
    assert (fake.fake_launches(b"mega_batch") == 0) == wavefront
    assert fake.fake_launches(b"wf_reduce") <= items * rays * spp >> 14


def test_pipelines_back_to_the_default(fake):
    from path_amd.datagen import set_pipelines
    from path_amd.renderer import Renderer
    r, scene, s = Renderer(0), _scene(20), _settings(kernel_approach="Streaming")
    for set_to, small, large in ((None, 1, 3), (4, 4, 4), (1, 1, 1), (0, 1, 3)):
        if set_to is not None:
            set_pipelines(r, set_to)
        for spp, n in ((16, small), (200, large)):
            r.render(scene, FTW, 64, 64, spp, s)
            assert r.last_stats().pipelines == n
    with pytest.raises(L.PathError):
        set_pipelines(r, 5)


def _image_call(r, scene):
    s = _settings()
    s.render_work_division.max_samples_per_thread = 1  # two sample blocks
    r.render(scene, FTW, 96, 64, 600, s, output="BGRA")


def _rays_call(r, scene):
    r.render_rays_batch([(scene, _rays(3000, i), None) for i in range(4)], 100, 8, _settings())


# Whatever of the wavefront's memory fits: a call that the mega-kernel alone can
# do is done, and leaves no more memory taken than the mega-kernel does
@pytest.mark.parametrize("call,mega", [(_image_call, b"mega"), (_rays_call, b"mega_batch")])
def test_hand_over_without_memory(fake, call, mega):
    from path_amd.renderer import Renderer
    scene = _scene(1100)

    def run(split, room):
        fake.fake_reset()
        gc.collect()
        start = fake.fake_live()
        fake.fake_limit(start + room)
        r = Renderer(0)
        r.set_megakernel_split(split)
        try:
            call(r, scene)
        except L.PathError:
            return None
        return fake.fake_live() - start, fake.fake_launches(mega) > 0
    alone, _ = run(False, 1 << 50)
    full, on_mega = run(True, 1 << 50)
    assert not on_mega and full > 2 * alone
    for room in (*np.linspace(alone, full, 60, endpoint=False).astype(int),
                 *range(full - 400, full, 40)):
        got = run(True, int(room))
        assert got is not None and got[1] and got[0] <= alone, room
    assert run(True, full) == (full, False)
    assert run(False, alone - 1) is None


# per-sample values of 0.8 GB and 0.6 GB are not kept; 10 MB are
@pytest.mark.parametrize("call,freed", [
    (lambda r, s: r.render(s, FTW, 1024, 1024, 64, _settings()), True),
    (lambda r, s: r.render(s, FTW, 1024, 1024, 2, _settings()), False),
    (lambda r, s: r.render_rays_batch([(s, _rays(200000), None)], 32, 8, _settings()), True),
    (lambda r, s: r.render_rays_batch([(s, _rays(9000), None)], 32, 3, _settings()), False)])
def test_large_values_are_given_back(fake, call, freed):
    from path_amd.renderer import Renderer
    r, scene = Renderer(0), _scene(1100)
    call(r, scene)
    assert fake.fake_launches(b"wf_trace") > 0
    values = fake.fake_largest()
    before = fake.fake_live()
    call(r, scene)
    assert fake.fake_live() == before
    assert (values > 512 << 20) == freed and (before < 900 << 20)


# errors after the rays' upload was queued: no Sobol table (there are no direction
# numbers), no room for the mega-kernel's outputs, launches that fail
@pytest.mark.parametrize("what", ["sobol", "memory", "wf_shade", "wf_reduce_batch", "mega_batch"])
def test_failed_ray_batch_leaves_no_copies(fake, what):
    from path_amd.renderer import Renderer
    r, scene = Renderer(0), _scene(20)
    r.set_megakernel_split(what not in ("memory", "mega_batch"))
    s = _settings(rng="Sobel" if what == "sobol" else "Uniform")
    items = [(scene, _rays(4096), None)]
    r.render_rays_batch(items, 8, 0, _settings())  # scene and staging are there
    fake.fake_fail(what.encode())
    if what == "memory":
        fake.fake_limit(fake.fake_live() + 50000)
    with pytest.raises(L.PathError):
        r.render_rays_batch(items, 128, 8, s)
    assert fake.fake_in_flight() == 0


def test_waiting_for_iterations_sleeps(fake):
    """Three pipelines of which each waits 0.3 s for its iteration."""
    import time
    from path_amd.renderer import Renderer
    r, scene = Renderer(0), _scene(20)
    s = _settings(kernel_approach="Streaming")
    r.render(scene, FTW, 256, 256, 16, s)
    fake.fake_report_delay(300)
    wall, cpu = time.perf_counter(), time.process_time()
    r.render(scene, FTW, 256, 256, 16, s)
    assert r.last_stats().pipelines == 3
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert wall > 0.3 and cpu < wall  # spinning: three times the wall time


@pytest.mark.parametrize("with_losses", [False, True])
def test_training_keeps_losses_only_when_asked(fake, with_losses):
    from path_amd.mlp import RadianceMLP
    m = RadianceMLP(0)
    m.set_dataset(np.zeros((10, 9), np.float32), np.zeros((10, 3), np.float32))
    live = []
    for steps in (1, 50000):
        losses = np.zeros(steps, np.float32) if with_losses else None
        L.check(fake.pt_mlp_train(m.handle, steps, 100, 1e-3, 1, L.fptr(losses), None))
        live.append(fake.fake_live())
    assert live[1] - live[0] == (4 * 49999 if with_losses else 0)


# the Streaming integrator's parameters, for which hand-overs were not measured
@pytest.mark.parametrize("params,pipes", [((16, 1, False), 0), ((0, 64, False), 0),
                                          ((0, 1, True), 0), ((0, 1, False), 1)])
def test_hand_over_takes_default_launch_parameters(fake, params, pipes):
    from path_amd.datagen import set_launch_params, set_pipelines
    from path_amd.renderer import Renderer
    r, scene = Renderer(0), _scene(1100)
    set_launch_params(r, *params)
    set_pipelines(r, pipes)
    for call, blocks in ((lambda: r.render(scene, FTW, 256, 256, 24, _settings()), 2048),
                         (lambda: r.render_rays_batch([(scene, _rays(4096), None)], 256, 0,
                                                      _settings()), 1536)):
        fake.fake_reset()
        call()
        assert r.last_stats().pipelines == fake.fake_launches(b"wf_shade") == 3
        assert fake.fake_blocks() == blocks
    set_launch_params(r, 5, 3, False)
    fake.fake_reset()
    r.render(scene, FTW, 64, 64, 16, _settings(kernel_approach="Streaming"))
    assert fake.fake_blocks() == 5 * 256 and fake.fake_launches(b"wf_shade") == 3
