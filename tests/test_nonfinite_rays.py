"""Rays with a NaN component or an infinite direction hit nothing: the
traversals skip them (ray_can_hit, core/geometry.h) instead of walking the
whole tree. The brute-force checker, which has no such rule, agrees."""
import ctypes as C
import itertools
import subprocess
from pathlib import Path

import numpy as np
import pytest


def nonfinite_rays():
    """Every choice of one or two bad components over axis-aligned and
    slanted rays."""
    base = [(0.3, 0.4, 2.0, 0.0, 0.0, -1.0), (0.1, 1.0, 0.2, 0.6, 0.0, 0.8),
            (-0.5, 0.5, 0.5, 0.267, -0.535, 0.802)]
    bad = [np.nan, np.inf, -np.inf]
    rows = []
    for b in base:
        for n in (1, 2):
            for at in itertools.combinations(range(6), n):
                for vals in itertools.product(bad, repeat=n):
                    r = list(b)
                    for i, v in zip(at, vals):
                        r[i] = v
                    if np.isnan(r).any() or np.isinf(r[3:]).any():
                        rows.append(r)
    return np.array(rows, np.float32)


def soup(seed, n, flat):
    rng = np.random.default_rng(seed)
    v = rng.uniform(-1, 1, (n, 3, 3))
    if flat:  # axis-aligned: zero edge components meet the infinities
        v[np.arange(n), :, rng.integers(0, 3, n)] = rng.uniform(-1, 1, (n, 1))
    return np.concatenate([v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]], 1).astype(np.float32)


def test_rule(tmp_path):
    so = tmp_path / "ray_check.so"
    subprocess.run(["g++", "-O2", "-std=c++20", "-ffp-contract=off", "-shared", "-fPIC",
                    str(Path(__file__).resolve().parent / "native" / "ray_check.cpp"),
                    "-o", str(so)], check=True)
    lib = C.CDLL(str(so))

    def can_hit(rays):
        rays = np.ascontiguousarray(rays, np.float32)
        out = np.zeros(len(rays), np.uint8)
        lib.rays_can_hit(rays.ctypes.data_as(C.c_void_p), len(rays),
                         out.ctypes.data_as(C.c_void_p))
        return out
    assert not can_hit(nonfinite_rays()).any()
    # finite components of every size, and infinite origins
    sizes = [0.0, -0.0, 1e-45, -1e-40, 1.2e-38, 0.7, -5.0, 1e20, 3.4028235e38, -3.4028235e38]
    assert can_hit(np.array(list(itertools.product(sizes, repeat=6)), np.float32)).all()
    assert can_hit([[np.inf, 0, -np.inf, 1, 0, 0]]).all()


@pytest.mark.parametrize("flat", [False, True])
def test_brute_force_finds_no_hit(flat):
    from oracle import oracle as O
    rays = nonfinite_rays()
    for seed in range(4):
        _, idx, _ = O.loopall(soup(seed, 64, flat), rays)
        assert (idx == 0xFFFFFFFF).all()


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["cornell", "cornell_sphere"])
def test_gpu_finds_no_hit(renderer, request, which):
    from oracle import oracle as O
    from tests.helpers import random_rays
    scene, _ = request.getfixturevalue(which)
    # among finite rays, whose hits stay what they were
    rays = random_rays(3000, -1.2, 2.2, seed=5)
    bad = nonfinite_rays()
    at = np.random.default_rng(1).choice(len(rays), len(bad), replace=False)
    rays[at] = bad
    _, idx, _ = renderer.intersect(scene, rays)
    _, ridx, _ = O.loopall(scene.flat()["tris"], rays)
    assert np.array_equal(idx, ridx)
    assert (idx[at] == 0xFFFFFFFF).all()


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [0, 3])
def test_ray_batch_of_the_wavefront(renderer, cornell_sphere, steps):
    """The wavefront's traversal writes such a ray's miss itself: a batch large
    enough for it equals the mega-kernel's render of the same rays."""
    from path_amd.renderer import Settings
    from tests.helpers import random_rays
    scene, _ = cornell_sphere
    rays = random_rays(3000, -1.2, 2.2, seed=5)
    bad = nonfinite_rays()
    rays[np.random.default_rng(1).choice(len(rays), len(bad), replace=False)] = bad
    s = Settings()
    s.kernel_approach = "MegaKernel"
    s.term_prob, s.n_iters = "NIters", 3
    spp = 96
    (got,) = renderer.render_rays_batch([(scene, rays, None)], spp, steps, s)
    assert renderer.last_stats().mega_launches == 0
    traced = renderer.last_stats().rays
    out = dict(output="OutputPerStep", n_steps=steps) if steps else {}
    ref, _ = renderer.render(scene, None, 0, 0, spp, s, rays=rays, **out)
    assert renderer.last_stats().mega_launches > 0 and renderer.last_stats().rays == traced
    got = np.asarray(got).reshape(max(steps, 1), len(rays), 3)
    ref = ref.reshape(got.shape)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    assert ref.sum() > 0
