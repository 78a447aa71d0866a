"""Rays with a NaN component or an infinite direction hit nothing: the
traversals skip them (ray_can_hit, core/geometry.h) instead of walking the
whole tree. The brute-force checker, which has no such rule, agrees."""
import itertools

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
