"""Radiance MLP on the GPU (BF16 MFMA kernels) against the numpy
restatement with the same BF16 rounding points."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def net():
    from path_amd.mlp import RadianceMLP
    return RadianceMLP(0, seed=3)


def _data(n, seed):
    rng = np.random.default_rng(seed)
    f = np.concatenate([rng.uniform(-1, 1, (n, 3)),
                        rng.normal(size=(n, 3)), rng.uniform(0, 1, (n, 3))], 1)
    f[:, 3:6] /= np.linalg.norm(f[:, 3:6], axis=1, keepdims=True)
    t = rng.uniform(0, 3, (n, 3))
    return f.astype(np.float32), t.astype(np.float32)


def test_weights_round_trip(net):
    w = net.get_weights()
    w2 = w.copy()
    w2[::7] *= 1.5
    net.set_weights(w2)
    assert np.array_equal(net.get_weights(), w2)
    net.set_weights(w)


@pytest.mark.parametrize("n", [1, 130, 1000])
def test_forward_matches_reference(net, n):
    from oracle import mlp_ref as M
    f, _ = _data(n, n)
    out = net.forward(f)
    ref, _, _ = M.forward(net.get_weights(), f, emulate=True)
    scale = np.abs(ref).max()
    err = np.abs(out - ref).max() / scale
    print("forward max err / max |y|", err)
    assert err <= 2e-2
    assert np.sqrt(((out - ref) ** 2).mean()) <= 3e-3 * scale


@pytest.mark.parametrize("n", [1, 128, 130, 5000])
def test_fused_forward_equals_layer_gemms(net, n):
    """The one-kernel inference forward (activations in LDS) returns the bits
    of the encoding kernel + one GEMM per layer."""
    f, _ = _data(n, 100 + n)
    w = net.get_weights()
    w2 = w * np.float32(1.7)   # larger activations than the initial weights give
    net.set_weights(w2)
    try:
        net.set_forward_kernel(True)
        fused = net.forward(f)
        net.set_forward_kernel(False)
        layered = net.forward(f)
    finally:
        net.set_forward_kernel(True)
        net.set_weights(w)
    assert np.abs(fused).max() > 0
    assert np.array_equal(fused.view(np.uint32), layered.view(np.uint32))


def test_gradient_matches_reference(net):
    from oracle import mlp_ref as M
    f, t = _data(2048, 7)
    w = net.get_weights()
    g, loss = net.gradient(f, t)
    rloss, rg = M.loss_and_grad(w, f, t, emulate=True)
    _, rg64 = M.loss_and_grad(w, f, t, emulate=False)
    assert abs(loss - rloss) <= 1e-3 * rloss
    offs = np.cumsum([0] + [o * i for o, i in M.SHAPES])
    for l in range(len(M.SHAPES)):
        a, b, c = g[offs[l]:offs[l + 1]], rg[offs[l]:offs[l + 1]], rg64[offs[l]:offs[l + 1]]
        e_emu = np.linalg.norm(a - b) / np.linalg.norm(b)
        e_64 = np.linalg.norm(a - c) / np.linalg.norm(c)
        print("layer", l, "rel err vs bf16 reference", e_emu, "vs fp64", e_64)
        assert e_emu <= 1e-2
        # BF16 operands alone (the emulated reference) account for this
        assert e_64 <= 0.15


# 32-row tiles below 24,576 rows, 64-row tiles up to 57,344, then 128-row ones;
# ragged last tiles, and fewer row stages than weight-gradient splits. The bounds are those of
# test_gradient_matches_reference, from the same roundings.
@pytest.mark.parametrize("n", [1, 31, 129, 700, 24449, 57300])
def test_gradient_over_tile_sizes(net, n):
    from oracle import mlp_ref as M
    f, t = _data(n, 40 + n)
    w = net.get_weights()
    g, loss = net.gradient(f, t)
    rloss, rg = M.loss_and_grad(w, f, t, emulate=True)
    assert abs(loss - rloss) <= 1e-3 * rloss
    offs = np.cumsum([0] + [o * i for o, i in M.SHAPES])
    for l in range(len(M.SHAPES)):
        a, b = g[offs[l]:offs[l + 1]], rg[offs[l]:offs[l + 1]]
        # one sample's gradient has no sum for its roundings to average in
        assert np.linalg.norm(a - b) <= (3e-2 if n < 32 else 1e-2) * np.linalg.norm(b)


def test_gradient_sums_of_a_large_batch(net):
    """262,144 rows against the FP64 mean of 128 gradients of 2,048 of them: with
    powers of two the roundings to BF16 are the same, so only the sums over the rows
    differ. Each weight's sum is a chain of at most rows / splits / 16 products of
    16 rows, splits / 4 partials and 4 wave sums (42 splits); each addition rounds by
    2^-24 of a partial sum, and here no partial sum is far above the whole."""
    n, c = 1 << 18, 1 << 11
    f, t = _data(n, 9)
    g, loss = net.gradient(f, t)
    parts = [net.gradient(f[i:i + c], t[i:i + c]) for i in range(0, n, c)]
    ref = np.mean([p[0].astype(np.float64) for p in parts], 0)
    bound = (n / 42 / 16 + 42 / 4 + 4) * 2.0 ** -24
    from oracle import mlp_ref as M
    offs = np.cumsum([0] + [o * i for o, i in M.SHAPES])
    for l in range(len(M.SHAPES)):
        a, b = g[offs[l]:offs[l + 1]], ref[offs[l]:offs[l + 1]]
        assert np.linalg.norm(a - b) <= bound * np.linalg.norm(b)
    assert abs(loss - np.mean([p[1] for p in parts])) <= bound * loss


def test_train_draws_rows_and_steps_like_train_step(net):
    """Training on the resident set equals host batches of the rows it draws
    (SplitMix64 of the row's number), step by step."""
    f, t = _data(5000, 3)
    w = net.get_weights()
    net.set_weights(w)  # Adam from its first step
    net.set_dataset(f, t)
    losses, _ = net.train(2, 900, 1e-3, seed=77)
    trained = net.get_weights()
    net.set_weights(w)
    with np.errstate(over="ignore"):
        for it in range(2):
            seed = np.uint64(77) + np.uint64(it) * np.uint64(0x632be59bd9b4e019)
            z = seed + np.uint64(0x9e3779b97f4a7c15) * np.arange(1, 901, dtype=np.uint64)
            z = (z ^ (z >> np.uint64(30))) * np.uint64(0xbf58476d1ce4e5b9)
            z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94d049bb133111eb)
            i = ((z ^ (z >> np.uint64(31))) % np.uint64(5000)).astype(np.int64)
            assert net.train_step(f[i], t[i], 1e-3) == losses[it]
    assert np.array_equal(net.get_weights(), trained)
    net.set_weights(w)


def test_training_reduces_loss():
    from path_amd.mlp import RadianceMLP
    m = RadianceMLP(0, seed=5)
    rng = np.random.default_rng(0)
    n = 1 << 16
    f, _ = _data(n, 11)
    # smooth target: light from +y, albedo-weighted, plus a position term
    t = f[:, 6:9] * (np.clip(f[:, 4:5], 0, None) * 2.0 + 0.2) + 0.3 * (f[:, 1:2] + 1.0)
    m.set_dataset(f, t.astype(np.float32))
    losses, secs = m.train(1000, 8192, 1e-3, seed=1)
    print("loss", losses[:5].mean(), "->", losses[-20:].mean(), "in", secs, "s")
    assert np.isfinite(losses).all()
    assert losses[-20:].mean() < 0.1 * losses[:5].mean()
    pred = m.forward(f[:4096])
    rel = np.sqrt(((pred - t[:4096]) ** 2).mean()) / np.sqrt((t[:4096] ** 2).mean())
    print("relative RMSE on training points", rel)
    assert rel < 0.1
