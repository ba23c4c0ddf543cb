"""The network's kernels at the sizes where their tilings can go wrong."""
import numpy as np
import pytest

from oracle import mlp_oracle


def _net(seed, rng):
    from chm_amd import pbsm3d as pb

    net = pb.Mlp(seed=seed)
    p = net.get_params()
    o = 0
    for r, c in mlp_oracle.SHAPES:  # biases that are not zero, output rows past the targets stay zero
        o += r * c
        p[o:o + (r if r == mlp_oracle.H else mlp_oracle.OUT)] = rng.normal(0, 0.2, r if r == mlp_oracle.H
                                                                            else mlp_oracle.OUT)
        o += r
    net.set_params(p)
    norm = (rng.normal(0, 1, 16), rng.uniform(0.5, 2, 16), rng.normal(0, 1, 11), rng.uniform(0.5, 2, 11))
    net.set_normalization(*norm)
    return net, p, tuple(np.asarray(v, dtype=np.float32) for v in norm)


# 16-sample MFMA blocks, 64-sample wave tiles, one tile per wave of the first workgroups, and one
# tile past a full round of 256 workgroups x 8 waves; offset 1: rows that are not 16-byte aligned
@pytest.mark.gpu
@pytest.mark.parametrize("n,offset", [(1, 0), (15, 1), (16, 0), (17, 1), (63, 0), (64, 1), (65, 0), (1000, 1),
                                      (16384 + 33, 0), (256 * 8 * 64 + 65, 0)])
def test_inference_matches_the_layer_by_layer_gemms(n, offset):
    import torch

    print(f"[case] mlp inference n={n} offset={offset}", flush=True)
    rng = np.random.default_rng(n)
    net, p, norm = _net(5, rng)
    X = (rng.normal(0, 1.5, (n, 16)) * norm[1] + norm[0]).astype(np.float32)
    flat = torch.empty(n * 16 + offset, dtype=torch.float32, device="cuda:0")
    Xd = flat[offset:].view(n, 16)
    Xd.copy_(torch.tensor(X))
    Y1 = torch.full((n, 11), np.nan, dtype=torch.float32, device="cuda:0")
    Y2 = torch.full_like(Y1, np.nan)
    net.predict(Xd, Y1, path=1)
    net.predict(Xd, Y2, path=2)
    assert torch.equal(Y1, Y2)
    k = min(n, 400)  # the first and last rows against the FP64 reference
    rows = np.r_[0:k, n - k:n]
    ref = mlp_oracle.predict(p, X[rows], norm, bf16=True)
    assert np.abs(Y1.cpu().numpy()[rows] - ref).max() <= 1e-2 * np.abs(ref).max()


# one 64-sample tile per workgroup, partial tiles, more tiles than workgroups (256 x 64 = 16384)
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 16, 63, 64, 65, 200, 4097, 16384, 16384 + 100, 3 * 16384 + 7])
def test_gradients_match_the_reference(n):
    print(f"[case] mlp gradients n={n}", flush=True)
    rng = np.random.default_rng(100 + n)
    net, p, norm = _net(6, rng)
    X = (rng.normal(0, 1.5, (n, 16)) * norm[1] + norm[0]).astype(np.float32)
    Y = rng.normal(0, 1, (n, 11)).astype(np.float32)
    loss, g = net.gradients(X, Y)
    rloss, rg = mlp_oracle.loss_and_grad(p, X, Y, norm, bf16=True)
    # the bound of the whole-batch check: BF16 roundings that fall the other way after an FP32 sum
    # in another order, 2^-9 of a value each
    assert abs(loss - rloss) <= 1e-3 * rloss
    o = 0
    for r, c in mlp_oracle.SHAPES:
        for size in (r * c, r):
            a, b = g[o:o + size], rg[o:o + size]
            assert np.linalg.norm(a - b) <= 2e-2 * np.linalg.norm(b) + 1e-7, (o, size)
            o += size


@pytest.mark.gpu
def test_training_step_is_adam_on_the_sampled_rows():
    """One batch of a one-batch epoch: the counter hash's rows, their gradient, Adam's first step."""
    import torch

    print("[case] mlp training step", flush=True)
    n, seed, lr = 333, 9, 1e-3
    rng = np.random.default_rng(7)
    net, p, norm = _net(8, rng)
    X = (rng.normal(0, 1.5, (n, 16)) * norm[1] + norm[0]).astype(np.float32)
    Y = rng.normal(0, 1, (n, 11)).astype(np.float32)
    loss = net.train(torch.tensor(X, device="cuda:0"), torch.tensor(Y, device="cuda:0"), epochs=1, batch=n, lr=lr,
                     seed=seed)
    m64, golden = (1 << 64) - 1, 0x9E3779B97F4A7C15

    def row(t):
        z = (seed * golden + t * golden) & m64
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m64
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m64
        return (z ^ (z >> 31)) % n

    rows = [row(t) for t in range(n)]
    rloss, rg = mlp_oracle.loss_and_grad(p, X[rows], Y[rows], norm, bf16=True)
    assert abs(loss - rloss) <= 1e-3 * rloss
    step = net.get_params() - p
    # Adam's first step is lr g / (|g| + eps): lr against the gradient's sign where it is not tiny
    # (the parameter's own rounding: 2^-24 of values up to 1.5, 1e-4 of lr)
    big = np.abs(rg) > 0.05 * np.abs(rg).max()
    np.testing.assert_allclose(step[big], -lr * np.sign(rg[big]), rtol=1e-3)
    # output rows past the eleven targets are never stepped
    o = p.size - 16 * 128 - 16
    assert np.all(step[o + 11 * 128:o + 16 * 128] == 0) and np.all(step[-5:] == 0)


def _uniform_net(seed):
    """A network whose parameters are exact multiples of uniform counters (no libm in their making)."""
    from chm_amd import meshgen
    from chm_amd import pbsm3d as pb

    u = meshgen.uniform(seed, 31, 37264 + 54)
    p, o = np.zeros(37264, dtype=np.float32), 0
    for r, c in mlp_oracle.SHAPES:
        rows = r if r == mlp_oracle.H else mlp_oracle.OUT  # output rows past the targets stay zero
        p[o:o + rows * c] = (u[o:o + rows * c] - 0.5) * (2.0 * np.sqrt(6.0 / c))
        o += r * c
        p[o:o + rows] = (u[o:o + rows] - 0.5) * 0.5
        o += r
    v = u[37264:]
    net = pb.Mlp(seed=seed)
    net.set_params(p)
    net.set_normalization(v[:16] - 0.5, 0.5 + v[16:32], v[32:43] - 0.5, 0.5 + v[43:54])
    return net


def _uniform_rows(seed, n):
    from chm_amd import meshgen

    X = (4.0 * meshgen.uniform(seed, 32, 16 * n) - 2.0).astype(np.float32).reshape(n, 16)
    return X, (4.0 * meshgen.uniform(seed, 33, 11 * n) - 2.0).astype(np.float32).reshape(n, 11)


def _digest(*arrays):
    import hashlib

    h = hashlib.sha256()
    for a in arrays:
        h.update(np.ascontiguousarray(a).tobytes())
    return h.hexdigest()[:16]


def _network_bits(what, n, batch):
    import torch

    net = _uniform_net(3)
    X, Y = _uniform_rows(n, n)
    Xd, Yd = torch.tensor(X, device="cuda:0"), torch.tensor(Y, device="cuda:0")
    if what == "predict":
        out = torch.full((n, 11), np.nan, dtype=torch.float32, device="cuda:0")
        net.predict(Xd, out)
        return _digest(out.cpu().numpy())
    if what == "gradients":
        loss, g = net.gradients(X, Y)
        return _digest(np.float64(loss), g)
    loss = net.train(Xd, Yd, epochs=3, batch=batch, lr=2e-3, seed=9)
    return _digest(np.float64(loss), net.get_params())


# Slabs of the weight gradients: one (n < 1024), ends inside a tile (1060), 9 of 576 rows (5000), 64
# (32768 and more); row blocks of the bias gradients: tiles, or across them (from 32769 on)
BITS = [
    ("predict", 1, 0, "751c4467ceb9c22b"),
    ("predict", 1000, 0, "d68a15674364c0a4"),
    ("predict", 131137, 0, "cffbd442bdfb2b2a"),
    ("gradients", 1, 0, "89909ec7c993f64f"),
    ("gradients", 200, 0, "e43fe30b3edb93a0"),
    ("gradients", 1060, 0, "aa5d2602d468d0d4"),
    ("gradients", 5000, 0, "280be4b727e95bf9"),
    ("gradients", 16484, 0, "9b767333a3ac39b5"),
    ("gradients", 32768, 0, "f170e5cd60941281"),
    ("gradients", 32769, 0, "c30b524f2549a11e"),
    ("gradients", 49159, 0, "f76b28e07e97963c"),
    ("train", 333, 333, "c094b065aa05a279"),
    ("train", 20000, 2048, "408658507db1c732"),
    ("train", 20000, 5000, "9b795a52f2569451"),
    ("train", 50000, 8192, "bc2d1e79e45b1bff"),
    ("train", 60000, 40000, "81b93b1810bb50a9"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("what,n,batch,want", BITS)
def test_network_bits(what, n, batch, want):
    """The kernels keep the bits of the trainer and forward that ran one launch per product, slab sum,
    column sum and elementwise step: the digests are of its outputs, recorded on an MI355X."""
    print(f"[case] network bits {what} n={n} batch={batch}", flush=True)
    assert _network_bits(what, n, batch) == want
