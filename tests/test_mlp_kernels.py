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
