"""Training kernels at the edges of their tiles: batches around the 32-sample workgroup, the 16-sample
block and the 256-sample chunk, against the FP64 oracle on the same BF16-rounded inputs and weights
(bars of test_gpu_surrogate.py: 5 % of the norm per tensor, loss within 2 %); and a minibatch drawn by
the training loop against the same rows given to the gradient hook."""
import numpy as np
import pytest

from cil_cuda_amd import abi, configs
from cil_cuda_amd.colony import HipMD
from oracle import mlp_oracle as M
from test_gpu_surrogate import bf16, flatten, random_params, rounded, unflatten

pytestmark = pytest.mark.gpu


def _ctx():
    p, box, col = configs.bulk_3d_mixed(n=600, seed=5)
    md = HipMD(p, box, [sp["capacity"] for sp in col.species])
    return md


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 33, 255, 256, 257, 273, 2049])
def test_gradient_at_tile_edges(gpu, n):
    md = _ctx()
    rng = np.random.default_rng(n)
    p = random_params(4)
    md.mlp_set_params(flatten(p))
    # a larger batch first: what it leaves in the work buffers must not show
    md.mlp_grad(rng.normal(0, 1, (2100, M.NFEAT)), rng.normal(0, 0.01, (2100, 3)))
    X, T = rng.normal(0, 1, (n, M.NFEAT)), rng.normal(0, 0.01, (n, 3))
    g, loss = md.mlp_grad(X, T)
    lr, gr = M.loss_and_grad(rounded(p), bf16(X), T.astype(np.float32).astype(np.float64) / M.OUT_SCALE)
    gg = unflatten(g)
    md.close()
    assert abs(loss - lr) <= 0.02 * abs(lr)
    for k in gr:
        assert np.linalg.norm(gg[k] - gr[k]) <= 0.05 * np.linalg.norm(gr[k]), k


def test_drawn_minibatch_matches_its_rows(gpu):
    """One Adam step on a drawn batch: its loss is the gradient hook's on the same rows (Philox keyed by
    (seed, step, row)), to FP32 rounding of the loss sum."""
    md = _ctx()
    rng = np.random.default_rng(3)
    md.mlp_set_params(flatten(random_params(7)))
    n, batch, seed = 1000, 300, 12345678901
    X, T = rng.normal(0, 1, (n, M.NFEAT)), rng.normal(0, 0.01, (n, 3))
    md.surrogate_set_samples(X, T)
    rows = [(_philox(i, 1, 0x5EED, 7, seed)) % n for i in range(batch)]
    _, want = md.mlp_grad(X[rows], T[rows])
    got = md.surrogate_train(1, batch=batch, lr=1e-3, seed=seed)[0]
    md.close()
    assert abs(got - want) <= 1e-5 * abs(want)


def _philox(c0, c1, c2, c3, seed):
    m = 0xFFFFFFFF
    k0, k1 = seed & m, seed >> 32
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c0, 0xCD9E8D57 * c2
        c0, c1, c2, c3 = (p1 >> 32) ^ c1 ^ k0, p1 & m, (p0 >> 32) ^ c3 ^ k1, p0 & m
        k0, k1 = (k0 + 0x9E3779B9) & m, (k1 + 0xBB67AE85) & m
    return (c0 << 32) | c1
