"""Training repeats itself bit for bit, from build to build: losses, weights and gradients against
recorded digests.  Adam moves a weight of a tiny gradient by a whole step, so any change of the products'
order, of a rounding point or of a sum shows in what a run learns; the arithmetic is fixed (K = 8 matrix
products in ascending K, SiLU' rounded to BF16, bias gradients and losses in sample order), whatever the
launches.  Recorded on an MI355X with the first training kernels (one launch per tensor)."""
import hashlib
import json
import os

import numpy as np
import pytest

from cil_cuda_amd import configs
from cil_cuda_amd.colony import HipMD

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "training_bits.json")

# (samples, batch, Adam steps): partial tiles, blocks, chunks and loss groups; more steps than the loss
# partials that are held; the largest batch
RUNS = [(1000, 1, 3), (1000, 33, 3), (1000, 300, 260), (5000, 2049, 5), (20000, 8192, 8), (20000, 65536, 2)]
GRADS = [1, 15, 17, 128, 129, 256, 273, 2049]


def _weights():
    rng = np.random.default_rng(11)
    return np.concatenate([rng.uniform(-1, 1, n) / np.sqrt(f) for n, f in
                           ((128 * 72, 72), (128, 72), (128 * 128, 128), (128, 128), (3 * 128, 128), (3, 128))]
                          ).astype(np.float32)


def _data(n):
    rng = np.random.default_rng(n)
    return rng.normal(0, 1, (n, 72)).astype(np.float32), rng.normal(0, 0.002, (n, 3)).astype(np.float32)


def _digest(*arrays):
    return hashlib.sha256(b"".join(np.ascontiguousarray(a).tobytes() for a in arrays)).hexdigest()[:16]


def _ctx():
    p, box, col = configs.bulk_3d_mixed(n=600, seed=5)
    return HipMD(p, box, [sp["capacity"] for sp in col.species])


def train_digest(samples, batch, steps):
    md = _ctx()
    md.mlp_set_params(_weights())
    md.surrogate_set_samples(*_data(samples))
    losses = [md.surrogate_train(k, batch=batch, lr=1e-3, seed=77) for k in (steps - 1, 1)]
    w = md.mlp_get_params()
    md.close()
    return _digest(*losses, w)


def grad_digest(n):
    md = _ctx()
    md.mlp_set_params(_weights())
    g, loss = md.mlp_grad(*_data(n))
    md.close()
    return _digest(g, np.float32(loss))


def _golden():
    with open(GOLDEN) as f:
        return json.load(f)


@pytest.mark.parametrize("samples,batch,steps", RUNS)
def test_training_bits(gpu, samples, batch, steps):
    assert train_digest(samples, batch, steps) == _golden()["train"][f"{samples},{batch},{steps}"]


@pytest.mark.parametrize("n", GRADS)
def test_gradient_bits(gpu, n):
    assert grad_digest(n) == _golden()["grad"][str(n)]
