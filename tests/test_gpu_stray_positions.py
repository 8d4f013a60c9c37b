"""Discs uploaded outside a periodic box, by a little or by several box lengths: each acts as its image in
the box, as the oracle's minimum image does.  Forces, pair sets and the first steps against the oracle, in
every stencil kernel and in neighbour-list mode.  Bars of the lane tests: 1e-12 (FP64) or 1e-5 (FP32, with a
floor of 1 % of the median pair scale) of (sum of |pair terms| + |F|)."""
import numpy as np
import pytest

from cil_cuda_amd import abi, configs
from cil_cuda_amd.colony import Colony, HipMD
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _colony(dim, n, L, periodic, seed):
    rng = np.random.default_rng(seed)
    p = configs.base_params(dim, 2, 1)
    for s in range(2):
        p.species[s].sig_well[0], p.species[s].eps_core[0], p.species[s].eps_well[0] = 0.5, 10.0, 1.0
    configs.set_law(p, abi.LAW_SC, 1.0)
    p.dt = 1e-4
    box = configs.make_box([L] * dim, periodic[:dim])
    col = Colony(dim, 1, [n, n], ncells=[n, n // 2])
    for sp in col.species:
        x = rng.uniform(0, L, (n, dim))
        k = rng.integers(-3, 4, (n, dim)) * (rng.random((n, 1)) < 0.3)  # whole box lengths, whatever the bin
        near = rng.random(n) < 0.1  # just outside, into the neighbouring image
        x[near, 0] = np.where(rng.random(near.sum()) < 0.5, L + 0.4, -0.4) * rng.uniform(0.5, 1.0, near.sum())
        sp["pos"][:, 0] = x + L * k * np.array(periodic[:dim])
        sp["sigma"][:] = rng.uniform(0.6, 1.25, (n, 1))
        sp["state"][:] = abi.CS_CRAWLING
    return p, box, col


@pytest.mark.parametrize("mode", ["fp64", "fp32", "generic32", "list32"])
@pytest.mark.parametrize("dim,n,L,periodic", [(2, 200, 17.0, (1, 1)), (2, 300, 2.2, (1, 1)), (2, 200, 17.0, (1, 0)),
                                              (3, 500, 9.0, (1, 1, 1)), (3, 500, 9.0, (0, 1, 1))])
def test_strays_act_as_their_images(gpu, mode, dim, n, L, periodic):
    p, box, col = _colony(dim, n, L, periodic, seed=dim + n)
    p.precision = abi.PREC_FP64 if mode == "fp64" else abi.PREC_FP32
    tol, floor, far = (1e-12, 0.0, 1e-9) if mode == "fp64" else (1e-5, 0.01, 1e-5)
    q = abi.Params.from_buffer_copy(p)
    q.precision = abi.PREC_FP64
    ref = col.copy()
    orc = O.Oracle(q, box, traversal=1)
    orc.forces(ref, 0)
    scale, fref = orc.force_scale(ref), ref.flat("frc").reshape(-1, dim)
    md = HipMD(p, box, [sp["capacity"] for sp in col.species])
    md.upload(col)
    if mode == "generic32":
        md.set_kernel(1)
    if mode == "list32":
        md.set_neighbour_list(True, 0.3, 1024)
    else:
        assert np.array_equal(md.pairs(), orc.pairs(col, 1))
    frc, _ = md.forces()
    bound = tol * (scale + np.linalg.norm(fref, axis=1) + floor * np.median(scale)) + 1e-300
    assert np.max(np.linalg.norm(frc - fref, axis=1) / bound) <= 1.0
    md.step(3, 0)
    orc.step(ref, 3, 0)
    got = col.copy()
    md.download(got)
    md.close()
    orc.close()
    d = (got.flat("pos") - ref.flat("pos")).reshape(-1, dim)
    for k in range(dim):
        if periodic[k]:
            d[:, k] -= L * np.round(d[:, k] / L)
    assert np.max(np.abs(d)) <= far
