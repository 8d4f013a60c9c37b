"""Divisions in one launch (small colonies) against the separate launches (large ones).

The path follows the context's cell slots, so the same colony in a large capacity takes the other one.
Events must be identical: counts, division steps, the append order (every daughter next to its mother's
mirror position) and the records of the division log.
"""
import numpy as np
import pytest

from cil_cuda_amd import abi, configs
from cil_cuda_amd.colony import Colony, HipMD

pytestmark = pytest.mark.gpu

LARGE = 40000  # more cell slots than the one-launch path takes


def _theta_together(n):
    """Every cell of both species reaches the end of its cycle within a few steps, many in the same one."""
    p, box, col = configs.theta_2d_hz(n_cells=1, L=2.2 * np.sqrt(n) + 4, seed=4, capacity=8)
    p.nspecies = 2
    p.species[1] = p.species[0]
    configs.set_law(p, abi.LAW_HZ, 1.0)
    rng = np.random.default_rng(5)
    n0 = n // 3
    two = Colony(2, 1, [2 * n0, 2 * (n - n0)], ncells=[n0, n - n0])
    for s, a, b in ((0, 0, n0), (1, n0, n)):
        sp, m = two.species[s], b - a
        k = np.arange(a, b)
        side = int(np.ceil(np.sqrt(n)))
        sp["pos"][:m, 0] = (np.stack([k % side, k // side], 1) + 0.5) * 2.2 + rng.uniform(-0.2, 0.2, (m, 2))
        sp["sigma"][:m, 0] = sp["sigma_t"][:m] = 1.4
        sp["state"][:m] = abi.CS_DIVIDING
        sp["rho"][:m] = 1.0
        sp["theta"][:m] = 1.0 - 0.05 * rng.integers(1, 4, m)
        sp["ang_vel"][:m] = 0.051
    return p, box, two


def _linear():
    return configs.channel_2d_hz(width=12.0, length=30.0, capacity=512, dt=1e-3, tau=0.05)


def _binary():
    return configs.binary_2d_fene(n_cells=150)


def _run(p, box, col, caps, steps):
    md = HipMD(p, box, caps)
    md.upload(col)
    md.set_division_log(True)
    md.forces(want=False)
    ts = 0
    for n in steps:  # eager steps and a captured chunk
        ts = md.step(n, ts)
    c = Colony(col.dim, col.nelem, caps)
    md.download(c)
    logs = [md.division_log(s) for s in range(col.nspec)]
    md.close()
    return c, logs


@pytest.mark.parametrize("build,steps", [(lambda: _theta_together(40), (1, 2, 9)), (lambda: _theta_together(1500), (1, 2, 9)),
                                         (_linear, (5, 200)), (_binary, (5, 300))])
def test_one_launch_divisions_match_separate_launches(gpu, build, steps):
    p, box, col = build()
    small = [sp["capacity"] for sp in col.species]
    a, la = _run(p, box, col, small, steps)
    b, lb = _run(p, box, col, [small[0] + LARGE] + small[1:], steps)
    assert a.ncells() == b.ncells() and a.total_cells() > col.total_cells()
    for f in ("t0", "state", "tswitch", "ang_vel"):
        assert np.array_equal(a.flat(f), b.flat(f)), f
    d = a.flat("pos").reshape(-1, 2) - b.flat("pos").reshape(-1, 2)
    for k in range(2):
        if box.periodic[k]:
            d[:, k] -= box.length[k] * np.round(d[:, k] / box.length[k])
    assert np.max(np.abs(d)) <= 1e-9  # the pair sums' order follows the particle slots too
    for (xa, ta), (xb, tb) in zip(la, lb):
        assert np.array_equal(ta, tb) and np.max(np.abs(xa - xb), initial=0.0) <= 1e-9
