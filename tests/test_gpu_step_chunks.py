"""Steps launched together against the same steps launched one by one: velocities kept only where they are
read until the chunk's last step, and noise drawn where the cell forces are evaluated, also when the
caller moves the step index between calls or steps the colony in a batch."""
import numpy as np
import pytest

from cil_cuda_amd import abi, configs
from cil_cuda_amd.colony import HipBatch, HipMD
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _plain(precision):
    return configs.plain_2d_sc(n_cells=130, L=16.0, seed=3, precision=precision)


def _theta():
    return configs.theta_2d_hz(n_cells=20, L=24.0, seed=6)


def _wiener(active=0, integrator=abi.INT_EULER):
    p, box, col = configs.binary_2d_fene(n_cells=60, L=14.0, integrator=integrator)
    p.division = abi.DIV_NONE
    p.active_noise = active
    p.species[0].d_noise_radial, p.species[0].d_noise_angular = 0.3, 0.2
    return p, box, col


BUILDS = [lambda: _plain(abi.PREC_FP64), lambda: _plain(abi.PREC_FP32), _theta, _wiener, lambda: _wiener(1),
          lambda: _wiener(1, abi.INT_HEUN)]


def _run(p, box, col, calls):
    md = HipMD(p, box, [sp["capacity"] for sp in col.species])
    md.upload(col)
    md.forces(want=False)
    ts = 0
    for n, jump in calls:
        ts = md.step(n, ts + jump)
    c = col.copy()
    md.download(c)
    md.close()
    return c


@pytest.mark.parametrize("build", BUILDS)
def test_chunked_steps_match_single_steps(gpu, build):
    p, box, col = build()
    a = _run(p, box, col, [(70, 0), (5, 0)])  # one captured chunk, then eager chunks
    b = _run(p, box, col, [(1, 0)] * 75)
    assert a.ncells() == b.ncells()
    for f in ("pos", "vel", "frc", "sigma", "pressure"):
        assert np.array_equal(a.flat(f), b.flat(f)), f


def test_replayed_stream_reads_every_velocity(gpu):
    """The reference's sequential stream (dSFMT): a single disc at rest draws a direction at every force
    pass, whatever its motility, so each step's velocity must be there for the next pass.  Discs too far
    apart to touch, no motility, dividing: chunked, single and the oracle's steps make the same draws."""
    p, box, col = configs.theta_2d_hz(n_cells=12, L=60.0, seed=6)
    p.species[0].motility[0] = 0.0
    p.rng = abi.RNG_DSFMT
    col.species[0]["pos"][:12, 0] = 8.0 + 15.0 * np.stack([np.arange(12) % 4, np.arange(12) // 4], 1)
    col.species[0]["vel"][:12, 0, 0] = 0.3
    a = _run(p, box, col, [(70, 0), (5, 0)])
    b = _run(p, box, col, [(1, 0)] * 75)
    ref = col.copy()
    orc = O.Oracle(p, box, traversal=1)
    orc.set_rng(O.RNG_DSFMT, p.seed)
    orc.forces(ref, 0)
    orc.step(ref, 75, 0)
    assert a.ncells() == b.ncells() == ref.ncells() and a.ncells()[0] > 12
    for f in ("pos", "vel", "frc", "sigma", "pressure", "theta", "ang_vel", "tswitch", "t0"):
        assert np.array_equal(a.flat(f), b.flat(f)), f
    assert np.array_equal(a.flat("t0"), ref.flat("t0"))
    # the spans come from the stream's normal draws: one draw more or less changes them altogether
    assert np.allclose(a.flat("ang_vel"), ref.flat("ang_vel"), rtol=1e-11)
    d = a.flat("pos") - ref.flat("pos")
    d -= box.length[0] * np.round(d / box.length[0])
    assert np.max(np.abs(d)) <= 1e-9


@pytest.mark.parametrize("active", [0, 1])
def test_noise_of_held_forces_keeps_its_step_index(gpu, active):
    """Forces held from index 0, then steps from index 40: the first step uses the noise drawn at 0."""
    p, box, col = _wiener(active)
    got = _run(p, box, col, [(12, 40)])
    ref = col.copy()
    orc = O.Oracle(p, box, traversal=1)
    orc.forces(ref, 0)
    orc.step(ref, 12, 40)
    d = got.flat("pos") - ref.flat("pos")
    d -= box.length[0] * np.round(d / box.length[0])
    assert np.max(np.abs(d)) <= 1e-9


@pytest.mark.parametrize("build", BUILDS[:5])
def test_batch_chunks_match_single_colonies(gpu, build):
    setups = [build(), build()]
    for k, (p, _, _) in enumerate(setups):
        p.seed = 70 + k
    members = []
    for p, box, col in setups:
        md = HipMD(p, box, [sp["capacity"] for sp in col.species])
        md.upload(col)
        md.forces(want=False)
        members.append(md)
    batch = HipBatch(members)
    ts = [0, 0]
    for n in (60, 3, 1, 9):
        ts = batch.step(n, ts)
    batch.close()
    for md, (p, box, col) in zip(members, setups):
        t = md.step(4, 73)  # and on alone, with the batch's last forces
        assert t == 77
        c = col.copy()
        md.download(c)
        md.close()
        one = _run(p, box, col, [(77, 0)])
        assert c.ncells() == one.ncells()
        for f in ("pos", "vel", "frc"):
            assert np.array_equal(c.flat(f), one.flat(f)), f
