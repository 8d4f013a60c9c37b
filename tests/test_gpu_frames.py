"""Frames copied to the host: every field of every active cell, bit for bit, at sizes on both sides of
the one-transfer frame and across staging parts; views that leave arrays out or are too small."""
import ctypes as C

import numpy as np
import pytest

from cil_cuda_amd import abi, configs
from cil_cuda_amd.colony import Colony, HipMD

pytestmark = pytest.mark.gpu

FIELDS = ("pos", "vel", "frc", "sigma") + Colony.DOUBLE_CELL + Colony.INT_CELL


def _filled(dim, nelem, caps, ncells, seed):
    rng = np.random.default_rng(seed)
    col = Colony(dim, nelem, caps, ncells=ncells)
    for sp in col.species:
        for f in FIELDS:
            a = sp[f]
            if a.dtype == np.int32:
                a[:] = rng.integers(0, 1 << 30, a.shape)
            else:
                a[:] = rng.uniform(0.5, 1.0, a.shape)
    return col


def _setup(dim, nelem, caps, ncells):
    p = configs.base_params(dim, len(caps), nelem)
    configs.set_law(p, abi.LAW_SC, 1.0)
    box = configs.make_box([50.0] * dim, [1] * dim)
    col = _filled(dim, nelem, caps, ncells, sum(ncells) + dim)
    md = HipMD(p, box, caps)
    md.upload(col, with_frc=True)
    return md, col


SIZES = [([1], [1]), ([3, 4], [0, 3]), ([700, 900, 64], [699, 0, 64]), ([40000, 1000], [39999, 17]), ([5000, 90000], [4000, 70001])]


@pytest.mark.parametrize("dim,nelem", [(2, 1), (2, 2), (3, 1)])
@pytest.mark.parametrize("caps,ncells", SIZES)
def test_frame_round_trip(gpu, dim, nelem, caps, ncells):
    md, col = _setup(dim, nelem, caps, ncells)
    for _ in range(2):  # the second download reuses the staging
        got = Colony(dim, nelem, caps)
        md.download(got)
        assert got.ncells() == ncells
        for a, b, n in zip(got.species, col.species, ncells):
            for f in FIELDS:
                assert np.array_equal(a[f][:n], b[f][:n]), f
    md.close()


@pytest.mark.parametrize("caps,ncells", SIZES[2:])
def test_frame_with_absent_arrays(gpu, caps, ncells):
    md, col = _setup(2, 2, caps, ncells)
    got = Colony(2, 2, caps)
    views = got.views()
    for v in views:
        v.pos, v.frc, v.theta, v.t0 = abi.PD(), abi.PD(), abi.PD(), abi.PI()
    req = (C.c_int * abi.MAX_SPECIES)()
    assert md.L.cil_hip_download(md.ctx, views, len(caps), req) == 0
    md.close()
    for a, b, n in zip(got.species, col.species, ncells):
        for f in FIELDS:
            if f in ("pos", "frc", "theta", "t0"):
                assert not a[f].any(), f
            else:
                assert np.array_equal(a[f][:n], b[f][:n]), f


def test_views_too_small_are_reported(gpu):
    md, _ = _setup(3, 1, [40000, 10], [39999, 5])
    small = Colony(3, 1, [39998, 10])
    req = (C.c_int * abi.MAX_SPECIES)()
    assert md.L.cil_hip_download(md.ctx, small.views(), 2, req) == -3
    assert list(req)[:2] == [39999, 5] and not small.species[0]["pos"].any()
    md.close()
