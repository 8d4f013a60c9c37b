"""The pair kernels with every number of lanes per particle, against the CPU oracle.

The lanes per particle follow the context's particle slots, so a large capacity puts a small colony
on the path of a large one.  Colonies: one particle, a partial last wave in each type, a box of one
bin, a box at the smallest stencil grid, and an open box with discs outside it (kept in the edge
bins until the drain takes them).  Bars as everywhere: 1e-12 (FP64) or 1e-5 (FP32) of (sum of |pair
terms| + |F|), FP32 with a floor of 1 % of the median pair scale.
"""
import numpy as np
import pytest

from cil_cuda_amd import abi, configs
from cil_cuda_amd.colony import Colony, HipBatch, HipMD
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _colony(dim, n, L, periodic, law, capacity, seed, stray=0):
    rng = np.random.default_rng(seed)
    p = configs.base_params(dim, 2, 1)
    for s in range(2):
        p.species[s].sig_well[0] = 0.5 + 0.2 * s
        p.species[s].eps_core[0] = 10.0
        p.species[s].eps_well[0] = 1.0
    p.species[1].cross_adhesion = 0.5
    configs.set_law(p, law, 2.0 if law == abi.LAW_LJ else 1.0)
    p.pressure = 1
    box = configs.make_box([L] * dim, [periodic] * dim)
    counts = [n - n // 2, n // 2]
    col = Colony(dim, 1, [capacity - capacity // 2, capacity // 2], ncells=counts)
    for sp, m in zip(col.species, counts):
        sp["pos"][:m, 0] = rng.uniform(0, L, (m, dim))
        sp["sigma"][:m] = rng.uniform(0.8, 1.25, (m, 1))
        sp["state"][:m] = abi.CS_CRAWLING
        k = min(stray, m)  # outside an open box, some near each other
        sp["pos"][:k, 0, dim - 1] = rng.uniform(-3.0, 0.2, k)
        sp["pos"][:k, 0, 0] = rng.uniform(L - 0.5, L + 1.5, k)
    return p, box, col


def _worst(p, box, col, tol, floor, skin=0.0, extra=0):
    dim = p.dim
    q = abi.Params.from_buffer_copy(p)
    q.precision = abi.PREC_FP64
    orc = O.Oracle(q, box, traversal=1)
    ref = col.copy()
    orc.forces(ref, 0)
    scale = orc.force_scale(ref)
    orc.close()
    md = HipMD(p, box, [extra + sp["capacity"] for sp in col.species])
    md.upload(col)
    if skin:
        md.set_neighbour_list(True, skin, 1024)
    frc, pr = md.forces()
    md.close()
    fref = ref.flat("frc").reshape(-1, dim)
    err = np.linalg.norm(frc - fref, axis=1)
    bound = tol * (scale + np.linalg.norm(fref, axis=1) + floor * float(np.median(scale))) + 1e-300
    return float(np.max(err / bound)), pr, ref.flat("pressure")


CASES = [(1, 12.0, 1, 0), (67, 9.0, 1, 0), (300, 2.2, 1, 0), (300, 5.0, 1, 0), (391, 9.0, 0, 40)]
CAPS64 = {2: (400, 50000, 100000, 200000), 3: (400, 10000, 20000, 40000, 80000)}
CAPS32 = {2: (400, 30000, 60000, 120000), 3: (400, 20000, 40000, 80000, 200000, 300000)}


@pytest.mark.parametrize("law", [abi.LAW_LJ, abi.LAW_SC, abi.LAW_HZ])
@pytest.mark.parametrize("dim,cap", [(d, c) for d in (2, 3) for c in CAPS64[d]])
def test_pair_lanes_fp64(gpu, dim, cap, law):
    for n, L, periodic, stray in CASES:
        p, box, col = _colony(dim, n, L, periodic, law, cap, seed=100 + n + law, stray=stray)
        worst, pr, prr = _worst(p, box, col, 1e-12, 0.0)
        assert worst <= 1.0, (n, L, periodic, worst)
        if law == abi.LAW_HZ:
            assert np.allclose(pr, prr, rtol=1e-11, atol=1e-11 * max(1.0, float(np.max(np.abs(prr)))))


# soft core and Hertz: these random colonies overlap, and the LJ r^-13 wall would turn FP32 coordinate
# rounding at near-zero distances into errors beyond the bar
@pytest.mark.parametrize("law", [abi.LAW_SC, abi.LAW_HZ])
@pytest.mark.parametrize("dim,cap", [(d, c) for d in (2, 3) for c in CAPS32[d]])
def test_pair_lanes_fp32(gpu, dim, cap, law):
    for n, L, periodic, stray in CASES:
        p, box, col = _colony(dim, n, L, periodic, law, cap, seed=100 + n + law, stray=stray)
        p.precision = abi.PREC_FP32
        # the floor stands for the absolute rounding of bin-local coordinates: ulp 2^-23 inside the
        # bins (up to 1.3 wide), 2^-22 for discs up to 3 outside them
        worst, _, _ = _worst(p, box, col, 1e-5, 0.02 if stray else 0.01)
        assert worst <= 1.0, (n, L, periodic, worst)


LIST_CAPS = (400, 20000, 100000, 300000)  # eight, four, two and one lane per particle in 3D


@pytest.mark.parametrize("law", [abi.LAW_SC, abi.LAW_HZ])
@pytest.mark.parametrize("cap", LIST_CAPS)
def test_list_lanes(gpu, cap, law):
    for n, L, periodic, stray in CASES:
        p, box, col = _colony(3, n, L, periodic, law, cap, seed=100 + n + law)
        p.precision = abi.PREC_FP32
        worst, _, _ = _worst(p, box, col, 1e-5, 0.01, skin=0.3)
        assert worst <= 1.0, (n, L, periodic, worst)


@pytest.mark.parametrize("cap", LIST_CAPS)
def test_two_level_list_lanes(gpu, cap):
    """The inner list keeps each lane's entries and their order: bit-identical to one level, through
    refreshes and rebuilds."""
    p, box, col = configs.relaxed_bulk_3d(4096, seed=3, precision=abi.PREC_FP32)
    ends = []
    for inner in (0.0, 0.05):
        md = HipMD(p, box, [cap + sp["capacity"] for sp in col.species])
        md.upload(col)
        md.set_neighbour_list(True, 0.15, 160, inner_skin=inner)
        md.forces(want=False)
        md.step(150, 0)
        c = col.copy()
        md.download(c)
        md.close()
        ends.append(c)
    for f in ("pos", "vel", "frc"):
        assert np.array_equal(ends[0].flat(f), ends[1].flat(f)), f


def test_list_capacity_is_the_particles(gpu):
    """The smallest list capacity that holds a colony is the same at eight, four, two and one lane per
    particle, and every larger one holds it."""
    p, box, col = configs.relaxed_bulk_3d(4096, seed=3, precision=abi.PREC_FP32)
    slots = list(range(48, 121, 4))
    accepted = []
    for cap in LIST_CAPS:
        codes = []
        for n in slots:
            md = HipMD(p, box, [cap + sp["capacity"] for sp in col.species])
            md.upload(col)
            md.set_neighbour_list(True, 0.15, n)
            try:
                md.forces(want=False)
                codes.append(n)
            except abi.CilError as e:
                assert e.code == -3
            md.close()
        accepted.append(codes)
    assert all(a == accepted[0] for a in accepted) and slots[0] < accepted[0][0]
    assert accepted[0] == list(range(accepted[0][0], 121, 4))


@pytest.mark.parametrize("mode", ["fp64", "fp32", "list32"])
@pytest.mark.parametrize("law", [abi.LAW_SC, abi.LAW_HZ, abi.LAW_EA])
@pytest.mark.parametrize("alike", [(1, 1), (1, 0), (0, 0)])
def test_two_disc_classes(gpu, mode, law, alike):
    """Two-disc species whose discs have the same law parameters (sorted as one class) or different ones
    (two classes): forces and pair sets against the oracle."""
    rng = np.random.default_rng(9 + law)
    n, L = 120, 13.0
    p = configs.base_params(2, 2, 2)
    for s in range(2):
        sp = p.species[s]
        sp.spring, sp.k_harm = abi.SPRING_HARMONIC, 3.0
        for e in range(2):
            sp.sig_well[e] = 0.4 + 0.1 * s + (0.0 if alike[s] else 0.15 * e)
            sp.eps_core[e] = 10.0 + (0.0 if alike[s] else 5.0 * e)
            sp.eps_well[e] = 0.5 + 0.5 * s
    p.species[1].cross_adhesion = 0.5
    configs.set_law(p, law, 1.0)
    p.precision = abi.PREC_FP64 if mode == "fp64" else abi.PREC_FP32
    box = configs.make_box([L, L], [1, 1])
    col = Colony(2, 2, [n, n], ncells=[n, n - 7])
    for sp in col.species:
        c = rng.uniform(0, L, (n, 2))
        u = rng.normal(size=(n, 2))
        u /= np.linalg.norm(u, axis=1, keepdims=True)
        sp["pos"][:, 0], sp["pos"][:, 1] = c, np.mod(c + 0.6 * u, L)
        sp["sigma"][:] = rng.uniform(0.8, 1.2, (n, 2))
        sp["sigma"][:, 1] *= 1.2  # the diameter bounds differ by disc
        sp["rest_len"][:] = 0.6
        sp["state"][:] = abi.CS_CRAWLING
    tol, floor = (1e-12, 0.0) if mode == "fp64" else (1e-5, 0.01)
    worst, _, _ = _worst(p, box, col, tol, floor, skin=0.3 if mode == "list32" else 0.0)
    assert worst <= 1.0, worst
    q = abi.Params.from_buffer_copy(p)
    q.precision = abi.PREC_FP64
    orc = O.Oracle(q, box, traversal=1)
    md = HipMD(p, box, [n, n])
    md.upload(col)
    assert np.array_equal(md.pairs(), orc.pairs(col))
    md.close()
    orc.close()


def test_crowded_merged_bucket(gpu):
    """More than 1,024 discs of a two-disc class in one bucket (each element type below that), in the
    one-launch sort and, with a large capacity, in the general one."""
    rng = np.random.default_rng(2)
    n, L = 700, 2.0
    for cap in (n, 40000):
        p = configs.base_params(2, 1, 2)
        p.species[0].spring, p.species[0].k_harm = abi.SPRING_HARMONIC, 1.0
        for e in range(2):
            p.species[0].sig_well[e], p.species[0].eps_core[e] = 0.5, 1.0
        configs.set_law(p, abi.LAW_SC, 1.0)
        box = configs.make_box([L, L], [1, 1])
        col = Colony(2, 2, [cap], ncells=[n])
        sp = col.species[0]
        sp["pos"][:n] = rng.uniform(0, L, (n, 2, 2))
        sp["sigma"][:n] = rng.uniform(0.9, 1.0, (n, 2))
        sp["rest_len"][:n] = 0.6
        worst, _, _ = _worst(p, box, col, 1e-12, 0.0)
        assert worst <= 1.0, (cap, worst)


@pytest.mark.parametrize("law", [abi.LAW_SC, abi.LAW_HZ])
@pytest.mark.parametrize("capacity", [65536, 65537, 200000, 600000])
@pytest.mark.parametrize("periodic", [0, 1])
def test_crowded_queues(gpu, law, capacity, periodic):
    """Far more partners in reach per lane than a lane's queue holds (FP32, 3D, eight lanes to one)."""
    p, box, col = _colony(3, 900, 6.0, periodic, law, capacity, 21, stray=0 if periodic else 9)
    p.precision = abi.PREC_FP32
    p.max_disp = 0.0
    worst, pr, ref = _worst(p, box, col, 1e-5, 0.01 if periodic else 0.02)
    assert worst <= 1.0, worst


@pytest.mark.parametrize("capacity", [400, 65536, 65537])
def test_generic_kernel_passes(gpu, capacity):
    """The generic FP32 kernel behind the one-launch sort, whose counts it clears, and behind the general
    one, which clears its own: repeated passes alone and in a batch, against the FP64 oracle's steps."""
    p, box, col = _colony(2, 300, 14.0, 1, abi.LAW_SC, capacity, 31)
    p.precision, p.dt = abi.PREC_FP32, 1e-4
    q = abi.Params.from_buffer_copy(p)
    q.precision = abi.PREC_FP64
    ref = col.copy()
    orc = O.Oracle(q, box, traversal=1)
    orc.forces(ref, 0)
    orc.step(ref, 12, 0)
    orc.close()
    mds = []
    for _ in range(3):
        md = HipMD(p, box, [sp["capacity"] for sp in col.species])
        md.upload(col)
        md.set_kernel(1)
        md.forces(want=False)
        mds.append(md)
    mds[0].step(12, 0)
    batch = HipBatch(mds[1:])
    batch.step(12, [0, 0])
    batch.close()
    ends = []
    for md in mds:
        c = col.copy()
        md.download(c)
        md.close()
        ends.append(c.flat("pos"))
    assert np.array_equal(ends[0], ends[1]) and np.array_equal(ends[0], ends[2])
    d = ends[0] - ref.flat("pos")
    d -= 14.0 * np.round(d / 14.0)
    # 12 steps of dt 1e-4: FP32 force errors of 1e-5 of forces up to a few hundred move a disc by 1e-5
    assert np.max(np.abs(d)) <= 1e-5


@pytest.mark.parametrize("caps", [(500, 16000, 33000, 70000), (16384, 16384, 12001, 16384, 16384),
                                  (16384, 16384, 16384, 16384, 16383, 20000, 40000, 300000)])
@pytest.mark.parametrize("law", ["lj", abi.LAW_HZ])
def test_batched_3d_members_keep_their_bits(gpu, law, caps):
    """3D FP32 colonies in a batch against the same alone: evaluated at once where the colony alone queues
    (over 32,768 slots), and in turns by fewer lanes where colonies of 32 lanes overfill the chip (over 65,536
    slots together)."""
    members, ends = [], []
    for c, cap in enumerate(caps):
        if law == "lj":
            p, box, col = configs.relaxed_bulk_3d(400, seed=c, precision=abi.PREC_FP32)
        else:
            p, box, col = _colony(3, 380 + c, 7.0, c & 1, law, cap, 40 + c)
            p.precision, p.dt = abi.PREC_FP32, 1e-5
        n = [sp["ncells"] for sp in col.species]
        room = [cap - n[1], n[1]]
        alone = HipMD(p, box, room)
        both = [alone, HipMD(p, box, room)]
        for md in both:
            md.upload(col)
            md.forces(want=False)
        members.append(both[1])
        alone.step(11, 0)
        end = Colony(3, 1, room)
        alone.download(end)
        alone.close()
        ends.append(end)
    batch = HipBatch(members)
    batch.step(11, [0] * len(caps))
    batch.close()
    for md, end in zip(members, ends):
        got = Colony(3, 1, [sp["capacity"] for sp in end.species])
        md.download(got)
        md.close()
        for f in ("pos", "vel", "frc", "pressure"):
            assert np.array_equal(got.flat(f), end.flat(f)), (f, end.species[0]["capacity"])


def _cutoff_pairs(seed):
    """The relaxed LJ / soft-core bulk with 60 disjoint LJ pairs moved to 1 +- 5e-6 .. 1e-10 of their cut-off,
    where FP32 distances cannot tell inside from outside."""
    p, box, col = configs.relaxed_bulk_3d(1200, seed=seed, precision=abi.PREC_FP32)
    L, rng = box.length[0], np.random.default_rng(seed)
    x, sig = col.species[0]["pos"][:, 0], col.species[0]["sigma"][:, 0]
    left, done = set(range(len(x))), 0
    for i in rng.permutation(len(x)):
        if i not in left or done == 60:
            continue
        d = x - x[i]
        d -= L * np.round(d / L)
        r, rc = np.linalg.norm(d, axis=1), 2.5 * 0.5 * (sig + sig[i])
        near = [j for j in np.nonzero(np.abs(r / rc - 1) < 0.01)[0] if j in left]
        if not near:
            continue
        j = near[0]
        delta = (1, -1)[done % 2] * (5e-6, 1e-7, 1e-10)[done % 3]
        x[j] = np.mod(x[i] + d[j] * (rc[j] * (1 + delta) / r[j]), L)
        left -= {i, j}
        done += 1
    assert done == 60
    return p, box, col


@pytest.mark.parametrize("mode", ["stencil", "list"])
@pytest.mark.parametrize("extra", [0, 10000, 20000, 50000, 130000, 300000])
def test_lj_cutoff_band(gpu, mode, extra):
    """FP32 LJ forces at every number of lanes, evaluated at once (extra slots up to 10,000 in each of two
    species) and from queues, and over lists, with pairs on the cut-off: their FP64 decision is the oracle's.
    A pair decided wrongly is off by the LJ force at the cut-off, 0.04: more than the bar of a particle whose
    terms sum to less than 4,000."""
    p, box, col = _cutoff_pairs(7)
    worst, _, _ = _worst(p, box, col, 1e-5, 0.01, skin=0.3 if mode == "list" else 0.0, extra=extra)
    assert worst <= 1.0, worst


@pytest.mark.parametrize("mode", ["stencil", "list"])
@pytest.mark.parametrize("extra", [0, 20000, 50000, 130000, 300000])
@pytest.mark.parametrize("partners", [4, 5])
def test_cutoff_band_limit_is_the_particles(gpu, mode, extra, partners):
    """Four pairs on the cut-off of one particle are decided, five reported, whatever the lanes."""
    p, box, _ = configs.bulk_3d_mixed(n=64, seed=1)
    for d in range(3):
        box.length[d] = 12.0
    u = np.array([[1, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0], [0, 0, 1]])[:partners]
    col = Colony(3, 1, [8 + extra, 8], ncells=[1 + partners, 0])
    col.species[0]["pos"][:1 + partners, 0] = np.concatenate([[[6, 6, 6]], 6 + 2.5 * (1 + 1e-7) * u])
    col.species[0]["sigma"][:] = 1.0
    md = HipMD(p, box, [sp["capacity"] for sp in col.species])
    md.upload(col)
    if mode == "list":
        md.set_neighbour_list(True, 0.3, 64)
    if partners == 4:
        md.forces()
    else:
        with pytest.raises(abi.CilError) as e:
            md.forces()
        assert "guard-band" in str(e.value)
    md.close()
