"""The step kernel (queue layout: the last list's pairs, the springs and the
integrator in one launch) against the separate kernels of the cluster layout,
and the spring rows it reads, where its parts change: clusters that are not
full, one stretch of 64 list words and more than the ring holds, the sizes at
which the number of waves per cluster changes, rows on both sides of the sort's
register path, several lists, compensated positions, fixed beads.

Both layouts sum the same terms in FP64 in another order (differences of about
1e-14), round the force once to FP32 and integrate in FP32, so a step may differ
by one rounding of the force: 6e-8 of the largest velocity change, grown over
three steps by the springs (a factor below 4); 1e-6 is allowed.
"""
import numpy as np
import pytest

from biospring_amd import _abi, workloads
from biospring_amd.network import SpringNetwork

pytestmark = pytest.mark.gpu

TOL = 1e-6


def _state(s, params, steps=3):
    net = SpringNetwork.from_system(s, params)
    net.run(steps)
    x, v = net.getState()
    return x, v, net.getEnergies()


def _compare(s, **over):
    got = []
    for layout in (_abi.PAIR_QUEUES, _abi.PAIR_CLUSTERS):
        p = s.params.copy()
        for k, v in over.items():
            setattr(p, k, v)
        p.pair_layout = layout
        got.append(_state(s, p))
    (xq, vq, eq), (xc, vc, ec) = got
    assert np.abs(vq - vc).max() <= TOL * max(np.abs(vc).max(), 1e-12)
    assert np.abs(xq - xc).max() <= TOL * max(np.abs(xc).max(), 1.0)
    # every energy to its own size (sums whose terms nearly cancel: to 1e-9)
    assert np.allclose(eq, ec, rtol=TOL, atol=1e-9)
    return xq, vq, eq


def _perturbed(config, n, seed):
    s = workloads.generate(config, seed=seed, n=n)
    rng = np.random.default_rng(seed)
    s.x = (s.x + rng.normal(scale=0.02, size=s.x.shape)).astype(np.float32)
    return s


# 16,384 and 40,960 beads are 2,048 and 5,120 clusters
@pytest.mark.parametrize("n", [9, 63, 1001, 16384, 16385, 40960, 40967])
def test_sizes(n):
    print("n", n, flush=True)
    _compare(_perturbed(1, n, 3))


@pytest.mark.parametrize("over", [
    {"steric_cutoff": 10.0, "dielectric_model": 0, "electrostatic_dielectric": 20.0},
    {"steric_mode": _abi.STERIC_ZACHARIAS_8_6, "dielectric_model": 0},
    {"steric_mode": _abi.STERIC_LEWITT_8_6, "compensated_positions": 1},
    {"steric_mode": _abi.STERIC_LINEAR, "hydrophobicity_enable": 1},
    {"steric_enable": 0},
    {"spring_enable": 0, "steric_cutoff": 6.0, "electrostatic_cutoff": 6.0},
], ids=["two_lists", "zacharias", "lewitt_comp", "linear_hydro", "coulomb_only", "no_springs"])
def test_terms(over):
    s = _perturbed(1, 1501, 5)
    rng = np.random.default_rng(5)
    s.flags = (rng.random(s.n) < 0.2).astype(np.uint8)
    if over.get("steric_mode") == _abi.STERIC_ZACHARIAS_8_6:
        s.radius = np.sqrt(s.radius).astype(np.float32)  # products of radii
    if over.get("hydrophobicity_enable"):
        # the force goes with h_i h_j: 100 times that of h = 1, which changes the
        # velocities (2e-3 at most) by 2e-7 in three steps
        s.hydro = rng.uniform(-10.0, 10.0, s.n).astype(np.float32)
    _, v, e = _compare(s, **over)
    if over.get("hydrophobicity_enable"):
        # the term is there to be compared: without it the energy is none and
        # the velocities differ by far more than the comparison allows
        assert abs(e[_abi.E_HYDROPHOBIC]) > 0.0
        p = s.params.copy()
        for k, w in over.items():
            setattr(p, k, w)
        p.hydrophobicity_enable = 0
        _, v0, e0 = _state(s, p)
        assert e0[_abi.E_HYDROPHOBIC] == 0.0
        assert np.abs(v - v0).max() >= 1e3 * TOL * np.abs(v).max()


def test_distant_beads_have_empty_lists():
    s = _perturbed(1, 200, 7)
    s.x[-30:] += np.float32(500.0) * np.repeat(np.arange(1, 11, dtype=np.float32), 3)
    far = set(range(190, 200))
    keep = np.array([a not in far and b not in far for a, b in zip(s.id1, s.id2)])
    s.id1, s.id2, s.l0, s.k = s.id1[keep], s.id2[keep], s.l0[keep], s.k[keep]
    _compare(s)


@pytest.mark.parametrize("spokes", [1, 7, 8, 255, 256, 257, 300, 512, 513, 1023, 1024, 1025])
def test_row_lengths(spokes):
    """One hub with `spokes` springs, given in a shuffled order: its force is
    their sum, and every spoke's the opposite."""
    rng = np.random.default_rng(spokes)
    n = spokes + 1
    x = rng.normal(size=(n, 3)).astype(np.float32) * 5.0
    x[0] = 0.0
    order = rng.permutation(spokes) + 1
    flip = rng.random(spokes) < 0.5
    a = np.where(flip, order, 0).astype(np.uint32)
    b = np.where(flip, 0, order).astype(np.uint32)
    l0 = rng.uniform(1.0, 4.0, spokes).astype(np.float32)
    k = rng.uniform(0.1, 1.0, spokes).astype(np.float32)
    p = _abi.default_params()
    p.spring_enable, p.timestep = 1, 1.0
    net = SpringNetwork(p)
    net.setParticles(x.reshape(-1))
    net.setSprings(a, b, l0, k)
    f, e = net.computeForces()
    d = x[order].astype(np.float64)
    r = np.linalg.norm(d, axis=1)
    c = 1.0e3 / 6.02214169e23 * 1.0e10 * (1.0e10 / 1.66054e-27 * 1e-30)
    pull = (k.astype(np.float64) * (r - l0) * c / r)[:, None] * d
    want = np.zeros((n, 3))
    want[0] = pull.sum(0)
    want[order] = -pull
    # FP64 sums rounded to FP32: half an ulp of each component
    assert np.abs(f - want).max() <= 1.2e-7 * np.abs(want).max()
    assert abs(e[_abi.E_SPRING] - (0.5 * k.astype(np.float64) * (r - l0) ** 2).sum()) <= 1e-9 * abs(e[_abi.E_SPRING])


@pytest.mark.parametrize("n,cutoff", [(900, 7.0), (1100, 12.0), (1400, 40.0)])
def test_exclusions_of_long_rows(n, cutoff):
    """The listed pairs are those inside the cutoff without a spring, whether
    a cluster's rows fit the exclusions' LDS copy (8,192 partners) or not:
    rows of 15 to 100, of 85 to 520, and of 1,260."""
    rng = np.random.default_rng(n)
    x = (rng.random((n, 3)) * 24.0).astype(np.float32)
    d = np.linalg.norm(x[:, None].astype(np.float64) - x[None], axis=2)
    i, j = np.triu_indices(n, 1)
    spring = (d[i, j] < cutoff) & (rng.random(len(i)) < 0.9)
    near = d[i, j] < 12.0
    order = rng.permutation(np.flatnonzero(spring))
    p = _abi.default_params()
    p.spring_enable, p.steric_enable, p.steric_mode, p.steric_cutoff = 1, 1, _abi.STERIC_LINEAR, 12.0
    net = SpringNetwork(p)
    net.setParticles(x.reshape(-1))
    net.setSprings(i[order].astype(np.uint32), j[order].astype(np.uint32), d[i, j][order].astype(np.float32),
                   np.ones(len(order), np.float32))
    got = {tuple(sorted(v)) for v in net.getPairs(_abi.NS_STERIC).tolist()}
    want = set(zip(i[near & ~spring].tolist(), j[near & ~spring].tolist()))
    assert got == want, (len(got), len(want), len(got ^ want))


@pytest.mark.parametrize("layout", [_abi.PAIR_QUEUES, _abi.PAIR_CLUSTERS])
@pytest.mark.parametrize("lost", [np.inf, np.nan])
@pytest.mark.parametrize("comp", [0, 1])
def test_a_fixed_bead_nowhere_adds_nothing(layout, lost, comp):
    """A fixed bead without springs at a position that is not finite (an atom
    that a structure lacks) leaves every force, energy and step as they are
    without it."""
    s = _perturbed(1, 1501, 9)
    gone = 700
    keep = (s.id1 != gone) & (s.id2 != gone)
    s.id1, s.id2, s.l0, s.k = s.id1[keep], s.id2[keep], s.l0[keep], s.k[keep]
    s.flags[gone] = _abi.FLAG_STATIC
    got = []
    for x in (1.0e4, lost):
        s.x.reshape(-1, 3)[gone] = x
        p = s.params.copy()
        p.pair_layout, p.compensated_positions, p.electrostatic_enable = layout, comp, 0
        net = SpringNetwork.from_system(s, p)
        f, e = net.computeForces()
        net.run(3)
        x3, v3 = net.getState()
        got.append((f, e, np.delete(x3, gone, 0), v3, net.getEnergies()))
    for a, b in zip(*got):
        assert np.isfinite(b).all()
        assert np.abs(a - b).max() <= TOL * max(np.abs(a).max(), 1e-12)


@pytest.mark.parametrize("mode", [_abi.STERIC_AMBER_12_6, _abi.STERIC_LEWITT_8_6])
@pytest.mark.parametrize("layout", [_abi.PAIR_QUEUES, _abi.PAIR_CLUSTERS])
def test_a_negative_radius_is_not_a_number(mode, layout):
    """sqrt(r_i r_j) of a negative and a positive radius is NaN, as in the
    reference (energy/steric.hpp), and not a size with a sign: the bead's
    forces and the steric energy say so, the beads out of its reach are as
    they were."""
    s = _perturbed(1, 1501, 4)
    p = s.params.copy()
    p.pair_layout, p.steric_mode, p.electrostatic_enable = layout, mode, 0
    f0, e0 = SpringNetwork.from_system(s, p).computeForces()
    bad = 17
    s.radius[bad] = -s.radius[bad]
    f, e = SpringNetwork.from_system(s, p).computeForces()
    d = np.linalg.norm(s.x.reshape(-1, 3).astype(np.float64) - s.x.reshape(-1, 3)[bad], axis=1)
    assert np.isnan(f[bad]).all() and np.isnan(e[_abi.E_STERIC]) and np.isfinite(e0).all()
    far = d > 1.0001 * p.steric_cutoff
    assert far.any() and np.array_equal(f[far], f0[far])


@pytest.mark.parametrize("clusters", [16384, 65536])
def test_list_build_blocks_change(clusters):
    """Long lists on both sides of the cluster counts at which the build's
    blocks change from four waves to one and back: eight beads far away add a
    cluster and no force, so the others' are the same (FP64 sums in another
    order, rounded once)."""
    n = 8 * clusters
    rng = np.random.default_rng(clusters)
    per = int(np.ceil(n ** (1 / 3)))
    site = np.stack(np.unravel_index(np.arange(n), (per, per, per)), 1)
    x = ((site + rng.uniform(-0.2, 0.2, (n, 3))) * 3.0).astype(np.float32)
    far = (np.full((8, 3), per * 3.0 + 100.0) + 40.0 * np.arange(8)[:, None]).astype(np.float32)
    p = _abi.default_params()
    p.steric_enable, p.steric_mode, p.steric_cutoff = 1, _abi.STERIC_LINEAR, 16.0
    got = []
    for beads in (x, np.concatenate([x, far])):
        net = SpringNetwork(p)
        net.setParticles(beads.reshape(-1), radius=np.full(len(beads), 5.0, np.float32))
        print("n", len(beads), flush=True)
        f, e = net.computeForces()
        assert net.counters()["list_cap"] >= 1024
        got.append((f[:n], e[_abi.E_STERIC], net.countPairs(_abi.NS_STERIC)))
        assert not f[n:].any()
        net.close()
    (fa, ea, pa), (fb, eb, pb) = got
    assert pa == pb and abs(ea - eb) <= 1e-9 * abs(ea)
    assert np.abs(fa - fb).max() <= 1.2e-7 * np.abs(fa).max()


@pytest.mark.parametrize("n", [63, 1001, 8192, 8193, 16384])
@pytest.mark.parametrize("cutoffs", [(12.0, 12.0), (10.0, 12.0)], ids=["one_list", "two_lists"])
def test_rebuilding_every_step(n, cutoffs):
    """Systems that rebuild in every step (an interval of 1, or no skin) leave
    the one-workgroup binning: the same steps as with the lists kept."""
    s = _perturbed(1, n, 6)
    got = []
    for interval, skin in ((0, 0.25), (1, 0.25), (0, 0.0)):
        p = s.params.copy()
        p.rebuild_interval, p.list_skin = interval, skin
        p.steric_cutoff, p.electrostatic_cutoff = cutoffs
        got.append(_state(s, p, 4))
    (x0, v0, e0) = got[0]
    for x, v, e in got[1:]:
        assert np.abs(v - v0).max() <= TOL * max(np.abs(v0).max(), 1e-12)
        assert np.abs(x - x0).max() <= TOL * max(np.abs(x0).max(), 1.0)
        assert np.allclose(e, e0, rtol=TOL, atol=1e-9)
