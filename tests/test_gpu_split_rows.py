"""Row splitting, tile sizing and the 16-bit list build against the CPU oracle, at the sizes where
they can go wrong.

* lists: rows shared by 8, 4, 2 and 1 lanes and stencils of one and two cells; lattices whose
  distances equal r_n exactly, which only the FP64 decision can place; column runs of more than 64
  candidates; records on the grid's faces.  Counts and neighbour sets are integers: equal.
* forces and energies of one- and two-type, capped and uncapped tables: a row of some 80 pairs
  summed in another order differs by about sqrt(80) roundings of 1.1e-16 of its largest term, and
  the largest term of a capped or lattice row is within a factor of a hundred of the largest
  force: 1e-12 of the largest force, as in the core tests.  Energies likewise, relative.
* the native loop in the store form (two-type and capped tables) equals the actions bit for bit.
* ensembles whose cells are so dense that tiles are one column wide, in boxes of two cells.
"""
import numpy as np
import pytest

import pyoracle as O
import test_gpu_batch as B
from mrmd_amd.lattice import maxwell_boltzmann

pytestmark = pytest.mark.gpu

RN = 2.8


@pytest.fixture(scope="module")
def M():
    import mrmd_amd
    return mrmd_amd


@pytest.fixture(scope="module")
def ctx(M):
    c = M.Context(0)
    yield c
    c.close()


def _jittered(n, density, seed):
    """n points of a jittered cubic lattice: no pair closer than about a third of the spacing"""
    g = np.random.default_rng(seed)
    side = int(np.ceil(n ** (1.0 / 3.0) - 1e-9))
    a = density ** (-1.0 / 3.0)
    i = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)
    p = (i[g.permutation(i.shape[0])[:n]] + 0.5 + g.uniform(-0.25, 0.25, (n, 3))) * a
    return p, side * a


def _lists(M, ctx, pos, rn, ratio, L, types=None):
    """the list over open-boundary atoms (no ghosts) on the device and in the oracle"""
    kw = {} if types is None else dict(type=types)
    g, c = M.Atoms.from_arrays(ctx, pos, **kw), O.Atoms.from_arrays(pos, **kw)
    vl, ov = M.HalfVerletList(ctx), O.Verlet()
    vl.build(g, 0, g.nlocal, rn, ratio, [0.0] * 3, [L] * 3)
    ov.build(c, c.nlocal, 0, c.nlocal, rn, ratio, [0.0] * 3, [L] * 3)
    return g, c, vl, ov


def _same_lists(vl, ov, n, sets):
    counts, _ = vl.half_counts(n)
    np.testing.assert_array_equal(counts, ov.counts()[:n])
    if sets:
        rows, ref = vl.half_rows(n), ov.neighbors()
        for i in range(n):
            assert rows[i] == set(ref[i, : counts[i]].tolist()), i


@pytest.mark.parametrize("n,density,ratio", [(1, 0.8, 1.0), (2, 0.8, 1.0), (65, 0.8, 1.0), (1025, 0.8, 0.5),
                                             (4097, 0.05, 1.0), (3000, 4.0, 1.0), (3000, 3.0, 0.5)])
def test_lists_match_oracle(M, ctx, n, density, ratio):
    pos, L = _jittered(n, density, n)
    L = max(L, RN)
    # some records on the faces of the grid
    pos[: n // 8, 0] = 0.0
    pos[n // 8: n // 4, 2] = L
    g, c, vl, ov = _lists(M, ctx, pos, RN, ratio, L)
    _same_lists(vl, ov, n, True)


@pytest.mark.parametrize("ratio", [1.0, 0.5])
@pytest.mark.parametrize("scale", [1.0, 0.7])
def test_lattice_at_exactly_the_radius(M, ctx, ratio, scale):
    """distances that equal r_n (3, 4, 5: also off the axes) to the last bit or miss it by one"""
    i = np.stack(np.meshgrid(*[np.arange(14)] * 3, indexing="ij"), -1).reshape(-1, 3)
    pos = i.astype(np.float64) * scale * 0.5
    g, c, vl, ov = _lists(M, ctx, pos, 2.5 * scale, ratio, 7.0 * scale)
    _same_lists(vl, ov, pos.shape[0], True)


@pytest.mark.parametrize("num_types", [1, 2])
@pytest.mark.parametrize("cap", [0.0, 0.9])
@pytest.mark.parametrize("n", [63, 1000, 16384, 16385, 32769, 65537])
def test_forces_match_oracle(M, ctx, n, cap, num_types):
    """8, 8, 8, 4, 2 and 1 lanes per row"""
    pos, L = _jittered(n, 0.8, 7 * n)
    if cap:
        pos[1:2] = pos[:1] + [[1e-3, 0.0, 0.0]]  # one pair far inside the capping distance
    types = None if num_types == 1 else (np.arange(n) % 3 == 0).astype(np.int64)
    g, c, vl, ov = _lists(M, ctx, pos, RN, 1.0, L, types)
    _same_lists(vl, ov, n, False)
    k = num_types * num_types
    sig, eps = [1.0, 0.93, 0.93, 0.86][:k], [1.0, 0.75, 0.75, 0.5][:k]
    lj = M.LennardJones(ctx, [2.5] * k, sig, eps, capping_distance=[cap] * k, num_types=num_types, shifted=True,
                        type_stride=num_types)
    olj = O.LJ([cap] * k, [2.5] * k, sig, eps, num_types, shifted=True, type_stride=num_types)
    g.set_force(0.0)
    lj.apply(g, vl)
    O.lib().or_set_threads(1)
    energy, virial = olj.apply(c, ov)
    F, ref = g.download(M.FORCE, n), c.get(O.FORCE, n)
    assert np.abs(F - ref).max() <= 1e-12 * np.abs(ref).max()
    E, W = lj.energy_virial()
    assert E == pytest.approx(energy, rel=1e-12) and W == pytest.approx(virial, rel=1e-12)


@pytest.mark.parametrize("num_types,cap", [(2, 0.0), (1, 0.8), (2, 0.8)])
def test_store_form_loop_equals_actions(M, ctx, num_types, cap):
    from mrmd_amd.drivers import LJSystem
    n = 2744
    pos, L = _jittered(n, 0.7, 5)
    k = num_types * num_types
    kw = dict(cap=cap)
    if num_types > 1:
        kw = dict(sigma=[1.0, 0.93, 0.93, 0.86], epsilon=[1.0, 0.75, 0.75, 0.5], cap=[cap] * k, num_types=num_types,
                  type_stride=num_types, types=(np.arange(n) % 2).astype(np.int64))
    out = []
    for native in (True, False):
        s = LJSystem(ctx, pos, maxwell_boltzmann(n, 1.0, 9), L, **kw)
        if native:
            s.run(40, 0.002)
        else:
            for _ in range(40):
                s.step(0.002)
        out.append((s.local(M.POS), s.local(M.VEL), s.local(M.FORCE), s.rebuilds))
    assert out[0][3] == out[1][3] > 1
    for a, b in zip(out[0][:3], out[1][:3]):
        np.testing.assert_array_equal(a, b)


def test_dense_replicas_in_boxes_of_two_cells(ctx):
    """tiles of one column, neighbours through both faces of an axis, rows of several lanes"""
    from mrmd_amd.ensemble import adress_box, cubic_box, relax, replica
    specs = [(230, 0.9, False), (500, 0.9, False), (1300, 0.9, True), (64, 0.35, False), (5000, 0.3, True)]
    reps, pos = [], []
    g = np.random.default_rng(3)
    for k, (n, rho, ad) in enumerate(specs):
        box = adress_box(n, rho) if ad else cubic_box(n, rho)
        if min(box) < 2.0 * RN:
            box = [max(b, 2.0 * RN + 1e-6) for b in box]
        reps.append(replica(n, box, 1.0, 50 + k, adress=ad, tf_every=50))
        pos.append(g.uniform(0.0, 1.0, (n, 3)) * np.asarray(box))
    pos, vel = relax(ctx, reps, pos)
    e = B._ensemble(ctx, reps, pos, vel)
    e.run(1, 0)
    P, F = e.positions(), e.forces()
    for k, r in enumerate(reps):
        ref = B._oracle_adress_forces(P[k], r) if r["adress"] else B._oracle_plain_forces(P[k], r["box"])
        assert np.abs(F[k] - ref).max() <= 1e-12 * np.abs(ref).max(), k
