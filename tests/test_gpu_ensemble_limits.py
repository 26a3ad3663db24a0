"""Ensembles at the limits of their lists and sums, and saved states that are none."""
import numpy as np
import pytest

from mrmd_amd.lattice import rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import mrmd_amd
    return mrmd_amd


@pytest.fixture(scope="module")
def ctx(M):
    c = M.Context(0)
    yield c
    c.close()


def _cold(M, ctx, pos, box, rc, **lj):
    """one plain replica at rest, without noise: a step leaves it where it is"""
    from mrmd_amd.ensemble import Ensemble, replica
    e = Ensemble(ctx, [replica(pos.shape[0], box, 0.0, 1)], rc, 0.3)
    e.set_lj(**lj)
    e.upload(M.POS, [pos])
    e.upload(M.VEL, [np.zeros_like(pos)])
    return e


@pytest.mark.parametrize("side", [21, 22])
def test_neighbourhoods_beyond_the_entries_are_refused(M, ctx, side):
    """a list entry holds 15 bits: in a box of two cells per axis the smallest tile's neighbourhood is
    27 cells, 27 / 8 of the atoms, so 9,261 atoms (31,255 records) still have lists and 10,648
    (35,937) have none"""
    rc = 0.5 * side - 0.31
    i = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)
    pos = i + 0.5 + rng(5).uniform(-0.2, 0.2, i.shape)
    e = _cold(M, ctx, pos, [float(side)] * 3, rc)
    if 27 * pos.shape[0] > 8 * 32768:
        with pytest.raises(M.MrmdError, match="neighbourhood"):
            e.run(1, 0)
        return
    e.run(1, 0)
    F = e.forces()[0]
    for k in range(0, pos.shape[0], 997):
        d = pos[k] - pos
        d -= side * np.round(d / side)
        r2 = np.sum(d * d, axis=1)
        w = np.where((r2 > 0.0) & (r2 <= rc * rc), r2, np.inf)
        f6 = 1.0 / w ** 3
        f = d * (f6 * (48.0 * f6 - 24.0) / w)[:, None]
        # 5,000 terms in another order: sqrt(5000) roundings of 1.1e-16 of the summed magnitudes
        assert np.abs(F[k] - f.sum(axis=0)).max() <= 1e-14 * np.abs(f).sum(axis=0).max()


@pytest.mark.parametrize("cap", [0.0, 1e-100])
def test_energy_of_an_overflowing_pair_is_infinite(M, ctx, cap):
    """two atoms 1e-60 apart: r^-12 and r^-6 overflow, and their difference is the first, not a NaN"""
    pos = np.array([[0.0, 0.0, 0.0], [1e-60, 0.0, 0.0], [3.0, 3.0, 3.0]])
    e = _cold(M, ctx, pos, [6.0] * 3, 2.5, cap=cap)
    e.run(1, 0)
    assert e.energies()[0][0] == np.inf


@pytest.mark.parametrize("bad", [-1, 300, 100, 1 << 30])
def test_states_with_foreign_atom_indices_are_refused(M, ctx, bad):
    """a negative index, one past the atoms, one of the other replica (or a second of its own) and one far
    beyond; the refused load leaves the ensemble as it was"""
    from mrmd_amd.ensemble import Ensemble, cubic_box, replica
    reps = [replica(n, cubic_box(n, 0.3), 1.0, n) for n in (200, 100)]
    g = rng(8)
    e = Ensemble(ctx, reps)
    e.set_lj(cap=0.7)
    e.upload(M.POS, [g.uniform(0.0, 1.0, (r["num_atoms"], 3)) * np.asarray(r["box"]) for r in reps])
    e.run(5, 0)
    state, pos = e.state(), np.concatenate(e.positions())
    header, n = 64, 300
    index = header + n * 32 + 6 * n * 8  # after the positions, three velocities and three forces
    order = state[index: index + 4 * n].view(np.int32)
    assert sorted(order.tolist()) == list(range(n))
    for place in (0, 250):
        broken = state.copy()
        broken[index + 4 * place: index + 4 * place + 4] = np.array([bad], np.int32).view(np.uint8)
        if broken.tobytes() == state.tobytes():
            continue
        with pytest.raises(M.MrmdError, match="indices"):
            e.load_state(broken)
    np.testing.assert_array_equal(np.concatenate(e.positions()), pos)
    e.load_state(state)
