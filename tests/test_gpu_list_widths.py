"""Verlet lists of any width against the CPU oracle: the width hint of a build changes neither the
list nor whether it is built, and rows longer than the list build's row buffers (96 entries) keep
every entry.  Counts and neighbour sets are integers: equal."""
import numpy as np
import pytest

import pyoracle as O
from test_gpu_split_rows import _jittered, _lists, _same_lists

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


def _ball(n, radius, center, seed):
    g = np.random.default_rng(seed)
    v = g.normal(size=(n, 3))
    r = radius * g.uniform(0.0, 1.0, (n, 1)) ** (1.0 / 3.0)
    return np.asarray(center) + v / np.linalg.norm(v, axis=1, keepdims=True) * r


@pytest.mark.parametrize("ratio", [1.0, 0.5])
def test_width_hints(M, ctx, ratio):
    pos, L = _jittered(4000, 0.8, 11)
    g, _, vl, ov = _lists(M, ctx, pos, RN, ratio, L)
    _same_lists(vl, ov, 4000, False)
    rows, counts = vl.full_rows(4000)
    entries = np.arange(rows.shape[1]) < counts[:, None]  # (what a row leaves over is not written)
    for hint in (60, 150, 300, 700, 2000):
        wide = M.HalfVerletList(ctx)
        wide.build(g, 0, g.nlocal, RN, ratio, [0.0] * 3, [L] * 3, hint)
        other, n = wide.full_rows(4000)
        np.testing.assert_array_equal(n, counts)
        np.testing.assert_array_equal(other[entries], rows[entries])


@pytest.mark.parametrize("ratio", [1.0, 0.5])
@pytest.mark.parametrize("density", [1.05, 1.6])
def test_rows_about_and_beyond_the_row_buffers(M, ctx, density, ratio):
    """rows of 40 to 110 and of 60 to 170 entries, in more tiles than take buffers of the list's width;
    the second build knows the widest row"""
    n = 30000
    pos, L = _jittered(n, density, 12)
    g, _, vl, ov = _lists(M, ctx, pos, RN, ratio, L)
    _same_lists(vl, ov, n, False)
    ref = ov.neighbors()
    sets = [set(ref[i, :c].tolist()) for i, c in enumerate(ov.counts()[:2000])]
    for _ in range(2):
        rows = vl.half_rows(n)
        assert all(rows[i] == s for i, s in enumerate(sets))
        vl.build(g, 0, n, RN, ratio, [0.0] * 3, [L] * 3)


@pytest.mark.parametrize("ratio", [1.0, 0.5])
@pytest.mark.parametrize("n", [600, 1500, 2040])
def test_clusters_within_the_radius(M, ctx, n, ratio):
    """everything neighbours everything; the same list object builds ordinary rows afterwards"""
    L = 14.0
    pos = _ball(n, 0.49 * RN, [0.45 * L] * 3, n)
    g, _, vl, ov = _lists(M, ctx, pos, RN, ratio, L)
    assert vl.num_pairs() == n * (n - 1) // 2
    _same_lists(vl, ov, n, n <= 600)
    pos, L = _jittered(1000, 0.8, 13)
    kw = (1000, RN, ratio, [0.0] * 3, [L] * 3)
    a, c, ov = M.Atoms.from_arrays(ctx, pos), O.Atoms.from_arrays(pos), O.Verlet()
    vl.build(a, 0, *kw)
    ov.build(c, 1000, 0, *kw)
    _same_lists(vl, ov, 1000, True)


def test_radius_far_below_the_cells(M, ctx):
    """a radius of less than a unit of the tiles' 16-bit coordinates (three cells of 10,000 radii an
    axis): every pair within a few units is decided on the records themselves, also across a cell
    face, where no column ties decide it"""
    g = np.random.default_rng(14)
    n, pos = 300, []
    for d in (0.004, 0.0095, 0.0105, 0.013, 0.02, 0.04):
        u = g.normal(size=(n, 3))
        u[:, 0] = np.abs(u[:, 0]) + 1.0
        u *= d / np.linalg.norm(u, axis=1, keepdims=True)
        base = g.uniform(5.0, 295.0, (n, 3))
        base[:, 0] = np.where(g.uniform(size=n) < 0.5, 100.0, 200.0) - u[:, 0] * g.uniform(0.1, 0.9, n)
        pos += [base, base + u]
    pos = np.concatenate(pos)
    _, _, vl, ov = _lists(M, ctx, pos, 0.01, 1e4, 300.0)
    assert ov.total() >= 2 * n
    _same_lists(vl, ov, pos.shape[0], True)
