"""The tile shape that a list build chooses: what a fresh list would choose, whatever the list object
has built before or was asked for, and the lists themselves are the same."""
import numpy as np
import pytest

from test_gpu_split_rows import _jittered

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


def _build(M, ctx, pos, L, vl=None, ratio=1.0):
    a = M.Atoms.from_arrays(ctx, pos)
    vl = vl or M.HalfVerletList(ctx)
    vl.build(a, 0, pos.shape[0], RN, ratio, [0.0] * 3, [L] * 3)
    return vl, vl.tiling()


@pytest.mark.parametrize("n", [4000, 70000])
def test_default_shape_can_be_asked_for(M, ctx, n):
    """4,000 atoms: one column by one cell; 70,000: two by two columns of three cells"""
    pos, L = _jittered(n, 0.8442, 3)
    fresh, shape = _build(M, ctx, pos, L)
    vl = M.HalfVerletList(ctx)
    for cells, columns in ((2, 3), (0, 1), (0, 2)):
        vl.set_tiling(cells, 256, columns)
        _, other = _build(M, ctx, pos, L, vl)
        if columns != 2:
            assert other["tile_columns"] == columns
    assert other == shape
    np.testing.assert_array_equal(vl.half_counts(n)[0], fresh.half_counts(n)[0])


def test_shape_follows_the_system(M, ctx):
    """a list object that has built another density, a wider stencil, a corner of the grid and a crowd whose
    tiles had to shrink; the shape after the crowd is back with the second ordinary build at the latest"""
    n = 70000
    pos, L = _jittered(n, 0.8442, 4)
    _, shape = _build(M, ctx, pos, L)
    vl = M.HalfVerletList(ctx)
    thin, thin_L = _jittered(n, 0.1, 5)
    for p, edge, ratio in ((thin, thin_L, 1.0), (pos, L, 0.5)):
        _, other = _build(M, ctx, p, edge, vl, ratio)
        assert other != shape
        assert _build(M, ctx, pos, L, vl)[1] == shape
    # as many atoms in a corner of the same grid
    corner, _ = _jittered(n, 0.8442 * 27, 5)
    assert _build(M, ctx, corner, L, vl)[1] != shape
    assert _build(M, ctx, pos, L, vl)[1] == shape
    g = np.random.default_rng(6)
    crowd = pos.copy()
    crowd[g.permutation(n)[:1500]] = 0.5 * L + g.uniform(-0.7, 0.7, (1500, 3))
    _, other = _build(M, ctx, crowd, L, vl)
    assert (other["tile_columns"], other["tile_cells"]) < (shape["tile_columns"], shape["tile_cells"])
    assert _build(M, ctx, crowd, L, vl)[1] == other
    _build(M, ctx, pos, L, vl)
    assert _build(M, ctx, pos, L, vl)[1] == shape


def test_tuners_try_the_default_shapes(M, ctx):
    """a system's or an ensemble's own choice is among the candidates, so tuning cannot lose it"""
    from mrmd_amd.autotune import ENSEMBLE_BLOCKS, ENSEMBLE_TARGETS, tune_lj_system
    from mrmd_amd.drivers import LJSystem
    from mrmd_amd.ensemble import Ensemble, cubic_box, replica
    pos, L = _jittered(4000, 0.8442, 7)
    s = LJSystem(ctx, pos, np.zeros_like(pos), L)
    s.rebuild()
    own, tried = s.vl.tiling(), []
    rebuild = s.rebuild

    def recorded():
        rebuild()
        tried.append(s.vl.tiling())

    s.rebuild = recorded
    tune_lj_system(s, force_reps=1)
    assert own in tried
    e = Ensemble(ctx, [replica(600, cubic_box(600, 0.8), 1.0, 1)])
    own = e.tiling()
    assert own["target_staged"] in ENSEMBLE_TARGETS and own["block"] in ENSEMBLE_BLOCKS


@pytest.mark.parametrize("n", [5000, 66000])
@pytest.mark.parametrize("num_types", [1, 2])
@pytest.mark.parametrize("cap", [0.0, 0.9])
def test_global_staging_gives_the_same_bits(M, ctx, n, num_types, cap):
    """rows of eight lanes and of one, every table, from a tile's slice of memory and from LDS"""
    pos, L = _jittered(n, 0.8442, n)
    pos[1] = pos[0] + [1e-3, 0.0, 0.0] if cap else pos[1]  # one pair far inside the capping distance
    types = (np.arange(n) % num_types).astype(np.int64)
    k = num_types * num_types
    lj = M.LennardJones(ctx, [2.5] * k, [1.0, 0.93, 0.93, 0.86][:k], [1.0, 0.75, 0.75, 0.5][:k],
                        capping_distance=[cap] * k, num_types=num_types, shifted=True, type_stride=num_types)
    out = []
    for limit in (0, 64):
        a = M.Atoms.from_arrays(ctx, pos, type=types)
        vl = M.HalfVerletList(ctx)
        vl.set_tiling(1, 256, 1)
        vl.set_stage_limit(limit)
        vl.build(a, 0, n, RN, 1.0, [0.0] * 3, [L] * 3)
        assert limit == 0 or vl.tiling()["max_staged"] > limit
        a.set_force(0.0)
        lj.apply(a, vl)
        out.append((a.download(M.FORCE, n), lj.energy_virial()))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]
