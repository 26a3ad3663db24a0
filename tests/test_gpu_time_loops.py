"""The native time loops where a step's work was enqueued ahead of the wait for the displacement and
the step rebuilds all the same, which voids it: a cold start with one close pair, whose largest
displacement grows by more than a third from one step to the next, and a skin that the guess keeps
within and the step exceeds.  Against the same actions called one by one."""
import numpy as np
import pytest

from mrmd_amd.lattice import fcc

pytestmark = pytest.mark.gpu

DT, STEPS = 0.01, 8


@pytest.fixture(scope="module")
def M():
    import mrmd_amd
    return mrmd_amd


@pytest.fixture(scope="module")
def ctx(M):
    c = M.Context(0)
    yield c
    c.close()


def _largest_moves(M, system, L, steps):
    """each step's largest displacement, from the positions"""
    L = np.asarray(L)
    out = []
    for _ in range(steps):
        was = system.local(M.POS)
        system.step(DT)
        d = system.local(M.POS) - was
        d -= L * np.round(d / L)
        out.append(np.sqrt((d * d).sum(axis=1).max()))
    return out


def _skin(moves):
    """twice the middle between what the guess at the second step reckons with (1.25 times the first
    step's displacement) and that step's displacement; the first step always rebuilds"""
    assert moves[1] > 1.35 * moves[0], moves
    return 1.25 * moves[0] + moves[1]


def _both_loops(make, skin):
    a, b = make(skin), make(skin)
    for _ in range(STEPS):
        a.step(DT)
    b.run(STEPS, DT)
    assert a.rebuilds == b.rebuilds and a.rebuilds >= 2
    return a, b


@pytest.mark.parametrize("kind", ["plain", "permuted", "two types, capped"])
def test_lj_loop_rebuilds_against_the_guess(M, ctx, kind):
    from mrmd_amd.drivers import LJSystem
    pos, L = fcc(7, 0.8442)
    pos[1] = pos[0] + 0.8 * (pos[1] - pos[0]) / np.linalg.norm(pos[1] - pos[0])
    n = pos.shape[0]
    kw = dict(permute=kind == "permuted")
    if kind == "two types, capped":
        kw = dict(sigma=[1.0, 0.93, 0.93, 0.86], epsilon=[1.0, 0.75, 0.75, 0.5], cap=[0.7] * 4, num_types=2,
                  type_stride=2, types=(np.arange(n) % 3 == 2).astype(np.int64))

    def make(skin):
        return LJSystem(ctx, pos, np.zeros((n, 3)), L, skin=skin, **kw)

    # (not permuted, so that an atom keeps its place between the two positions)
    free = LJSystem(ctx, pos, np.zeros((n, 3)), L, skin=0.6, **{k: v for k, v in kw.items() if k != "permute"})
    a, b = _both_loops(make, _skin(_largest_moves(M, free, [L] * 3, 2)))
    for field in (M.POS, M.VEL, M.FORCE):
        np.testing.assert_array_equal(a.local(field), b.local(field))
    assert a.lj.energy_virial() == b.lj.energy_virial()


def test_adress_loop_rebuilds_against_the_guess(M, ctx):
    """ghost partners' forces are added by atomics, so the last bits can differ between any two runs:
    1e-9 after 8 steps, as in the other comparisons of the two loops"""
    from mrmd_amd.drivers import AdResSSystem
    L = [40.0, 12.0, 12.0]
    grid = np.stack(np.meshgrid(np.arange(32) * 1.25, np.arange(10) * 1.2, np.arange(10) * 1.2, indexing="ij"), -1)
    pos = grid.reshape(-1, 3) + 0.3
    at = np.argmin(np.abs(pos - [20.0, 6.0, 6.0]).sum(axis=1))
    pos[at + 1] = pos[at] + [0.0, 0.0, 0.8]

    def make(skin):
        return AdResSSystem(ctx, pos, np.zeros_like(pos), L, 8.0, 5.0, 1, temperature=0.0, skin=skin, tf_every=3)

    a, b = _both_loops(make, _skin(_largest_moves(M, make(0.6), L, 2)))
    assert a.ljig.run_counter == b.ljig.run_counter and a.tf.samples == b.tf.samples
    assert a.energy == pytest.approx(b.energy, rel=1e-10)
    for field in (M.POS, M.VEL):
        d = a.local(field) - b.local(field)
        d -= np.asarray(L) * np.round(d / np.asarray(L))
        assert np.abs(d).max() < 1e-9
    assert np.abs(a.tf.get_force() - b.tf.get_force()).max() < 1e-9
