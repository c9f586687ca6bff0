"""The default choice between the persistent step and the step graph, per loaded table: few
meshes with small dabs, a mesh without dabs, dabs that cover their meshes, and tables on
both sides of the rule loaded into one batch in turn.  Whatever is chosen, the bits and
totals are the step graph's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _table(sg, meshes, steps, rmin, rmax, seed, empty=()):
    rng = np.random.default_rng(seed)
    return [[None if m in empty else
             sg.make_dab(tool=(1, 2, 4, 5)[(s + m) % 4], location=co[rng.integers(len(co))],
                         radius=float(rng.uniform(rmin, rmax)), strength=0.6, smooth_iterations=1 + s % 4,
                         grab_delta=rng.normal(size=3) * 0.01) for m, (co, _) in enumerate(meshes)]
            for s in range(steps)]


@pytest.mark.parametrize("levels,tables", [  # per table: radii, meshes without dabs, the choice
    ((3, 4), [(0.05, 0.2, (), True)]),
    ((7,), [(0.4, 0.9, (), False), (0.01, 0.03, (), True), (0.5, 0.8, (), False)]),
    ((4, 7, 2), [(0.02, 0.1, (1,), True), (0.5, 1.5, (), False), (0.02, 0.05, (0, 2), True)]),
])
def test_default_choice_keeps_the_bits(sg, levels, tables):
    meshes = [sg.noisy_icosphere(lv, seed=50 + i, amplitude=0.02) for i, lv in enumerate(levels)]
    a, b = sg.Batch(meshes, leaf_limit=64), sg.Batch(meshes, leaf_limit=64)
    b.set_persistent(False)
    for i, (rmin, rmax, empty, persistent) in enumerate(tables):
        table = _table(sg, meshes, 6, rmin, rmax, i, empty)
        a.run(table)
        b.run(table)
        assert a.info()["persistent"] == persistent and not b.info()["persistent"], i
        for m in range(len(meshes)):
            assert np.array_equal(a.positions(m).view(np.uint32), b.positions(m).view(np.uint32)), (i, m)
            assert np.array_equal(a.normals(m).view(np.uint32), b.normals(m).view(np.uint32)), (i, m)
    assert a.totals() == b.totals()
    a.close()
    b.close()


@pytest.mark.parametrize("persistent", [False, True])
def test_tables_of_other_step_counts_in_one_batch(sg, persistent):
    """Tables that need other kernels in the step graph than the one before them (Smooth steps,
    odd and even) against the same dabs on each mesh alone."""
    meshes = [sg.noisy_icosphere(lv, seed=60 + lv, amplitude=0.02) for lv in (4, 5)]
    b = sg.Batch(meshes, leaf_limit=64)
    b.set_persistent(persistent)
    alone = [sg.PBVH(co, tris, leaf_limit=64) for co, tris in meshes]
    rng = np.random.default_rng(5)
    for tool, k in ((1, 1), (2, 4), (2, 16), (2, 3), (2, 1), (4, 1), (2, 64)):
        table = [[sg.make_dab(tool=tool, location=co[rng.integers(len(co))], radius=0.3, strength=0.5,
                              smooth_iterations=k) for co, _ in meshes] for _ in range(3)]
        b.run(table)
        for m, p in enumerate(alone):
            p.stroke([row[m] for row in table])
            assert np.array_equal(b.positions(m).view(np.uint32), p.positions().view(np.uint32)), (tool, k, m)
            assert np.array_equal(b.normals(m).view(np.uint32), p.normals().view(np.uint32)), (tool, k, m)
    b.close()
    for p in alone:
        p.close()


def test_choice_by_tool_and_steps(sg):
    """A wide Draw dab on one mesh beside Smooth dabs on the other: with a few steps the graph
    is the shorter one, with 64 it has 63 kernels more in every step."""
    meshes = [sg.noisy_icosphere(7, seed=50, amplitude=0.02), sg.noisy_icosphere(4, seed=51, amplitude=0.02)]
    b = sg.Batch(meshes, leaf_limit=64)
    for k, persistent in ((2, False), (64, True), (1, False)):
        b.load([[sg.make_dab(tool=1, location=meshes[0][0][9], radius=0.25, strength=0.5),
                 sg.make_dab(tool=2, location=meshes[1][0][9], radius=0.04, strength=0.5, smooth_iterations=k)]] * 4)
        assert b.info()["persistent"] == persistent, k
    b.set_persistent(False)
    assert not b.info()["persistent"]
    b.close()
