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


@pytest.mark.parametrize("levels,tables", [
    ((3, 4), [(0.05, 0.2, ())]),
    ((7,), [(0.4, 0.9, ()), (0.01, 0.03, ())]),
    ((4, 7, 2), [(0.02, 0.1, (1,)), (0.5, 1.5, ()), (0.02, 0.05, (0, 2))]),
])
def test_default_choice_keeps_the_bits(sg, levels, tables):
    meshes = [sg.noisy_icosphere(lv, seed=50 + i, amplitude=0.02) for i, lv in enumerate(levels)]
    a, b = sg.Batch(meshes, leaf_limit=64), sg.Batch(meshes, leaf_limit=64)
    b.set_persistent(False)
    for i, (rmin, rmax, empty) in enumerate(tables):
        table = _table(sg, meshes, 6, rmin, rmax, i, empty)
        a.run(table)
        b.run(table)
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
