"""The learned brush's tiles (16 vertices a workgroup) against the batched kernel's (a wave a
tile), bit for bit: leaves below, at and above a tile and above eight tiles, brushes that
cover one vertex or the mesh, dabs that are rejected."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaf,radius", [(9, 0.15), (16, 0.4), (64, 0.02), (128, 0.3), (400, 0.25), (3000, 3.0)])
def test_single_and_batch(sg, leaf, radius):
    from dune_sculpt_amd import learned as L

    m = sg.MLP.load(L.MODEL_PATH)
    meshes = [sg.noisy_torus(41, 17, seed=2, amplitude=0.01), sg.noisy_icosphere(4, seed=3, amplitude=0.02)]
    rng = np.random.default_rng(5)
    at = [co[rng.integers(len(co), size=6)] for co, _ in meshes]
    row = lambda i: [sg.make_dab(tool=sg.TOOL_SMOOTH, location=c[i], radius=radius, strength=0.2 + 0.15 * i,
                                 smooth_iterations=4) for c in at]
    table = [L.learned_dabs(row(i)) for i in range(6)]
    b = sg.Batch(meshes, leaf_limit=leaf)
    b.set_learned(m)
    b.run(table)
    for j, (co, tris) in enumerate(meshes):
        p = sg.PBVH(co, tris, leaf_limit=leaf)
        p.set_learned(m)
        p.stroke([t[j] for t in table])
        assert p.positions().tobytes() == b.positions(j).tobytes()
        assert p.normals().tobytes() == b.normals(j).tobytes()
        p.close()
    b.close()
