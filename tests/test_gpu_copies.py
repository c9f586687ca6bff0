"""Checkpoints copied as one launch: restored bit for bit over sizes around the copy's
chunk (16 KiB) and over element counts whose arrays end off a 16-byte boundary."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nu,nv", [(9, 9), (31, 33), (64, 64), (67, 61), (205, 101)])
def test_restore_faces(sg, nu, nv):
    co, tris = sg.noisy_torus(nu, nv, seed=2, amplitude=0.01)
    p = sg.PBVH(co, tris, leaf_limit=64)
    boxes = lambda: np.array([p.node_bb(i) for i in range(p.tree_info()["nodes"])], np.float32)
    before = p.positions(), p.normals(), boxes()
    p.snapshot()
    dabs = [sg.make_dab(tool=t, location=co[0], radius=0.6, strength=0.5, grab_delta=(0.05, 0, 0)) for t in (1, 2, 5)]
    for _ in range(3):
        p.stroke(dabs)
        assert p.positions().tobytes() != before[0].tobytes()
        p.restore()
        assert all(a.tobytes() == b.tobytes() for a, b in zip(before, (p.positions(), p.normals(), boxes())))
    p.close()


@pytest.mark.parametrize("n,level", [(1, 2), (2, 3), (3, 4), (5, 3)])
def test_restore_grids(sg, n, level):
    from dune_sculpt_amd import grids as gr

    co, off, pv = gr.quad_sphere(n)
    g = gr.Grids(co, off, pv, level=level)
    g.recalc_normals()
    p = gr.GridPBVH(g, leaf_limit=500)
    d = sg.make_dab(tool=1, location=g.co()[0], radius=0.7, strength=0.6)
    p.snapshot()
    before = p.state()[:2]
    p.dab(d)
    once = p.state()[:2]
    assert once[0].tobytes() != before[0].tobytes()
    p.restore()
    assert all(a.tobytes() == b.tobytes() for a, b in zip(before, p.state()[:2]))
    p.dab(d)
    assert all(a.tobytes() == b.tobytes() for a, b in zip(once, p.state()[:2]))


def test_restore_batch(sg):
    meshes = [sg.noisy_torus(20 + i, 13, seed=i, amplitude=0.01) for i in range(3)]
    b = sg.Batch(meshes, leaf_limit=64)
    b.snapshot()
    before = [(b.positions(m), b.normals(m)) for m in range(3)]
    table = [[sg.make_dab(tool=1, location=co[0], radius=0.5, strength=0.6) for co, _ in meshes]] * 2
    b.run(table)
    b.restore()
    for m in range(3):
        assert b.positions(m).tobytes() == before[m][0].tobytes()
        assert b.normals(m).tobytes() == before[m][1].tobytes()
    b.close()
