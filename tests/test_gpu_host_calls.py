"""Calls that hand data to the host through pinned memory, at the size where they change
to staged copies, and the open undo step's count read on the device."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return (-3 * d).astype(np.float32), d.astype(np.float32)


@pytest.mark.parametrize("n", [1, 63, 4097, 23831, 23832, 30000])  # 2 MiB of rays and hits between 23831 and 23832
def test_rays_in_parts(sg, n):
    co, tris = sg.noisy_icosphere(4, seed=3, amplitude=0.02)
    p = sg.PBVH(co, tris, leaf_limit=64)
    s, d = _rays(n, n)
    whole = p.raycast(s, d)
    parts = np.concatenate([p.raycast(s[i:i + 7001], d[i:i + 7001]) for i in range(0, n, 7001)])
    assert whole["hit"].all()
    for f in whole.dtype.names:
        if f != "reserved":
            assert whole[f].tobytes() == parts[f].tobytes()
    p.close()


@pytest.mark.parametrize("nu,nv", [(9, 9), (1021, 171), (1025, 171)])  # 2 MiB of coordinates between the last two
def test_read_positions(sg, nu, nv):
    co, tris = sg.noisy_torus(nu, nv, seed=2, amplitude=0.01)
    p = sg.PBVH(co, tris)
    for _ in range(2):
        assert p.positions().tobytes() == co.tobytes()
    p.close()


def test_restore_original_of_an_overflowed_step_changes_nothing(sg):
    co, tris = sg.noisy_icosphere(4, seed=3, amplitude=0.02)
    p = sg.PBVH(co, tris, leaf_limit=64)
    p.undo_begin(max_verts=20)
    p.dab(sg.make_dab(tool=1, location=co[0], radius=0.5, strength=0.7))
    after = p.positions(), p.normals()
    with pytest.raises(RuntimeError):
        p.undo_restore_original()
    assert all(a.tobytes() == b.tobytes() for a, b in zip(after, (p.positions(), p.normals())))
    with pytest.raises(RuntimeError):
        p.undo_end()
    p.close()


def test_custom_curves_of_one_stroke(sg):
    """Two curves in one stroke, graph and stream launches, refit at the end and after each dab."""
    co, tris = sg.noisy_icosphere(4, seed=3, amplitude=0.02)
    t = np.linspace(0, 1, sg.CM_TABLE + 1)
    dabs = [sg.make_dab(tool=1, location=co[9 * i], radius=0.3, strength=0.5, falloff=sg.CURVE_CUSTOM,
                        curve_table=(t ** (1 + i % 2)).astype(np.float32)) for i in range(6)]
    got = []
    for how in ({"graph": True}, {"graph": False}, {"refit_each": True}, {"graph": False, "refit_each": True}, None):
        p = sg.PBVH(co, tris, leaf_limit=64)
        if how is None:
            for d in dabs:
                p.dab(d)
        else:
            p.stroke(dabs, **how)
        got.append([p.positions().tobytes(), p.normals().tobytes(), p.last_affected().tobytes(),
                    p.last_stats()[:2].tobytes()])
        p.close()
    assert all(g == got[-1] for g in got)
