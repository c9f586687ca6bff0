"""Ray-placed strokes as fused dabs against the separate kernels, bit for bit: lengths around
the modulo-3 lists, rays that miss, Smooth over several launches, dabs in between that are
not fused, masks, hidden vertices, an open undo step, logged counts, replays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dabs(sg, n, seed, ks, orig=False):
    rng = np.random.default_rng(seed)
    t = np.linspace(0, 1, sg.CM_TABLE + 1).astype(np.float32)
    dabs = []
    for i in range(n):
        kw = {"falloff": sg.CURVE_CUSTOM, "curve_table": t ** (1 + i % 2)} if i % 3 == 1 else {}
        if orig and i % 4 == 3:
            kw["flag"] = sg.DAB_ORIGINAL
        dabs.append(sg.make_dab(tool=(1, 4, 2, 5)[i % 4], location=(0, 0, 0), radius=float(rng.uniform(0.08, 0.35)),
                                strength=float(rng.uniform(0.2, 1.0)), smooth_iterations=ks[i % len(ks)], **kw))
    a = np.linspace(0, 2.0, n) + seed
    d = np.stack([np.cos(a), np.sin(a), 0.3 * np.sin(3 * a)], -1)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    start, dirs = 3 * d, -d
    dirs[4::7] *= -1  # these miss
    return dabs, start.astype(np.float32), dirs.astype(np.float32)


def _run(sg, fused, n, ks, how, orig=False):
    co, tris = sg.noisy_icosphere(5, seed=7, amplitude=0.02)
    p = sg.PBVH(co, tris, leaf_limit=64, hidden=co[:, 2] > 0.6)
    p.set_mask(np.clip(0.5 - co[:, 1], 0, 1).astype(np.float32))
    p.set_fused(fused)
    dabs, s, d = _dabs(sg, n, 1, ks, orig)
    out = []

    def state():
        boxes = np.array([np.concatenate([p.node_bb(i), p.node_bb(i, original=True)])
                          for i in range(p.tree_info()["nodes"])], np.float32)
        out.extend([p.positions(), p.normals(), boxes, p.last_affected(), p.last_gathered(), p.last_stats()[:2]])

    if how == "prepared":
        st = p.prepare_placed(dabs, s, d, log=True)
        p.undo_begin()
        st.launch()
        st.launch(sync=False)
        st.launch()
        p.undo_end()
        out.append(p.stroke_log(n)[:, :5])
        state()
        p.undo()
        out.extend([p.positions(), p.normals()])
    else:
        for _ in range(2):
            p.stroke_placed(dabs, s, d, log=True, **how)
            out.append(p.stroke_log(n)[:, :5])
            state()
        p.stroke(dabs[:2])  # centre 0: gathers nothing, then a dab that reads what the stroke left
        p.dab(sg.make_dab(tool=4, location=co[100], radius=0.4, strength=0.5))
        state()
    p.close()
    return out


@pytest.mark.parametrize("n,ks", [(1, (2,)), (2, (3,)), (3, (4,)), (4, (1,)), (5, (5,)), (7, (8, 2)), (24, (3, 4, 9))])
@pytest.mark.parametrize("how", [{"graph": True}, {"graph": False}, {"graph": False, "refit_each": True}, "prepared"])
def test_placed(sg, n, ks, how):
    a, b = _run(sg, True, n, ks, how), _run(sg, False, n, ks, how)
    assert all(x.tobytes() == y.tobytes() for x, y in zip(a, b))


def test_broken_by_dabs_that_are_not_fused(sg):
    a, b = _run(sg, True, 24, (3,), "prepared", True), _run(sg, False, 24, (3,), "prepared", True)
    assert all(x.tobytes() == y.tobytes() for x, y in zip(a, b))
