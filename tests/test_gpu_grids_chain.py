"""Strokes on grids, where each dab searches for the next and the faces fit a workgroup,
against the oracle and against the same dabs one by one, bit for bit: small and large
grids (level 6: the kernels per leaf), more leaves than one workgroup searches, faces whose
grids lie in several leaves, coordinates that are zero (boxes with a side of either sign)."""
import numpy as np
import pytest

from dune_sculpt_amd import grids as gr
from test_gpu_grids import noisy_sphere_grids, oracle_of, stroke

pytestmark = pytest.mark.gpu


def _all(p):
    co, no, mk = p.state()
    vb, ob = p.boxes()
    return [co, no, vb, ob, p.last_affected(), p.last_gathered(), p.last_stats()[:2]] + ([mk] if mk is not None else [])


@pytest.mark.parametrize("n,level,leaf_limit,amp,mask", [
    (1, 2, 10, 0.02, False), (3, 3, 100, 0.0, False), (4, 5, 1500, 0.02, True), (2, 6, 4000, 0.02, False),
    (20, 2, 40, 0.02, False), (9, 4, 100, 0.0, True)])
def test_stroke(sg, po, n, level, leaf_limit, amp, mask):
    dabs = stroke(sg, 3, 21, 0.1, 0.5)
    got = []
    for how in ("graph", "stream", "dabs"):
        g, mesh = noisy_sphere_grids(sg, n, level, seed=5, amp=amp, mask=mask)
        if mask:
            g.set_mask(np.clip(g.co()[:, 0], 0, 1).astype(np.float32))
        if how == "graph":
            o = oracle_of(po, g, mesh, leaf_limit)
            for d in dabs + dabs:
                o.dab(po.to_orc(d))
            want = [*o.state()[:2], *o.boxes()]
            o.close()
        p = gr.GridPBVH(g, leaf_limit=leaf_limit)
        if how == "dabs":
            for d in dabs + dabs:
                p.dab(d)
        elif how == "stream":
            p.stroke(dabs, graph=False)
            p.stroke(dabs, graph=False)
        else:
            s = p.prepare(dabs)
            s.launch(sync=False)
            s.launch()
        got.append(_all(p))
        p.close()
    for a in got:
        for x, y in zip(a[:4], want):
            assert np.array_equal(np.ascontiguousarray(x).view(np.uint32), np.ascontiguousarray(y).view(np.uint32))
        for x, y in zip(a, got[0]):
            assert np.asarray(x).tobytes() == np.asarray(y).tobytes()


def test_single_dab_after_strokes_and_edits(sg, po):
    """The counters and marks a stroke leaves: a dab, a host edit's updates, a replay."""
    dabs = stroke(sg, 3, 5, 0.2, 0.4)
    got = []
    for chained in (True, False):
        g, _ = noisy_sphere_grids(sg, 5, 4, seed=5)
        p = gr.GridPBVH(g, leaf_limit=1000)
        run = (lambda: p.stroke(dabs, graph=False)) if chained else (lambda: [p.dab(d) for d in dabs])
        run()
        p.dab(dabs[2])
        p.snapshot()
        run()
        p.restore()
        run()
        got.append(_all(p))
        p.close()
    assert all(np.asarray(x).tobytes() == np.asarray(y).tobytes() for x, y in zip(*got))


def test_dabs_of_few_leaves_before_wide_ones_beside_other_work(sg):
    """The refit's last workgroup searches for the next dab while others of its launch may not
    have started: dabs that gather nothing or a leaf or two (few workgroups take part) before
    dabs over most leaves, with another stream keeping the chip busy."""
    wide, narrow = stroke(sg, 3, 30, 0.5, 1.2), stroke(sg, 4, 30, 0.01, 0.02)
    away = sg.make_dab(tool=1, location=(9, 9, 9), radius=0.1, strength=0.5)
    dabs = [d for i in range(30) for d in (narrow[i], away, wide[i])]
    co, tris = sg.noisy_icosphere(7, seed=3, amplitude=0.02)
    other = sg.PBVH(co, tris, leaf_limit=64)
    cover = other.prepare([sg.make_dab(tool=2, location=co[0], radius=3.0, strength=0.5, smooth_iterations=8)] * 40)
    got = []
    for busy in (True, False, None):
        g, _ = noisy_sphere_grids(sg, 16, 3, seed=5)
        p = gr.GridPBVH(g, leaf_limit=200)
        assert p.nodes > 200
        for _ in range(2):
            if busy:
                for _ in range(4):
                    cover.launch(sync=False)
            if busy is None:  # each dab with a search of its own
                for d in dabs:
                    p.dab(d)
            else:
                p.stroke(dabs)
        got.append(_all(p))
        p.close()
    cover.launch()
    other.close()
    for x in got[:2]:
        assert all(np.asarray(u).tobytes() == np.asarray(w).tobytes() for u, w in zip(x, got[2]))


@pytest.mark.parametrize("bad", [{"tool": 21}, {"tool": 2, "flag": "SMOOTH_LEARNED"}])
def test_stroke_with_a_refused_dab(sg, bad):
    """A stroke stops at a dab that grids do not cover; what ran before it stays, and the next
    calls (a captured stroke that is not launched yet, a dab, the stroke) see clean counters."""
    dabs = stroke(sg, 3, 6, 0.3, 0.6)
    kw = {k: getattr(sg, v) if isinstance(v, str) else v for k, v in bad.items()}
    no = sg.make_dab(location=(0, 0, 1), radius=0.3, strength=0.5, **kw)
    got = []
    for refused in (True, False):
        g, _ = noisy_sphere_grids(sg, 12, 3, seed=5)
        p = gr.GridPBVH(g, leaf_limit=200)
        if refused:
            with pytest.raises(RuntimeError):
                p.stroke([dabs[0], no, dabs[1]], graph=False)
            with pytest.raises(RuntimeError):
                p.prepare([dabs[0], no])
        else:
            p.dab(dabs[0])
        st = p.prepare(dabs[2:])
        p.dab(dabs[1])
        st.launch()
        got.append(_all(p))
        p.close()
    assert all(np.asarray(x).tobytes() == np.asarray(y).tobytes() for x, y in zip(*got))


@pytest.mark.parametrize("level,leaf_limit", [(2, 10000), (3, 2500)])
def test_many_faces(sg, po, level, leaf_limit):
    """A base of 66 k faces, past the line where faces and edges are tested four to a line and
    small dabs run per leaf: both kinds of dab in one stroke, against the oracle."""
    g, mesh = noisy_sphere_grids(sg, 105, level, seed=5)
    o = oracle_of(po, g, mesh, leaf_limit)
    p = gr.GridPBVH(g, leaf_limit=leaf_limit)
    small, wide = stroke(sg, 3, 8, 0.01, 0.03), stroke(sg, 4, 8, 0.1, 0.4)
    dabs = [d for i in range(8) for d in (small[i], wide[i], small[(i + 1) % 8])]
    p.stroke(dabs)
    for d in dabs:
        o.dab(po.to_orc(d))
    for x, y in zip(p.state()[:2], o.state()[:2]):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    for x, y in zip(p.boxes(), o.boxes()):
        assert np.array_equal(x, y)
    p.close()
    o.close()
