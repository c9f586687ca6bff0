"""Chained fused dabs (one launch per dab that also searches for the next one) against the
separate kernels, bit for bit: positions, normals, every node box, the last dab's affected
vertices and gathered leaves, per-dab logged counts.  At the chain's own edges: every
position of the modulo-3 lists (lengths 1..7), chains broken by dabs that are not fused,
meshes of fewer leaves than list segments, radii that jump (the next dab's area normal
then comes from leaves the dab before did not touch), area spheres larger than the brush,
hidden leaves, refit after every dab, replays, undo and what reads the mesh after it."""
import numpy as np
import pytest

from parity_util import n_bit_diff

pytestmark = pytest.mark.gpu


def _state(p):
    n = p.tree_info()["nodes"]
    boxes = np.array([np.concatenate([p.node_bb(i), p.node_bb(i, original=True)]) for i in range(n)], np.float32)
    return p.positions(), p.normals(), boxes


def _same(a, b):
    return all(n_bit_diff(x, y) == 0 for x, y in zip(a, b))


def _path(sg, n, seed, radii, tools, ks=(2,), spacing=0.3, **kw):
    """Overlapping dabs along a great circle of the unit sphere."""
    radii = np.asarray(radii, np.float32)
    c = sg.great_circle_centres(seed, radii, spacing_frac=spacing)
    rng = np.random.default_rng(seed)
    return [sg.make_dab(tool=tools[i % len(tools)], location=c[i], radius=float(radii[i]),
                        strength=float(rng.uniform(0.2, 1.0)), smooth_iterations=int(ks[i % len(ks)]),
                        grab_delta=rng.normal(size=3) * 0.02, **kw) for i in range(n)]


def _check(sg, co, tris, dabs, leaf=64, hidden=None, mask=None, **how):
    a = sg.PBVH(co, tris, leaf_limit=leaf, hidden=hidden)
    b = sg.PBVH(co, tris, leaf_limit=leaf, hidden=hidden)
    assert a.set_fused(True)
    b.set_fused(False)
    for p in (a, b):
        if mask is not None:
            p.set_mask(mask)
        p.stroke(dabs, log=True, **how)
        p.stroke(dabs[::-1], log=True, **how)  # on what the first one left
    assert np.array_equal(a.stroke_log(len(dabs))[:, :5], b.stroke_log(len(dabs))[:, :5])
    assert np.array_equal(a.last_affected(), b.last_affected())
    assert np.array_equal(a.last_gathered(), b.last_gathered())
    assert np.array_equal(a.last_stats()[:2], b.last_stats()[:2])
    assert _same(_state(a), _state(b))
    a.close()
    b.close()


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("graph", [True, False])
def test_lengths(sg, n, graph):
    co, tris = sg.noisy_icosphere(5, seed=3, amplitude=0.02)
    _check(sg, co, tris, _path(sg, n, n, np.full(n, 0.2), (1, 4, 2, 5)), graph=graph)


@pytest.mark.parametrize("tools,ks", [((1,), (1,)), ((1, 2), (4,)), ((2,), (1, 5, 4, 9)), ((4, 5, 1), (1,)),
                                      ((1, 2, 2), (3, 6))])
def test_broken_chains(sg, tools, ks):
    """Smooth with more steps than a launch covers, as several launches between dabs of one."""
    co, tris = sg.noisy_icosphere(5, seed=4, amplitude=0.02)
    _check(sg, co, tris, _path(sg, 24, 2, np.full(24, 0.15), tools, ks))


@pytest.mark.parametrize("level,leaf", [(1, 128), (2, 128), (2, 20), (3, 9), (4, 300)])
def test_few_and_odd_leaves(sg, level, leaf):
    co, tris = sg.noisy_icosphere(level, seed=5, amplitude=0.02)
    _check(sg, co, tris, _path(sg, 12, 6, np.full(12, 0.5), (1, 2, 4, 5)), leaf=leaf)


@pytest.mark.parametrize("factor", [0.25, 0.5, 1.0, 1.7])
def test_area_normal_of_jumping_radii(sg, factor):
    co, tris = sg.noisy_icosphere(6, seed=6, amplitude=0.02)
    radii = np.tile([0.05, 0.6, 0.1, 0.02, 0.9, 0.05], 4)
    _check(sg, co, tris, _path(sg, 24, 7, radii, (1,), normal_radius_factor=factor), leaf=32)


@pytest.mark.parametrize("k", [5, 6, 7, 8, 9, 13, 64])
def test_smooth_over_several_launches(sg, k):
    """More steps than one launch covers, beside other tools, with a mask."""
    co, tris = sg.noisy_icosphere(5, seed=10, amplitude=0.02)
    mask = np.clip(0.5 - co[:, 1], 0, 1).astype(np.float32)
    _check(sg, co, tris, _path(sg, 9, 3, np.full(9, 0.25), (2, 1, 2, 2, 5), (k,)), mask=mask)
    _check(sg, co, tris, _path(sg, 1, 3, [0.4], (2,), (k,)), graph=False)


def _quad_torus(sg, nu, nv, mixed):
    """Quads of a torus; with `mixed` every third one split into two triangles."""
    co, _ = sg.noisy_torus(nu, nv, seed=3, amplitude=0.02)
    i, j = np.meshgrid(np.arange(nu), np.arange(nv), indexing="ij")
    q = np.stack([i * nv + j, (i + 1) % nu * nv + j, (i + 1) % nu * nv + (j + 1) % nv, i * nv + (j + 1) % nv], -1)
    faces = []
    for n, f in enumerate(q.reshape(-1, 4).tolist()):
        faces += [f[:3], [f[0], f[2], f[3]]] if mixed and n % 3 == 0 else [f]
    off = np.concatenate([[0], np.cumsum([len(f) for f in faces])]).astype(np.int32)
    return co, (off, np.concatenate(faces).astype(np.int32), np.ones(len(faces), np.uint8),
                np.zeros(len(faces), np.int16))


@pytest.mark.parametrize("nu,nv,leaf,mixed", [(40, 13, 64, False), (40, 13, 64, True), (9, 9, 128, True),
                                              (101, 31, 17, False)])
def test_quads(sg, nu, nv, leaf, mixed):
    co, polys = _quad_torus(sg, nu, nv, mixed)
    rng = np.random.default_rng(4)
    dabs = [sg.make_dab(tool=(1, 4, 2, 5)[i % 4], location=co[rng.integers(len(co))], radius=float(rng.uniform(0.1, 0.5)),
                        strength=0.6, smooth_iterations=1 + i % 6, grab_delta=rng.normal(size=3) * 0.02)
            for i in range(20)]
    got = []
    for fused in (True, False):
        p = sg.PBVH(co, None, leaf_limit=leaf, polys=polys)
        assert p.set_fused(fused), "triangles and quads have halo tables"
        p.stroke(dabs, log=True)
        got.append([*_state(p), p.last_affected(), p.last_gathered(), p.stroke_log(20)[:, :5]])
        p.close()
    for x, y in zip(*got):
        assert x.tobytes() == y.tobytes()


def test_ngons_keep_the_separate_kernels(sg):
    """A pentagon's corners do not fit a face record: no halo tables, the dab still runs."""
    t = np.linspace(0, 2 * np.pi, 6)[:5]
    co = np.concatenate([np.stack([np.cos(t), np.sin(t), 0 * t], -1), [[0, 0, 1]]]).astype(np.float32)
    faces = [[4, 3, 2, 1, 0]] + [[i, (i + 1) % 5, 5] for i in range(5)]
    off = np.concatenate([[0], np.cumsum([len(f) for f in faces])]).astype(np.int32)
    p = sg.PBVH(co, None, polys=(off, np.concatenate(faces).astype(np.int32), np.zeros(6, np.uint8),
                                 np.zeros(6, np.int16)))
    assert not p.set_fused(True)
    p.stroke([sg.make_dab(tool=1, location=(0, 0, 1), radius=0.8)] * 2)
    assert p.positions()[5, 2] > 1.0
    p.close()


def test_hidden_masked_refit_each(sg):
    co, tris = sg.noisy_icosphere(5, seed=8, amplitude=0.02)
    hidden = co[:, 2] > 0.55
    mask = np.clip(co[:, 0], 0, 1).astype(np.float32)
    dabs = _path(sg, 30, 11, np.random.default_rng(1).uniform(0.05, 0.4, 30), (1, 4, 2, 5), (1, 4))
    _check(sg, co, tris, dabs, hidden=hidden, mask=mask, refit_each=True)


def test_replay_undo_and_readers(sg):
    """A captured stroke replayed over a changed mesh, an undo step around it, then the
    draw buffers and rays: as after the separate kernels."""
    co, tris = sg.noisy_icosphere(5, seed=9, amplitude=0.02)
    dabs = _path(sg, 17, 13, np.random.default_rng(2).uniform(0.05, 0.3, 17), (1, 2, 4, 5), (4,))
    dirs = np.random.default_rng(3).normal(size=(200, 3))
    dirs = (dirs / np.linalg.norm(dirs, axis=1, keepdims=True)).astype(np.float32)
    got = []
    for fused in (True, False):
        p = sg.PBVH(co, tris, leaf_limit=64)
        p.set_fused(fused)
        p.draw_build(np.ones(len(tris), np.int32))
        st = p.prepare(dabs)
        p.undo_begin()
        st.launch()
        p.dab(dabs[3])
        st.launch(sync=False)
        st.launch()
        p.undo_end()
        out = [*_state(p)]
        p.draw_update()
        leaf = [i for i in range(p.tree_info()["nodes"]) if p.node_flag(i) & sg.PBVH_Leaf]
        out.append(np.concatenate([p.draw_leaf(i)[0].reshape(-1) for i in leaf]))
        p.stroke_placed(dabs[:6], -3 * dirs[:6], dirs[:6])
        h = p.raycast(-3 * dirs, dirs)
        out += [h[f] for f in ("hit", "depth", "looptri")] + [*_state(p)]
        p.undo()
        out += [*_state(p)]
        got.append(out)
        p.close()
    for x, y in zip(*got):
        assert x.tobytes() == y.tobytes()


def test_area_normal_of_leaves_whose_boxes_lag(sg, po):
    """Host edits whose normals were updated and bounds not: a leaf that the dab before did
    not touch is gathered by its old box, and every vertex of it counts for the area normal,
    wherever it lies now."""
    co, tris = sg.noisy_icosphere(5, seed=9, amplitude=0.02)
    c, r = co[123], 0.6
    dabs = [sg.make_dab(tool=1, location=-c, radius=0.1, strength=0.5),
            sg.make_dab(tool=1, location=c, radius=r, strength=0.7, normal_radius_factor=0.5)]
    o = po.Oracle(co, tris, leaf_limit=64)
    near = {n: np.linalg.norm(co[o.node_verts(n)] - c, axis=1).min() for n in o.leaves_dfs()}
    far = [n for n in near if 0.36 < near[n] < 0.55]
    assert len(far) > 3
    moved = np.unique(np.concatenate([o.node_verts(n) for n in far]))
    got = []
    for fused in (True, False):
        p = sg.PBVH(co, tris, leaf_limit=64)
        assert p.set_fused(fused)
        if fused:
            o.set_normals(p.normals())
        mv = p.mverts()
        for v in moved:
            mv[v] = (c + 0.2 * (co[v] - c)).astype(np.float32)
            if fused:
                o.set_vert(v, mv[v])
        for n in far:
            p.node_mark_update(n)
        p.update_normals()  # uploads the edit; no vertex is marked, and no bounds update follows
        p.stroke(dabs, log=True)
        got.append([p.stroke_log(2)[:, :6], p.positions(), p.normals()])
        p.close()
    assert all(x.tobytes() == y.tobytes() for x, y in zip(*got))
    for d in dabs:
        o.dab(d)
    assert np.abs(got[0][1] - o.positions()).max() <= 1e-5
    o.close()


@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_vertices_that_are_no_numbers(sg, value):
    """A vertex of some leaves is NaN or infinite: its leaf's box folds over it, its neighbours'
    normals and Smooth steps take it up, and the chain decides as the separate kernels do."""
    co, tris = sg.noisy_icosphere(5, seed=9, amplitude=0.02)
    dabs = _path(sg, 16, 5, np.resize([0.5, 0.1, 0.6], 16), (1, 4, 1, 2, 5), (3, 6))
    at = np.stack([d.location for d in dabs[:4]]).astype(np.float32)
    bad = [int(np.argsort(np.linalg.norm(co - c, axis=1))[j]) for c in at for j in (60, 140)]
    got = []
    for fused in (True, False):
        p = sg.PBVH(co, tris, leaf_limit=64)
        p.set_fused(fused)
        mv = p.mverts()
        for v in bad:
            mv[v] = (co[v][0], value, co[v][2])
            p.vert_mark_update(v)
        for i in range(p.tree_info()["nodes"]):
            if p.node_flag(i) & sg.PBVH_Leaf:
                p.node_mark_update(i)
        p.update_bounds(sg.PBVH_UpdateBB | sg.PBVH_UpdateOriginalBB)
        p.stroke(dabs, log=True)
        got.append([p.stroke_log(16)[:, :6], *_state(p), p.last_affected()])
        p.close()
    for x, y in zip(*got):
        assert np.array_equal(x, y, equal_nan=x.dtype == np.float32)
    assert np.isnan(got[0][1]).any() or np.isinf(got[0][1]).any()


@pytest.mark.parametrize("nu,nv,leaf", [(64, 28, 1900), (60, 30, 1800), (62, 30, 1900)])
def test_largest_fused_leaves(sg, nu, nv, leaf):
    """Two leaves whose vertices, ring and faces take 60.5 to 62.8 KiB of LDS for a Draw dab
    are still one launch a dab (no normals kernel of its own)."""
    co, tris = sg.noisy_torus(nu, nv, seed=2, amplitude=0.01)
    dabs = [sg.make_dab(tool=(1, 4, 5)[i % 3], location=co[37 * i], radius=0.3, strength=0.5, grab_delta=(0.01, 0, 0))
            for i in range(7)]
    _check(sg, co, tris, dabs, leaf=leaf)
    p = sg.PBVH(co, tris, leaf_limit=leaf)
    p.set_profile(True)
    p.stroke(dabs, graph=False)
    assert [v[1] for k, v in p.profile_read().items() if "post" in k] == [0]
    p.close()


@pytest.mark.parametrize("breaks", ["orig", "elastic"])
@pytest.mark.parametrize("run", [1, 2, 3, 4])
@pytest.mark.parametrize("how", [{"graph": True}, {"graph": False}, {"refit_each": True}])
def test_chains_between_dabs_that_are_not_fused(sg, breaks, run, how):
    """Chains of 1 to 4 dabs before each Grab from the original coordinates or elastic deform,
    whose search takes in the chain's results and counters."""
    co, tris = sg.noisy_icosphere(5, seed=4, amplitude=0.02)
    dabs = _path(sg, 15, 2, np.full(15, 0.25), (1, 2, 4, 5), (3, 6))
    other = {"orig": dict(tool=5, flag=sg.DAB_ORIGINAL),
             "elastic": dict(tool=sg.TOOL_ELASTIC_DEFORM, elastic_type=sg.ELASTIC_GRAB)}[breaks]
    for i in range(run, 15, run + 1):
        dabs[i] = sg.make_dab(location=dabs[i].location, radius=0.3, strength=0.5, grab_delta=(0.01, 0.02, 0), **other)
    _check(sg, co, tris, dabs, **how)
