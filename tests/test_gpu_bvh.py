"""GPU BVH build / refit / skinning parity: node bytes, Morton order and
triangle arrays identical to the oracle's build of the same scene."""
import numpy as np
import pytest

from srt_amd import scenes
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


def _soup(n, seed, spread=10.0, size=0.5):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-spread, spread, size=(n, 3))
    v = (c[:, None, :] + rng.normal(scale=size, size=(n, 3, 3))).reshape(-1, 3).astype(np.float32)
    idx = np.arange(3 * n, dtype=np.uint32).reshape(n, 3)
    mats = np.asarray([scenes.material()], scenes.MAT_DTYPE)
    return scenes.SceneData(positions=v, indices=idx, mesh_first=np.array([0, n], np.int32),
                            mesh_material=np.array([0], np.int32), materials=mats)


def _compare(ctx, s, max_leaf=4, cluster_size=0):
    h = ctx.upload(s)
    ctx.build_bvh(h, max_leaf=max_leaf, cluster_size=cluster_size)
    nodes, order, tris, info = ctx.bvh_download(h)
    ob = O.Bvh(O.Scene(s), max_leaf=max_leaf, cluster_size=cluster_size)
    n2, o2, t2, _ = ob.arrays()
    oi = ob.info()
    ctx.release(h)
    assert info["root"] == oi["root"]
    assert info["max_depth"] == oi["max_depth"]
    assert info["clusters"] == oi["clusters"]
    np.testing.assert_array_equal(order, o2)
    assert np.array_equal(tris.view(np.uint32), t2.view(np.uint32))
    assert nodes.shape == n2.shape
    bad = np.nonzero((nodes != n2).any(axis=1))[0]
    assert bad.size == 0, f"{bad.size} nodes differ, first {bad[:5]}"
    return info


@pytest.mark.parametrize("n", [1, 2, 3, 7, 64, 65, 1000])
def test_small_soups(ctx, n):
    _compare(ctx, _soup(n, seed=n))


@pytest.mark.parametrize("n", [255, 257, 4096, 4097, 4098, 8193, 12290])
def test_pieces_of_the_level_order(ctx, n):
    """Radix trees and binary trees whose node counts lie around a multiple of
    the level order's pieces (4096 nodes, 256 threads): the tree equals the
    oracle's, and the closest hits found through its 4-wide form equal those of
    the oracle's tree."""
    s = _soup(n, seed=n)
    _compare(ctx, s)
    rng = np.random.default_rng(n)
    h = ctx.upload(s)
    ctx.build_bvh(h)
    o = rng.uniform(-12, 12, size=(512, 3))
    d = rng.normal(size=(512, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    got = ctx.trace(h, o, d)
    ctx.release(h)
    osc = O.Scene(s)
    want = O.trace(osc, o, d, bvh=O.Bvh(osc))
    assert np.array_equal(got[3], want[3])
    assert np.array_equal(got[0], want[0])


@pytest.mark.parametrize("cluster", [8, 16, 100])
def test_top_level_sah(ctx, cluster):
    info = _compare(ctx, _soup(5000, seed=9), cluster_size=cluster)
    assert info["clusters"] > 1


@pytest.mark.parametrize("leaf", [1, 2, 8])
def test_leaf_sizes(ctx, leaf):
    _compare(ctx, _soup(3000, seed=4), max_leaf=leaf, cluster_size=64)


def _points(c, size=0.01):
    """Small triangles around the given centres."""
    c = np.asarray(c, np.float64)
    v = c[:, None, :] + size * np.array([[-1, -1, 0], [1, -1, 0], [0, 2, 0]])
    n = len(c)
    return scenes.SceneData(positions=v.reshape(-1, 3).astype(np.float32),
                            indices=np.arange(3 * n, dtype=np.uint32).reshape(n, 3),
                            mesh_first=np.array([0, n], np.int32), mesh_material=np.array([0], np.int32),
                            materials=np.asarray([scenes.material()], scenes.MAT_DTYPE))


# one triangle per cluster: pairs, one wave's subtrees (21 items), nodes of one
# wave and of four (256), with and without wide levels (1024, 512 per chunk)
@pytest.mark.parametrize("n", [2, 3, 20, 21, 22, 23, 45, 255, 256, 257, 258, 1023, 1024, 1025, 1537, 2048, 2050, 9001])
def test_top_level_node_sizes(ctx, n):
    info = _compare(ctx, _soup(n, seed=100 + n), max_leaf=1, cluster_size=1)
    assert info["clusters"] == n


@pytest.mark.parametrize("n", [2, 5, 21, 22, 257, 1025, 3000])
@pytest.mark.parametrize("kind", ["one_point", "line", "two_points", "skewed"])
def test_top_level_degenerate_items(ctx, kind, n):
    """Items that no boundary separates (one centroid: halves in order), a
    single axis with an extent, many items in two places, and distances that
    shrink by a constant factor (deep, unbalanced trees)."""
    i = np.arange(n, dtype=np.float64)
    if kind == "one_point":
        c = np.zeros((n, 3))
    elif kind == "line":
        c = np.stack([0 * i, i, 0 * i], 1)
    elif kind == "two_points":
        c = np.stack([(i % 2) * 5, 0 * i, (i % 2) * -3], 1)
    else:
        c = np.stack([4.0 ** -(i % 40), np.sin(i) * 1e-3, 2.0 ** -(i % 70)], 1)
    _compare(ctx, _points(c), max_leaf=1, cluster_size=1)


def test_cluster_size_below_leaf_size_is_raised(ctx):
    info = _compare(ctx, _soup(2000, seed=11), max_leaf=8, cluster_size=2)
    assert info["cluster_size"] == 8


def test_cornell(ctx):
    _compare(ctx, scenes.cornell())


def test_rebuilds_with_kept_scratch(ctx):
    """Builds take the device scratch chunks kept by earlier builds (larger and
    smaller scenes, the same scene again): every tree equals the oracle's, and
    with keep_build_scratch 0 the chunks are freed."""
    _compare(ctx, _soup(40000, seed=21))
    _compare(ctx, _soup(3000, seed=22))
    s = _soup(20000, seed=23)
    h = ctx.upload(s)
    ctx.build_bvh(h)
    first = ctx.bvh_download(h)
    for _ in range(2):
        ctx.build_bvh(h)
        again = ctx.bvh_download(h)
        for a, b in zip(first[:3], again[:3]):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    kept = ctx.lib.srt_hbm_used(ctx.h)
    ctx.set_option("keep_build_scratch", 0)
    try:
        assert ctx.lib.srt_hbm_used(ctx.h) < kept
        ctx.build_bvh(h)
        assert ctx.lib.srt_hbm_used(ctx.h) < kept
        again = ctx.bvh_download(h)
        for a, b in zip(first[:3], again[:3]):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    finally:
        ctx.set_option("keep_build_scratch", 1)
        ctx.release(h)
    _compare(ctx, _soup(5000, seed=24), cluster_size=16)


def test_spheres_1m(ctx):
    info = _compare(ctx, scenes.spheres(), max_leaf=2)     # the library's defaults
    assert info["triangles"] == 1000008
    assert info["clusters"] > 100


def test_refit_identity_and_skin(ctx):
    s = scenes.tube()
    h = ctx.upload(s)
    ctx.build_bvh(h)
    nodes0, order0, tris0, _ = ctx.bvh_download(h)
    ctx.set_skin(h, s.skin["bone_ids"], s.skin["bone_weights"])
    ident = np.tile(np.eye(4, dtype=np.float32)[:3], (s.skin["num_bones"], 1, 1))
    ctx.skin_refit(h, ident)
    nodes1, order1, tris1, _ = ctx.bvh_download(h)
    # identity bones: weights sum to 1 in float only approximately, so compare to the oracle
    osc = O.Scene(s)
    ob = O.Bvh(osc)
    n0, _, _, _ = ob.arrays()
    assert np.array_equal(nodes0, n0)
    for frame in (0, 17, 42):
        M = s.skin["matrices"](frame)
        ctx.skin_refit(h, M)
        p, n, t = ctx.download_vertices(h, s.positions.shape[0], normals=True, tangents=True)
        p2, n2, t2 = O.skin(s.positions, s.normals, s.tangents, s.skin["bone_ids"], s.skin["bone_weights"], M)
        assert np.array_equal(p.view(np.uint32), p2.view(np.uint32))
        assert np.array_equal(n.view(np.uint32), n2.view(np.uint32))
        assert np.array_equal(t.view(np.uint32), t2.view(np.uint32))
        osc.set_vertices(p2, n2, t2)
        ob.refit()
        nodes, order, tris, _ = ctx.bvh_download(h)
        nr, orr, tr, _ = ob.arrays()
        np.testing.assert_array_equal(order, orr)
        assert np.array_equal(tris.view(np.uint32), tr.view(np.uint32))
        assert np.array_equal(nodes, nr)
    ctx.release(h)


def test_refused_rebuild_leaves_no_half_built_tree():
    """A rebuild that the memory budget refuses part-way leaves the scene with
    its old tree or with none (the next render builds the default one): over a
    sweep of budgets every later frame is one of the two trees' or SRT_E_OOM."""
    from srt_amd import abi
    s = scenes.tube()

    def session(budget, rebuild):
        c = abi.Context(0, budget)
        c.set_option("keep_build_scratch", 0)
        h = c.upload(s)
        img = None
        try:
            c.build_bvh(h, cluster_size=0 if rebuild is None else 64)
            c.render(h, s.camera, 64, 36, 1, 3, 4, 1, 1, 2)
        except abi.SrtError:
            c.close()
            return "first", None
        state, used = "built", c.hbm_used()
        if rebuild:
            try:
                c.build_bvh(h, max_leaf=1, cluster_size=1)
            except abi.SrtError as e:
                assert e.code == -4
                state = "refused"
        try:
            img = c.render(h, s.camera, 64, 36, 1, 3, 4, 1, 1, 2)
        except abi.SrtError as e:
            assert e.code == -4 and state == "refused"
        c.close()
        return state, img if budget else (img, used)

    default = session(0, None)[1][0]
    old, used = session(0, False)[1]
    states = []
    for mb in range(30, 160, 2):
        state, img = session(used + (mb << 20), True)
        states.append(state)
        if state == "refused" and img is not None:
            assert np.array_equal(img, old) or np.array_equal(img, default), mb
    assert states.count("refused") >= 5 and states[-1] == "built"
