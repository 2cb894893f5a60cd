"""GPU parity of the grid builds against the oracle: every array bit-exact.

Inputs are the seeded synthetic workloads; the oracle builds the same scene
with the same parameters on the CPU.
"""
import numpy as np
import pytest

import shinobi_amd as sa
from shinobi_amd import workloads as W

pytestmark = pytest.mark.gpu


def _gpu_build(ctx, soa9, kind, **kw):
    scene = sa.FaceSoup(ctx, soa9)
    B = sa.FastTwoLevelGridBuilder if kind == 1 else sa.FastSimpleGridBuilder
    b = B(ctx, keep_debug=1, **kw)
    b.init(scene)
    g = b.build()
    return scene, g


def _assert_same_params(info, og):
    assert info.status == 0
    assert tuple(info.res) == tuple(og.res)
    np.testing.assert_array_equal(info.bmin, og.bmin)
    np.testing.assert_array_equal(info.bmax, og.bmax)
    np.testing.assert_array_equal(info.cell_size, og.cs)
    np.testing.assert_array_equal(info.build_rcp, og.rcp_build)
    np.testing.assert_array_equal(info.cell_size_rcp, og.cell_rcp)
    assert (info.C1, info.P1, info.P1_valid) == (og.C1, og.P1, og.P1_valid)


def _assert_top_level(g, og):
    np.testing.assert_array_equal(g.download("tri_counts"), og.tri_counts)
    np.testing.assert_array_equal(g.download("top_keys"), og.top_keys)
    np.testing.assert_array_equal(g.download("top_vals"), og.top_vals)
    np.testing.assert_array_equal(g.download("top_ranges"), og.top_ranges)


def _assert_leaf_level(g, og):
    info = g.info()
    assert (info.C2, info.P2, info.P2_valid) == (og.C2, og.P2, og.P2_valid)
    np.testing.assert_array_equal(g.download("leaf_counts"), og.leaf_counts)
    np.testing.assert_array_equal(g.download("top_cells"), og.top_cells)
    np.testing.assert_array_equal(g.download("pair_counts"), og.pair_counts)
    np.testing.assert_array_equal(g.download("leaf_keys"), og.leaf_keys)
    np.testing.assert_array_equal(g.download("leaf_vals"), og.leaf_vals)
    np.testing.assert_array_equal(g.download("leaves"), og.leaves)
    np.testing.assert_array_equal(g.download("indices"), og.indices)


def test_uniform_soup10k_bit_exact(ctx, oracle):
    w = W.soup10k()
    og = oracle.build_uniform(w.scene, **w.oracle)
    assert og.status == 0
    _, g = _gpu_build(ctx, w.scene, 0, **w.build)
    _assert_same_params(g.info(), og)
    _assert_top_level(g, og)
    np.testing.assert_array_equal(g.download("indices"), og.indices)


@pytest.mark.parametrize("grid", [64, 256])
def test_twolevel_heightfield_small_bit_exact(ctx, oracle, grid):
    w = W.heightfield2m(grid=grid, res_x=64, res_y=32)
    og = oracle.build_twolevel(w.scene, **w.oracle)
    assert og.status == 0
    _, g = _gpu_build(ctx, w.scene, 1, **w.build)
    _assert_same_params(g.info(), og)
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)


def test_twolevel_heightfield2m_bit_exact(ctx, oracle):
    w = W.heightfield2m(res_x=64, res_y=32)
    assert w.scene.shape[1] == 2_093_058
    og = oracle.build_twolevel(w.scene, **w.oracle)
    assert og.status == 0
    _, g = _gpu_build(ctx, w.scene, 1, **w.build)
    _assert_same_params(g.info(), og)
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)


def test_twolevel_cluster_bit_exact(ctx, oracle):
    """the cluster's dense top cell is a leaf tile too large for LDS: its
    pairs take the parallel emission and the global leaf sort, in the build
    and in every rebuild"""
    w = W.cluster(n_small=60_000, n_large=400, res_x=32, res_y=32)
    og = oracle.build_twolevel(w.scene, **w.oracle)
    _, g = _gpu_build(ctx, w.scene, 1, **w.build)
    info = g.info()
    assert info.status == og.status
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)
    g.rebuild()
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)


def test_twolevel_cluster_full_size_bit_exact(ctx, oracle):
    """the dense-cluster configuration at full size (500,000 tiny triangles
    in a sphere of radius 0.02 plus 2,000 large ones in [0, 10]^3): every
    top- and leaf-level array equals the oracle's, after the build and after
    a rebuild"""
    w = W.cluster(res_x=16, res_y=16)
    assert w.scene.shape[1] == 502_000
    og = oracle.build_twolevel(w.scene, **w.oracle)
    assert og.status == 0
    _, g = _gpu_build(ctx, w.scene, 1, **w.build)
    _assert_same_params(g.info(), og)
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)
    g.rebuild()
    _assert_same_params(g.info(), og)
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)


def test_rebuild_into_an_oversize_tile(ctx, oracle):
    """a grid built without oversize leaf tiles and rebuilt after 5,000 of its
    triangles moved into one top cell: the one-block emission of such tiles
    (used until a build of the grid has met one) gives the oracle's grid"""
    a = sa.gen_soup(71, 20_000, 0.01)
    b = a.copy()
    k = 5_000
    c = np.float32(0.301)
    for j in range(3):   # shrink triangles 0..k-1 around (0.301, 0.301, 0.301)
        b[3 * j:3 * j + 3, :k] = c + (a[3 * j:3 * j + 3, :k] - np.float32(0.5)) * np.float32(0.004)
    scene, g = _gpu_build(ctx, a, 1, lam=5.0, lambda_leaf=2.0)
    res = tuple(g.info().res)
    scene.upload_vertices(b)
    g.rebuild()
    og = oracle.build_twolevel(b, lam=5.0, top_divisor=6, lambda_leaf=2.0, res_override=res)
    info = g.info()
    assert info.status == og.status == 0
    assert tuple(info.res) == tuple(og.res)
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)
    # the traversal reads the reference records the block wrote for the
    # oversize tile: rays through the dense cell hit what the oracle hits
    rays = sa.gen_random_rays(72, 30_000, 0.28, 0.32)
    pg, tg = g.trace_host(rays)
    po, to = og.trace(rays)
    assert (po != sa.MISS).sum() > 1000
    np.testing.assert_array_equal(pg, po)
    np.testing.assert_array_equal(tg.view(np.uint32), to.view(np.uint32))


def _dense_cell_with_wide_boxes(n_small):
    """n_small tiny triangles in a sphere of radius 0.02 (one finely divided
    top cell) and 300 large ones, ten of which cross it: seven at random
    angles, one on a coordinate plane, one collinear, one almost a point"""
    a = sa.gen_cluster(11, n_small, 300)
    rng = np.random.default_rng(12)
    big = (0.5 + rng.uniform(-0.4, 0.4, (7, 3, 3))).astype(np.float32)
    big[:, 0] = 1.5 - big[:, 1] / 2 - big[:, 2] / 2 - 0.5   # around the cell
    flat = [[0.2, 0.2, 0.5], [0.9, 0.3, 0.5], [0.4, 0.8, 0.5]]
    line = [[0.25, 0.25, 0.25], [0.5, 0.5, 0.5], [0.75, 0.75, 0.75]]
    dot = [[0.5, 0.5, 0.5], [0.5, 0.5, 0.5000001], [0.5, 0.5000001, 0.5]]
    for k, t in enumerate(list(big) + [flat, line, dot]):
        a[:, n_small + 5 + k] = np.asarray(t, np.float32).reshape(9)
    return a


@pytest.mark.parametrize("n_small", [3_000, 30_000, 200_000])
def test_wide_leaf_boxes_bit_exact(ctx, oracle, n_small):
    """large triangles across a finely divided top cell: leaf boxes below and
    far above the size from which a block visits a box together"""
    a = _dense_cell_with_wide_boxes(n_small)
    kw = dict(lam=5.0, top_divisor=6, lambda_leaf=2.0, leaf_min_refs=16)
    og = oracle.build_twolevel(a, **kw)
    assert og.status == 0
    assert og.pair_counts.max() > n_small // 25
    _, g = _gpu_build(ctx, a, 1, **kw)
    for _ in range(2):
        _assert_same_params(g.info(), og)
        _assert_top_level(g, og)
        _assert_leaf_level(g, og)
        g.rebuild()


def _dense_cells_under_large_triangles(n_cells, n_small, n_large):
    """n_cells groups of n_small tiny triangles, each within a cell of a 21^3
    lattice of the unit cube and crossed by n_large tilted triangles"""
    r = np.random.default_rng(7)
    m = 21
    k = r.permutation(m ** 3)[:n_cells]
    o = (np.stack([k % m, (k // m) % m, k // m // m], 1) + 0.1) / m
    n = n_cells * n_small
    small = (np.repeat(o, n_small, 0) + r.random((n, 3)) * 0.8 / m)[None] + (r.random((3, n, 3)) - 0.5) * 0.02 / m
    q = r.random((3, n_cells * n_large, 3)) * 0.1 + np.array([[0, 0, 0], [.81, .18, .81], [.09, .81, .72]])[:, None]
    large = np.repeat(o, n_large, 0)[None] + q * 0.8 / m
    ends = np.array([[[0, 0, 0], [1, 1, 1]], [[.001, 0, 0], [.999, 1, 1]], [[0, .001, 0], [1, .999, 1]]])
    v = np.concatenate([small, large, ends], 1)
    return np.ascontiguousarray(v.transpose(0, 2, 1).reshape(9, -1), dtype=np.float32)


@pytest.mark.parametrize("n_cells,n_small,n_large", [(60, 2_000, 5), (230, 2_000, 6)])
def test_many_wide_leaf_boxes_bit_exact(ctx, oracle, n_cells, n_small, n_large):
    """more wide boxes than blocks count them, and more than are counted by
    blocks (1,024); the tiles are not oversize, so one launch counts and scans"""
    a = _dense_cells_under_large_triangles(n_cells, n_small, n_large)
    kw = dict(lam=5.0, top_divisor=6, lambda_leaf=2.0, res_override=(21, 21, 21))
    og = oracle.build_twolevel(a, **kw)
    assert og.status == 0 and (og.pair_counts >= 1024).sum() > (1_024 if n_cells > 200 else 128)
    _, g = _gpu_build(ctx, a, 1, **kw)
    for _ in range(3):
        _assert_top_level(g, og)
        _assert_leaf_level(g, og)
        g.rebuild()


@pytest.mark.parametrize("n_small", [3_000, 30_000])
def test_rebuild_into_wide_leaf_boxes(ctx, oracle, n_small):
    """the same meshes met first by a rebuild: the grid is built while the
    small triangles are spread over the scene, so one block emits and sorts
    the dense cell's tile"""
    b = _dense_cell_with_wide_boxes(n_small)
    a = b.copy()
    rng = np.random.default_rng(13)
    a[:, :n_small] += np.tile(rng.uniform(0, 9, (3, n_small)), (3, 1)).astype(np.float32)
    scene, g = _gpu_build(ctx, a, 1, lam=5.0, lambda_leaf=2.0, capacity_slack=4.0)
    res = tuple(g.info().res)
    scene.upload_vertices(b)
    g.rebuild()
    og = oracle.build_twolevel(b, lam=5.0, top_divisor=6, lambda_leaf=2.0, res_override=res)
    info = g.info()
    assert info.status == og.status == 0
    assert og.pair_counts.max() >= (1024 if n_small > 10_000 else 64)
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)


def _clumps(n_clump, spread):
    """20,000 small triangles, n_clump of them moved into one top cell:
    spread 0 puts them all on one place (every leaf list as long as the
    clump), otherwise over spread times the cell"""
    a = sa.gen_soup(71, 20_000, 0.01)
    at = np.float32(0.301)
    for j in range(3):
        own = a[3 * j:3 * j + 3, :n_clump].copy()
        if spread == 0.0:
            own = np.repeat(own[:, :1], n_clump, axis=1)
        a[3 * j:3 * j + 3, :n_clump] = at + (own - np.float32(0.5)) * np.float32(max(spread, 0.004))
    return a


@pytest.mark.parametrize("keep", [0, 1])
@pytest.mark.parametrize("case", [
    ("clump", 400, 0.05), ("clump", 2_000, 0.05), ("clump", 2_200, 0.05), ("clump", 11_200, 0.05),
    ("clump", 11_600, 0.05), ("clump", 190, 0.0), ("clump", 200, 0.0), ("clump", 1_700, 0.0), ("clump", 9_000, 0.0),
    ("sphere", 30_000, 0.0), ("sphere", 200_000, 0.0), ("coarse", 4_000, 0.0)], ids=lambda c: f"{c[0]}{c[1]}-{c[2]}")
def test_leaf_tile_forms_bit_exact(ctx, oracle, case, keep):
    """leaf tiles at the edges of the emission's forms: more top pairs than a
    small and than a sliced tile holds, lists on both sides of the length from
    which a wave sorts them, boxes of more than 32 cells (large triangles over
    a finely divided cell), tiles in several slices"""
    name, n, spread = case
    kw = dict(lam=5.0, top_divisor=6, lambda_leaf=2.0)
    if name == "clump":
        a = _clumps(n, spread)
    elif name == "sphere":
        a = W.sphere_mesh(n)
    else:   # few large triangles over a grid of few, finely divided top cells
        a = sa.gen_soup(73, n, 0.3)
        kw = dict(res_override=(2, 2, 3), lambda_leaf=4.0)
    og = oracle.build_twolevel(a, **kw)
    assert og.status == 0
    scene = sa.FaceSoup(ctx, a)
    b = sa.FastTwoLevelGridBuilder(ctx, keep_debug=keep, **kw)
    b.init(scene)
    g = b.build()
    rays = sa.gen_random_rays(72, 20_000, 0.0, 1.0)
    po, to = og.trace(rays)
    for _ in range(2):
        info = g.info()
        assert info.status == 0
        assert (info.C2, info.P2, info.P2_valid) == (og.C2, og.P2, og.P2_valid)
        names = ["top_keys", "top_vals", "top_cells", "leaf_vals", "leaves", "indices"]
        for k in names + (["leaf_keys", "pair_counts"] if keep else []):
            np.testing.assert_array_equal(g.download(k), getattr(og, k), err_msg=k)
        pg, tg = g.trace_host(rays)   # reads the reference records
        np.testing.assert_array_equal(pg, po)
        np.testing.assert_array_equal(tg.view(np.uint32), to.view(np.uint32))
        g.rebuild()


def _plates(n):
    """triangles without extent along z, across many leaf cells of a plane"""
    a = sa.gen_soup(74, n, 0.3)
    a[5], a[8] = a[2], a[2]
    a[2, :2], a[5, :2], a[8, :2] = [0.0, 1.0], [0.0, 1.0], [0.0, 1.0]
    return a


@pytest.mark.parametrize("keep", [0, 1])
@pytest.mark.parametrize("case", [
    ("soup", 20_000, 0.06, 2.0), ("soup", 60_000, 0.04, 2.0),       # stored boxes, tiles of several chunks
    ("soup", 20_000, 0.01, 30.0), ("soup", 20_000, 0.01, 64.0),     # tiles of several windows of leaf cells
    ("soup", 20_000, 0.03, 20.0),                                   # both
    ("cells", 60, 200, 3), ("cells", 40, 600, 3),                   # boxes below and above those a wave visits
    ("plates", 1_500, 0.0, 6.0),                                    # boxes without a plane test
    ("one", 600, 0.9, 1.5), ("one", 1_400, 0.9, 1.5),               # more stored boxes than the pool's part holds
], ids=lambda c: "-".join(str(x) for x in c))
def test_stored_boxes_windows_and_chunks_bit_exact(ctx, oracle, case, keep):
    """boxes of 33 to 1,023 leaf cells, stored by the count and listed from
    there, and tiles beyond one window of leaf cells or one chunk of pairs"""
    name, n, x, y = case
    kw = dict(lam=5.0, top_divisor=6, lambda_leaf=float(y))
    if name == "soup":
        a = sa.gen_soup(75, n, x)
    elif name == "cells":
        a = _dense_cells_under_large_triangles(n, x, y)
        kw = dict(lam=5.0, lambda_leaf=2.0, res_override=(21, 21, 21))
    elif name == "plates":
        a = _plates(n)
        kw = dict(lambda_leaf=y, res_override=(3, 3, 2))
    else:
        a = sa.gen_soup(76, n, x)
        kw = dict(lambda_leaf=y, res_override=(1, 1, 1))
    og = oracle.build_twolevel(a, **kw)
    assert og.status == 0
    if x != 0.01:
        assert ((og.pair_counts > 32) & (og.pair_counts < 1024)).sum() > 100
    scene = sa.FaceSoup(ctx, a)
    b = sa.FastTwoLevelGridBuilder(ctx, keep_debug=keep, **kw)
    b.init(scene)
    g = b.build()
    rays = sa.gen_random_rays(72, 20_000, 0.0, 1.0)
    po, to = og.trace(rays)
    for _ in range(2):
        assert g.info().status == 0
        for k in ("top_cells", "leaves", "leaf_vals", "indices") + (("leaf_keys", "pair_counts") if keep else ()):
            np.testing.assert_array_equal(g.download(k), getattr(og, k))
        pg, tg = g.trace_host(rays)
        np.testing.assert_array_equal(pg, po)
        np.testing.assert_array_equal(tg.view(np.uint32), to.view(np.uint32))
        g.rebuild()


def test_twolevel_reference_leaf_lambda(ctx, oracle):
    """lambda_leaf = 1.2 (TwoLevelBuildKernels.h:49) on the 10k soup"""
    w = W.soup10k()
    og = oracle.build_twolevel(w.scene, lam=5.0, top_divisor=6, lambda_leaf=1.2, leaf_min_refs=16)
    _, g = _gpu_build(ctx, w.scene, 1, lam=5.0, top_divisor=6, lambda_leaf=1.2, leaf_min_refs=16)
    _assert_same_params(g.info(), og)
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)


@pytest.mark.parametrize("radix_bits", [4, 6, 8])
def test_radix_width_does_not_change_the_grid(ctx, oracle, radix_bits):
    w = W.heightfield2m(grid=200, res_x=8, res_y=8)
    og = oracle.build_twolevel(w.scene, **w.oracle)
    _, g = _gpu_build(ctx, w.scene, 1, radix_bits=radix_bits, **w.build)
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)


def test_build_is_deterministic_and_rebuild_matches(ctx, oracle):
    w = W.heightfield2m(grid=300, res_x=8, res_y=8)
    scene, g = _gpu_build(ctx, w.scene, 1, **w.build)
    first = {k: g.download(k) for k in ("top_keys", "top_vals", "leaf_keys", "leaf_vals", "leaves", "top_cells")}
    g.rebuild()
    for k, v in first.items():
        np.testing.assert_array_equal(g.download(k), v)
    # move the vertices (same topology); rebuild keeps the resolution
    res = g.info().res
    moved = w.scene.copy()
    moved[2] *= np.float32(1.1)
    moved[5] *= np.float32(1.1)
    moved[8] *= np.float32(1.1)
    scene.upload_vertices(moved)
    g.rebuild()
    og = oracle.build_twolevel(moved, res_override=res, **w.oracle)
    info = g.info()
    assert info.status == 0 and tuple(info.res) == tuple(og.res)
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)


def test_edge_scenes(ctx, oracle):
    # one triangle
    one = np.array([[0.], [0.], [0.], [1.], [0.], [0.2], [0.], [1.], [0.5]], np.float32)
    for kind in (0, 1):
        og = (oracle.build_twolevel if kind else oracle.build_uniform)(one, lam=5.0, top_divisor=6 if kind else 1)
        _, g = _gpu_build(ctx, one, kind, lam=5.0)
        _assert_top_level(g, og)
        if kind:
            _assert_leaf_level(g, og)
    # degenerate (zero-area) triangles mixed in: plane test rejects them when they span cells
    w = sa.gen_soup(7, 3000, 0.05)
    w[3:6, ::7] = w[0:3, ::7]
    w[6:9, ::7] = w[0:3, ::7] + np.float32(0.2)
    og = oracle.build_twolevel(w, lam=5.0, top_divisor=6, lambda_leaf=2.0)
    _, g = _gpu_build(ctx, w, 1, lam=5.0, lambda_leaf=2.0)
    _assert_top_level(g, og)
    _assert_leaf_level(g, og)


def test_invalid_scenes_are_reported(ctx):
    flat = sa.gen_soup(3, 100, 0.01)
    flat[[2, 5, 8]] = 0.25      # zero extent in z
    scene = sa.FaceSoup(ctx, flat)
    b = sa.FastSimpleGridBuilder(ctx)
    b.init(scene)
    with pytest.raises(sa.ShinobiError) as e:
        b.build()
    assert e.value.status == 2


def test_rebuild_many_graph_matches_oracle(ctx, oracle):
    """sg_rebuild_many over six grids of both kinds, captured into a graph
    (concurrent branches) and replayed: after every replay each grid equals
    the oracle's build of its moved vertices at the grid's resolution, and
    the traversal after the join reads the rebuilt grids"""
    specs = [(0, 3_000, 81), (1, 40_000, 82), (0, 12_000, 83), (1, 2_000, 84), (1, 25_000, 85), (0, 80_000, 86)]
    items = []
    for kind, n, seed in specs:
        a = sa.gen_soup(seed, n, 0.01)
        kw = dict(lam=5.0, lambda_leaf=2.0) if kind else dict(lam=3.0)
        scene, g = _gpu_build(ctx, a, kind, **kw)
        moved = a.copy()
        for j in (2, 5, 8):
            moved[j] *= np.float32(1.1)
        items.append((kind, kw, scene, g, a, moved, tuple(g.info().res)))
    for kind, kw, scene, g, a, moved, res in items:
        scene.upload_vertices(moved)
    rays = sa.gen_random_rays(87, 20_000, 0.0, 1.0)
    rb = sa.RayBatch(ctx, rays)
    outs = [(sa.DeviceBuffer(ctx, 4 * rb.n), sa.DeviceBuffer(ctx, 4 * rb.n)) for _ in items]
    batch = sa.Batch(ctx, len(items))
    for it, (p, t) in zip(items, outs):
        batch.add(it[3], rb, p, t)
    batch.commit()
    ctx.sync()
    with sa.Graph.capture(ctx) as graph:
        batch.rebuild(branches=4)
        batch.launch()
    expect = []
    for kind, kw, scene, g, a, moved, res in items:
        if kind:
            og = oracle.build_twolevel(moved, top_divisor=6, res_override=res, **kw)
        else:
            og = oracle.build_uniform(moved, top_divisor=1, res_override=res, **kw)
        assert og.status == 0
        expect.append(og)
    for rep in range(2):
        # eager work between replays: grid 1 rebuilt from the original
        # vertices, the outputs poisoned
        items[1][2].upload_vertices(items[1][4])
        items[1][3].rebuild()
        items[1][2].upload_vertices(items[1][5])
        for p, _ in outs:
            p.upload(np.full(rb.n, 7, np.uint32))
        graph.launch()
        ctx.sync()
        for (kind, kw, scene, g, a, moved, res), og, (p, t) in zip(items, expect, outs):
            assert g.info().status == 0 and tuple(g.info().res) == res
            _assert_top_level(g, og)
            if kind:
                _assert_leaf_level(g, og)
            else:
                np.testing.assert_array_equal(g.download("indices"), og.indices)
            po, to = og.trace(rays)
            np.testing.assert_array_equal(p.download(np.uint32, rb.n), po, err_msg=f"replay {rep}")
            np.testing.assert_array_equal(t.download(np.float32, rb.n).view(np.uint32), to.view(np.uint32))
    graph.close()
    # sg_rebuild_many itself, eager, on 1 and on 4 branches (the original
    # vertices back in between): every grid again equals the oracle's
    for branches in (1, 4):
        for it in items:
            it[2].upload_vertices(it[4])
        sa.rebuild_many(ctx, [it[3] for it in items], branches=2)
        for it in items:
            it[2].upload_vertices(it[5])
        sa.rebuild_many(ctx, [it[3] for it in items], branches=branches)
        ctx.sync()
        for (kind, kw, scene, g, a, moved, res), og in zip(items, expect):
            _assert_top_level(g, og)
            if kind:
                _assert_leaf_level(g, og)
            else:
                np.testing.assert_array_equal(g.download("indices"), og.indices)
    # the argument checks
    sa.rebuild_many(ctx, [], branches=4)
    with pytest.raises(sa.ShinobiError):
        sa.rebuild_many(ctx, [items[0][3], items[0][3]])
    with pytest.raises(sa.ShinobiError):
        sa.rebuild_many(ctx, [items[0][3]], branches=17)
    ctx.sync()
    # a grid rebuilt from another scene (same triangle count) after the
    # commit: the batch refuses to rebuild until it is committed again, a
    # cleared batch rebuilds nothing, and after the new commit the grid is
    # rebuilt from the new scene
    kind, kw, scene, g, a, moved, res = items[0]
    assert kind == 0
    other = sa.gen_soup(91, a.shape[1], 0.01)
    oscene = sa.FaceSoup(ctx, other)
    sa.check(ctx._l.sg_rebuild(ctx.h, oscene.h, g.h, ctx.stream), "sg_rebuild")
    with pytest.raises(sa.ShinobiError):
        batch.rebuild(branches=4)
    batch.clear()
    batch.rebuild(branches=4)
    # a cleared batch launches nothing: the outputs keep what they hold
    outs[0][0].upload(np.full(rb.n, 5, np.uint32))
    batch.launch()
    ctx.sync()
    assert (outs[0][0].download(np.uint32, rb.n) == 5).all()
    for it, (p, t) in zip(items, outs):
        batch.add(it[3], rb, p, t)
    batch.commit()
    oscene.upload_vertices(other * np.float32(0.9))
    batch.rebuild(branches=4)
    ctx.sync()
    og = oracle.build_uniform(other * np.float32(0.9), top_divisor=1, res_override=res, **kw)
    assert og.status == 0
    _assert_top_level(g, og)
    np.testing.assert_array_equal(g.download("indices"), og.indices)
    batch.clear()


@pytest.mark.parametrize("n,size", [
    (1, 0.1), (255, 0.05), (256, 0.05), (257, 0.05),
    (1_000, 0.4),                                  # more pairs in a tile than it stages
    (2**19 - 1, 0.002), (2**19, 0.002), (2**19 + 1, 0.002)])   # one triangle or four per thread
def test_top_emission_forms_at_their_edges(ctx, oracle, n, size):
    a = sa.gen_soup(91, n, size)
    og = oracle.build_uniform(a, lam=5.0, top_divisor=1)
    assert og.status == 0
    _, g = _gpu_build(ctx, a, 0, lam=5.0)
    _assert_same_params(g.info(), og)
    _assert_top_level(g, og)
    g.rebuild()
    _assert_top_level(g, og)


def _bar(n, seed, axis, thin, pile):
    """n small triangles in the unit cube, the two other axes scaled by thin,
    the first `pile` of them crowded into the lower half of the axis"""
    r = np.random.default_rng(seed)
    c = r.random((3, n)).astype(np.float32)
    c[axis, : int(pile * n)] *= np.float32(0.45)
    v = np.clip(c[None] + (r.random((3, 3, n)) - 0.5).astype(np.float32) * np.float32(0.01), 0, 1).astype(np.float32)
    v *= np.array([1.0 if k == axis else thin for k in range(3)], np.float32)[:, None]
    v[0, :, 0], v[0, axis, 1] = 0.0, 1.0
    return np.ascontiguousarray(v.reshape(9, n), dtype=np.float32)


@pytest.mark.parametrize("first", ["build", "rebuild"])
@pytest.mark.parametrize("n,axis,thin,lam,cells,pile", [
    (2060, 0, 1 / 64, 2.0, 1, 0.0),      # 256 leaf cells along the axis: the packed byte is 0
    (2060, 2, 1 / 64, 3.0, 1, 0.0),      # 293: the byte is 37
    (8000, 1, 1 / 256, 2.0, 3, 0.0),     # three top cells of more pairs than a small leaf tile holds
    (900, 2, 1 / 256, 10.0, 3, 0.0),     # two top cells in a tile, one in the next
    (300, 0, 1 / 256, 30.0, 3, 0.0),     # tiles of the small kernel
    (12000, 1, 1 / 64, 2.0, 2, 0.95),    # rebuilt: an oversize tile that the grid's build did not meet
])
def test_leaf_ranges_beyond_the_packed_resolutions(ctx, oracle, n, axis, thin, lam, cells, pile, first):
    """a grid flagged for leaf resolutions beyond 255, built or reached by a
    rebuild: the reserved leaf cells that no tile writes are empty"""
    res = tuple(cells if k == axis else 1 for k in range(3))
    opt = dict(lam=5.0, top_divisor=1, lambda_leaf=lam, leaf_min_refs=16, res_override=res)
    bar = _bar(n, 5, axis, thin, pile)
    og = oracle.build_twolevel(bar, **opt)
    assert og.status != 0
    scene = sa.FaceSoup(ctx, bar if first == "build" else _bar(n, 6, axis, 1.0, 0.0))
    b = sa.FastTwoLevelGridBuilder(ctx, **opt)
    b.init(scene)
    g = b.build()
    if first == "rebuild":
        assert g.info().status == 0
        scene.upload_vertices(bar)
        g.rebuild()
    info = g.info()
    assert info.status != 0 and (info.C2, info.P2, info.P2_valid) == (og.C2, og.P2, og.P2_valid)
    np.testing.assert_array_equal(g.download("top_cells"), og.top_cells)
    np.testing.assert_array_equal(g.download("leaves"), og.leaves)
    np.testing.assert_array_equal(g.download("indices"), og.indices)
    rays = sa.gen_random_rays(98, 20_000, -0.1, 1.1)
    for k in range(3):
        if k != axis:
            rays[[k, 3 + k]] *= np.float32(thin)
    for shadow in (False, True):
        if shadow:
            rays[6] = 1.0
        pg, tg = g.trace_host(rays, shadow=shadow)
        po, to = og.trace(rays, shadow=shadow)[:2]
        np.testing.assert_array_equal(pg, po)
        np.testing.assert_array_equal(tg.view(np.uint32), to.view(np.uint32))


def test_cell_words_only_where_they_are_read(ctx, oracle):
    """a uniform grid of 2^17 cells holds cell words (half a byte a cell), a
    smaller one does not; both trace as the oracle"""
    v = np.array([[0, 0, 0], [0.01, 0, 0.01], [0, 0.01, 0.01]], np.float32)
    soa = np.ascontiguousarray(np.stack([v, 1 - v], 2).reshape(9, 2))
    rays = sa.gen_random_rays(99, 4000, 0.0, 0.02)
    size = []
    for rz in (31, 32):
        kw = dict(lam=5.0, res_override=(64, 64, rz))
        scene, g = _gpu_build(ctx, soa, 0, **kw)
        size.append(g.info().device_bytes)
        po, to = oracle.build_uniform(soa, **kw).trace(rays)[:2]
        pg, tg = g.trace_host(rays)
        np.testing.assert_array_equal(pg, po)
        np.testing.assert_array_equal(tg.view(np.uint32), to.view(np.uint32))
    ranges, words = 64 * 64 * 8, 64 * 64 * 32 // 2
    assert abs(size[1] - size[0] - ranges - words) <= 2048
