"""GPU parity of the leafwise and levelwise growers against the CPU oracle.

Quantized trees are bit-exact (same quantized gradients); FP32 trees are bit-exact
against the oracle restating the device's fixed summation order.
"""
import numpy as np
import pytest

from oracle_lib import CHUNK_ADAPTIVE, DEVICE_CHUNK, HIST_F32_FIXED, HIST_INT, cfg as orc_cfg
from test_gpu_depthwise import assert_same_tree, ctx_for, grad_of, tall_data

pytestmark = pytest.mark.gpu

# Leafwise FP32 histograms sum over leaf-sized units (at most 256 per built node at these
# shapes); the oracle follows the same rule.
LW_F32_CHUNK = CHUNK_ADAPTIVE | 256


@pytest.fixture(scope="module")
def tall():
    return tall_data(40000, seed_cfg=2)


def wide_data(n=6000, f=300):
    from bonsai_amd import synth
    from oracle_lib import load_oracle
    orc = load_oracle()
    X, y = synth.wide_bins(n, f)
    cuts = [orc.fit_cuts(X[:, j], 255) for j in range(f)]
    bins = np.stack([orc.transform(cuts[j], X[:, j]) for j in range(f)], axis=1)
    nb = np.array([c.size for c in cuts], np.uint16)
    return bins, nb, X, y


@pytest.fixture(scope="module")
def wide():
    return wide_data()


@pytest.mark.parametrize("leaves,depth", [(2, 12), (31, 12), (63, 5), (255, 12)])
def test_grow_leafwise_int_bit_exact(hip, orc, tall, leaves, depth):
    bins, nb, X, y = tall
    g, h = grad_of(orc, y, seed=leaves)
    ctx = ctx_for(hip, bins, nb, grower="hip_leafwise", quantized=True, max_depth=depth, max_leaves=leaves)
    gq, hq, sc = ctx.set_gradients(g, h)
    nodes, lor = ctx.grow_tree()
    ref, rlor = orc.grow_leafwise(bins, nb, gq=gq, hq=hq, scales=sc,
                                  c=orc_cfg(max_depth=depth, max_leaves=leaves), mode=HIST_INT)
    assert_same_tree(nodes, ref)
    assert np.array_equal(lor, rlor)


@pytest.mark.parametrize("leaves,depth", [(31, 12), (127, 7)])
def test_grow_leafwise_f32_matches_device_order_oracle(hip, orc, tall, leaves, depth):
    bins, nb, X, y = tall
    g, h = grad_of(orc, y, seed=100 + leaves)
    ctx = ctx_for(hip, bins, nb, grower="hip_leafwise", quantized=False, max_depth=depth, max_leaves=leaves)
    ctx.set_gradients(g, h)
    nodes, lor = ctx.grow_tree()
    ref, rlor = orc.grow_leafwise(bins, nb, g=g, h=h, c=orc_cfg(max_depth=depth, max_leaves=leaves),
                                  mode=HIST_F32_FIXED, chunk=LW_F32_CHUNK)
    assert_same_tree(nodes, ref)
    assert np.array_equal(lor, rlor)


@pytest.fixture(scope="module")
def tall600k():
    return tall_data(600000, seed_cfg=3)


# Large enough that the leaf-sized work units leave their minimum sizes: the root's
# partition chunks are 768 rows, the first children's 512, and a quantized child of
# more than 262,144 rows gets histogram units above 1024 rows, with many partials.
@pytest.mark.parametrize("quantized", [True, False])
@pytest.mark.parametrize("leaves,depth", [(15, 10), (63, 12)])
def test_grow_leafwise_600k_rows(hip, orc, tall600k, quantized, leaves, depth):
    bins, nb, X, y = tall600k
    g, h = grad_of(orc, y, seed=7 + leaves)
    ctx = ctx_for(hip, bins, nb, grower="hip_leafwise", quantized=quantized, max_depth=depth, max_leaves=leaves)
    c = orc_cfg(max_depth=depth, max_leaves=leaves)
    if quantized:
        gq, hq, sc = ctx.set_gradients(g, h)
        ref, rlor = orc.grow_leafwise(bins, nb, gq=gq, hq=hq, scales=sc, c=c, mode=HIST_INT)
    else:
        ctx.set_gradients(g, h)
        ref, rlor = orc.grow_leafwise(bins, nb, g=g, h=h, c=c, mode=HIST_F32_FIXED, chunk=LW_F32_CHUNK)
    nodes, lor = ctx.grow_tree()
    ctx.close()
    assert_same_tree(nodes, ref)
    assert np.array_equal(lor, rlor)


def levelwise_view(nodes, D):
    """Perfect dense tree -> (level splits, leaf values, leaf covers)."""
    levels = np.array([[nodes[(1 << k) - 1]["feature"], nodes[(1 << k) - 1]["bin"],
                        nodes[(1 << k) - 1]["default_left"]] for k in range(D)], np.int64).reshape(D, 3)
    leaves = nodes[(1 << D) - 1:]
    return levels, leaves["value"], leaves["cover"]


def check_levelwise(hip, orc, bins, nb, g, h, depth, quantized):
    ctx = ctx_for(hip, bins, nb, grower="hip_levelwise", quantized=quantized, max_depth=depth)
    if quantized:
        gq, hq, sc = ctx.set_gradients(g, h)
    else:
        ctx.set_gradients(g, h)
    nodes, lor = ctx.grow_tree()
    if quantized:
        levels, lv, lc, gains, rlor = orc.grow_levelwise(bins, nb, gq=gq, hq=hq, scales=sc,
                                                         c=orc_cfg(max_depth=depth), mode=HIST_INT)
    else:
        levels, lv, lc, gains, rlor = orc.grow_levelwise(bins, nb, g=g, h=h, c=orc_cfg(max_depth=depth),
                                                         mode=HIST_F32_FIXED)
    D = levels.shape[0]
    assert len(nodes) == (2 << D) - 1
    dl, dv, dc = levelwise_view(nodes, D)
    assert np.array_equal(dl, levels.astype(np.int64))
    assert np.array_equal(dv.view(np.uint32), lv.view(np.uint32))
    assert np.array_equal(dc, lc)
    assert np.array_equal(lor - ((1 << D) - 1), rlor)


@pytest.mark.parametrize("depth", [1, 4, 8])
def test_grow_levelwise_int_bit_exact(hip, orc, tall, depth):
    bins, nb, X, y = tall
    g, h = grad_of(orc, y, seed=200 + depth)
    check_levelwise(hip, orc, bins, nb, g, h, depth, True)


@pytest.mark.parametrize("depth", [3, 6])
def test_grow_levelwise_f32_matches_device_order_oracle(hip, orc, tall, depth):
    bins, nb, X, y = tall
    g, h = grad_of(orc, y, seed=300 + depth)
    check_levelwise(hip, orc, bins, nb, g, h, depth, False)


@pytest.mark.parametrize("quantized", [True, False])
def test_grow_levelwise_wide_rows(hip, orc, wide, quantized):
    """300 features: rows wider than the register-resident scatter, three feature slices."""
    bins, nb, X, y = wide
    rng = np.random.default_rng(3)
    g, h = orc.mse_grad(rng.normal(0, 1, y.size).astype(np.float32), y)
    check_levelwise(hip, orc, bins, nb, g, h, 6, quantized)


@pytest.mark.parametrize("quantized", [True, False])
def test_grow_depthwise_wide_rows(hip, orc, wide, quantized):
    bins, nb, X, y = wide
    rng = np.random.default_rng(4)
    g, h = orc.mse_grad(rng.normal(0, 1, y.size).astype(np.float32), y)
    ctx = ctx_for(hip, bins, nb, quantized=quantized, max_depth=5)
    if quantized:
        gq, hq, sc = ctx.set_gradients(g, h)
        ref, rlor = orc.grow_depthwise(bins, nb, gq=gq, hq=hq, scales=sc, c=orc_cfg(max_depth=5), mode=HIST_INT)
    else:
        ctx.set_gradients(g, h)
        ref, rlor = orc.grow_depthwise(bins, nb, g=g, h=h, c=orc_cfg(max_depth=5), mode=HIST_F32_FIXED)
    nodes, lor = ctx.grow_tree()
    assert_same_tree(nodes, ref)
    assert np.array_equal(lor, rlor)


@pytest.mark.parametrize("pair", [1, 0])
def test_grow_depthwise_int_50_features(hip, orc, pair):
    """52-byte rows: paired levels with 13 dwords per row in the histogram lanes."""
    bins, nb, X, y = wide_data(n=30000, f=50)
    rng = np.random.default_rng(5)
    g, h = orc.mse_grad(rng.normal(0, 1, y.size).astype(np.float32), y)
    ctx = ctx_for(hip, bins, nb, quantized=True, max_depth=6, min_data_in_leaf=5)
    ctx.set_tuning(pair_levels=pair)
    gq, hq, sc = ctx.set_gradients(g, h)
    ref, rlor = orc.grow_depthwise(bins, nb, gq=gq, hq=hq, scales=sc, c=orc_cfg(max_depth=6, min_data=5),
                                   mode=HIST_INT)
    nodes, lor = ctx.grow_tree()
    assert_same_tree(nodes, ref)
    assert np.array_equal(lor, rlor)


@pytest.mark.parametrize("quantized", [True, False])
@pytest.mark.parametrize("f,n,depth", [(65, 1025, 3), (127, 3001, 7), (128, 9000, 6), (129, 2047, 9), (257, 900, 8)])
def test_wide_row_edges(hip, orc, f, n, depth, quantized):
    """Rows of row ids (over 64 bytes) at slice and chunk edges: feature counts around the
    histogram's slices, bin counts 2 .. 256 with and without missing cells, levels deep
    enough for nodes without rows; a levelwise tree, a depthwise tree and one on a row
    subset, all bit-exact."""
    rng = np.random.default_rng(f)
    nb = rng.choice([2, 3, 17, 64, 255, 256], f).astype(np.uint16)
    bins = np.stack([rng.integers(0, int(b) - (j & 1), n) if b > 2 else np.full(n, j & 1)
                     for j, b in enumerate(nb)], axis=1).astype(np.uint8)
    y = (bins[:, 3] > nb[3] // 3).astype(np.float32) + rng.normal(0, 0.3, n).astype(np.float32)
    g, h = orc.mse_grad(np.zeros(n, np.float32), y)
    check_levelwise(hip, orc, bins, nb, g, h, depth, quantized)
    c = orc_cfg(max_depth=depth, min_data=3)
    for rows in (np.arange(n), np.sort(rng.permutation(n)[:n // 2 + 1])):
        ctx = ctx_for(hip, bins, nb, quantized=quantized, max_depth=depth, min_data_in_leaf=3)
        if quantized:
            gq, hq, sc = ctx.set_gradients(g, h)
            ref, rlor = orc.grow_depthwise(bins[rows], nb, gq=gq[rows], hq=hq[rows], scales=sc, c=c, mode=HIST_INT)
        else:
            ctx.set_gradients(g, h)
            ref, rlor = orc.grow_depthwise(bins[rows], nb, g=g[rows], h=h[rows], c=c, mode=HIST_F32_FIXED,
                                           scales=(orc.fx_shift(g), orc.fx_shift(h)))
        if rows.size < n:
            ctx.set_row_subset(rows.astype(np.uint32))
        nodes, lor = ctx.grow_tree()
        ctx.close()
        assert_same_tree(nodes, ref)
        assert np.array_equal(lor[rows], rlor)


@pytest.mark.parametrize("quantized", [True, False])
@pytest.mark.parametrize("f,top", [(65, 256), (66, 17), (100, 255), (257, 64), (513, 3)])
def test_wide_histogram_of_row_lists(hip, orc, f, top, quantized):
    """Row lists of one to several histogram units over more than 64 features: slices are
    narrowed by the units there are, cells bit for bit."""
    rng = np.random.default_rng(f)
    n = 40_000
    nb = rng.integers(1, top + 1, f).astype(np.uint16)
    nb[f // 2] = top
    bins = (rng.random((n, f)) * nb).astype(np.uint8)
    g, h = orc.mse_grad(np.zeros(n, np.float32), rng.normal(0, 1, n).astype(np.float32))
    ctx = ctx_for(hip, bins, nb, quantized=quantized, max_depth=3)
    gq, hq, _ = ctx.set_gradients(g, h)
    for m in (1, 100, 8_193, 40_000):
        rows = np.sort(rng.permutation(n)[:m]).astype(np.uint32)
        got = ctx.histogram(rows)
        if quantized:
            assert np.array_equal(got.ravel(), np.asarray(orc.hist_int(bins, rows, gq, hq, top)).ravel())
        else:
            want = orc.hist_f32(bins, rows, g, h, top, HIST_F32_FIXED, DEVICE_CHUNK)
            assert np.array_equal(got.view(np.uint32).ravel(), want.view(np.uint32).ravel())
    ctx.close()


@pytest.mark.parametrize("quantized", [True, False])
@pytest.mark.parametrize("f,n", [(65, 100), (70, 8192), (131, 20_001)])
def test_wide_single_bin_histogram(hip, orc, f, n, quantized):
    """Planes of more than 64 features with one bin each: every feature's only cell holds
    the rows' sums, which a finder that skips the first features takes its totals from."""
    rng = np.random.default_rng(f)
    bins, nb = np.zeros((n, f), np.uint8), np.ones(f, np.uint16)
    g, h = orc.mse_grad(np.zeros(n, np.float32), rng.normal(0, 1, n).astype(np.float32))
    ctx = ctx_for(hip, bins, nb, quantized=quantized, max_depth=2)
    gq, hq, sc = ctx.set_gradients(g, h)
    rows = np.arange(n, dtype=np.uint32)
    got = ctx.histogram(rows)
    mask = np.zeros(f, np.uint8)
    mask[f - 1] = 1
    ctx.set_feature_mask(mask)
    nodes, _ = ctx.grow_tree()
    ctx.close()
    orc.set_feature_mask(mask)
    try:
        if quantized:
            want = orc.hist_int(bins, rows, gq, hq, 1)
            ref, _ = orc.grow_depthwise(bins, nb, gq=gq, hq=hq, scales=sc, c=orc_cfg(max_depth=2), mode=HIST_INT)
        else:
            want = orc.hist_f32(bins, rows, g, h, 1, HIST_F32_FIXED, DEVICE_CHUNK)
            ref, _ = orc.grow_depthwise(bins, nb, g=g, h=h, c=orc_cfg(max_depth=2), mode=HIST_F32_FIXED,
                                        scales=(orc.fx_shift(g), orc.fx_shift(h)))
    finally:
        orc.set_feature_mask(None)
    assert np.array_equal(got.reshape(f, 2), np.reshape(want, (f, 2)))
    assert_same_tree(nodes, ref)


@pytest.mark.parametrize("grower", ["hip_leafwise", "hip_levelwise"])
def test_train_graph_equals_eager(hip, orc, tall, grower):
    bins, nb, X, y = tall
    res = []
    for use_graph in (True, False):
        ctx = ctx_for(hip, bins, nb, grower=grower, quantized=True, max_depth=6, max_leaves=31,
                      use_graph=use_graph, learning_rate=0.1)
        ctx.upload_labels(y)
        ctx.set_scores(np.full(y.size, orc.init_score(1, y), np.float32))
        ctx.train(3)
        ctx.train(2)
        res.append((ctx.trees(), ctx.get_scores()))
        ctx.close()
    (ta, sa), (tb, sb) = res
    assert len(ta) == len(tb) == 5
    for a, b in zip(ta, tb):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    assert np.array_equal(sa.view(np.uint32), sb.view(np.uint32))


@pytest.mark.parametrize("quantized", [True, False])
@pytest.mark.parametrize("leaves", [2, 9, 10, 13])
def test_grow_leafwise_chain(hip, orc, leaves, quantized):
    """Labels that triple from group to group: every split peels one group off, so each pop
    waits for the last one's children and 13 leaves need more rounds than a tree is first
    given (6); leaf counts around one round's eight.  The tree, then a fit by graph and
    eagerly, bit-exact."""
    n, f = 6500, 3
    rng = np.random.default_rng(5)
    group = rng.integers(0, 13, n)
    bins = np.stack([group, rng.integers(0, 13, n), rng.integers(0, 13, n)], axis=1).astype(np.uint8)
    nb = np.full(f, 14, np.uint16)
    y = (3.0 ** group).astype(np.float32)
    g, h = orc.mse_grad(np.zeros(n, np.float32), y)
    kw = dict(grower="hip_leafwise", quantized=quantized, max_depth=12, max_leaves=leaves, min_data_in_leaf=1)
    c = orc_cfg(max_depth=12, max_leaves=leaves, min_data=1)
    ctx = ctx_for(hip, bins, nb, **kw)
    if quantized:
        gq, hq, sc = ctx.set_gradients(g, h)
        ref, rlor = orc.grow_leafwise(bins, nb, gq=gq, hq=hq, scales=sc, c=c, mode=HIST_INT)
    else:
        ctx.set_gradients(g, h)
        ref, rlor = orc.grow_leafwise(bins, nb, g=g, h=h, c=c, mode=HIST_F32_FIXED, chunk=LW_F32_CHUNK)
    nodes, lor = ctx.grow_tree()
    ctx.close()
    assert_same_tree(nodes, ref)
    assert np.array_equal(lor, rlor)
    fits = []
    for use_graph in (True, False):
        ctx = ctx_for(hip, bins, nb, use_graph=use_graph, learning_rate=0.5, **kw)
        ctx.upload_labels(y)
        ctx.set_scores(np.zeros(n, np.float32))
        ctx.train(3)
        fits.append((ctx.trees(), ctx.get_scores()))
        ctx.close()
    for a, b in zip(fits[0][0], fits[1][0]):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    assert np.array_equal(fits[0][1].view(np.uint32), fits[1][1].view(np.uint32))


@pytest.mark.parametrize("quantized", [True, False])
def test_grow_leafwise_wide_row_chunks(hip, orc, quantized):
    """Leaves on both sides of the wide rows' cap of 1,024 rows a chunk: the leaf-sized rule
    reaches it past 262,144 rows."""
    n, f = 300_000, 66
    rng = np.random.default_rng(66)
    bins = rng.integers(0, 32, (n, f), dtype=np.uint8)
    nb = np.full(f, 33, np.uint16)
    y = ((bins[:, 3] > 4) * 2.0 + bins[:, 7] / 16.0 + rng.normal(0, 0.3, n)).astype(np.float32)
    g, h = orc.mse_grad(np.zeros(n, np.float32), y)
    ctx = ctx_for(hip, bins, nb, grower="hip_leafwise", quantized=quantized, max_depth=6, max_leaves=12)
    c = orc_cfg(max_depth=6, max_leaves=12)
    if quantized:
        gq, hq, sc = ctx.set_gradients(g, h)
        ref, rlor = orc.grow_leafwise(bins, nb, gq=gq, hq=hq, scales=sc, c=c, mode=HIST_INT)
    else:
        ctx.set_gradients(g, h)
        ref, rlor = orc.grow_leafwise(bins, nb, g=g, h=h, c=c, mode=HIST_F32_FIXED, chunk=LW_F32_CHUNK)
    nodes, lor = ctx.grow_tree()
    ctx.close()
    assert_same_tree(nodes, ref)
    assert np.array_equal(lor, rlor)


@pytest.mark.parametrize("quantized", [True, False])
def test_grow_leafwise_wide_rows(hip, orc, quantized):
    """1,500-byte rows: partitions order row ids, in chunks of the leaf-sized rule's 256-row
    minimum at this many rows."""
    bins, nb, X, y = wide_data(n=4000, f=1500)
    rng = np.random.default_rng(6)
    g, h = orc.mse_grad(rng.normal(0, 1, y.size).astype(np.float32), y)
    ctx = ctx_for(hip, bins, nb, grower="hip_leafwise", quantized=quantized, max_depth=8, max_leaves=20,
                  min_data_in_leaf=5)
    c = orc_cfg(max_depth=8, max_leaves=20, min_data=5)
    if quantized:
        gq, hq, sc = ctx.set_gradients(g, h)
        ref, rlor = orc.grow_leafwise(bins, nb, gq=gq, hq=hq, scales=sc, c=c, mode=HIST_INT)
    else:
        ctx.set_gradients(g, h)
        ref, rlor = orc.grow_leafwise(bins, nb, g=g, h=h, c=c, mode=HIST_F32_FIXED, chunk=LW_F32_CHUNK)
    nodes, lor = ctx.grow_tree()
    ctx.close()
    assert_same_tree(nodes, ref)
    assert np.array_equal(lor, rlor)
