"""GPU parity of predict, TreeSHAP and the serving loop.

predict: bit-equal to the oracle's bin-space walk (the reference's contract,
test_cuda_predict.cpp:88-140).  TreeSHAP: within 1e-5 relative of the oracle's
Algorithm 2 in double, additivity sum(phi) = margin within 1e-5 relative
(test_cuda_shap.cpp:55,137-158), golden ice-cream tree against brute-force Shapley.
Serving: every request's result identical alone and inside any batch.
"""
import itertools
import math

import numpy as np
import pytest

from oracle_lib import HIST_F32_OMP, NODE_DTYPE, cfg as orc_cfg
from test_gpu_depthwise import tall_data

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model():
    from oracle_lib import load_oracle
    orc = load_oracle()
    bins, nb, X, y = tall_data(30000, seed_cfg=4)
    trees, init, _ = orc.train_depthwise(bins[:20000], nb, y[:20000], 1, 40, 0.1, orc_cfg(max_depth=6),
                                         mode=HIST_F32_OMP, n_threads=4)
    return trees, init, bins[20000:], nb


def test_predict_bit_equal(hip, orc, model):
    trees, init, held, nb = model
    p = hip.Predictor(trees, nb, 0.1, init)
    dev = p.predict(held)
    ref = orc.predict(trees, held, nb, 0.1, init)
    assert np.array_equal(dev.view(np.uint32), ref.view(np.uint32))
    # truncated ensembles and a single row
    p5 = hip.Predictor(trees[:5], nb, 0.1, init)
    assert np.array_equal(p5.predict(held[:1]), orc.predict(trees[:5], held[:1], nb, 0.1, init))


def test_shap_matches_algorithm2_and_is_additive(hip, orc, model):
    trees, init, held, nb = model
    rows = held[:257]
    p = hip.Predictor(trees, nb, 0.1, init)
    dev = p.shap(rows)
    ref = orc.pred_contribs(trees, rows, nb, 0.1, init, 6)
    scale = np.abs(ref).sum(axis=1, keepdims=True)
    assert np.max(np.abs(dev - ref) / scale) <= 1e-5
    margin = p.predict(rows).astype(np.float64)
    assert np.max(np.abs(dev.sum(axis=1) - margin) / np.maximum(1.0, np.abs(margin))) <= 1e-5


def ice_cream_tree():
    """The reference's ice-cream tree (tests/unit/test_shap_paths.cpp:421-434):
    covers 100 / 50 50 / 25 25 25 25, leaves 0 10 0 90, both features split at bin 0."""
    t = np.zeros(7, NODE_DTYPE)
    t[0] = (1, 0, 0, 1, 2, 0.0, 100.0, 1.0)
    t[1] = (0, 0, 0, 3, 4, 0.0, 50.0, 1.0)
    t[2] = (0, 0, 0, 5, 6, 0.0, 50.0, 1.0)
    for i, v in zip(range(3, 7), (0.0, 10.0, 0.0, 90.0)):
        t[i] = (-1, 0, 0, 0, 0, v, 25.0, 0.0)
    return t


def brute_shapley(orc, tree, row, nb):
    F = row.size
    last = (np.asarray(nb, np.uint16) - 1).astype(np.uint16)
    import ctypes as C
    from oracle_lib import P
    phi = np.zeros(F)
    tr = np.ascontiguousarray(tree)
    rb = np.ascontiguousarray(row, np.uint8)

    def ev(mask):
        s = np.array([(mask >> f) & 1 for f in range(F)], np.uint8)
        return orc.L.orc_cond_expectation(P(tr), P(rb), P(last), P(s))

    for mask in range(1 << F):
        size = bin(mask).count("1")
        for f in range(F):
            if (mask >> f) & 1:
                continue
            w = math.factorial(size) * math.factorial(F - size - 1) / math.factorial(F)
            phi[f] += w * (ev(mask | (1 << f)) - ev(mask))
    return phi


def test_shap_golden_ice_cream(hip, orc):
    tree = ice_cream_tree()
    nb = np.array([3, 3], np.uint16)   # bins 0, 1 and the missing bin 2
    p = hip.Predictor([tree], nb, 1.0, 0.0)
    rows = np.array(list(itertools.product([0, 1, 2], repeat=2)), np.uint8)
    dev = p.shap(rows)
    for r in range(rows.shape[0]):
        exact = brute_shapley(orc, tree, rows[r], nb)
        assert np.allclose(dev[r, :2], exact, rtol=0, atol=1e-4)
    # bias = expected value of the tree = (0 + 10 + 0 + 90) / 4
    assert np.allclose(dev[:, 2], 25.0)


def test_serve_results_identical_alone_and_in_the_mix(hip, orc, model):
    trees, init, held, nb = model
    p = hip.Predictor(trees, nb, 0.1, init)
    rng = np.random.default_rng(9)
    sizes = np.clip(np.round(rng.lognormal(np.log(64), 1.0, 60)).astype(np.int64), 1, 2000)
    idx = rng.integers(0, held.shape[0], sizes.sum())
    rows = held[idx]
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    arrival = np.cumsum(rng.exponential(1 / 2000.0, sizes.size))
    pred, shap, lat, stats = p.serve(rows, offs, arrival, n_slots=3, do_shap=True, max_batch_rows=4096,
                                     hbm_budget=64 << 20)
    assert stats["requests"] == sizes.size and stats["rows"] == sizes.sum()
    assert np.all(lat > 0) and stats["p99_ms"] >= stats["p50_ms"] > 0
    for r in range(sizes.size):
        a, b = int(offs[r]), int(offs[r + 1])
        alone = p.predict(rows[a:b])
        assert np.array_equal(alone.view(np.uint32), pred[a:b].view(np.uint32))
        sa = p.shap(rows[a:b])
        assert np.array_equal(sa.view(np.uint64), shap[a:b].view(np.uint64))


def test_serve_overlaps_batches_on_the_device(hip, orc, model):
    """Requests that arrive together are admitted into every free slot (several in
    flight at once) and their kernels run on the device at the same time: the device-time
    spans of batches on different streams intersect.  Results stay identical to the
    requests served alone."""
    trees, init, held, nb = model
    p = hip.Predictor(trees, nb, 0.1, init)
    rng = np.random.default_rng(12)
    n_req, size = 16, 6000
    idx = rng.integers(0, held.shape[0], n_req * size)
    rows = held[idx]
    offs = (np.arange(n_req + 1) * size).astype(np.uint64)
    arrival = np.zeros(n_req)                      # a burst: everything arrives at once
    pred, shap, lat, stats = p.serve(rows, offs, arrival, n_slots=4, do_shap=True, max_batch_rows=size,
                                     hbm_budget=1 << 30)
    assert stats["max_inflight"] >= 2
    assert stats["max_device_concurrency"] >= 2
    assert stats["device_overlap_ms"] > 0.0
    for r in (0, 7, n_req - 1):
        a, b = int(offs[r]), int(offs[r + 1])
        assert np.array_equal(p.predict(rows[a:b]).view(np.uint32), pred[a:b].view(np.uint32))
        assert np.array_equal(p.shap(rows[a:b]).view(np.uint64), shap[a:b].view(np.uint64))
    p.close()


def test_shap_split_launch_equals_single_pass(hip, orc, model):
    """A batch of 65,536 or more rows runs one workgroup per 32-row block over every path;
    smaller batches split each block's path groups over several workgroups that add their
    fixed-point sums with 64-bit integer atomics.  Both give the same bits for every row."""
    trees, init, held, nb = model
    p = hip.Predictor(trees, nb, 0.1, init)
    rng = np.random.default_rng(21)
    big = held[rng.integers(0, held.shape[0], 65_536 + 37)]
    whole = p.shap(big)                               # single pass: 2,050 row blocks
    for a, b in ((0, 1), (5, 262), (65_000, 65_573), (1_000, 33_000)):
        part = p.shap(big[a:b])                       # split launches (1 to 1,000 row blocks)
        assert np.array_equal(part.view(np.uint64), whole[a:b].view(np.uint64)), (a, b)
    ref = orc.pred_contribs(trees, big[:64], nb, 0.1, init, 6)
    scale = np.abs(ref).sum(axis=1, keepdims=True)
    assert np.max(np.abs(whole[:64] - ref) / scale) <= 1e-5
    p.close()


def random_trees(rng, n_trees, depth, n_features, nb, p_leaf, zero_cover=False):
    """Trees of exactly `depth` levels on one path, other nodes leaves with p_leaf."""
    trees = []
    for _ in range(n_trees):
        nodes = []

        def grow(level, cover, spine):
            i = len(nodes)
            nodes.append(None)
            if level == depth or (not spine and rng.random() < p_leaf):
                nodes[i] = (-1, 0, 0, 0, 0, rng.normal(0, 0.1), cover, 0.0)
                return i
            f = int(rng.integers(0, n_features))
            b = int(rng.integers(0, max(1, nb[f] - 1)))
            cl = float(np.round(cover * rng.uniform(0.05, 0.95)))
            if zero_cover and rng.random() < 0.2:
                cl = 0.0
            side = rng.random() < 0.5
            left = grow(level + 1, cl, spine and side)
            right = grow(level + 1, cover - cl, spine and not side)
            nodes[i] = (f, b, int(rng.integers(0, 2)), left, right, 0.0, cover, 1.0)
            return i

        grow(0, 1e6, True)
        trees.append(np.array(nodes, NODE_DTYPE))
    return trees


@pytest.mark.parametrize("depth,n_features,used,n_rows,p_leaf", [
    (1, 1, 1, 1, 0.0), (2, 3, 3, 64, 0.0), (3, 5, 5, 65, 0.3), (4, 28, 28, 63, 0.0), (5, 28, 4, 130, 0.2),
    (8, 28, 28, 257, 0.0), (8, 28, 6, 100, 0.1), (8, 256, 256, 31, 0.0), (9, 28, 28, 70, 0.3), (10, 10, 10, 33, 0.2),
    (12, 40, 40, 65, 0.35), (12, 28, 3, 20, 0.3), (13, 28, 12, 20, 0.4)])
def test_shap_tree_form_matches_packed_form(hip, orc, depth, n_features, used, n_rows, p_leaf):
    """Ensembles of up to 12 levels, 12 features per path and 256 features are served by
    the tree form, others by the packed form: a plane with unused features up to 257 takes
    the same trees through the packed form.  Both sum float path terms exactly, so they
    agree with the double oracle to a few float roundings per path element (1e-5 of the
    row's mass, the bound of the other TreeSHAP tests)."""
    rng = np.random.default_rng([depth, n_features, used])
    nb = rng.integers(2, 257, n_features).astype(np.uint16)
    nb[0] = 2
    for zero_cover in (False, True):
        trees = random_trees(rng, 5, depth, used, nb, p_leaf, zero_cover)
        trees.append(np.array([(-1, 0, 0, 0, 0, 0.5, 10.0, 0.0)], NODE_DTYPE))   # a single leaf
        rows = (rng.random((n_rows, n_features)) * nb).astype(np.uint8)
        p = hip.Predictor(trees, nb, 0.3, 0.25)
        got = p.shap(rows)
        wide = np.zeros((n_rows, 257), np.uint8)
        wide[:, :n_features] = rows
        wnb = np.full(257, 2, np.uint16)
        wnb[:n_features] = nb
        packed = hip.Predictor(trees, wnb, 0.3, 0.25).shap(wide)
        mass = np.abs(packed).sum(axis=1, keepdims=True)
        assert np.max(np.abs(got[:, :n_features] - packed[:, :n_features]) / mass) <= 1e-5
        assert np.array_equal(got[:, -1], packed[:, -1])
        assert np.array_equal(p.shap(rows[-1:])[0], got[-1])
        if not zero_cover:
            ref = orc.pred_contribs(trees, rows, nb, 0.3, 0.25, depth)
            assert np.max(np.abs(got - ref) / mass) <= 1e-5


@pytest.mark.parametrize("depth,used,p_leaf", [
    (4, 28, 0.0), (5, 28, 0.0), (6, 3, 0.3), (7, 28, 0.2), (8, 28, 0.0), (9, 6, 0.3), (10, 10, 0.1), (11, 28, 0.4),
    (12, 12, 0.35), (12, 3, 0.25)])
def test_shap_split_trees_equal_whole_walks(hip, depth, used, p_leaf):
    """A handful of rows take a lane a block, few row blocks x trees may give each tree a
    workgroup whose waves walk its subtrees; 1,300 rows x 60 trees walk whole trees.  The
    same bits for every row."""
    rng = np.random.default_rng([7, depth, used])
    nb = rng.integers(2, 257, 28).astype(np.uint16)
    trees = random_trees(rng, 57, depth, used, nb, p_leaf, True) + random_trees(rng, 3, 2, used, nb, 0.2)
    rows = (rng.random((1300, 28)) * nb).astype(np.uint8)
    p = hip.Predictor(trees, nb, 0.3, 0.25)
    whole = p.shap(rows)
    for a, b in ((0, 1), (3, 68), (1200, 1300)):
        assert np.array_equal(p.shap(rows[a:b]).view(np.uint64), whole[a:b].view(np.uint64)), (a, b)


@pytest.mark.parametrize("depth,n_features,n_trees,p_leaf", [
    (1, 1, 3, 0.0), (4, 28, 1, 0.0), (8, 28, 37, 0.0), (9, 28, 130, 0.3), (6, 256, 70, 0.1), (12, 60, 9, 0.2),
    (3, 257, 5, 0.0), (13, 5, 2, 0.0)])
def test_predict_tiles_match_the_walk(hip, orc, depth, n_features, n_trees, p_leaf):
    """Large batches walk trees from LDS tiles (256 or 1,024 rows per workgroup here);
    smaller ones, more than 256 features and trees past a tile walk from memory.  Every
    row is bit-equal to the oracle's walk in each."""
    rng = np.random.default_rng([depth, n_features, n_trees])
    nb = rng.integers(2, 257, n_features).astype(np.uint16)
    trees = random_trees(rng, n_trees, depth, n_features, nb, p_leaf)
    trees.append(np.array([(-1, 0, 0, 0, 0, 0.5, 10.0, 0.0)], NODE_DTYPE))
    for t in trees[::3]:
        inner = t["feature"] >= 0
        t["bin"][inner] = np.maximum(t["bin"][inner], nb[t["feature"][inner]].astype(np.uint32) - 1)  # past every cut
    p = hip.Predictor(trees, nb, 0.1, -0.5)
    for n in (1, 33, 1_025, 2_047, 2_049, 20_001, 131_073, 262_145):
        if n > 3_000 and (n_trees > 40 or n_features > 30):
            continue
        rows = (rng.random((n, n_features)) * nb).astype(np.uint8)
        dev = p.predict(rows)
        ref = orc.predict(trees, rows, nb, 0.1, -0.5)
        assert np.array_equal(dev.view(np.uint32), ref.view(np.uint32)), n
    p.close()


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("at", [0, 1, -1])
@pytest.mark.parametrize("depth,n_rows", [(3, 5), (6, 70), (6, 20_000)])
def test_shap_nonfinite_leaf(hip, depth, n_rows, at, value):
    """A leaf that is not finite, wherever it stands, makes every contribution NaN."""
    rng = np.random.default_rng([depth, n_rows])
    nb = np.full(9, 60, np.uint16)
    trees = random_trees(rng, 4, depth, 9, nb, 0.2)
    leaves = np.flatnonzero(trees[2]["feature"] < 0)
    trees[2]["value"][leaves[at]] = value
    rows = (rng.random((n_rows, 9)) * nb).astype(np.uint8)
    p = hip.Predictor(trees, nb, 0.3, 0.25)
    assert np.isnan(p.shap(rows)[:, :-1]).all()
    p.close()


@pytest.mark.parametrize("depth,n_rows", [(4, 3), (4, 20_000), (7, 5), (7, 20_000), (10, 70)])
def test_shap_small_leaves_beside_a_large_one(hip, orc, depth, n_rows):
    """One leaf of 1e6 and a subtree of leaves around 1e-6 on the root's other side: the
    grid is Sum |leaf| / 2^59 or finer, so the subtree's features (each on at most 2^(depth
    - 1) nodes, half a grid step apiece) keep their digits: that and 64 float roundings
    of terms that sum to at most twice the subtree's largest leaf."""
    rng = np.random.default_rng([depth, n_rows])
    nb = np.full(9, 60, np.uint16)
    sub = random_trees(rng, 1, depth - 1, 8, nb[1:], 0.1)[0]
    small = sub["value"] * 1e-5
    sub["value"] = small
    inner = sub["feature"] >= 0
    sub["feature"][inner] += 1
    sub["left"][inner] += 2
    sub["right"][inner] += 2
    root = np.array([(0, 30, 1, 1, 2, 0.0, 3e6, 1.0), (-1, 0, 0, 0, 0, 1e6, 2e6, 0.0)], NODE_DTYPE)
    trees = [np.concatenate([root, sub])]
    rows = (rng.random((n_rows, 9)) * nb).astype(np.uint8)
    rows[:, 0] = np.where(np.arange(n_rows) % 2 == 0, 40, 3)  # into the subtree, or beside it
    p = hip.Predictor(trees, nb, 1.0, 0.0)
    got = p.shap(rows)
    m = min(n_rows, 300)
    ref = orc.pred_contribs(trees, rows[:m], nb, 1.0, 0.0, depth)
    leaf_sum = float(np.abs(trees[0]["value"][trees[0]["feature"] < 0]).sum())
    tol = 2 ** (depth - 1) * 0.5 * leaf_sum / 2 ** 59 + 64 * 2 ** -24 * 2 * float(np.abs(small).max())
    assert np.max(np.abs(got[:m, 1:9] - ref[:, 1:9])) <= tol
    assert np.array_equal(p.shap(rows[:2]), got[:2])
    p.close()


@pytest.mark.parametrize("used,longest", [(8, 8), (9, 9), (16, 12)])
@pytest.mark.parametrize("n_rows", [1, 33, 3_000])
def test_shap_packed_path_lengths(hip, orc, used, longest, n_rows):
    """The packed form's kernels for paths of up to 8 and up to 16 features, on either side
    of the line (257 features keep the tree form off), within 1e-5 of the row's mass."""
    rng = np.random.default_rng([used, n_rows])
    nb = rng.integers(3, 257, 257).astype(np.uint16)
    trees = random_trees(rng, 6, longest, used, nb, 0.3)
    rows = (rng.random((n_rows, 257)) * nb).astype(np.uint8)
    p = hip.Predictor(trees, nb, 0.3, 0.25)
    got = p.shap(rows)
    m = min(n_rows, 200)
    ref = orc.pred_contribs(trees, rows[:m], nb, 0.3, 0.25, longest)
    mass = np.abs(ref).sum(axis=1, keepdims=True)
    assert np.max(np.abs(got[:m] - ref) / mass) <= 1e-5
    assert np.array_equal(p.shap(rows[-1:])[0], got[-1])
    p.close()


@pytest.mark.parametrize("depth,n_features,n_trees,sizes", [
    (8, 28, 37, (2_500, 5_003, 17_000, 300_000)),   # walked, then tiles of 64, 256 and 1,024 rows
    (12, 28, 5, (5_003, 16_385, 90_000)),           # a tile a tree: walked until the rows pay for it
    (13, 28, 4, (1_000, 16_383, 70_000)),           # trees past a tile
    (3, 100, 1, (33, 8_192, 100_001)),              # fewer values a row than a tile of trees
    (4, 257, 70, (2_049, 16_383, 16_384)),          # 8 rows a workgroup at most
    (3, 257, 500, (2_559, 2_560, 16_383, 16_385)),  # 16 rows and 256 trees, then a row per lane
    (3, 9_000, 3, (1, 9, 16_385))])                 # rows that leave LDS for few of them
def test_predict_shapes_match_the_walk(hip, orc, depth, n_features, n_trees, sizes):
    """Both sides of every line between the launch shapes, bit-equal to the oracle."""
    rng = np.random.default_rng([depth, n_features, n_trees])
    nb = rng.integers(2, 257, n_features).astype(np.uint16)
    trees = random_trees(rng, n_trees, depth, n_features, nb, 0.05)
    p = hip.Predictor(trees, nb, 0.1, -0.5)
    for n in sizes:
        rows = (rng.random((n, n_features), np.float32) * nb).astype(np.uint8)
        assert np.array_equal(p.predict(rows).view(np.uint32), orc.predict(trees, rows, nb, 0.1, -0.5).view(np.uint32)), n
    p.close()


@pytest.mark.parametrize("depth,used,n_features,n_trees,p_leaf", [
    (1, 1, 1, 3, 0.0), (3, 5, 5, 70, 0.2), (4, 28, 28, 300, 0.0), (5, 9, 9, 40, 0.5), (6, 28, 28, 130, 0.0),
    (7, 3, 28, 33, 0.2), (8, 28, 28, 60, 0.0), (8, 200, 200, 20, 0.1), (9, 12, 12, 30, 0.3), (10, 28, 28, 40, 0.0),
    (10, 40, 256, 9, 0.1), (11, 10, 28, 7, 0.3), (12, 28, 28, 12, 0.2), (12, 28, 28, 1, 0.0)])
def test_shap_bits_do_not_depend_on_the_batch(hip, depth, used, n_features, n_trees, p_leaf):
    """Batches of 1 to 700 rows go to lanes, subtrees or whole walks by what they cost, and
    share their trees over one or several workgroups: every row has the bits it has among
    1,500 rows, with leaves of one size and with one far above the others (either grid)."""
    rng = np.random.default_rng([11, depth, used, n_trees])
    nb = rng.integers(2, 257, n_features).astype(np.uint16)
    rows = (rng.random((1500, n_features)) * nb).astype(np.uint8)
    for large in (False, True):
        trees = random_trees(rng, n_trees, depth, used, nb, p_leaf, True)
        trees.insert(1, np.array([(-1, 0, 0, 0, 0, 0.5, 10.0, 0.0)], NODE_DTYPE))  # a single leaf
        if large:
            trees[0]["value"][np.flatnonzero(trees[0]["feature"] < 0)[0]] = 1e5
        p = hip.Predictor(trees, nb, 0.3, 0.25)
        whole = p.shap(rows).view(np.uint64)
        for a, b in ((0, 1), (5, 7), (9, 16), (0, 33), (64, 128), (100, 165), (0, 130), (200, 450), (0, 700)):
            assert np.array_equal(p.shap(rows[a:b]).view(np.uint64), whole[a:b]), (a, b)
        p.close()
