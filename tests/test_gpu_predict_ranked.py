"""Prediction by ranks (the route of large inputs) against the per-node kernel, which restates the reference's loop, bit for
bit: remainders of row tiles, tree chunks and feature groups, values equal to thresholds, trees that end early."""
import numpy as np
import pytest
import torch

from lbtree import _lib, ops

pytestmark = pytest.mark.gpu


def _ensemble(rs, n_trees, depth, f, k, dtype, levels):
    """Trees of at most `depth` levels, in turn complete, with early leaves, and of fewer levels; thresholds are drawn from
    `levels` values (0: none repeats), a few of them infinite or NaN."""
    trees = []
    for t in range(n_trees):
        d = depth if t % 3 != 2 else rs.randint(1, depth + 1)
        n, inner = 2 ** (d + 1) - 1, 2 ** d - 1
        feature = np.full(n, -1, np.int32)
        feature[:inner] = rs.randint(0, f, inner)
        if t % 3 == 1:
            feature[1:inner][rs.rand(inner - 1) < 0.2] = -1
        split = np.zeros(n)
        split[:inner] = rs.rand(inner) if levels == 0 else rs.randint(0, levels, inner) / levels
        odd = rs.rand(inner) < 0.02
        split[:inner][odd] = rs.choice([np.inf, -np.inf, np.nan, 0.0, -0.0], odd.sum())
        trees.append((torch.from_numpy(rs.randn(n, k)).cuda(), torch.from_numpy(feature).cuda(), torch.from_numpy(split).cuda()))
    return trees


def _rows(rs, n, f, dtype, levels):
    X = rs.rand(n, f) if levels == 0 else rs.randint(0, levels, (n, f)) / levels
    odd = rs.rand(n, f) < 0.01
    X[odd] = rs.choice([np.inf, -np.inf, np.nan, 0.0, -0.0, 1e300], odd.sum())
    with np.errstate(over="ignore"):
        return torch.from_numpy(X.astype(dtype)).cuda()


def _takes_ranks(X, trees, k):
    nodes = np.array([t[1].shape[0] for t in trees], np.int32)
    dt = ops._DT[X.dtype]
    plain = _lib.lib.lbt_predict_workspace_bytes(len(trees), int(nodes.sum()), k, dt)
    return _lib.lib.lbt_predict_rows_workspace_bytes(X.shape[0], X.shape[1], len(trees), nodes.ctypes.data, k, dt) > plain


@pytest.mark.parametrize("n,f,k,n_trees,depth,dtype,levels", [
    (600_011, 5, 1, 130, 6, np.float32, 0),     # 1024 rows a tile
    (900_011, 8, 1, 90, 8, np.float64, 7),      # few distinct thresholds: ties everywhere
    (400_007, 100, 1, 160, 8, np.float32, 0),   # 512 rows
    (140_001, 203, 1, 130, 8, np.float64, 0),   # 256 rows, no 16-byte rows
    (140_001, 256, 8, 120, 8, np.float32, 16),
    (66_000, 481, 3, 300, 8, np.float32, 0),    # 128 rows
    (40_003, 700, 1, 500, 7, np.float64, 0),    # 64 rows
    (3_000_003, 1, 1, 120, 3, np.float32, 0),   # one feature, shallow
    (150_003, 30, 5, 260, 10, np.float32, 0),   # deep
    (160_001, 64, 2, 301, 5, np.float64, 0),
    (70_003, 520, 1, 40, 5, np.float32, 0),     # few thresholds on many features
])
def test_ranks_give_the_sums_of_the_per_node_walk(n, f, k, n_trees, depth, dtype, levels):
    rs = np.random.RandomState(n % 1000 + f)
    trees = _ensemble(rs, n_trees, depth, f, k, dtype, levels)
    X = _rows(rs, n, f, dtype, levels)
    assert _takes_ranks(X, trees, k)
    want = ops.predict(X, trees, k, tiled=False)
    assert torch.equal(ops.predict(X, trees, k), want)


@pytest.mark.parametrize("n_trees,share,dtype", [(400, 0.3, np.float32), (250, 0.3, np.float64), (400, 0.8, np.float32)])
def test_thresholds_that_crowd_one_feature(n_trees, share, dtype):
    """255 thresholds a tree on eight features, a share of them on the first: more than its sort holds (counted instead), or
    more than 16-bit ranks tell apart, which only the device finds out."""
    rs = np.random.RandomState(int(10 * share))
    trees = []
    for _ in range(n_trees):
        feature = np.full(511, -1, np.int32)
        feature[:255] = np.where(rs.rand(255) < share, 0, rs.randint(0, 8, 255))
        trees.append((torch.from_numpy(rs.randn(511, 1)).cuda(), torch.from_numpy(feature).cuda(),
                      torch.from_numpy(rs.rand(511)).cuda()))
    X = _rows(rs, 600_001, 8, dtype, 0)
    assert _takes_ranks(X, trees, 1)
    assert torch.equal(ops.predict(X, trees, 1), ops.predict(X, trees, 1, tiled=False))


@pytest.mark.parametrize("n,f,n_trees,depth,nan_from", [
    (700_001, 40, 200, 8, 32),  # the last features have NaN thresholds only
    (600_011, 9, 200, 8, 8),
    (100_003, 520, 60, 5, 512),  # features by the cache line
    (3_000_003, 1, 120, 3, 0),  # and here there are no others at all
])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_nan_thresholds_on_features_without_others(n, f, n_trees, depth, nan_from, dtype):
    """No value is <= NaN, so every row steps to the right there, whatever the workspace held before."""
    rs = np.random.RandomState(f)
    trees = _ensemble(rs, n_trees, depth, f, 1, dtype, 0)
    for t in trees:
        t[2][t[1] >= nan_from] = float("nan")
    X = _rows(rs, n, f, dtype, 0)
    assert _takes_ranks(X, trees, 1)
    want = ops.predict(X, trees, 1, tiled=False)
    for byte in (0, 255):
        leaf_p, feat_p, split_p, nodes, _, keep = ops._tree_arrays(trees, 1)
        nbytes = _lib.lib.lbt_predict_rows_workspace_bytes(n, f, n_trees, nodes, 1, ops._DT[X.dtype])
        ws = torch.full((nbytes,), byte, dtype=torch.uint8, device="cuda")
        out = torch.empty((n, 1), dtype=torch.float64, device="cuda")
        _lib.check(_lib.lib.lbt_predict(ops._stream(), X.data_ptr(), ops._DT[X.dtype], n, f, n_trees, leaf_p, feat_p, split_p,
                                        nodes, 1, out.data_ptr(), ws.data_ptr(), nbytes))
        assert torch.equal(out, want)


@pytest.mark.parametrize("f", [513, 515, 516, 518, 543])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_last_features_of_a_cache_line(f, dtype):
    """Features by the cache line, a few at a time: the last line has one, some of a step's, a step's and more, all but one."""
    rs = np.random.RandomState(f)
    trees = _ensemble(rs, 40, 5, f, 1, dtype, 0)
    X = _rows(rs, 70_003, f, dtype, 0)
    assert _takes_ranks(X, trees, 1)
    assert torch.equal(ops.predict(X, trees, 1), ops.predict(X, trees, 1, tiled=False))


@pytest.mark.parametrize("f,n_trees,dtype", [(400, 100, np.float32), (403, 100, np.float32), (100, 40, np.float64), (103, 41, np.float64), (200, 50, np.float64)])
@pytest.mark.parametrize("share", [0.0, 0.33, 0.6, 0.9])
@pytest.mark.parametrize("last", [False, True])
def test_thresholds_that_crowd_one_cache_line(f, n_trees, dtype, share, last):
    """255 thresholds a tree, a share of them on the features of the first or of the last line of 128 bytes. Evenly all lines' tables lie
    in the LDS beside the rows (46,592 bytes; 63,232 beside turns of 128 rows, of 40 trees on doubles). A line of 9810 floats (0.33), 6770
    (0.6 of 40 trees) or 4900 doubles (0.33 of 50) has fewer cells, one of 16,000 floats, 9200 or 8000 doubles is searched in memory."""
    rs = np.random.RandomState(f + int(100 * share))
    line = 128 // np.dtype(dtype).itemsize
    crowd = np.arange((f - 1) // line * line, f) if last else np.arange(line)
    trees = []
    for _ in range(n_trees):
        feature = np.full(511, -1, np.int32)
        feature[:255] = np.where(rs.rand(255) < share, rs.choice(crowd, 255), rs.randint(0, f, 255))
        trees.append((torch.from_numpy(rs.randn(511, 1)).cuda(), torch.from_numpy(feature).cuda(),
                      torch.from_numpy(rs.rand(511)).cuda()))
    X = _rows(rs, 50_001, f, dtype, 0)
    assert _takes_ranks(X, trees, 1)
    assert torch.equal(ops.predict(X, trees, 1), ops.predict(X, trees, 1, tiled=False))


@pytest.mark.parametrize("n,f,n_trees,depth", [(1_000_000, 8, 130, 6), (70_000, 516, 40, 5)])
def test_a_start_off_a_16_byte_boundary(n, f, n_trees, depth):
    rs = np.random.RandomState(5)
    trees = _ensemble(rs, n_trees, depth, f, 1, np.float32, 0)
    base = _rows(rs, n + 1, f, np.float32, 0).reshape(-1)
    X = base[1:1 + n * f].view(n, f)
    assert X.data_ptr() % 16 != 0 and _takes_ranks(X, trees, 1)
    assert torch.equal(ops.predict(X, trees, 1), ops.predict(X, trees, 1, tiled=False))
