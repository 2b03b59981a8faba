"""The update of many trees in one call against one tree after the other (gradient, lbt_update_tree, prediction update), which the
oracle covers: remainders of row tiles, passes over the trees, rows staged and not, objectives, outputs, weights."""
import numpy as np
import pytest
import torch

import lbtree as lb
from lbtree import ops

pytestmark = pytest.mark.gpu


def _trees(rs, n_trees, depth, f, mixed):
    out = []
    for t in range(n_trees):
        d = depth if not mixed or t % 2 == 0 else rs.randint(0, depth + 1)
        m, inner = 2 ** (d + 1) - 1, 2 ** d - 1
        feat = -np.ones(m, np.int32)
        feat[:inner] = rs.randint(0, f, inner)
        if inner > 4:
            feat[rs.randint(0, inner, 2)] = -1
        out.append((torch.from_numpy(feat).cuda(), torch.from_numpy(rs.rand(m)).cuda(), 0.01 * (t % 3), 1.0))
    return out


@pytest.mark.parametrize("n,f,k,n_trees,depth,dtype,objective,weighted", [
    (1, 3, 1, 2, 1, np.float32, "squared_error", False),
    (1025, 7, 1, 35, 5, np.float64, "log_loss", True),       # three passes, 33 descriptors and more
    (70001, 50, 1, 10, 8, np.float32, "squared_error", True),
    (4099, 64, 3, 5, 6, np.float32, "log_loss", False),      # rows of whole words
    (4099, 30, 9, 4, 5, np.float64, "log_loss", True),       # any number of outputs
    (2049, 9, 2, 17, 4, np.float32, "squared_error", False),
    (3001, 900, 1, 3, 7, np.float64, "squared_error", False),  # rows walked in memory
    (5003, 9, 1, 4, 11, np.float64, "log_loss", False),      # one tree's nodes fill the LDS
    (63, 130, 8, 3, 8, np.float32, "log_loss", False),
    (8_400_001, 1, 1, 16, 2, np.float32, "squared_error", False),  # passes of seven trees
])
def test_rounds_match_one_tree_at_a_time(n, f, k, n_trees, depth, dtype, objective, weighted):
    """Both sum in double in no fixed order: a node's sum of n terms below g is off by at most n * 2^-53 of n * g, a leaf by n * g * 2^-53
    (its hessian grows with its rows), and every later round starts from the errors so far."""
    rs = np.random.RandomState(n % 100 + k)
    X = torch.from_numpy(rs.rand(n, f).astype(dtype)).cuda()
    trees = _trees(rs, n_trees, depth, f, True)
    if objective == "log_loss":
        y = torch.from_numpy(rs.randint(0, max(k, 2), n).astype(np.float64)).cuda()
    else:
        y = torch.from_numpy(rs.rand(n, k)).cuda()
    w = torch.from_numpy(0.5 + rs.rand(n)).cuda() if weighted else None
    pred = torch.from_numpy(0.1 * rs.randn(n, k)).cuda()
    want_pred = pred.clone()
    yk = y if objective == "log_loss" and k > 1 else y.reshape(n, k)
    got = ops.update_trees(X, yk, w, objective, 0.3, pred, trees)
    assert len(got) == n_trees
    tol = 8 * n * 2.0 ** -53 * n_trees
    for (leaf, hess), (feat, split, l1, l2) in zip(got, trees):
        g, h = ops.weighted_gradient(objective, yk, want_pred, w, 0.3)
        want_leaf, want_hess, rows = ops.update_tree(X, g, h, feat, split, l1, l2, row_leaf=True)
        ops.add_leaf_values(want_pred, want_leaf, rows)
        assert torch.allclose(hess, want_hess, rtol=tol, atol=tol)
        assert torch.allclose(leaf, want_leaf, rtol=tol, atol=tol)
    assert torch.allclose(pred, want_pred, rtol=tol, atol=tol)


def test_trees_that_are_updated_one_at_a_time():
    """More sums than the LDS holds, or a tree that is not of whole levels: the call takes nothing and does nothing."""
    rs = np.random.RandomState(0)
    X = torch.from_numpy(rs.rand(100, 4)).cuda()
    y, pred = torch.zeros(100, 3, dtype=torch.float64).cuda(), torch.zeros(100, 3, dtype=torch.float64).cuda()
    assert ops.update_trees(X, y, None, "squared_error", 0.1, pred, _trees(rs, 2, 11, 4, False)) is None
    feat, split, l1, l2 = _trees(rs, 1, 3, 4, False)[0]
    assert ops.update_trees(X, y, None, "squared_error", 0.1, pred, [(feat[:14].contiguous(), split[:14].contiguous(), l1, l2)]) is None
    assert not pred.any()


@pytest.mark.parametrize("kind,outputs", [("regression", 1), ("regression", 3), ("classification", 1), ("classification", 4)])
def test_an_estimator_updates_as_with_a_tree_that_brings_its_own_update(kind, outputs):
    class Own(lb.models.Tree):
        def update(self, X, g, h):
            return super().update(X, g, h)

    rs = np.random.RandomState(outputs)
    X = rs.rand(3000, 6).astype(np.float32)
    s = X @ rs.randn(6, max(outputs, 2))
    y = (s[:, 0] if outputs == 1 else s[:, :outputs]) if kind == "regression" else s.argmax(axis=1).astype(np.float64)
    X2, y2 = X[::2].copy(), y[::2].copy()
    out = []
    for tree in (lb.models.Tree, Own):
        cls = lb.LBRegressor if kind == "regression" else lb.LBClassifier
        m = cls(n_estimators=5, base_models=(tree(max_depth=4),), random_state=1).fit(X, y)
        old = [t.leaf_value for t in m]
        m.update(X2, y2)
        assert all(not o.any() for o in old)  # cleared, and replaced
        out.append([(t.leaf_value, t.hessian) for t in m])
    for (a, b), (c, d) in zip(*out):
        assert torch.allclose(a, c, rtol=1e-9, atol=1e-12) and torch.allclose(b, d, rtol=1e-9, atol=1e-12)
