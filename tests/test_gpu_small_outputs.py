"""Trees of several outputs on few rows, bit for bit against the oracle: every width of a scan workgroup, levels with more nodes than it
has threads, rows and features that fill no whole turn, features that are left out."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,f,k,depth,samples,dtype", [
    (601, 70, 8, 10, 128, np.float32),    # more nodes than the 256 threads
    (1024, 41, 5, 6, 256, np.float64),
    (1025, 300, 2, 5, 64, np.float32),
    (2047, 130, 8, 7, 256, np.float32),
    (4096, 60, 3, 8, 256, np.float32),
    (4097, 270, 4, 7, 256, np.float32),   # more workgroups than CUs
    (7001, 300, 2, 11, 64, np.float32),
    (63, 9, 16, 6, 16, np.float64),
])
def test_few_rows_with_outputs(n, f, k, depth, samples, dtype):
    import gpu_util as gu

    rs = np.random.RandomState(n + k)
    X = rs.normal(size=(n, f)).astype(dtype)
    X[:, ::3] = rs.randint(0, 4, X[:, ::3].shape)  # many rows in a bin
    g, h = rs.normal(size=(n, k)), 0.01 + rs.rand(n, k)
    allowed = np.ones(f, bool)
    allowed[1::7] = False
    gr, cr = gu.both(X, g, h, max_depth=depth, split_samples=samples, seed=3, feature_set=allowed)
    gu.assert_tree_parity(gr, cr)


@pytest.mark.parametrize("polls", [-1, 0, 1])
@pytest.mark.parametrize("n,f,depth,s,dtype,kind", [
    (1, 3, 2, 16, np.float32, "plain"),
    (2, 1, 1, 1, np.float64, "plain"),
    (1000, 10, 8, 256, np.float64, "plain"),
    (1023, 16, 10, 64, np.float32, "few_values"),
    (1024, 17, 9, 512, np.float32, "first_excluded"),
    (1025, 32, 10, 100, np.float32, "many_excluded"),
    (2048, 33, 8, 256, np.float32, "plain"),
    (2049, 64, 8, 2048, np.float64, "few_values"),
    (4095, 5, 10, 256, np.float32, "l1"),
    (4096, 64, 1, 32, np.float32, "many_excluded"),
    (4096, 40, 7, 256, np.float32, "first_excluded"),
    (600, 8, 6, 128, np.float32, "none_left"),
    (700, 7, 9, 128, np.float32, "noise"),
])
def test_all_levels_in_one_launch(n, f, depth, s, dtype, kind, polls):
    """One output, few rows, around the sizes of the workgroups and of the lanes that decide a node. polls: looks a workgroup takes at
    the others' results before it takes a feature over; with none it does so as soon as a feature is late, and keeps several features' orders in memory."""
    import gpu_util as gu
    import oracle_lib as orc
    import torch
    from lbtree import _lib, ops

    rs = np.random.RandomState(n + f)
    X = rs.normal(size=(n, f)).astype(dtype)
    if kind == "few_values":
        X = np.round(X)
    g = (np.sin(3 * X[:, :1]) + 0.3 * rs.normal(size=(n, 1))).astype(np.float64)
    if kind == "noise":
        g = rs.normal(size=(n, 1))
    h = 0.1 + rs.rand(n, 1)
    kw = dict(max_depth=depth, split_samples=s, seed=5)
    if kind == "l1":
        kw["min_split_gain"] = 0.01
    mask = None
    if kind in ("first_excluded", "many_excluded", "none_left"):
        mask = np.ones(f, bool)
        mask[0] = False
        if kind == "many_excluded":
            mask[rs.permutation(f)[: f * 3 // 4]] = False
        if kind == "none_left":
            mask[:] = False
    l1 = 0.5 if kind == "l1" else 0.0
    want = orc.build_tree(X, g, h, feature_set=mask, l1=l1, **kw)
    Xd, gd, hd = (torch.from_numpy(a).cuda() for a in (X, g, h))
    for turn in range(3):
        _lib.lib.lbt_small_levels_polls(polls)
        try:
            got = ops.build_tree(Xd, gd, hd, feature_set=None if mask is None else torch.from_numpy(mask), row_leaf=True, wait=turn == 0,
                                 l1_regularization=l1, **kw)
        finally:
            _lib.lib.lbt_small_levels_polls(-1)
        torch.cuda.synchronize()
        for name in ("feature", "split_value", "gain"):
            assert np.array_equal(gu.cpu(getattr(got, name)), getattr(want, name)), (turn, name)
        assert np.allclose(gu.cpu(got.leaf_value), want.leaf_value, rtol=1e-12, atol=0)
        assert np.allclose(gu.cpu(got.hessian), want.hessian, rtol=1e-12, atol=0)
        gu.check_row_leaf(got, X)
