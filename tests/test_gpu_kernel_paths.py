"""Kernel variants that a rule on sizes or data selects, each at the sizes and values where it can go wrong,
bit for bit against the CPU oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _column(kind, n, rs):
    if kind == "uniform":
        return rs.random_sample(n)
    if kind == "normal":
        return rs.randn(n)
    if kind == "lognormal":
        return np.exp(2.0 * rs.randn(n))
    if kind == "negative_tail":
        return -np.exp(2.0 * rs.randn(n))
    if kind == "cauchy":
        return np.clip(rs.standard_cauchy(n), -1e30, 1e30)
    if kind == "two_clusters":
        return np.where(rs.random_sample(n) < 0.5, 1.0, 1e6) + 1e-3 * rs.randn(n)
    if kind == "tiny":
        return 1e-40 * rs.randn(n)
    if kind == "whole":
        return rs.randint(0, 16, n).astype(np.float64)
    x = rs.randn(n)
    x[::5] = np.inf
    x[1::7] = -np.inf
    x[3::13] = 3e38
    return x


@pytest.mark.parametrize("kinds", [
    ["uniform"] * 5 + ["whole"],                    # every feature straight: the plain cell function
    ["uniform"] * 4 + ["lognormal"],                # one bent feature: the whole search group is looked up bent
    ["lognormal", "negative_tail", "cauchy", "two_clusters", "tiny", "special", "normal", "whole", "uniform"],
])
@pytest.mark.parametrize("dtype,samples", [(np.float32, 256), (np.float64, 300)])
def test_cell_functions_of_the_bin_search(kinds, dtype, samples):
    import gpu_util as gu
    import oracle_lib as orc

    rs = np.random.RandomState(len(kinds) + samples)
    n = 6000
    X = np.stack([_column(k, n, rs) for k in kinds], axis=1).astype(dtype)
    # NaN falls into bin 0; not among the split candidates (their order would be unspecified) and not in a column
    # that splits (a traversal sends NaN to the right): the histograms show where it went
    nan_rows = np.setdiff1d(np.arange(0, n, 9), orc.row_samples(77, n, samples))
    X[nan_rows, 0] = np.nan
    usable = np.arange(len(kinds)) > 0
    g, h = rs.randn(n, 1), rs.rand(n, 1) + 0.5
    gr, cr = gu.both(X, g, h, levels=True, max_depth=4, split_samples=samples, seed=77, feature_set=usable)
    gu.assert_tree_parity(gr, cr, levels=True)


def _assert_tree(got, cr):
    import gpu_util as gu

    assert np.array_equal(gu.cpu(got.feature), cr.feature)
    for name in ("split_value", "gain", "leaf_value", "hessian"):
        gu.assert_same_floats(gu.cpu(getattr(got, name)), getattr(cr, name), name)


@pytest.mark.parametrize("n,f,k,depth,s,dtype", [
    (1, 1, 1, 1, 1, np.float32),
    (2, 1, 1, 13, 256, np.float64),
    (63, 3, 1, 4, 7, np.float32),
    (64, 2, 2, 5, 64, np.float64),
    (1000, 10, 1, 8, 256, np.float64),
    (1024, 5, 1, 6, 512, np.float32),      # one workgroup width of rows, and one more
    (1025, 5, 3, 6, 513, np.float32),      # samples sorted by counting, and by the bitonic network
    (2048, 70, 1, 9, 2048, np.float64),
    (2049, 4, 16, 5, 256, np.float32),
    (4095, 33, 1, 10, 100, np.float32),
    (4097, 300, 1, 7, 256, np.float32),
    (8191, 6, 4, 12, 1024, np.float64),
    (8192, 9, 4, 8, 256, np.float32),      # the most rows and entries the few-rows builder takes
    (8193, 9, 1, 8, 256, np.float32),      # one row more
    (8192, 3, 5, 4, 64, np.float32),       # more entries than it takes
    (500, 4, 1, 14, 64, np.float32),       # deeper than it takes
    (7732, 3, 1, 13, 64, np.float32),      # the most rows whose thirteen levels fit the scan's LDS, one more, and
    (7733, 3, 1, 13, 64, np.float32),      # the most rows at all
    (8192, 3, 1, 13, 64, np.float64),
    (8192, 4, 4, 13, 32, np.float32),
    (8192, 5, 4, 11, 64, np.float32),      # deeper than the medium builder takes: several outputs at the most rows,
    (2049, 4, 16, 11, 256, np.float32),    # and the most outputs
    (6900, 10, 1, 8, 256, np.float32),     # either side of where the medium builder is the faster one
    (7300, 10, 1, 8, 256, np.float32),
    (1500, 20, 4, 6, 256, np.float32),
    (2000, 20, 4, 6, 256, np.float64),
    (600, 3, 16, 2, 64, np.float32),
])
def test_few_rows(n, f, k, depth, s, dtype):
    """The builder for few rows at the edges of what it takes (and just past them), with constant and
    two-valued columns, ties between features, a feature set, an offset and regularisation in turn."""
    import gpu_util as gu
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(n + 7 * f + depth)
    X = rs.randn(n, f).astype(dtype)
    if f > 2:
        X[:, 1] = rs.randint(0, 3, n)
        X[:, 2] = X[:, 0]  # the same splits twice: the tie rule decides between features
    if f > 4:
        X[:, 3] = 1.25
    g = rs.randn(n, k)
    h = rs.rand(n, k) + 0.1
    if n > 100:
        h[n // 2:] = 0.0  # rows left out, as row subsampling leaves them
        g[n // 2:] = 0.0
    fs = None
    if f > 5:
        fs = rs.rand(f) < 0.7
        fs[0] = False
    opt = dict(l1_regularization=0.05, l2_regularization=0.5, min_split_gain=1e-3) if depth % 2 else {}
    cr = orc.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=n, feature_set=fs, l1=opt.get("l1_regularization", 0.0),
                        l2=opt.get("l2_regularization", 1.0), min_split_gain=opt.get("min_split_gain", 0.0))
    for wait in (True, False):
        got = ops.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=n, feature_set=fs, row_leaf=True,
                             wait=wait, **opt)
        torch.cuda.synchronize()
        _assert_tree(got, cr)
        gu.check_row_leaf(got, X)


@pytest.mark.parametrize("n,f,depth,dtype", [(1024, 16, 8, np.float32), (1025, 17, 9, np.float64), (4096, 64, 7, np.float32), (4097, 10, 6, np.float32),
                                             (3001, 65, 6, np.float32), (37, 1, 8, np.float64), (700, 33, 10, np.float32), (2048, 32, 8, np.float64)])
@pytest.mark.parametrize("stops", [False, True])
def test_few_rows_whose_scans_decide(n, f, depth, dtype, stops):
    """Levels that are decided by the next one's scan, either side of the rows, features, lanes and nodes up to which they are,
    in turn with levels that are not; rows that end at every level, features that are not used, ties between features."""
    import gpu_util as gu
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(n + f)
    X = rs.randn(n, f).astype(dtype)
    if f > 8:
        X[:, 5] = X[:, 0]
        X[:, 7] = rs.randint(0, 2, n)
    g, inside = rs.randn(n, 1), np.ones(n, bool)
    if stops:
        g *= 0.2
        for level in range(depth):
            inside &= X[:, level % f] > (0 if level < f else 0.3)
            g[:, 0] += inside
    kw = dict(max_depth=depth, split_samples=100, seed=3, min_split_gain=0.5 if stops else 0.0)
    h = 0.5 + rs.rand(n, 1)
    for fs in (None, np.arange(f) % 3 != 0) if f > 3 else (None,):
        cr = orc.build_tree(X, g, h, feature_set=fs, **kw)
        got = ops.build_tree(X, g, h, feature_set=fs, row_leaf=True, **kw)
        _assert_tree(got, cr)
        gu.check_row_leaf(got, X)


@pytest.mark.parametrize("case", ["negative_hessian", "zero_hessian", "all_zero", "constant_target"])
def test_few_rows_special_gradients(case):
    """Rows whose rounded hessian is not positive need the reference's unscanned bins: such data take the other
    builder, whatever the size."""
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(5)
    n, f, k = 3000, 7, 2
    X = rs.randn(n, f).astype(np.float32)
    X[:, 0] = np.round(X[:, 0])
    g, h = rs.randn(n, k), rs.rand(n, k) + 0.1
    if case == "negative_hessian":
        h[::5] *= -1.0
    elif case == "zero_hessian":
        h[::3] = 0.0
    elif case == "all_zero":
        g[:], h[:] = 0.0, 0.0
    else:
        g[:] = 1.0
        h[:] = 1.0
    cr = orc.build_tree(X, g, h, max_depth=6, split_samples=64, seed=3)
    _assert_tree(ops.build_tree(X, g, h, max_depth=6, split_samples=64, seed=3), cr)


def test_few_rows_takes_the_chunk_sums_of_the_gradient_pass():
    from lbtree import ops

    rs = np.random.RandomState(8)
    n, k = 6000, 3
    X = torch.from_numpy(rs.randn(n, 12).astype(np.float32)).cuda()
    pred, y = torch.from_numpy(rs.randn(n, k)).cuda(), torch.from_numpy(rs.randn(n, k)).cuda()
    g, h, sums = ops.weighted_gradient("squared_error", y, pred, None, 0.1, sums=True)
    a = ops.build_tree(X, g, h, max_depth=5, split_samples=64, seed=4)
    b = ops.build_tree(X, g, h, max_depth=5, split_samples=64, seed=4, abs_sum_chunks=sums)
    for name in ("leaf_value", "feature", "split_value", "gain", "hessian"):
        assert torch.equal(getattr(a, name), getattr(b, name)), name


@pytest.mark.parametrize("n,f,k,depth,s,dtype,options", [
    (8200, 4, 1, 1, 256, np.float32, {}),
    (9000, 33, 1, 6, 256, np.float32, {"features": 0.7}),
    (8448, 7, 1, 8, 64, np.float64, {}),                    # rows a multiple of the binning tile
    (20001, 32, 1, 7, 256, np.float32, {"zeros": True}),
    (16385, 5, 1, 9, 512, np.float32, {"l1": True}),        # two-byte bins, two tiles of bins in the scan
    (12000, 3, 1, 10, 2048, np.float64, {}),                # most bins, deepest tree, blocks of nodes
    (9001, 70, 3, 5, 100, np.float32, {"features": 0.5}),   # several outputs
    (8300, 11, 16, 4, 300, np.float64, {"l1": True}),
    (40000, 130, 1, 5, 256, np.float32, {}),
    (8193, 6, 2, 10, 256, np.float32, {"zeros": True}),
    (9000, 6, 1, 11, 64, np.float32, {}),                   # deeper than the builder for medium sizes takes
])
def test_medium_sizes(n, f, k, depth, s, dtype, options):
    """The builder that leaves rows in their own order, at the edges of its tiles and plans."""
    import gpu_util as gu
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(n + 7 * f + depth)
    X = rs.randn(n, f).astype(dtype)
    if f > 3:
        X[:, 1] = rs.randint(0, 3, n)
        X[:, 2] = X[:, 0]
        X[:, 3] = np.exp(2.0 * rs.randn(n))
    g = rs.randn(n, k) + X[:, :1]
    h = rs.rand(n, k) + 0.1
    if options.get("zeros"):
        h[::3] = 0.0
        g[::3] = 0.0
    fs = rs.rand(f) < options["features"] if "features" in options else None
    kw = dict(l1=0.05, l2=0.5, min_split_gain=1e-3) if options.get("l1") else {}
    kw2 = dict(l1_regularization=0.05, l2_regularization=0.5, min_split_gain=1e-3) if kw else {}
    cr = orc.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=n, feature_set=fs, **kw)
    for wait in (True, False):
        got = ops.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=n, feature_set=fs, row_leaf=True,
                             wait=wait, **kw2)
        torch.cuda.synchronize()
        _assert_tree(got, cr)
        gu.check_row_leaf(got, X)


@pytest.mark.parametrize("n,f,k,depth,s", [(9001, 43, 1, 9, 256), (8500, 260, 1, 5, 64), (156250, 64, 1, 4, 64), (156251, 64, 1, 4, 64), (200003, 61, 1, 4, 64),
                                           (20002, 10, 2, 8, 128), (30011, 17, 3, 6, 256), (78125, 64, 1, 4, 64), (78126, 64, 1, 4, 64), (9000, 512, 1, 4, 64), (9000, 514, 1, 4, 64),
                                           (31250, 20, 8, 4, 64), (31251, 20, 8, 4, 64)])
def test_medium_sizes_whose_rows_stop_at_every_level(n, f, k, depth, s):
    """Histogram workgroups that find their rows' nodes, by themselves or after the launch that decides many nodes, either side
    of the number of rows where they do (one workgroup to a CU, and two), in turn with levels that do not: rows end at every level,
    at most nodes of the last ones no row is left."""
    import gpu_util as gu
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(n + f)
    X = rs.randn(n, f).astype(np.float32)
    g, inside = 0.3 * rs.randn(n, k), np.ones(n, bool)
    for level in range(depth):  # half of what is left is told from the rest, and goes on
        inside &= X[:, level % f] > (0 if level < f else 0.5)
        g[:, 0] += inside
    h = 0.5 + rs.rand(n, k)
    kw = dict(max_depth=depth, split_samples=s, seed=9, min_split_gain=2.0)
    cr = orc.build_tree(X, g, h, **kw)
    got = ops.build_tree(X, g, h, row_leaf=True, **kw)
    _assert_tree(got, cr)
    gu.check_row_leaf(got, X)
    ends = [int((cr.feature[2 ** d - 1:2 ** (d + 1) - 1] < 0).sum()) for d in range(depth)]
    assert ends[depth // 2] > 0 and int((cr.feature >= 0).sum()) >= depth


def test_medium_sizes_under_an_explicit_budget():
    """Budgets either side of what the builder's histograms and images take, in a workspace of the size the query
    names for the budget: the same tree, by that builder or by the general one."""
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(12)
    n, f, k, depth, s = 12000, 14, 2, 6, 200
    X, g, h = rs.randn(n, f).astype(np.float32), rs.randn(n, k), rs.rand(n, k) + 0.1
    cr = orc.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=2)
    two_levels = 2 * 2 ** (depth - 1) * k * f * s * 16
    for budget in (1, two_levels - 1, two_levels + (64 << 20), 10 ** 9):
        ops._workspace.clear()
        _assert_tree(ops.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=2, hist_cache_bytes=budget), cr)


@pytest.mark.parametrize("case", ["one_sign", "one_row", "negative_hessian", "all_zero"])
def test_medium_sizes_special_gradients(case):
    """Sums at the edge of the packed 32 bits (all gradients of one sign in one bin; nearly the whole mass in one
    row) and data that the other builder has to take."""
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(6)
    n, f = 30000, 5
    X = rs.randn(n, f).astype(np.float32)
    X[:, 0] = (rs.rand(n) < 1e-3).astype(np.float32)  # nearly all rows in one bin
    g, h = rs.rand(n, 1) + 0.1, rs.rand(n, 1) + 0.1
    if case == "one_row":
        g = rs.randn(n, 1) * 1e-6
        g[4321] = -5.0
        h = np.full((n, 1), 1e-3)
        h[17] = 900.0
    elif case == "negative_hessian":
        h[::7] *= -1.0
    elif case == "all_zero":
        g[:], h[:] = 0.0, 0.0
    for sign in (1.0, -1.0):
        cr = orc.build_tree(X, sign * g, h, max_depth=4, split_samples=64, seed=5)
        _assert_tree(ops.build_tree(X, sign * g, h, max_depth=4, split_samples=64, seed=5), cr)


@pytest.mark.parametrize("rows", [(700, 900), (700, 9000), (9000, 9500)])
def test_builds_of_one_thread_on_two_streams(rows):
    """All builds of a thread hear from their kernels through the same pinned words. Calls without observation points
    beside calls that want the number of bins, in turn on two streams and with the words given back in between: every
    call has to get its own answer, and no store of an earlier one may come after it has returned."""
    from lbtree import _lib, ops

    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    calls, want = [], []
    for i, n in enumerate(rows):
        rs = np.random.RandomState(n)
        X, g, h = (torch.from_numpy(a).cuda() for a in (rs.randn(n, 20).astype(np.float32), rs.randn(n, 1), 0.1 + rs.rand(n, 1)))
        calls.append((X, g, h, dict(max_depth=5, split_samples=64, seed=i, row_leaf=i == 1, wait=False)))
        want.append(ops.build_tree(X, g, h, **dict(calls[i][3], wait=True)))
    torch.cuda.synchronize()
    for turn in range(100):
        got = [None, None]
        for i in ((0, 1) if turn % 2 else (1, 0)):
            X, g, h, kw = calls[i]
            with torch.cuda.stream(streams[i]):
                got[i] = ops.build_tree(X, g, h, **kw)
        if turn % 10 == 0:
            assert _lib.lib.lbt_release_thread_resources() == 0
        torch.cuda.synchronize()
        for i in range(2):
            for name in ("leaf_value", "feature", "split_value", "gain", "hessian"):
                assert torch.equal(getattr(got[i], name), getattr(want[i], name)), (turn, i, name)


@pytest.mark.parametrize("n,f,k,depth,hessian", [(1, 2, 1, 1, -0.3), (900, 12, 3, 7, -0.3), (5000, 9, 1, 13, -0.3),
                                                 (900, 12, 3, 7, 1e-13), (5000, 9, 1, 13, 1e-13),
                                                 (9000, 9, 1, 1, -0.3), (40000, 21, 2, 10, -0.3)])
def test_data_for_the_other_builder_leave_the_queue(n, f, k, depth, hessian):
    """Negative hessians (for the builder for few rows also those that round to 0) are met when the levels of the
    builders for few rows and medium sizes are being queued: what is queued does nothing, and the general builder's
    tree is the result, call after call without a wait between."""
    import gpu_util as gu
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(n + f)
    X = rs.randn(n, f).astype(np.float32)
    g, h = rs.randn(n, k), rs.rand(n, k) + 0.1
    bad = h.copy()
    bad[n // 2:] = hessian
    Xd, gd, hd, bd = (torch.from_numpy(a).cuda() for a in (X, g, h, bad))
    kw = dict(max_depth=depth, split_samples=32, seed=9)
    got = []
    for turn in range(3):
        got.append(ops.build_tree(Xd, gd, bd, wait=False, row_leaf=True, **kw))
        got.append(ops.build_tree(Xd, gd, hd, wait=False, row_leaf=turn == 1, **kw))
    torch.cuda.synchronize()
    want = [orc.build_tree(X, g, a, **kw) for a in (bad, h)]
    for i, r in enumerate(got):
        _assert_tree(r, want[i % 2])
        if i % 2 == 0:
            gu.check_row_leaf(r, X)


@pytest.mark.parametrize("n,f,k,depth,s,kind,dtype", [
    (9000, 6, 1, 5, 64, "low", np.float32),
    (12000, 33, 1, 8, 256, "span", np.float32),
    (20001, 7, 2, 6, 300, "most", np.float32),
    (8200, 5, 3, 10, 512, "output", np.float64),
    (30000, 12, 1, 9, 100, "most", np.float32),
])
def test_medium_sizes_with_hessians_that_round_to_zero(n, f, k, depth, s, kind, dtype):
    """Rows with a gradient whose hessian rounds to 0 make the reference leave bins unscanned, and their siblings'
    histograms differ by them (in every one of these cases the tree is another one without that rule). The medium
    builder keeps to it where the reference would hold all histograms; an explicit budget under which it would not
    gives the tree of that budget."""
    import gpu_util as gu
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(n + f)
    X = rs.randn(n, f).astype(dtype)
    X[:, 0] = np.round(2 * X[:, 0]) / 2
    g, h = rs.randn(n, k), rs.rand(n, k) + 0.1
    if kind == "low":  # no hessian where a feature is small: its first bins have a sum of gradients only
        h[X[:, 1] < -0.5] = 1e-12
    elif kind == "most":
        h[rs.rand(n) < 0.95] = 1e-12
    elif kind == "span":
        h = 10.0 ** (-10 * rs.rand(n, k))
    else:  # of one output, of another one
        h[::3, 0] = 0.0
        h[X[:, 2] < 0, k - 1] = 1e-12
    for budget in (0, f * s * k * 16 * 5):
        cr = orc.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=n, hist_cache_bytes=budget)
        assert ((cr.quantised[..., 1] == 0) & (cr.quantised[..., 0] != 0)).any()
        got = ops.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=n, row_leaf=True, hist_cache_bytes=budget)
        _assert_tree(got, cr)
        gu.check_row_leaf(got, X)


@pytest.mark.parametrize("f,k", [(13, 2), (13, 4), (13, 5), (13, 8), (13, 9), (100, 8), (100, 9), (100, 17), (200, 2),
                                 (200, 16), (200, 17), (200, 33)])
def test_predict_shares_the_outputs_out_among_the_lanes_of_a_row(f, k):
    """Output counts around one and two per lane and around a whole walk, for 4, 8 and 16 lanes per row; few trees,
    a batch that is not full, and several batches. Sums are formed in tree order: equal to the oracle's."""
    import gpu_util as gu
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(f + k)
    X = rs.rand(777, f).astype(np.float32)
    trees_c, trees_g = [], []
    for t in range(45):
        depth = [6, 2, 8, 4][t % 4]
        m, inner = 2 ** (depth + 1) - 1, 2 ** depth - 1
        feat = -np.ones(m, np.int32)
        feat[:inner] = rs.randint(0, f, inner)
        trees_c.append((rs.randn(m, k), feat, rs.rand(m)))
        trees_g.append(tuple(ops.as_device(a) for a in trees_c[-1]))
    for n_trees in (1, 3, 18, 45):
        want = orc.predict(X, trees_c[:n_trees], k)
        assert np.array_equal(gu.cpu(ops.predict(X, trees_g[:n_trees], k)), want), n_trees


@pytest.mark.parametrize("n,f,k,s,depth", [(9001, 60, 8, 512, 9), (9001, 50, 1, 512, 12)])
@pytest.mark.parametrize("zero_hessians", [False, True])
def test_levels_that_outgrow_the_histogram_budget_give_the_same_tree(n, f, k, s, depth, zero_hessians):
    """The library's own budget (parents kept, only built siblings cleared) against explicit budgets (every level
    that outgrows them starts an empty buffer), and against observed builds, whose levels are all in memory and built as
    the reference builds them (the deep case's otherwise stay in the LDS under any budget). With rows that have no
    hessian the tree depends on the budget (the reference leaves bins unscanned), and the library's own is the
    reference's."""
    from lbtree import ops

    rs = np.random.RandomState(f)
    X = torch.from_numpy(rs.randn(n, f).astype(np.float32)).cuda()
    g = torch.from_numpy(rs.randn(n, k)).cuda()
    h = torch.from_numpy(0.1 + rs.random_sample((n, k))).cuda()
    if zero_hessians:
        h[::97] = 0.0
    got = ops.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=3, row_leaf=True)
    for budget in (10 ** 9,) if zero_hessians else (10 ** 9, 4 * 10 ** 7):
        for observed in (False, True):
            want = ops.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=3, row_leaf=True, hist_cache_bytes=budget,
                                  taps=observed)
            for name in ("leaf_value", "feature", "split_value", "gain", "hessian", "row_leaf"):
                assert torch.equal(getattr(got, name), getattr(want, name)), (budget, observed, name)


@pytest.mark.parametrize("n,f,k,s,depth", [(9001, 60, 8, 512, 9), (8200, 40, 3, 2048, 9), (9001, 50, 1, 512, 12)])
@pytest.mark.parametrize("share,sign", [(0.02, 0), (0.5, 0), (0.5, -1), (0.97, -1)])
def test_levels_that_outgrow_the_budget_with_hessians_of_zero(n, f, k, s, depth, share, sign):
    """Unscanned bins in few and in most nodes of the levels above: siblings are derived below the reference's buffer only where
    their parent's histogram is what its rows add up to. Equal to the reference's budget, whose levels are added up from all rows, and to its observed
    build, bit for bit."""
    from lbtree import ops

    rs = np.random.RandomState(n + k)
    X = rs.randn(n, f).astype(np.float32)
    X[:, 1] = np.round(X[:, 1])
    g, h = rs.randn(n, k), 0.1 + rs.random_sample((n, k))
    h[rs.rand(n, k) < share] = 0.0
    if sign:
        g = np.where(rs.rand(n, k) < 0.9, -np.abs(g), g)
    X, g, h = (torch.from_numpy(a).cuda() for a in (X, g, h))
    kw = dict(max_depth=depth, split_samples=s, seed=3, row_leaf=True)
    got = ops.build_tree(X, g, h, **kw)
    for observed in (False, True):
        want = ops.build_tree(X, g, h, hist_cache_bytes=10 ** 9, taps=observed, **kw)
        for name in ("leaf_value", "feature", "split_value", "gain", "hessian", "row_leaf"):
            assert torch.equal(getattr(got, name), getattr(want, name)), (observed, name)


def test_a_build_does_without_the_room_that_it_cannot_have(monkeypatch):
    """Where the room for the library's own budget of histograms cannot be had the build takes place in the
    reference's, and gives the same tree; an explicit budget is not cut."""
    from lbtree import _lib, ops

    rs = np.random.RandomState(1)
    n, f, k, depth, s = 9001, 60, 8, 9, 512
    X, g, h = (torch.from_numpy(a).cuda() for a in (rs.randn(n, f).astype(np.float32), rs.randn(n, k), 0.1 + rs.rand(n, k)))
    kw = dict(max_depth=depth, split_samples=s, seed=3)
    want = ops.build_tree(X, g, h, **kw)
    full, least = (_lib.lib.lbt_build_tree_workspace_bytes(n, f, k, depth, s, _lib.LBT_F32, b) for b in (0, 10 ** 9))
    assert full > least + 10 ** 9
    plain, asked = ops._get_workspace, []

    def scarce(nbytes, device):
        asked.append(nbytes)
        if nbytes > least:
            raise torch.OutOfMemoryError("not that much")
        return plain(nbytes, device)

    ops._workspace.clear()
    monkeypatch.setattr(ops, "_get_workspace", scarce)
    got = ops.build_tree(X, g, h, **kw)
    assert asked == [full, least]
    for name in ("leaf_value", "feature", "split_value", "gain", "hessian"):
        assert torch.equal(getattr(got, name), getattr(want, name)), name
    with pytest.raises(torch.OutOfMemoryError):
        ops.build_tree(X, g, h, hist_cache_bytes=4 * 10 ** 9, **kw)


def test_every_thread_and_stream_has_a_workspace_of_its_own():
    """Builds that may overlap do not share scratch; a thread's is reused call after call, and given back."""
    import threading

    from lbtree import ops

    device = torch.device("cuda", torch.cuda.current_device())

    def scratch():
        return ops._get_workspace(1000, device)

    ops.release_workspace()
    first, side = scratch(), torch.cuda.Stream()
    with torch.cuda.stream(side):
        second = scratch()
        assert scratch() is second
    others = []
    t = threading.Thread(target=lambda: others.append(scratch()))
    t.start()
    t.join()
    assert len({first.data_ptr(), second.data_ptr(), others[0].data_ptr()}) == 3
    assert scratch() is first and ops._get_workspace(900, device) is first and ops._get_workspace(2000, device) is not first
    ops.release_workspace()
    assert not ops._workspace.held


@pytest.mark.parametrize("n,f,k,depth,dtype", [(1, 3, 1, 1, np.float32), (1023, 7, 1, 5, np.float64),
                                               (1025, 50, 8, 8, np.float32), (70001, 13, 3, 8, np.float32),
                                               (5003, 9, 9, 8, np.float64), (5003, 9, 1, 11, np.float32), (3001, 200, 1, 5, np.float32),
                                               (3001, 9, 2, 11, np.float64)])
def test_update_tree_and_the_rows_leaves(n, f, k, depth, dtype):
    """Node sums that fit the LDS and that do not (more than 8192 doubles), rows around a workgroup: leaves within
    rounding of the oracle's sequential sums (n additions of one sign: n * 2^-53 relative), rows as predict walks."""
    import gpu_util as gu
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(n + k)
    X = rs.rand(n, f).astype(dtype)
    m, inner = 2 ** (depth + 1) - 1, 2 ** depth - 1
    feat = -np.ones(m, np.int32)
    feat[:inner] = rs.randint(0, f, inner)
    feat[rs.randint(0, inner, 2) if inner > 4 else []] = -1
    split = rs.rand(m)
    g, h = 0.5 + rs.rand(n, k), 0.5 + rs.rand(n, k)
    leaf_c, hess_c = orc.update_tree(X, g, h, feat, split, 0.0, 1.0)
    Xd, gd, hd, fd, sd = (ops.as_device(a) for a in (X, g, h, feat, split))
    leaf, hess, rows = ops.update_tree(Xd, gd, hd, fd, sd, 0.0, 1.0, row_leaf=True)
    tol = 4 * n * 2.0 ** -53
    assert np.allclose(gu.cpu(hess), hess_c, rtol=tol, atol=0)
    assert np.allclose(gu.cpu(leaf), leaf_c, rtol=2 * tol, atol=0)
    pred = torch.zeros((n, k), dtype=torch.float64, device="cuda")
    ops.add_leaf_values(pred, leaf, rows)
    assert torch.equal(pred, ops.predict(Xd, [(leaf, fd, sd)], k))
    plain = ops.update_tree(Xd, gd, hd, fd, sd, 0.0, 1.0)
    assert len(plain) == 2 and torch.allclose(plain[1], hess, rtol=tol, atol=0)


@pytest.mark.parametrize("n,f,s,depth,kind", [(9001, 50, 512, 12, "plain"), (20011, 33, 200, 12, "feature_set"),
                                              (9001, 7, 257, 13, "weighted"), (30011, 130, 256, 11, "whole")])
def test_levels_without_histograms_in_memory_give_the_oracles_tree(n, f, s, depth, kind):
    """Deep levels whose histograms stay in the LDS against an observed build, which keeps them in memory, and the
    oracle's tree: bins of one and two bytes, features that end inside a 16-byte piece, several record groups,
    unusable features, gradients that reach far into 32 bits, columns of few values (long empty runs)."""
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(depth)
    X = rs.randn(n, f).astype(np.float32)
    if kind == "whole":
        X[:, ::2] = rs.randint(0, 5, X[:, ::2].shape)
    g = rs.randn(n, 1)
    h = 0.5 + rs.random_sample((n, 1))
    if kind == "weighted":
        g[:3] *= 3000.0
    fs = rs.random_sample(f) < 0.6 if kind == "feature_set" else None
    Xd, gd, hd = (torch.from_numpy(a).cuda() for a in (X, g, h))
    kw = dict(max_depth=depth, split_samples=s, seed=5, feature_set=fs)
    got = ops.build_tree(Xd, gd, hd, row_leaf=True, **kw)
    want = ops.build_tree(Xd, gd, hd, row_leaf=True, taps=True, **kw)  # observed: histograms in memory
    for name in ("leaf_value", "feature", "split_value", "gain", "hessian", "row_leaf"):
        assert torch.equal(getattr(got, name), getattr(want, name)), name
    _assert_tree(got, orc.build_tree(X, g, h, **kw))


@pytest.mark.parametrize("n,f,s,depth,kind", [(9001, 9, 511, 12, "one_sign"), (9001, 6, 254, 11, "near_ties"), (20001, 5, 509, 12, "near_ties"),
                                              (12001, 17, 61, 11, "equal_columns"), (9001, 8, 512, 12, "l2"),
                                              (9001, 9, 64, 11, "one_sign"), (20001, 6, 64, 11, "near_ties"), (9001, 6, 65, 11, "near_ties")])
def test_deep_levels_whose_estimates_do_not_decide(n, f, s, depth, kind):
    """Sums of grads that leave 32 bits with their sign, bins whose estimates lie closer together than they are right, equal
    columns, a penalty far above the hessians; bins that are no multiple of the four a lane takes, and up to 64 bins, of which it takes
    one: the oracle's tree."""
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(s)
    X = rs.randn(n, f).astype(np.float32)
    g, h = rs.randn(n, 1), np.ones((n, 1))
    kw, l2 = dict(max_depth=depth, split_samples=s, seed=6), 1.0
    if kind == "one_sign":
        g = 1.0 + 0.2 * rs.rand(n, 1)
    elif kind == "near_ties":
        g = np.where(X[:, :1] > 0, 1.0, -1.0) * (1.0 + 1e-6 * rs.rand(n, 1))
    elif kind == "equal_columns":
        X[:, 1::2] = X[:, :1]
    else:
        l2 = 1e5
    Xd, gd, hd = (torch.from_numpy(a).cuda() for a in (X, g, h))
    _assert_tree(ops.build_tree(Xd, gd, hd, l2_regularization=l2, **kw), orc.build_tree(X, g, h, l2=l2, **kw))


@pytest.mark.parametrize("n,f,s,depth,kind", [(8193, 4, 256, 11, "outliers"), (12300, 2, 512, 12, "noise"), (16385, 3, 64, 11, "outliers"), (30001, 7, 256, 11, "outliers"), (60000, 5, 300, 12, "noise"),
                                              (70001, 20, 512, 11, "one_split"), (65536, 70, 64, 11, "stopped")])
def test_deep_levels_with_one_large_node(n, f, s, depth, kind):
    """Trees that are not balanced: nodes of more rows than one workgroup takes, which begin and end inside a range of
    positions, beside small ones and behind rows that have stopped. Call after call: the sums of a large node have to
    be zero again when the next one begins."""
    import gpu_util as gu
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(n)
    X = rs.randn(n, f).astype(np.float32)
    g, h = rs.randn(n, 1), 0.5 + rs.rand(n, 1)
    if kind == "outliers":
        g = g ** 9
    elif kind == "one_split":
        g = 0.1 * g + 5.0 * (X[:, :1] > 3.0)
    elif kind == "stopped":  # a third of the rows ends in leaves early, the others stay together for long
        g = np.where(X[:, :1] > 0.5, 1e6, g ** 9)
    kw = dict(max_depth=depth, split_samples=s, seed=4)
    cr = orc.build_tree(X, g, h, **kw)
    Xd, gd, hd = (torch.from_numpy(a).cuda() for a in (X, g, h))
    for _ in range(3):
        got = ops.build_tree(Xd, gd, hd, row_leaf=True, **kw)
        _assert_tree(got, cr)
    gu.check_row_leaf(got, Xd)


@pytest.mark.parametrize("f,k,n_trees", [(13, 1, 45), (13, 3, 45), (13, 1, 3), (100, 1, 45), (100, 9, 7), (200, 1, 45)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_predict_takes_more_lanes_per_row_for_few_rows(f, k, n_trees, dtype):
    """Row counts either side of the two limits, ensembles laid out for 4, 8 and 16 lanes, few trees and several
    outputs: equal to the per-node kernel."""
    from lbtree import ops

    rs = np.random.RandomState(f + k)
    gen = torch.Generator(device="cuda").manual_seed(f)
    X = torch.rand((33001, f), generator=gen, device="cuda", dtype=torch.float64).to(
        torch.float32 if dtype == np.float32 else torch.float64)
    trees = []
    for t in range(n_trees):
        depth = [6, 2, 8, 4][t % 4]
        m, inner = 2 ** (depth + 1) - 1, 2 ** depth - 1
        feat = -np.ones(m, np.int32)
        feat[:inner] = rs.randint(0, f, inner)
        trees.append(tuple(ops.as_device(a) for a in (rs.randn(m, k), feat, rs.rand(m))))
    want = ops.predict(X, trees, k, tiled=False)
    packed = ops.PackedEnsemble(trees, k, f, X.dtype) if f <= 100 else None
    for rows in (1, 63, 65, 16384, 16385, 32768, 32769, 33001):
        assert torch.equal(ops.predict(X[:rows], trees, k), want[:rows]), rows
        if packed is not None:
            assert torch.equal(packed.predict(X[:rows]), want[:rows]), rows


@pytest.mark.parametrize("f,k,n_trees,depth,dtype", [(13, 1, 17, 3, np.float32), (13, 1, 129, 6, np.float32), (160, 1, 300, 8, np.float64),
                                                     (7, 64, 40, 4, np.float32), (7, 65, 40, 4, np.float32), (300, 5, 33, 8, np.float64),
                                                     (31, 8, 1000, 3, np.float32),
                                                     # turns of one batch and of two, several outputs with few trees a batch and with more
                                                     (32, 1, 150, 8, np.float32), (100, 1, 117, 7, np.float32), (10, 1, 60, 8, np.float64),
                                                     (12, 8, 34, 9, np.float64), (22, 2, 60, 8, np.float32)])
def test_predict_of_few_rows(f, k, n_trees, depth, dtype):
    """Up to 4096 rows and more than 16 trees: rows around a workgroup's 16, trees around the 128 of a turn, outputs around the 64 that
    its threads add, ensembles of one and of many turns: equal to the per-node kernel."""
    from lbtree import ops

    rs = np.random.RandomState(f + n_trees)
    X = ops.as_device(rs.rand(4097, f).astype(dtype))
    trees = []
    for t in range(n_trees):
        d = depth if t % 3 else rs.randint(1, depth + 1)
        m, inner = 2 ** (d + 1) - 1, 2 ** d - 1
        feat = -np.ones(m, np.int32)
        feat[:inner] = rs.randint(0, f, inner)
        if t % 2 and inner > 4:
            feat[rs.randint(1, inner, 2)] = -1
        trees.append(tuple(ops.as_device(a) for a in (rs.randn(m, k), feat, rs.rand(m))))
    want = ops.predict(X, trees, k, tiled=False)
    for rows in (1, 15, 16, 17, 255, 4095, 4096, 4097):
        assert torch.equal(ops.predict(X[:rows], trees, k), want[:rows]), rows
    if f <= 160 and dtype == np.float32:
        packed = ops.PackedEnsemble(trees, k, f, X.dtype)
        for rows in (1, 17, 4096):
            assert torch.equal(packed.predict(X[:rows]), want[:rows]), rows


@pytest.mark.parametrize("n,f,s,depth", [(1024, 300, 64, 9), (4096, 257, 128, 8), (4097, 257, 64, 11), (8192, 260, 256, 9), (7999, 30, 256, 11),
                                         (2049, 256, 32, 10)])
def test_few_rows_with_the_nodes_staged_or_not(n, f, s, depth):
    """Either side of the sizes at which the scan keeps the nodes in the LDS (levels whose nodes do not fit beside the rows) and at
    which two of its workgroups share a CU (more features than CUs), rows around its numbers of places."""
    import gpu_util as gu
    import oracle_lib as orc

    rs = np.random.RandomState(n + f)
    X = rs.randn(n, f).astype(np.float32)
    g, h = rs.randn(n, 1), 0.5 + rs.rand(n, 1)
    kw = dict(max_depth=depth, split_samples=s, seed=3)
    got = gu.gpu_build(X, g, h, taps=False, **kw)
    cr = orc.build_tree(X, g, h, **kw)
    _assert_tree(got, cr)


# A level of up to 512 (node, feature) pairs is scanned by four or eight waves a pair (up to 64 bins, or 128 and one output,
# by one), a wider one by one wave: tiles of 64 bins that do not divide evenly among the waves, fewer tiles than waves, features of one bin, levels on both
# sides of the line, outputs whose hessians vanish, a penalty and features that are not to be split.
@pytest.mark.parametrize("f,k,s,depth,kind", [(64, 1, 512, 5, "plain"), (64, 3, 129, 5, "plain"), (5, 8, 300, 4, "l1"), (513, 1, 65, 2, "plain"),
                                              (128, 2, 64, 4, "plain"), (9, 64, 257, 3, "plain"), (33, 5, 256, 6, "feature_set"),
                                              (17, 4, 400, 5, "zero_output"), (40, 1, 449, 5, "zero_hessians"),
                                              (40, 1, 128, 4, "plain"), (40, 1, 129, 4, "plain"), (40, 2, 128, 4, "plain")])
def test_waves_that_share_a_scan(f, k, s, depth, kind):
    import gpu_util as gu

    rs = np.random.RandomState(f + k + s)
    n = 6001
    X = rs.randn(n, f).astype(np.float32)
    X[:, 0] = 1.0  # one bin
    X[:, 1] = rs.randint(0, 70, n)
    g, h = rs.randn(n, k), rs.rand(n, k) + 0.5
    if kind == "zero_output":
        g[:, k - 1] = h[:, k - 1] = 0.0
    if kind == "zero_hessians":
        h[rs.rand(n) < 0.3] = 0.0
    more = {"l1_regularization": 3.0} if kind == "l1" else {}
    if kind == "feature_set":
        more["feature_set"] = rs.rand(f) < 0.5
    for levels in (True, False):
        gr, cr = gu.both(X, g, h, levels=levels, max_depth=depth, split_samples=s, seed=f, **more)
        gu.assert_tree_parity(gr, cr, levels=levels)


# The prefix counts of a level's partition: one slab of 2048 rows, edges of slabs, more slabs than threads that
# scan them (1024), more than a thread asks for at once (8192), more parents than waves of a workgroup, than rows.
@pytest.mark.parametrize("n,level", [(1, 0), (2047, 1), (2048, 0), (2049, 2), (5000, 5), (3000, 11), (70001, 8), (2_100_000, 3), (17_000_003, 4)])
def test_partition_of_a_level_is_the_stable_sort(n, level):
    from lbtree import ops

    gen = torch.Generator(device="cuda").manual_seed(n + level)
    first, parents = (1 << level) - 1, 1 << level
    X = torch.rand((n, 1), device="cuda", generator=gen)
    node = torch.randint(-1, parents, (n,), device="cuda", generator=gen, dtype=torch.int32)
    node[node % 7 == 3] = -1  # retired rows, and parents without rows
    node = torch.where(node < 0, node, node + first).sort().values
    rows = torch.randperm(n, device="cuda", generator=gen).to(torch.int32)
    feature = torch.zeros(2 * parents + first, device="cuda", dtype=torch.int32)
    feature[first + 5 :: 6] = -1  # leaves
    split = torch.rand(feature.shape[0], device="cuda", generator=gen, dtype=torch.float64)
    positions = torch.stack([node, rows], dim=1).contiguous()

    at = node.clamp(min=0).long()
    left = X[rows.long(), 0].double() <= split[at]
    want = torch.where((node < 0) | (feature[at] < 0), -1, 2 * node + 2 - left.int())
    order = torch.sort(want, stable=True).indices
    want = torch.stack([want[order], rows[order]], dim=1).to(torch.int32)
    ops.update_positions(X, positions, feature, split, level)
    assert torch.equal(positions, want)


# Rounded gradients of one output: fewer rows than a workgroup, ragged ends of a thread's four rows, and hessians that
# round to zero in the last row only, which decides how the levels after the root may be built.
@pytest.mark.parametrize("n", [1, 1023, 262145, 3 * 262144 + 77, 1_300_000])
def test_rounding_of_one_output(n):
    import gpu_util as gu

    rs = np.random.RandomState(n % 1000)
    X = rs.randn(n, 3).astype(np.float32)
    g, h = rs.randn(n, 1), rs.rand(n, 1) + 0.5
    h[-1] = 1e-13
    gr, cr = gu.both(X, g, h, levels=True, max_depth=3, split_samples=32, seed=7)
    gu.assert_tree_parity(gr, cr, levels=True)


# Levels without histograms in memory estimate the gains and form few of them exactly: against the oracle where many are
# equal (columns of two values, copies of a column, plateaus of more than 64 empty bins), with penalties that rule the
# estimate out, gains that a min_split_gain cuts off, and gradients whose squares nearly leave the doubles.
@pytest.mark.parametrize("kind", ["copies", "two_values", "long_tails", "l1", "min_split_gain", "no_l2", "large_l2", "huge", "tiny", "one_sign"])
def test_estimated_gains_choose_the_oracles_splits(kind):
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(len(kind))
    n, f, s = 9001, 50, 512
    X = rs.randn(n, f).astype(np.float32)
    g, h = rs.randn(n, 1), 0.1 + rs.random_sample((n, 1))
    kw = dict(max_depth=11, split_samples=s, seed=9)
    if kind == "copies":
        X[:, 1::2] = X[:, ::2]
        X[:, 4] = -X[:, 0]
    elif kind == "two_values":
        X[:, ::3] = rs.randint(0, 2, X[:, ::3].shape)
        g = np.sign(g)
        h[:] = 1.0
    elif kind == "long_tails":
        X = np.exp(4 * X).astype(np.float32)
        g[: n // 2] *= 1e-4
    elif kind == "l1":
        kw["l1_regularization"] = 2.0
    elif kind == "min_split_gain":
        kw["min_split_gain"] = 0.5
    elif kind == "no_l2":
        kw["l2_regularization"] = 0.0
    elif kind == "large_l2":
        kw["l2_regularization"] = 1e9
        g *= 1e9
    elif kind in ("huge", "tiny"):
        g *= 1e150 if kind == "huge" else 1e-70
        h *= 1e120 if kind == "huge" else 1e-65
    elif kind == "one_sign":
        g = np.abs(g)
    Xd, gd, hd = (torch.from_numpy(a).cuda() for a in (X, g, h))
    got = ops.build_tree(Xd, gd, hd, **kw)
    names = {"l1_regularization": "l1", "l2_regularization": "l2"}
    _assert_tree(got, orc.build_tree(X, g, h, **{names.get(k, k): v for k, v in kw.items()}))


# The best of a wave's candidates where many gains are equal: the order of ties is the oracle's. Copies of columns,
# columns of two values, long runs of empty bins; one wave per node and fewer lanes (more than 16 nodes).
@pytest.mark.parametrize("n,f,k,s,depth", [(20001, 40, 1, 256, 7), (20001, 130, 1, 64, 5), (12001, 20, 3, 300, 6)])
def test_ties_of_medium_sizes(n, f, k, s, depth):
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(f)
    X = rs.randn(n, f).astype(np.float32)
    X[:, 1::2] = X[:, ::2]
    X[:, ::5] = rs.randint(0, 2, X[:, ::5].shape)
    g, h = np.sign(rs.randn(n, k)), np.ones((n, k))
    kw = dict(max_depth=depth, split_samples=s, seed=4)
    got = ops.build_tree(*(torch.from_numpy(a).cuda() for a in (X, g, h)), **kw)
    _assert_tree(got, orc.build_tree(X, g, h, **kw))


# Rows of a level find their sides in runs of eight positions a thread (up to 2^20 rows, or 4 nodes) or in positions
# apart: ragged ends, slabs that end inside a run, nodes that change inside one, bins of one and of two bytes.
@pytest.mark.parametrize("n,s,depth", [(7, 8, 3), (2047, 64, 9), (2052, 300, 9), (6145, 256, 9), (20003, 400, 8),
                                       (1 << 20, 40, 5), ((1 << 20) + 5, 40, 5), ((1 << 20) + 2047, 300, 4)])
def test_sides_of_a_levels_rows(n, s, depth):
    import gpu_util as gu

    rs = np.random.RandomState(n)
    X = rs.randn(n, 6).astype(np.float32)
    g, h = rs.randn(n, 1), rs.rand(n, 1) + 0.1
    gr, cr = gu.both(X, g, h, levels=True, max_depth=depth, split_samples=s, seed=2)
    gu.assert_tree_parity(gr, cr, levels=True)


# The bin counts reach the host from a kernel up to 4096 features and by a copy beyond.
@pytest.mark.parametrize("f", [4095, 4096, 4097])
def test_bin_counts_for_the_host(f):
    import gpu_util as gu

    rs = np.random.RandomState(f)
    X = rs.randint(0, 9, (9000, f)).astype(np.float32)
    g, h = rs.randn(9000, 1), rs.rand(9000, 1) + 0.5
    gr, cr = gu.both(X, g, h, levels=True, max_depth=2, split_samples=8, seed=1)
    gu.assert_tree_parity(gr, cr, levels=True)


# The tile plan of a level: one node a thread (up to 256) and several, nodes without rows, tiles that end inside one.
@pytest.mark.parametrize("n,depth,hist_cache_bytes", [(3, 2, 0), (5000, 9, 0), (20001, 10, 0), (9001, 10, 200_000)])
def test_tile_plans(n, depth, hist_cache_bytes):
    import gpu_util as gu

    rs = np.random.RandomState(n)
    X = rs.randn(n, 4).astype(np.float32)
    g, h = rs.randn(n, 1), rs.rand(n, 1) + 0.1
    gr, cr = gu.both(X, g, h, levels=True, max_depth=depth, split_samples=33, seed=6, hist_cache_bytes=hist_cache_bytes)
    gu.assert_tree_parity(gr, cr, levels=True)


# groups of 33 to 64 features: 12, 13, 14 or 16 bins of a row per lane (one output: up to 56), and what lies beside; 100 is 52 and 48
@pytest.mark.parametrize("f,k,s,dtype", [(32, 1, 256, np.float32), (33, 1, 256, np.float32), (33, 2, 256, np.float64), (43, 1, 200, np.float32),
                                         (47, 3, 256, np.float32), (48, 1, 256, np.float32), (49, 1, 256, np.float32), (49, 3, 256, np.float64),
                                         (50, 1, 64, np.float64), (50, 2, 256, np.float32), (52, 1, 100, np.float32), (52, 5, 256, np.float32),
                                         (53, 1, 256, np.float32), (53, 2, 64, np.float32), (54, 3, 256, np.float64), (56, 1, 256, np.float32),
                                         (56, 2, 256, np.float32), (57, 1, 256, np.float32), (57, 2, 256, np.float32), (64, 1, 8, np.float32),
                                         (64, 2, 256, np.float32), (65, 2, 32, np.float32), (80, 1, 256, np.float32), (90, 2, 256, np.float32),
                                         (100, 1, 256, np.float32), (100, 3, 256, np.float32), (111, 2, 256, np.float32), (130, 1, 256, np.float32)])
# one gradient that fills the packed sums within a tile (every row is then added by itself), after one, or never
@pytest.mark.parametrize("share", [0.0, 1.0 / 1500.0, 0.5])
def test_bins_spread_over_the_lanes_of_a_row(f, k, s, dtype, share):
    import gpu_util as gu

    n = 7001
    rs = np.random.RandomState(f + k + s)
    X = rs.randn(n, f).astype(dtype)
    X[:, ::7] = np.floor(3 * X[:, ::7])
    g, h = rs.randn(n, k), rs.rand(n, k) + 0.5
    if share > 0:
        g[n // 3, k - 1] = 0.0
        g[n // 3, k - 1] = np.abs(g).sum() * share / (1.0 - share)
    gr, cr = gu.both(X, g, h, levels=True, max_depth=4, split_samples=s, seed=f)
    gu.assert_tree_parity(gr, cr, levels=True)
    assert (cr.feature != -1).sum() > 5


@pytest.mark.parametrize("kind", ["plain", "l1", "tiny", "huge", "signs", "zero_hessians"])
@pytest.mark.parametrize("n,f,k,s", [(3000, 7, 1, 100), (2500, 5, 3, 300), (20000, 3, 8, 64)])
def test_scanned_levels_in_32_bits(n, f, k, s, kind):
    """Running sums formed in their lower halves and quotients without the special cases of a division: penalties, scales at the ends of
    the exponents (the general division), grads of one sign whose sums reach 2^31, hessians of both signs and of zero, whose
    running sums are not positive and leave bins as they are: the oracle's histograms and gains bit for bit."""
    import gpu_util as gu

    rs = np.random.RandomState(n + k)
    X = rs.normal(size=(n, f)).astype(np.float32)
    X[:, 0] = rs.randint(0, 3, n)
    g, h = rs.normal(size=(n, k)), 0.01 + rs.rand(n, k)
    kw = {}
    if kind == "l1":
        kw = dict(l1_regularization=0.7)
    elif kind == "tiny":
        g, h = g * 1e-75, h * 1e-75
    elif kind == "huge":
        g, h = g * 1e75, h * 1e70
    elif kind == "signs":
        g, h = np.abs(g) * np.where(np.arange(k) % 2, 1, -1), rs.normal(size=(n, k))
        h[:, 0] = np.abs(h[:, 0]) + 0.5
    elif kind == "zero_hessians":
        h[rs.rand(n, k) < 0.6] = 0.0
        g = -np.abs(g)
    gr, cr = gu.both(X, g, h, max_depth=6, split_samples=s, seed=5, **kw)
    gu.assert_tree_parity(gr, cr)
    # and unobserved, by the builders for few and for medium rows where they take it
    from lbtree import ops
    got = ops.build_tree(*(torch.from_numpy(v).cuda() for v in (X, g, h)), max_depth=6, split_samples=s, seed=5, row_leaf=True, **kw)
    _assert_tree(got, cr)


@pytest.mark.parametrize("n,f,k,s,depth,kind", [
    (9001, 60, 1, 512, 12, "plain"),        # more nodes than a slab decides, at last
    (9001, 513, 2, 64, 11, "plain"),        # more candidates than a slab reads: a launch of its own
    (8200, 100, 3, 256, 10, "empty"),       # most nodes without rows
    (20479, 90, 1, 256, 11, "retired"),     # rows that stop early lie in front
    (20480, 80, 1, 300, 11, "zero"),
    (20481, 80, 2, 300, 10, "negative"),    # splits of nodes without rows: a launch of its own
])
def test_levels_of_the_general_builder_that_begin_in_one_launch(n, f, k, s, depth, kind):
    """Splits found where rows are classified, tiles planned and histograms cleared where they are scattered: equal to the observed build,
    whose histograms and levels the oracle's tests cover, in everything that both return."""
    import gpu_util as gu
    from lbtree import ops

    rs = np.random.RandomState(n + f)
    X = rs.randn(n, f).astype(np.float32)
    g, h = rs.randn(n, k), 0.1 + rs.random_sample((n, k))
    if kind == "empty":
        X = np.round(X)
        g = np.repeat((X[:, :1] > 1) * 5.0, k, axis=1)
    elif kind == "retired":
        g = np.where(X[:, :1] > 0, np.sign(X[:, :1]), g)
    elif kind == "zero":
        h[rs.rand(n, k) < 0.3] = 0.0
    elif kind == "negative":
        h[rs.rand(n, k) < 0.3] *= -0.5
    Xd, gd, hd = (torch.from_numpy(a).cuda() for a in (X, g, h))
    kw = dict(max_depth=depth, split_samples=s, seed=2, row_leaf=True, hist_cache_bytes=10 ** 9)
    want = ops.build_tree(Xd, gd, hd, taps=True, **kw)
    got = ops.build_tree(Xd, gd, hd, **kw)
    for name in ("leaf_value", "feature", "split_value", "gain", "hessian", "row_leaf"):
        assert torch.equal(getattr(got, name), getattr(want, name)), name
    gu.check_row_leaf(got, X)
    assert _takes_the_general_builder(lambda: ops.build_tree(Xd, gd, hd, **kw))


def _takes_the_general_builder(build):
    """The other builders round the gradients in a launch that does more, and report none of this class."""
    from lbtree import _lib

    _lib.profile_reset()
    _lib.profile_enable(1)
    try:
        build()
        return _lib.profile_get()["quantise"]["launches"] == 1
    finally:
        _lib.profile_enable(0)
        _lib.profile_reset()


def test_which_builder_a_profile_tells():
    from lbtree import ops

    for n, f, depth, general in ((1000, 5, 4, False), (9001, 9, 6, False), (9001, 50, 11, True)):
        X, g = torch.rand((n, f), device="cuda"), torch.rand((n, 1), device="cuda", dtype=torch.float64)
        assert _takes_the_general_builder(lambda: ops.build_tree(X, g - 0.5, g + 0.1, max_depth=depth, split_samples=64, seed=1)) == general


@pytest.mark.parametrize("n,f,k,s,depth,kind", [
    (9000, 64, 1, 1, 6, "plain"),            # one bin, one tile
    (9001, 65, 1, 64, 6, "plain"),           # a full tile; workgroups of which some waves have nothing left
    (9001, 31, 1, 65, 9, "zeros"),           # one bin in the second tile
    (12000, 131, 1, 256, 5, "excluded"),
    (8200, 33, 2, 300, 7, "l1"),             # two-byte bins, a tile that is not full
    (70000, 40, 3, 129, 7, "zeros"),         # ranges of rows past those asked for ahead
    (9001, 128, 16, 32, 5, "excluded"),      # the most outputs
    (9001, 130, 8, 100, 5, "zeros"),         # tiles and many outputs in turn
    (8193, 130, 1, 2048, 5, "l1"),
    (200000, 16, 5, 257, 6, "plain"),        # by workgroups: 16 ranges and more, a second tile of bins, several outputs
])
def test_scans_of_wide_levels(n, f, k, s, depth, kind):
    """Scans of a wave for a pair of siblings and a feature, with their neighbours: tiles and outputs in turn, loads one item ahead."""
    import gpu_util as gu
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(n + f)
    X = rs.randn(n, f).astype(np.float32)
    X[:, 1] = np.round(X[:, 1])
    g = rs.randn(n, k) + np.sin(2 * X[:, :1]) + X[:, 2:3] * X[:, 3:4]
    h = rs.rand(n, k) + 0.1
    if kind == "zeros":
        h[rs.rand(n, k) < 0.4] = 0.0
    mask = rs.rand(f) < 0.6 if kind == "excluded" else None
    kw = dict(l1=0.05, l2=0.5, min_split_gain=1e-3) if kind == "l1" else {}
    kw2 = dict(l1_regularization=0.05, l2_regularization=0.5, min_split_gain=1e-3) if kw else {}
    cr = orc.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=n, feature_set=mask, **kw)
    got = ops.build_tree(X, g, h, max_depth=depth, split_samples=s, seed=n, feature_set=mask, row_leaf=True, **kw2)
    _assert_tree(got, cr)
    gu.check_row_leaf(got, X)


@pytest.mark.parametrize("n,f,k,s,dtype", [(1, 1, 1, 1, np.float32), (4096, 7, 1, 2, np.float64), (4097, 9, 1, 2048, np.float64), (1365, 8, 3, 257, np.float32),
                                           (1366, 65, 3, 256, np.float32), (30000, 300, 1, 5, np.float32), (9000, 900, 2, 64, np.float32)])
def test_a_tree_of_the_general_builder_begins_in_two_launches(n, f, k, s, dtype):
    """Samples, chunks of the absolute sums (whole, one entry more) and the state side by side, few and many tables of the host: proposals,
    rounded gradients and the tree are the oracle's."""
    import gpu_util as gu

    rs = np.random.RandomState(n + f)
    X = np.round(rs.randn(n, f), 2).astype(dtype)
    g, h = rs.randn(n, k), rs.rand(n, k) + 0.5
    gr, cr = gu.both(X, g, h, levels=True, max_depth=3, split_samples=s, seed=n)
    gu.assert_tree_parity(gr, cr, levels=True)
    assert np.array_equal(gu.cpu(gr.row_pointers), cr.row_pointers) and np.array_equal(gu.cpu(gr.proposals), cr.proposals)
    assert np.array_equal(gu.cpu(gr.quantised), cr.quantised)


@pytest.mark.parametrize("s", [1, 2, 7, 8, 9, 33, 63, 64, 65, 128, 255, 256, 257, 511, 512, 513, 1025])
@pytest.mark.parametrize("n,dtype", [(700, np.float32), (900, np.float64), (9001, np.float32), (9001, np.float64)])
def test_samples_sorted_by_counting(n, dtype, s):
    """Split proposals of the builders for few and for medium rows, of columns with ties, zeros of either sign, NaN, infinities, one value: the tree is the
    general builder's, whose proposals a network sorts."""
    from lbtree import ops

    rs = np.random.RandomState(s + n)
    X = np.empty((n, 9), dtype)
    X[:, 0] = rs.randn(n)
    X[:, 1] = rs.randint(-2, 3, n)
    X[:, 2] = np.where(rs.rand(n) < 0.5, 0.0, -0.0) * 1.0
    X[:, 3] = np.where(rs.rand(n) < 0.3, -0.0, rs.randn(n))
    X[:, 4] = np.where(rs.rand(n) < 0.3, 0.0, rs.randn(n))
    X[:, 5] = 3.0
    X[:, 6] = np.where(rs.rand(n) < 0.1, np.inf, np.where(rs.rand(n) < 0.1, -np.inf, rs.randn(n)))
    X[:, 7] = rs.randint(0, 300, n)
    X[:, 8] = np.where(rs.rand(n) < 0.2, np.nan, np.round(rs.randn(n)))
    if s > 1:
        X[:, 1] = np.where(rs.rand(n) < 0.5, -X[:, 1], X[:, 1])
    g, h = rs.randn(n, 1) + np.nan_to_num(X[:, :1]) + (X[:, 7:8] > 150) * X[:, 1:2], rs.rand(n, 1) + 0.1
    Xd, gd, hd = (torch.from_numpy(a).cuda() for a in (X, g, h))
    mask = torch.ones(9, dtype=torch.bool)
    mask[8] = False  # (no split on the column with NaN: a traversal sends it to the right)
    kw = dict(max_depth=4, split_samples=s, seed=s, feature_set=mask)
    want = ops.build_tree(Xd, gd, hd, taps=True, **kw)
    got = ops.build_tree(Xd, gd, hd, **kw)
    for name in ("feature", "split_value", "gain", "leaf_value", "hessian"):
        assert torch.equal(getattr(got, name), getattr(want, name)), name


@pytest.mark.parametrize("n", [1, 4096, 4097, 4096 * 4096, 4096 * 4096 + 1])
def test_scales_of_the_absolute_sums(n):
    """One, two and three levels of the fixed-order sum of |g| and |h|: the scales have the bits of the same additions on the host."""
    from lbtree import ops

    def level(a):
        chunks = -(-len(a) // 4096)
        a = np.concatenate([a, np.zeros(chunks * 4096 - len(a))]).reshape(chunks, 16, 256)
        lanes = np.zeros((chunks, 256))
        for j in range(16):  # a lane's entries in their order (one that is missing adds zero)
            lanes = lanes + a[:, j]
        while lanes.shape[1] > 1:
            half = lanes.shape[1] // 2
            lanes = lanes[:, :half] + lanes[:, half:]
        return lanes[:, 0]

    gen = torch.Generator(device="cuda").manual_seed(n % 1000)
    g = torch.randn((n, 1), generator=gen, device="cuda", dtype=torch.float64)
    h = torch.rand((n, 1), generator=gen, device="cuda", dtype=torch.float64)
    q, sums, scales = ops.quantise_gradients(g, h, 3)
    for at, a in ((0, g), (1, h)):
        s = level(np.abs(a.cpu().numpy().reshape(-1)))
        while len(s) > 1:
            s = level(s)
        assert scales[at].item() == 2147483647.0 / s[0] and scales[2 + at].item() == 1.0 / scales[at].item()
    assert torch.equal(sums, q.to(torch.int64).sum(dim=0))


@pytest.mark.parametrize("f,s", [(2047, 3), (2048, 2), (2049, 5), (4097, 33), (10_001, 2)])
def test_proposals_of_many_features_are_placed(f, s):
    """One feature a workgroup, and runs of several: row pointers and proposals are the oracle's."""
    import gpu_util as gu
    import oracle_lib as orc
    from lbtree import ops

    rs = np.random.RandomState(f)
    X = np.round(rs.randn(40, f) * 2).astype(np.float32)
    props, rp = ops.select_split_samples(torch.from_numpy(X).cuda(), s, 7)
    want_props, want_rp = orc.split_proposals(X, 7, s)
    assert np.array_equal(gu.cpu(rp), want_rp) and np.array_equal(gu.cpu(props), want_props)


def test_placing_proposals_does_not_grow_with_the_square_of_the_features():
    """8 times the features may take 16 times as long: 32,768 and 262,144 of them 41 and 278 us (6.8 times), 165 and 6974 (42 times) with a sum
    over all features in front for each."""
    from lbtree import _lib, ops

    def best_us(f):
        X = torch.zeros((4, f), device="cuda")
        ws = torch.empty(_lib.lib.lbt_select_split_samples_workspace_bytes(f, 2, 0), dtype=torch.uint8, device="cuda")
        props, rp = torch.empty(2 * f, device="cuda"), torch.empty(f + 1, dtype=torch.int32, device="cuda")
        best = float("inf")
        for _ in range(6):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            for _ in range(4):
                _lib.check(_lib.lib.lbt_select_split_samples(ops._stream(), X.data_ptr(), 0, 0, 4, f, 2, 3, 4, props.data_ptr(), rp.data_ptr(),
                                                             ws.data_ptr(), ws.numel()))
            end.record()
            end.synchronize()
            best = min(best, begin.elapsed_time(end) / 4 * 1e3)
        return best

    few, many = best_us(32_768), best_us(262_144)
    assert many < 16 * few, (few, many)
