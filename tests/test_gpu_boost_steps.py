"""What a fit and a prediction do either side of the trees, against the operators they stand for (legateboost.py:189-224,
507-529, objectives.py:131-147 and :489-531)."""
import ctypes as C
import math

import numpy as np
import pytest
import torch


def test_calls_check_their_arguments():
    from lbtree import _lib

    lib, one, two = _lib.lib, C.c_void_p(16), C.c_void_p(32)
    assert lib.lbt_class_probabilities(None, one, one, 10, 0, two) == -1
    assert lib.lbt_class_probabilities(None, one, one, 10, 1, one) == -1
    assert lib.lbt_class_probabilities(None, one, one, 10, 1, C.c_void_p(40)) == -1
    assert b"aligned" in lib.lbt_last_error()
    assert lib.lbt_class_probabilities(None, None, None, 0, 3, None) == 0
    assert lib.lbt_weighted_mean_workspace_bytes(256) > 0 and lib.lbt_weighted_mean_workspace_bytes(257) == 0
    assert lib.lbt_weighted_mean(None, one, None, 0, 1, one, one, 1 << 20) == -1
    assert lib.lbt_weighted_mean(None, one, None, 10, 1, one, one, 8) == -3
    assert lib.lbt_label_counts(None, None, 10, one) == -1
    assert lib.lbt_label_priors(None, one, 10, 257, one) == -1
    assert lib.lbt_keep_rows(None, one, 0.5, 10, 1, two, two) == -1
    assert lib.lbt_keep_rows(None, None, 0.5, 0, 1, None, None) == 0


@pytest.mark.parametrize("init,out,refused", [(512, 512, True), (512 + 8 * 29, 512, True), (512, 512 + 8 * 2, True),
                                              (512 - 8 * 3, 512, False), (512 + 8 * 30, 512, False)])
def test_initial_predictions_may_not_lie_in_the_output(init, out, refused):
    """10 rows of 3 outputs. What is not refused here goes on to the next check, a tree without nodes."""
    from lbtree import _lib

    ptr, nodes = (C.c_void_p * 1)(16), (C.c_int32 * 1)(0)
    rc = _lib.lib.lbt_predict_from(None, C.c_void_p(16), _lib.LBT_F32, 10, 4, 1, ptr, ptr, ptr, nodes, 3, C.c_void_p(init),
                                   C.c_void_p(out), None, 0)
    assert rc == -1
    assert (b"overlap" in _lib.lib.lbt_last_error()) == refused


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(1, 1), (257, 1), (1, 2), (255, 3), (513, 8), (300, 10), (1000, 16), (70, 7), (40, 19), (3, 300),
                                 (255, 9), (131, 12), (77, 13), (130, 24), (65, 25), (9, 33), (33, 48), (17, 49), (5, 64), (7, 65),
                                 (9, 128), (5, 129), (3, 256), (5, 257), (2, 1000)])
def test_class_probabilities(n, k):
    """exp and the sums of up to 1000 terms round differently from torch's: (k + 8) 2^-52 of each probability."""
    from lbtree import ops

    gen = torch.Generator(device="cuda").manual_seed(n + k)
    raw = 4 * torch.randn((n, k), generator=gen, device="cuda", dtype=torch.float64)
    raw[0] = 600.0
    raw[-1, 0] = -600.0
    init = torch.randn(k, generator=gen, device="cuda", dtype=torch.float64)
    v = init + raw
    if k == 1:
        p = 1.0 / (1.0 + torch.exp(-v))
        want = torch.cat([1.0 - p, p], dim=1)
    else:
        want = torch.softmax(v, dim=1)
    got = ops.class_probabilities(raw, init)
    assert got.shape == want.shape
    # an exponent rounded to 2^-53 of up to 1200 is off by 2^-43
    assert torch.allclose(got, want, rtol=(k + 8) * 2.0 ** -52, atol=2.0 ** -52)
    bad = raw.clone()
    bad[n // 2, k - 1] = float("nan")
    assert torch.equal(torch.isnan(ops.class_probabilities(bad, init)).all(dim=1),
                       torch.arange(n, device="cuda") == n // 2)


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(1, 1), (1023, 1), (1000003, 1), (5, 3), (40000, 7), (33, 256), (700, 130)])
@pytest.mark.parametrize("weighted", [False, True])
def test_weighted_mean(n, k, weighted):
    """Against exactly rounded sums: a thread adds up to n / 2^18 + 1 terms and a tree joins the threads."""
    from lbtree import ops

    rs = np.random.RandomState(n + k)
    y, w = 1.0 + rs.rand(n, k), 0.5 + rs.rand(n) if weighted else None
    got = ops.weighted_mean(torch.from_numpy(y).cuda(), None if w is None else torch.from_numpy(w).cuda()).cpu().numpy()
    ones = np.ones(n) if w is None else w
    for c in range(0, k, max(1, k // 5)):
        want = math.fsum(y[:, c] * ones) / math.fsum(ones)
        assert abs(got[c] - want) <= (n / 2.0 ** 18 + 600) * 2.0 ** -53 * want


@pytest.mark.gpu
@pytest.mark.parametrize("n,classes", [(1, 1), (1025, 2), (100003, 2), (5000, 8), (3000, 256)])
def test_labels_and_priors(n, classes):
    from lbtree import ops

    y = np.random.RandomState(n).randint(0, classes, n).astype(np.float64)
    stats = ops.label_counts(torch.from_numpy(y).cuda())
    count = np.bincount(y.astype(int), minlength=256)
    assert stats.tolist() == [0, int(y.max()), 0] + count.tolist()
    k = classes if classes > 2 else 1
    with np.errstate(divide="ignore"):
        share = count / n
        want = -np.log(1 / share[1:2] - 1) if k == 1 else np.log(share[:k])
    assert np.allclose(ops.label_priors(stats, n, k).cpu().numpy(), want, rtol=4 * 2.0 ** -52, atol=0)
    for value, at in ((0.5, 0), (-1.0, 0), (float("nan"), 0), (256.0, 2), (float("inf"), 2)):
        bad = y.copy()
        bad[n // 2] = value
        got = ops.label_counts(torch.from_numpy(bad).cuda()).tolist()
        assert [got[0], got[2]] == [int(at == 0), int(at == 2)]


@pytest.mark.gpu
def test_labels_beyond_the_counted_ones_still_fit():
    import lbtree as lb

    gen = torch.Generator(device="cuda").manual_seed(1)
    X = torch.rand((600, 3), generator=gen, device="cuda")
    y = torch.arange(600, device="cuda", dtype=torch.float64) % 300
    model = lb.LBClassifier(n_estimators=1, base_models=(lb.models.Tree(max_depth=2),), random_state=0).fit(X, y)
    assert model.predict_proba(X).shape == (600, 300)
    assert torch.allclose(model.model_init_, torch.full((300,), math.log(1 / 300), dtype=torch.float64, device="cuda"))
    with pytest.raises(ValueError, match="whole numbers"):
        lb.LBClassifier(n_estimators=1).fit(X, y - 0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(1, 1), (257, 1), (300, 5)])
def test_keep_rows(n, k):
    from lbtree import ops

    gen = torch.Generator(device="cuda").manual_seed(n)
    g, h, draw = (torch.randn(s, generator=gen, device="cuda", dtype=torch.float64) for s in ((n, k), (n, k), (n,)))
    mask = (draw < 0.3).to(torch.float64)[:, None]
    want = g * mask, h * mask
    ops.keep_rows(draw, 0.3, g, h)
    assert torch.equal(g, want[0]) and torch.equal(h, want[1])


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n_trees,k", [(1, 17, 1), (300, 105, 1), (300, 104, 3), (4096, 30, 1), (4097, 209, 1), (50000, 60, 1), (20, 3, 2),
                                            (33, 700, 1), (100, 0, 2)])
def test_predict_from_an_initial_prediction(rows, n_trees, k):
    """init + the sums, by the kernel for few rows and behind the others; trees either side of what one launch packs, batches of
    more than its first ones: bit for bit the sum of the two."""
    from lbtree import ops

    rs = np.random.RandomState(rows + n_trees)
    f = 12
    trees = []
    for t in range(n_trees):
        m, inner = 2 ** (4 + t % 5) - 1, 2 ** (3 + t % 5) - 1
        feat = -np.ones(m, np.int32)
        feat[:inner] = rs.randint(0, f, inner)
        trees.append(tuple(ops.as_device(a) for a in (rs.randn(m, k), feat, rs.rand(m))))
    init = ops.as_device(rs.randn(k))
    for dtype in (np.float32, np.float64):
        X = ops.as_device(rs.rand(rows, f).astype(dtype))
        want = ops.predict(X, trees, k, tiled=False)
        assert torch.equal(ops.predict(X, trees, k), want)
        assert torch.equal(ops.predict(X, trees, k, init=init), init + want)
        assert torch.equal(ops.predict(X, trees, k, tiled=False, init=init), init + want)
        if n_trees:
            packed = ops.PackedEnsemble(trees, k, f, X.dtype)
            assert torch.equal(packed.predict(X), want)


@pytest.mark.gpu
@pytest.mark.parametrize("n,k", [(1, 1), (5000, 1), (4099, 3), (4096, 2)])
@pytest.mark.parametrize("off", [0, 1])
def test_predict_from_into_an_output_that_begins_off_16_bytes(n, k, off):
    """The initial prediction is added two entries at a time where the output lies on 16 bytes: odd counts, and outputs that do not."""
    from lbtree import _lib, ops

    rs = np.random.RandomState(n + k)
    X = ops.as_device(rs.rand(n, 5))
    tree = tuple(ops.as_device(a) for a in (rs.randn(7, k), np.array([0, 1, 2, -1, -1, -1, -1], np.int32), rs.rand(7)))
    init = ops.as_device(rs.randn(k))
    room = torch.full((n * k + 3,), 7.0, dtype=torch.float64, device="cuda")
    ptrs = [(C.c_void_p * 1)(a.data_ptr()) for a in tree]
    _lib.check(_lib.lib.lbt_predict_from(ops._stream(), X.data_ptr(), _lib.LBT_F64, n, 5, 1, *ptrs, (C.c_int32 * 1)(7), k,
                                         init.data_ptr(), room.data_ptr() + 8 * off, None, 0))
    got = room[off:off + n * k].reshape(n, k)
    assert torch.equal(got, init + ops.predict(X, [tree], k, tiled=False))
    assert bool((room[off + n * k:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("task", ["regression", "classification"])
def test_fit_with_the_gradient_passes_sums(task):
    """From four million rows on the gradient pass leaves the quantiser's sums: the same model as tree by tree without them."""
    import lbtree as lb

    gen = torch.Generator(device="cuda").manual_seed(4)
    n = 4000003
    X = torch.rand((n, 4), generator=gen, device="cuda")
    y = X[:, 0].to(torch.float64) + 0.1 * torch.randn(n, generator=gen, device="cuda", dtype=torch.float64)
    kind = lb.LBRegressor if task == "regression" else lb.LBClassifier
    y = y if task == "regression" else (y > 0.6).to(torch.float64)

    class Stepwise(kind):
        def _get_weighted_gradient(self, *args):
            return super()._get_weighted_gradient(*args)

    models = [k(n_estimators=3, base_models=(lb.models.Tree(max_depth=5),), learning_rate=0.3, random_state=2).fit(X, y)
              for k in (kind, Stepwise)]
    assert torch.equal(models[0]._train_pred, models[1]._train_pred)
    for a, b in zip(*models):
        assert all(torch.equal(getattr(a, name), getattr(b, name)) for name in ("feature", "split_value", "leaf_value", "gain", "hessian"))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [5000, 4000000])
def test_fits_and_updates_call_a_replaced_gradient_step(monkeypatch, rows):
    """Replaced on the class that defines it, not on a subclass: the fits that form the gradients themselves must not pass it by."""
    import lbtree as lb
    from lbtree.boosting import LBBase

    seen, own = [], LBBase._get_weighted_gradient

    def step(self, y, pred, sample_weight, learning_rate):
        seen.append(tuple(sample_weight.shape))
        return own(self, y, pred, sample_weight, learning_rate)

    gen = torch.Generator(device="cuda").manual_seed(3)
    X = torch.rand((rows, 4), generator=gen, device="cuda")
    model = lb.LBRegressor(n_estimators=2, base_models=(lb.models.Tree(max_depth=2, split_samples=16),), random_state=1)
    monkeypatch.setattr(LBBase, "_get_weighted_gradient", step)
    model.fit(X, X[:, 0].double())
    assert seen == 2 * [(rows,)]
    model.update(X, X[:, 1].double())
    assert seen == 4 * [(rows,)]


@pytest.mark.gpu
@pytest.mark.parametrize("owner,name", [("LBBase", "_predict"), ("LogLossObjective", "transform"), ("Tree", "batch_predict")])
def test_predictions_call_what_has_been_replaced(monkeypatch, owner, name):
    import lbtree as lb
    from lbtree import boosting

    gen = torch.Generator(device="cuda").manual_seed(4)
    X = torch.rand((300, 4), generator=gen, device="cuda")
    model = lb.LBClassifier(n_estimators=2, base_models=(lb.models.Tree(max_depth=2, split_samples=16),), random_state=1)
    model.fit(X, (X[:, 0] > 0.5).double())
    want = model.predict_proba(X)
    cls, calls = getattr(boosting, owner), []
    own = getattr(cls, name)

    def replaced(*args):
        calls.append(name)
        return own(*args)

    monkeypatch.setattr(cls, name, staticmethod(replaced) if name == "batch_predict" else replaced)
    assert torch.allclose(model.predict_proba(X), want, rtol=0, atol=1e-15) and len(calls) == 1
    model._predict(X)
    assert len(calls) == (1 if name == "transform" else 2)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [2, 3, 4, 5, 8, 9, 10, 16, 33, 64, 127, 128, 129])
@pytest.mark.parametrize("weighted", [False, True])
def test_softmax_gradients_by_entry_and_by_row(k, weighted):
    """Rows that straddle stages and chunks, with and without the chunk sums (which ask for a thread per entry at any size): the same
    bits, torch's softmax to rounding, and the sums in the quantiser's order."""
    from lbtree import ops

    torch.manual_seed(k)
    for n in (1, 2, 2048 // k + 1, 4096 // k, 12345 // k + 2, 40000 // k + 1):
        pred = torch.randn(n, k, dtype=torch.float64).cuda() * 4
        y = torch.randint(0, k, (n,)).double().cuda()
        w = torch.rand(n, dtype=torch.float64).cuda() if weighted else None
        g, h = ops.weighted_gradient("log_loss", y, pred, w, 0.5)
        gs, hs, sums = ops.weighted_gradient("log_loss", y, pred, w, 0.5, sums=True)
        assert torch.equal(g, gs) and torch.equal(h, hs)
        q = torch.softmax(pred, dim=1)
        weight = w[:, None] if weighted else 1.0
        # a quotient: an argument within 1 ulp of up to 32, k additions, exponentials and the division to an ulp each
        bound = (k + 80) * 2.0 ** -52
        assert ((gs - 0.5 * weight * (q - torch.nn.functional.one_hot(y.long(), k))).abs() <= bound).all()
        assert ((hs - (weight * q * (1 - q)).clamp(min=1e-8)).abs() <= bound).all()  # (hessians are at least 1e-8)
        for a, got in ((gs, sums[0]), (hs, sums[1])):
            flat = torch.zeros(got.numel() * 4096, dtype=torch.float64)
            flat[: n * k] = a.cpu().reshape(-1).abs()
            lanes = torch.zeros(got.numel(), 256, dtype=torch.float64)
            for part in flat.reshape(-1, 16, 256).unbind(1):
                lanes = lanes + part
            while lanes.shape[1] > 1:
                lanes = lanes[:, : lanes.shape[1] // 2] + lanes[:, lanes.shape[1] // 2:]
            assert torch.equal(lanes[:, 0], got.cpu())


@pytest.mark.gpu
def test_softmax_gradients_of_many_entries():
    """Enough entries for a thread each without the sums too, in rows that a thread holds otherwise."""
    from lbtree import ops

    torch.manual_seed(1)
    n, k = 800_003, 5
    pred = torch.randn(n, k, dtype=torch.float64).cuda()
    y = torch.randint(0, k, (n,)).double().cuda()
    g, h = ops.weighted_gradient("log_loss", y, pred, None, 1.0)
    some = 700_001  # fewer entries: a thread per row
    g1, h1 = ops.weighted_gradient("log_loss", y[:some].contiguous(), pred[:some].contiguous(), None, 1.0)
    assert torch.equal(g[:some], g1) and torch.equal(h[:some], h1)
    g2, h2 = ops.weighted_gradient("log_loss", y[some:].contiguous(), pred[some:].contiguous(), None, 1.0)
    assert torch.equal(g[some:], g2) and torch.equal(h[some:], h2)


@pytest.mark.gpu
@pytest.mark.parametrize("task,n,k,asked", [("classes", 66_000, 128, True), ("classes", 66_000, 129, False), ("values", 66_000, 129, True),
                                            ("classes", 60_000, 128, False)])
def test_which_fits_ask_for_the_gradient_passes_sums(monkeypatch, task, n, k, asked):
    """Eight million entries or more, and of a softmax rows of up to 128 outputs: beyond, the pass with the sums costs a fit of 1000
    classes more than the trees do."""
    import lbtree as lb
    from lbtree import ops

    own, seen = ops.weighted_gradient, []

    def watched(*args, sums=False, **kw):
        seen.append(sums)
        return own(*args, sums=sums, **kw)

    monkeypatch.setattr(ops, "weighted_gradient", watched)
    torch.manual_seed(0)
    X = torch.rand(n, 3).cuda()
    tree = lb.models.Tree(max_depth=2, split_samples=8)
    if task == "classes":
        y = (torch.arange(n) % k).double().cuda()
        lb.LBClassifier(n_estimators=1, base_models=(tree,), random_state=1).fit(X, y)
    else:
        lb.LBRegressor(n_estimators=1, base_models=(tree,), random_state=1).fit(X, torch.rand(n, k, dtype=torch.float64).cuda())
    assert seen == [asked]


@pytest.mark.gpu
@pytest.mark.parametrize("n,f,k,dtype,kind", [
    (1000, 7, 1, torch.float32, "plain"), (1000, 7, 3, torch.float64, "plain"), (999, 5, 1, torch.float32, "strided"),
    (999, 5, 2, torch.float64, "single_gradients"), (500, 4, 1, torch.float32, "on_the_host"), (9000, 9, 1, torch.float32, "mask"),
    (300, 3, 1, torch.float32, "vector_targets"), (1, 1, 1, torch.float64, "plain"),
])
def test_a_round_in_native_code_is_the_one_in_python(n, f, k, dtype, kind, monkeypatch):
    """Gradient, tree and prediction update through lbtree._host, and for what that does not take through Python: the same bits."""
    from lbtree import ops

    gen = torch.Generator(device="cuda").manual_seed(n + k)
    X = torch.randn((n, f), generator=gen, device="cuda", dtype=dtype)
    y = torch.randn((n, k), generator=gen, device="cuda", dtype=torch.float64)
    pred = torch.randn((n, k), generator=gen, device="cuda", dtype=torch.float64)
    w = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)
    mask = None
    if kind == "strided":
        X, y = X.t().contiguous().t(), y.t().contiguous().t()
    elif kind == "single_gradients":
        y = y.to(torch.float32)
    elif kind == "on_the_host":
        X = X.cpu().numpy()
    elif kind == "vector_targets":
        y = y.reshape(-1)
    elif kind == "mask":
        mask = ops.feature_mask(np.arange(f) % 3 != 1, "cuda")
        assert mask.tolist() == [int(i % 3 != 1) for i in range(f)]
    out = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(ops, "_NATIVE", None)
        p = pred.clone()
        g, h = ops.weighted_gradient("squared_error", y, p, w, 0.1)
        g2 = g.to(torch.float32) if kind == "single_gradients" else g
        r = ops.build_tree(X, g2, h, max_depth=5, split_samples=64, seed=4, feature_set=mask, row_leaf=True, wait=False,
                           l2_regularization=np.float32(1.0))
        assert ops.add_leaf_values(p, r.leaf_value, r.row_leaf) is p
        out.append((g, h, r.leaf_value, r.feature, r.split_value, r.gain, r.hessian, r.row_leaf, p))
    for a, b in zip(*out):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.gpu
def test_a_refused_round_is_refused_as_before(monkeypatch):
    from lbtree import _lib, ops

    X = torch.zeros((10, 2), device="cuda")
    g = torch.ones((10, 1), device="cuda", dtype=torch.float64)
    for bad in (dict(max_depth=-1), dict(split_samples=0), dict(split_samples=4096), dict(max_depth=3.5)):
        kw = dict(max_depth=3, split_samples=16, seed=1, wait=False)
        kw.update(bad)
        said = []
        for native in (True, False):
            with monkeypatch.context() as m:
                if not native:
                    m.setattr(ops, "_NATIVE", None)
                with pytest.raises(Exception) as e:
                    ops.build_tree(X, g, g, **kw)
                said.append((type(e.value), str(e.value)))
        assert said[0] == said[1], bad
    with pytest.raises(_lib.LbtError):
        ops.build_tree(X, g[:5], g, max_depth=2, split_samples=16, seed=1, wait=False)
    with pytest.raises(_lib.LbtError):
        ops.add_leaf_values(g, g[:3].reshape(1, 3), torch.zeros(10, dtype=torch.int32, device="cuda"))


def test_a_plain_tree_is_copied_by_its_numbers():
    from lbtree import boosting
    from lbtree.models import Tree

    class Own(Tree):
        pass

    plain = Tree(max_depth=3)
    copied = boosting._copy_of(plain)
    assert type(copied) is Tree and vars(copied) == vars(plain) and copied is not plain
    listed = Tree(max_depth=3)
    listed.note = [1]
    copied = boosting._copy_of(listed)
    assert copied.note == [1] and copied.note is not listed.note
    assert type(boosting._copy_of(Own(max_depth=2))) is Own



@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 256, 257, 4096, 4097, 70_000])
@pytest.mark.parametrize("objective,k", [("squared_error", 1), ("squared_error", 3), ("log_loss", 1), ("log_loss", 4)])
@pytest.mark.parametrize("weighted,sums,native", [(False, False, True), (True, True, True), (True, False, False)])
def test_the_next_gradient_is_the_two_calls(n, objective, k, weighted, sums, native, monkeypatch):
    """Leaf values and gradients in one call: the bits of lbt_add_leaf_values and lbt_weighted_gradient(_sums); a row of no leaf keeps its
    prediction."""
    from lbtree import ops

    gen = torch.Generator(device="cuda").manual_seed(n + k)
    double = dict(device="cuda", dtype=torch.float64, generator=gen)
    pred, leaf = torch.randn((n, k), **double), torch.randn((31, k), **double)
    rows = torch.randint(0, 31, (n,), device="cuda", dtype=torch.int32, generator=gen)
    rows[n // 2] = -1 if n % 2 else 31
    labels = objective == "log_loss" and k > 1
    y = torch.randint(0, max(k, 2), (n, 1 if labels else k), device="cuda", generator=gen).double()
    w = torch.rand(n, **double) if weighted else None
    if not native:
        monkeypatch.setattr(ops, "_NATIVE", None)
    want = ops.add_leaf_values(pred.clone(), leaf, rows)
    told = ops.weighted_gradient(objective, y, want, w, 0.3, sums=sums)
    got, g, h = pred.clone(), torch.zeros_like(pred), torch.zeros_like(pred)
    part = torch.zeros_like(told[2]) if sums else None
    ops.next_gradient(objective, leaf, rows, got, y, w, 0.3, g, h, part)
    assert torch.equal(got, want) and torch.equal(g, told[0]) and torch.equal(h, told[1])
    assert not sums or torch.equal(part, told[2])
    assert torch.equal(got[n // 2], pred[n // 2])


@pytest.mark.gpu
@pytest.mark.parametrize("task", ["values", "two", "classes"])
def test_rounds_in_one_pass_are_the_rounds_step_by_step(monkeypatch, task):
    """Whose next gradients are formed with the prediction update, and whose are not: trees of another kind in between, a sample of the
    rows, a method replaced."""
    import lbtree as lb
    from lbtree import boosting, ops

    class OwnTree(lb.models.Tree):
        def fit_update_predictions(self, X, g, h, pred):
            return super().fit_update_predictions(X, g, h, pred)

    X = torch.randn((3000, 6), generator=torch.Generator().manual_seed(3)).cuda()
    y = {"values": X[:, 0] * 2 + X[:, 1], "two": (X[:, 0] > 0), "classes": (X[:, 0] * 2).round().clamp(0, 3)}[task].double()
    estimator = lb.LBRegressor if task == "values" else lb.LBClassifier
    calls = []
    own_step = ops.next_gradient
    monkeypatch.setattr(ops, "next_gradient", lambda *a, **kw: (calls.append(1), own_step(*a, **kw))[1])

    def fit(own, **kw):
        base = tuple((OwnTree if o else lb.models.Tree)(max_depth=4, split_samples=32) for o in own)
        del calls[:]
        m = estimator(n_estimators=5, base_models=base, random_state=4, **kw).fit(X, y)
        return [t.leaf_value for t in m] + [m._train_pred], len(calls)

    want, n = fit([True])
    assert n == 0
    for own, expected in (([False], 4), ([False, True], 0), ([False, False, True], 2)):
        got, n = fit(own)
        assert n == expected
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert fit([False], subsample=0.5)[1] == 0
    monkeypatch.setattr(boosting.LBBase, "_get_weighted_gradient", lambda *a: boosting._DEFINED[boosting.LBBase]["_get_weighted_gradient"](*a))
    got, n = fit([False])
    assert n == 0 and all(torch.equal(a, b) for a, b in zip(got, want))


def test_the_next_gradient_checks_its_arguments():
    from lbtree import _lib

    call, one, two, three, four = _lib.lib.lbt_next_gradient, *(C.c_void_p(v) for v in (1 << 20, 2 << 20, 3 << 20, 4 << 20))
    assert call(None, 7, one, 3, one, two, one, None, 0.1, 10, 1, three, four, None) == -1
    assert call(None, 0, None, 3, one, two, one, None, 0.1, 10, 1, three, four, None) == -1
    assert call(None, 0, one, 0, one, two, one, None, 0.1, 10, 1, three, four, None) == -1
    assert call(None, 0, two, 3, one, two, one, None, 0.1, 10, 1, three, four, None) == -1
    assert call(None, 0, one, 3, one, two, one, None, 0.1, 10, 1, two, four, None) == -1
    assert call(None, 0, one, 3, one, two, one, None, 0.1, 10, 1, three, four, C.c_void_p(3 << 20)) == -1
    assert call(None, 0, None, 3, None, None, None, None, 0.1, 0, 1, None, None, None) == 0
    assert _lib.lib.lbt_feature_mask(None, None, 3, one) == -1 and _lib.lib.lbt_feature_mask(None, one, 3, None) == -1


@pytest.mark.parametrize("objective,k", [(0, 1), (0, 3), (1, 1), (1, 4)])
def test_the_next_gradient_refuses_outputs_that_overlap_what_it_reads(objective, k):
    """The predictions are written while targets, weights, leaves and leaf values are read: whole arrays, first and last entries."""
    from lbtree import _lib

    n, nodes = 10, 3
    size = {"leaf": 8 * nodes * k, "rows": 4 * n, "pred": 8 * n * k, "y": 8 * n * (1 if objective == 1 and k > 1 else k), "w": 8 * n,
            "g": 8 * n * k, "h": 8 * n * k, "sums": 16}
    at = {name: (i + 1) << 20 for i, name in enumerate(size)}

    def refused(**moved):
        a = dict(at, **moved)
        p = {name: C.c_void_p(v) for name, v in a.items()}
        rc = _lib.lib.lbt_next_gradient(None, objective, p["leaf"], nodes, p["rows"], p["pred"], p["y"], p["w"], 0.1, n, k, p["g"], p["h"], p["sums"])
        return rc == -1 and b"alias" in _lib.lib.lbt_last_error()

    for out in ("pred", "g", "h", "sums"):
        for name in size:
            if name != out:
                for shift in (0, size[out] - 4, 4 - size[name]):
                    assert refused(**{name: at[out] + shift}), (out, name, shift)
