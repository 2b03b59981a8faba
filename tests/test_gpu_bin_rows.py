"""Root histograms against a direct count: the binning pass with its tables, probes and record layouts at the edges of
its lanes (features that are no whole lanes, pieces or records), for planes of several search groups, and for proposals that crowd
into few cells."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _columns(n, f, dtype, rs):
    X = rs.normal(size=(n, f))
    X[:, 1::5] = np.exp(3 * X[:, 1::5])                # a long tail
    X[:, 2::5] = rs.randint(0, 7, X[:, 2::5].shape)    # few values
    X[:, 3::5] = np.where(rs.rand(*X[:, 3::5].shape) < 0.9, 1 + 1e-6 * X[:, 3::5], 1e6 * X[:, 3::5])  # nearly all in one cell
    X[:, 4::5] = rs.rand(*X[:, 4::5].shape)
    X = X.astype(dtype)
    for value in (np.nan, np.inf, -np.inf, 0.0, -0.0):
        X[rs.randint(0, n, f), np.arange(f)] = value
    return X


def _proposals(X, samples, rs):
    """Distinct finite values of sampled rows, the last one replaced by +inf, as build_tree.cu:867-964 leaves them."""
    out, rp = [], [0]
    for c in range(X.shape[1]):
        v = X[rs.randint(0, X.shape[0], samples), c]
        v = np.unique(v[np.isfinite(v)] + 0.0)
        if v.size == 0:
            v = np.zeros(1, X.dtype)
        v[-1] = np.inf
        out.append(v)
        rp.append(rp[-1] + v.size)
    return np.concatenate(out).astype(X.dtype), np.array(rp, np.int32)


@pytest.mark.parametrize("n,f,k,dtype,samples", [
    (700, 1, 1, np.float32, 256), (700, 2, 1, np.float32, 256), (700, 2, 2, np.float32, 300), (701, 3, 1, np.float64, 64),
    (1, 4, 1, np.float32, 16), (33, 4, 1, np.float64, 256), (5000, 5, 1, np.float32, 256), (5000, 5, 3, np.float64, 300),
    (4097, 22, 1, np.float32, 128), (4097, 24, 1, np.float32, 256), (4097, 24, 2, np.float32, 256), (4097, 25, 1, np.float64, 256),
    (4099, 43, 1, np.float32, 256), (4099, 43, 2, np.float64, 64), (4099, 50, 1, np.float32, 512), (4099, 50, 1, np.float64, 512),
    (9001, 64, 1, np.float32, 256), (9001, 96, 1, np.float32, 256), (9001, 100, 1, np.float32, 256), (9001, 101, 1, np.float32, 256),
    (3001, 200, 2, np.float32, 256), (3001, 200, 1, np.float64, 256), (3001, 210, 1, np.float32, 256), (2001, 333, 1, np.float32, 512),
    (1001, 500, 3, np.float32, 64), (901, 40, 1, np.float32, 2048),
])
def test_root_histogram_of_binned_rows(n, f, k, dtype, samples):
    from lbtree import ops

    rs = np.random.RandomState(n + f)
    X = _columns(n, f, dtype, rs)
    props, rp = _proposals(X, samples, rs)
    q = rs.randint(-1000, 1000, (n, k, 2)).astype(np.int32)
    q[:, :, 1] = np.abs(q[:, :, 1]) + 1
    pos = np.stack([np.zeros(n, np.int32), np.arange(n, dtype=np.int32)], axis=1)
    sums = q.astype(np.int64).sum(axis=0)[None]
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (X, q, props, rp, pos, sums)]
    hist = torch.zeros((1, k, int(rp[-1]), 2), dtype=torch.int64, device="cuda")
    ops.histogram_level(dev[0], dev[1], dev[2], dev[3], samples, dev[4], 0, (0, 1), dev[5], (0, 1), hist)
    got = hist.cpu().numpy()[0]
    want = np.zeros_like(got)
    for c in range(f):
        # proposals below the value; none for NaN
        b = np.where(np.isnan(X[:, c]), 0, np.searchsorted(props[rp[c]:rp[c + 1]], X[:, c], side="left"))
        for j in range(k):
            np.add.at(want[j], rp[c] + b, q[:, j].astype(np.int64))
    assert np.array_equal(got, want)


@pytest.mark.parametrize("f", [1, 2, 3, 4, 5, 7, 8, 9, 11, 12, 13, 16, 17])
@pytest.mark.parametrize("samples", [256, 300])
@pytest.mark.parametrize("k,dtype", [(1, np.float32), (1, np.float64), (2, np.float32)])
def test_rows_whose_lanes_share_a_record(f, samples, k, dtype):
    """One, two and four lanes to a record of 32 bytes, some of them without features, bins of one and two bytes; 17: no longer."""
    test_root_histogram_of_binned_rows(4099 + f, f, k, dtype, samples)


@pytest.mark.parametrize("f", [1, 2, 3, 4, 8, 16])
def test_rows_whose_lanes_share_a_record_off_a_16_byte_boundary(f, monkeypatch):
    from lbtree import ops

    own = ops.histogram_level

    def moved(X, *args):
        base = torch.empty(X.numel() + 1, dtype=X.dtype, device=X.device)
        at = base[1:].view(X.shape)
        at.copy_(X)
        assert at.data_ptr() % 16 != 0
        return own(at, *args)

    monkeypatch.setattr(ops, "histogram_level", moved)
    test_root_histogram_of_binned_rows(2049, f, 1, np.float32, 256)


@pytest.mark.parametrize("n,f,k,dtype", [(301, 2051, 1, np.float32), (301, 4100, 1, np.float64), (301, 2048, 3, np.float32)])
def test_rows_of_as_many_lanes_as_a_search_group_has(n, f, k, dtype):
    """Few proposals a feature: what bounds a search group is its lanes, beside which those of the records have their place."""
    test_root_histogram_of_binned_rows(n, f, k, dtype, 3)


@pytest.mark.parametrize("n,f,k,dtype,samples", [
    (8447, 33, 1, np.float32, 256), (9000, 17, 1, np.float64, 300), (12345, 65, 1, np.float32, 64), (8961, 1, 2, np.float32, 16),
    (140000, 5, 1, np.float32, 512), (10241, 3, 3, np.float64, 1024),
])
def test_medium_builder_bins(n, f, k, dtype, samples):
    """The builder for medium sizes: blocks of features of even width, tiles and samples that fill no whole turn."""
    import gpu_util as gu

    rs = np.random.RandomState(n)
    X = np.abs(_columns(n, f, dtype, rs))
    X[~np.isfinite(X)] = 1  # (which samples are taken is up to the seed)
    g, h = rs.normal(size=(n, k)), 0.5 + rs.rand(n, k)
    gr, cr = gu.both(X, g, h, max_depth=3, split_samples=samples, seed=5)
    gu.assert_tree_parity(gr, cr)


@pytest.mark.parametrize("f", [1, 2, 3, 4, 7, 8, 9, 16])
@pytest.mark.parametrize("n,dtype", [(150_001, np.float32), (150_257, np.float64)])
def test_medium_builder_bins_of_few_features(n, f, dtype):
    """Tiles whose rows take some of a thread's turns, and some of the waves; the last one has one row."""
    test_medium_builder_bins(n, f, 1, dtype, 256)
