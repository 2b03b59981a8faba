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
