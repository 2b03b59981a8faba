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
