"""Prediction of large and small inputs and the update of many trees on a stream that is not the default one, behind work
that is still running there, and from two threads at a time."""
import threading

import numpy as np
import pytest
import torch

from lbtree import ops

pytestmark = pytest.mark.gpu

N_LARGE, F, TREES = 600_011, 8, 130  # rows enough for the ranks


def _trees(seed, depth=6):
    rs = np.random.RandomState(seed)
    m, inner = 2 ** (depth + 1) - 1, 2 ** depth - 1
    trees = []
    for _ in range(TREES):
        feat = -np.ones(m, np.int32)
        feat[:inner] = rs.randint(0, F, inner)
        trees.append(tuple(torch.from_numpy(a).cuda() for a in (rs.randn(m, 1), feat, rs.rand(m))))
    return trees


def _calls(X, y, trees, rounds):
    """Predictions by ranks, of few rows (estimator's call and packed) and an update of `rounds` trees."""
    packed = ops.PackedEnsemble(trees, 1, F, dtype=X.dtype)
    pred   = torch.zeros((X.shape[0], 1), dtype=torch.float64, device="cuda")
    new    = ops.update_trees(X, y, None, "squared_error", 0.3, pred, [(f, s, 0.0, 1.0) for _, f, s in trees[:rounds]])
    return [ops.predict(X, trees, 1), ops.predict(X[:1000], trees, 1), packed.predict(X[:256]), pred] + [a for t in new for a in t]


def _same(got, want):
    assert all(torch.equal(a, b) for a, b in zip(got[:3], want[:3]))
    # sums of n terms below 2 in no fixed order, in rounds that start from one another's errors
    tol = 8 * N_LARGE * 2.0 ** -53 * 6
    assert all(torch.allclose(a, b, rtol=tol, atol=tol) for a, b in zip(got[3:], want[3:]))


def test_calls_follow_what_is_queued_on_their_stream():
    gen    = torch.Generator(device="cuda").manual_seed(1)
    source = torch.rand((N_LARGE, F), generator=gen, device="cuda")
    target = torch.rand((N_LARGE, 1), generator=gen, device="cuda", dtype=torch.float64)
    trees  = _trees(1)
    want   = _calls(source, target, trees, 6)
    X, y   = torch.full_like(source, 2.0), torch.zeros_like(target)
    late   = [tuple(torch.zeros_like(a) for a in t) for t in trees]
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        torch.cuda._sleep(20_000_000)  # about 10 ms: inputs and trees come after the calls have been made
        X.copy_(source)
        y.copy_(target)
        for a, b in zip(late, trees):
            for to, of in zip(a, b):
                to.copy_(of)
        got = _calls(X, y, late, 6)
    stream.synchronize()
    _same(got, want)


def test_two_threads_with_a_stream_each():
    gen  = torch.Generator(device="cuda").manual_seed(2)
    work = [(torch.rand((N_LARGE, F), generator=gen, device="cuda"),
             torch.rand((N_LARGE, 1), generator=gen, device="cuda", dtype=torch.float64), _trees(seed)) for seed in (2, 3)]
    want = [_calls(*w, 6) for w in work]
    torch.cuda.synchronize()
    got, together = [None, None], threading.Barrier(2, timeout=60)

    def run(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            together.wait()
            got[i] = [_calls(*work[i], 6) for _ in range(3)]
        stream.synchronize()

    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(2):
        assert got[i] is not None
        for g in got[i]:
            _same(g, want[i])
