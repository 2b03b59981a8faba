"""lbtree._host.tree_arrays, the native look at an ensemble's arrays: what it does not take is left to the Python form."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from lbtree import _lib, ops


def test_anything_but_plain_device_arrays_is_left_to_the_caller():
    take = _lib._host.tree_arrays
    cpu = (torch.zeros(7, 1, dtype=torch.float64), torch.zeros(7, dtype=torch.int32), torch.zeros(7, dtype=torch.float64))
    assert take([], 1) == (b"", b"", b"", b"")
    for trees in ([cpu], [(1, 2, 3)], [cpu[:2]], [list(cpu)], [None], iter([cpu]), [(np.zeros((7, 1)),) + cpu[1:]]):
        assert take(trees, 1) is None
    assert take([], 0) is None
    with pytest.raises(TypeError):
        take([cpu])


@pytest.mark.parametrize("module", ["None", "types.SimpleNamespace(torch_version='0.0', tree_arrays=None)"])
def test_the_package_imports_without_the_native_look(module):
    """Not built, or built against another torch: said so, and looked over in Python."""
    code = ("import sys, types, warnings\n"
            "sys.modules['lbtree._host'] = %s\n"
            "with warnings.catch_warnings(record=True) as told:\n"
            "    warnings.simplefilter('always')\n"
            "    from lbtree import _lib, ops\n"
            "assert _lib._host is None and any('_host.so' in str(w.message) for w in told)\n"
            "assert ops._tree_arrays([], 1)[4] == 0\n" % module)
    package = os.path.dirname(os.path.dirname(os.path.abspath(_lib.__file__)))
    subprocess.run([sys.executable, "-c", code], check=True, env=dict(os.environ, PYTHONPATH=package))


@pytest.mark.gpu
def test_the_python_form_gives_the_same(monkeypatch):
    rs = np.random.RandomState(3)
    trees = [(torch.from_numpy(rs.randn(15, 2)).cuda(), torch.from_numpy(np.r_[rs.randint(0, 5, 7), -np.ones(8)].astype(np.int32)).cuda(),
              torch.from_numpy(rs.rand(15)).cuda()) for _ in range(20)]
    X = torch.rand(300, 5).cuda()
    want = ops.predict(X, trees, 2)
    monkeypatch.setattr(_lib, "_host", None)
    assert torch.equal(ops.predict(X, trees, 2), want)
    assert torch.equal(ops.PackedEnsemble(trees, 2, 5).predict(X), want)


@pytest.mark.gpu
def test_plain_arrays_and_those_that_are_not():
    take = _lib._host.tree_arrays
    leaf = torch.randn(7, 2, dtype=torch.float64).cuda()
    feat = torch.tensor([0, 1, 0, -1, -1, -1, -1], dtype=torch.int32).cuda()
    split = torch.rand(7, dtype=torch.float64).cuda()
    trees = [(leaf, feat, split), (leaf[:3], feat[:3], split[:3])]
    got = take(trees, 2)
    assert [np.frombuffer(b, np.uint64).tolist() for b in got[:3]] == [[t[i].data_ptr() for t in trees] for i in range(3)]
    assert np.frombuffer(got[3], np.int32).tolist() == [7, 3]
    wide = torch.randn(7, 4, dtype=torch.float64).cuda()
    for bad in ((wide[:, :2], feat, split), (leaf.float(), feat, split), (leaf, feat.long(), split), (leaf[:6], feat, split),
                (leaf, feat, split[:6]), (leaf[:, 0], feat, split), (leaf, feat, torch.rand(14, dtype=torch.float64).cuda()[::2])):
        assert take([bad], 2) is None
    assert take(trees, 1) is None
    # and the caller converts or refuses, as without it
    X = torch.rand(50, 2).cuda()
    want = ops.predict(X, trees, 2)
    strided = torch.stack([split, split], dim=1)[:, 0]
    mixed = [(leaf.cpu(), feat.long(), strided), tuple(t.cpu().numpy() for t in trees[1])]
    assert torch.equal(ops.predict(X, mixed, 2), want)
    assert torch.equal(ops.PackedEnsemble(mixed, 2, 2).predict(X), want)
    for bad in ((leaf[:6], feat, split), (leaf[:, :1], feat, split)):
        with pytest.raises(_lib.LbtError):
            ops.predict(X, [bad], 2)


def test_models_that_are_no_trees_are_left_to_the_caller():
    take = _lib._host.model_arrays
    names = ("a", "b", "c")

    class Model:
        a, b, c = torch.zeros(7, 1, dtype=torch.float64), torch.zeros(7, dtype=torch.int32), torch.zeros(7, dtype=torch.float64)

    class Bare:
        a = 1

    assert take([], Model, names, 1) == (b"", b"", b"", b"", [])
    for models in ([Model()], [Bare()], [None], iter([])):  # arrays of the CPU, others, none
        assert take(models, Model, names, 1) is None
    assert take([Bare()], Bare, names, 1) is None
    assert take([], Model, names, 0) is None and take([], 1, names, 1) is None and take([], Model, names[:2], 1) is None
    assert _lib._host.predict_packed(np.zeros((2, 2)), 0, 0, 0, 0, 1) is None
    assert _lib._host.predict_packed(torch.zeros(2, 2), 0, 0, 0, 0, 1) is None
    with pytest.raises(TypeError):
        _lib._host.predict_packed(torch.zeros(2, 2), 0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("k", [1, 3])
def test_a_packed_prediction_in_native_code_and_through_python(monkeypatch, dtype, k):
    rs = np.random.RandomState(k)
    trees = [(torch.from_numpy(rs.randn(15, k)).cuda(), torch.from_numpy(np.r_[rs.randint(0, 5, 7), -np.ones(8)].astype(np.int32)).cuda(),
              torch.from_numpy(rs.rand(15)).cuda()) for _ in range(20)]
    packed = ops.PackedEnsemble(trees, k, 5, dtype)
    wide = torch.rand(300, 10, dtype=dtype).cuda()
    good = [wide[:, :5].contiguous(), wide[:, :5], wide[:, ::2], wide[:5].t(), wide[:0, :5], wide[:1, :5].clone().requires_grad_(),
            wide[:, :5].cpu(), wide[7:9, :5].cpu().numpy()]
    bad = [wide, wide[0, :5], wide[:, :5].to(torch.float32 if dtype == torch.float64 else torch.float64), wide[:, :5].long()]
    got = [packed.predict(X) for X in good]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        aside = packed.predict(good[0])
    stream.synchronize()
    refused = []
    for X in bad:
        with pytest.raises(_lib.LbtError) as e:
            packed.predict(X)
        refused.append(str(e.value))
    with pytest.raises(Exception):
        torch.func.vmap(packed.predict)(wide[:4, :5].reshape(2, 2, 5))
    monkeypatch.setattr(ops, "_predict_packed", None)
    for X, out in zip(good, got):
        want = packed.predict(X)
        assert torch.equal(out, want) and out.dtype == want.dtype and out.device == want.device and not out.requires_grad
    assert torch.equal(aside, got[0])
    for X, told in zip(bad, refused):
        with pytest.raises(_lib.LbtError) as e:
            packed.predict(X)
        assert str(e.value) == told
    with pytest.raises(Exception):
        torch.func.vmap(packed.predict)(wide[:4, :5].reshape(2, 2, 5))


def test_code_behind_an_attribute_of_a_model():
    """It may change the list of models, raise, or look at every list there is: the caller then looks closer, and no list is seen
    before it is complete."""
    import gc

    take = _lib._host.model_arrays
    names = ("a", "b", "c")
    seen = []

    class Model:
        def __init__(self, act):
            self.act = act

        @property
        def a(self):
            self.act()
            return 1

    def interrupted():
        raise KeyboardInterrupt

    def wrong():
        raise ValueError

    def look():
        # (the size alone: an element that is not there yet could not be touched)
        seen.extend(len(o) for o in gc.get_objects() if type(o) is list and len(o) == 3 * 1237)

    with pytest.raises(KeyboardInterrupt):
        take([Model(interrupted)], Model, names, 1)
    assert take([Model(wrong)], Model, names, 1) is None
    models = []
    models.extend(Model(models.clear) for _ in range(3))
    assert take(models, Model, names, 1) is None and models == []
    assert take([Model(look)] * 1237, Model, names, 1) is None and seen == []


@pytest.mark.gpu
@pytest.mark.parametrize("change", ["append", "pop"])
def test_a_list_of_models_that_changes_while_it_is_read(change):
    """The library is told as many trees as there are addresses of."""
    rs = np.random.RandomState(3)
    arrays = (torch.from_numpy(rs.randn(15, 2)).cuda(), torch.from_numpy(np.r_[rs.randint(0, 5, 7), -np.ones(8)].astype(np.int32)).cuda(),
              torch.from_numpy(rs.rand(15)).cuda())

    class Model:
        leaf_value, feature = arrays[:2]
        act = None

        @property
        def split_value(self):
            if self.act is not None:
                act, self.act = self.act, None
                act()
            return arrays[2]

    models = [Model() for _ in range(20)]
    first = models[0]
    first.act = (lambda: models.append(Model())) if change == "append" else models.pop
    assert _lib._host.model_arrays(models, Model, ops._ARRAYS, 2) is None
    X = torch.rand(300, 5).cuda()
    first.act = (lambda: models.append(Model())) if change == "append" else models.pop
    got = ops.predict_models(X, models, Model, 2)
    assert torch.equal(got, ops.predict(X, [arrays] * len(models), 2))


def test_models_of_which_the_first_is_no_tree_are_refused():
    from lbtree.models import Tree

    class Other:
        pass

    with pytest.raises(AssertionError):
        Tree.batch_predict([Other()], torch.zeros(2, 2))
    with pytest.raises(IndexError):
        Tree.batch_predict([], torch.zeros(2, 2))


# ---------------------------------------------------------------- calls of the library from native code


def _native_calls(entry, first):
    """The calls of lbtree._host that enter the library, with another entry and another first argument (a stream's address)."""
    import ctypes as C

    n, k = 10, 1
    double = dict(device="cuda", dtype=torch.float64)
    X, g, h, y, pred = torch.zeros((n, 2), device="cuda"), *(torch.ones((n, k), **double) for _ in range(4))
    rows, leaf = torch.zeros(n, dtype=torch.int32, device="cuda"), torch.zeros((3, k), **double)
    address, host = C.cast(entry, C.c_void_p).value, _lib._host
    return {
        "predict_packed": lambda: host.predict_packed(X, address, first, 0, 0, k),
        "build_tree": lambda: host.build_tree(X, g, h, None, ops._get_workspace, address, ops._BUILD_BYTES, first, 0, 2, 4, 1, 0, 1, 0.0, 1.0, 0.0),
        "weighted_gradient": lambda: host.weighted_gradient(y, pred, None, address, first, 0, 0.1),
        "add_leaf_values": lambda: host.add_leaf_values(pred, leaf, rows, address, first),
        "next_gradient": lambda: host.next_gradient(pred, leaf, rows, y, None, g, h, None, address, first, 0, 0.1),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["predict_packed", "build_tree", "weighted_gradient", "add_leaf_values", "next_gradient"])
def test_an_exception_of_the_library_comes_back_with_the_lock_held(name):
    """An entry that throws (std::bad_alloc): None, the caller's way through Python, and an interpreter that goes on."""
    import ctypes as C

    thrower = C.CDLL("libstdc++.so.6")._ZSt17__throw_bad_allocv
    call = _native_calls(thrower, 0)[name]
    for _ in range(3):
        assert call() is None
    assert C.pythonapi.PyGILState_Check() == 1


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["predict_packed", "build_tree", "weighted_gradient", "add_leaf_values", "next_gradient"])
def test_other_threads_run_while_the_library_is_called(name):
    """An entry that sleeps for 0.3 s (a launch waits like that while the stream's queue is full): another thread takes its turns."""
    import ctypes as C
    import threading
    import time

    call = _native_calls(C.CDLL("libc.so.6").usleep, 300000)[name]
    turns, ended = [0], threading.Event()

    def count():
        while not ended.wait(0.002):
            turns[0] += 1

    other = threading.Thread(target=count)
    other.start()
    try:
        before = turns[0]
        call()
        while_it_slept = turns[0] - before
    finally:
        ended.set()
        other.join()
    assert while_it_slept >= 10  # with the lock held none or one


def test_numbers_that_are_none_are_left_to_the_caller():
    """A learning rate of another type: no error of the native call's own (the Python form says what is wrong with it)."""
    t = torch.zeros(2, 1, dtype=torch.float64)
    for rate in ("0.1", None, 10 ** 400, [1]):
        assert _lib._host.weighted_gradient(t, t, None, 0, 0, 0, rate) is None
        assert _lib._host.next_gradient(t, t, t, t, None, t, t, None, 0, 0, 0, rate) is None
    assert _lib._host.add_leaf_values(t, t, t, 0, "0") is None


@pytest.mark.gpu
@pytest.mark.parametrize("rate,taken", [("0.1", True), (np.float32(0.1), True), (None, False), (10 ** 400, False)])
def test_a_learning_rate_is_taken_or_refused_as_in_python(monkeypatch, rate, taken):
    y, pred = (torch.rand((4, 1), dtype=torch.float64, device="cuda") for _ in range(2))
    said = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(ops, "_NATIVE", None)
        try:
            said.append(ops.weighted_gradient("squared_error", y, pred, None, rate)[0].tolist())
        except Exception as e:
            said.append((type(e), str(e)))
    assert said[0] == said[1] and isinstance(said[0], list) == taken


def test_the_package_imports_without_a_native_module_of_an_older_source():
    """Built for this torch, but without the calls of a round: said so, and Python takes them all."""
    code = ("import sys, types, warnings, torch\n"
            "old = types.SimpleNamespace(torch_version=str(torch.__version__), **{n: print for n in ('tree_arrays', 'model_arrays', 'predict_packed')})\n"
            "sys.modules['lbtree._host'] = old\n"
            "with warnings.catch_warnings(record=True) as told:\n"
            "    warnings.simplefilter('always')\n"
            "    from lbtree import _lib, ops\n"
            "assert _lib._host is None and ops._NATIVE is None and ops._predict_packed is None\n"
            "assert any('without build_tree' in str(w.message) for w in told)\n")
    package = os.path.dirname(os.path.dirname(os.path.abspath(_lib.__file__)))
    subprocess.run([sys.executable, "-c", code], check=True, env=dict(os.environ, PYTHONPATH=package))


def test_every_native_call_of_the_package_is_asked_for():
    import re

    source = open(os.path.join(os.path.dirname(os.path.abspath(_lib.__file__)), "ops.py")).read()
    called = set(re.findall(r"(?:_NATIVE|_lib\._host)\.([a-z_]+)", source))
    assert called == set(_lib._HOST_CALLS) and all(callable(getattr(_lib._host, name)) for name in called)
