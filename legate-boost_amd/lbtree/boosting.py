"""The boosting loop that drives the tree learner: the part of
legateboost/legateboost.py (`_get_weighted_gradient` :189-224, `_partial_fit`
:254-298, `_predict` :507-529, `update` :306-386) and of objectives.py
(squared error :131-147, log loss :489-531) that feeds BuildTreeTask and
consumes PredictTask. Elementwise work runs as float64 torch ops on the device
that holds X; the tree tasks go through liblbtree.so."""
from copy import deepcopy

import numpy as np
import torch

from . import ops
from .models import Tree


def _check_random_state(seed):
    if seed is None or isinstance(seed, (int, np.integer)):
        return np.random.RandomState(seed)
    if isinstance(seed, np.random.RandomState):
        return seed
    raise ValueError("%r cannot be used to seed a RandomState" % seed)


def _as_defined(obj, owner, *names):
    """Whether these methods of obj are the ones this package defines for `owner`: overridden by no subclass and replaced neither
    on the object nor on a class. What bypasses a method asks this first."""
    cls, own, defined = type(obj), vars(obj), _DEFINED[owner]
    for n in names:
        if n in own or getattr(cls, n) is not defined[n]:
            return False
    return True


def _float64_on_device(a):
    """Whether the library's kernels can take `a` as it is, and no gradient is recorded through it."""
    return (isinstance(a, torch.Tensor) and a.dtype == torch.float64 and a.is_cuda and a.is_contiguous()
            and not a.requires_grad)


def _copy_of(model):
    """deepcopy(model). A tree whose attributes are numbers and names, as one that is not fitted has, is copied by them."""
    if type(model) is Tree and not hasattr(Tree, "__deepcopy__"):
        attributes = vars(model)
        if all(type(v) in _NUMBERS for v in attributes.values()):
            new = Tree.__new__(Tree)
            vars(new).update(attributes)
            return new
    return deepcopy(model)


_NUMBERS = (int, float, str, bool, type(None))


class SquaredErrorObjective:
    fused = "squared_error"  # ops.weighted_gradient computes transform + gradient + weighting in one pass

    def gradient(self, y, pred):
        return pred - y, torch.ones_like(pred)

    def transform(self, pred):
        return pred

    def initialise_prediction(self, y, w, boost_from_average):
        if boost_from_average:
            per_row = w is None or (w.dim() == 1 and w.shape[0] == y.shape[0] and not w.requires_grad)
            if y.is_cuda and 0 < y.shape[0] and 0 < y.shape[1] <= ops.MAX_MEAN_OUTPUTS and per_row and not y.requires_grad:
                return ops.weighted_mean(y, w)
            w = torch.ones(y.shape[0], dtype=torch.float64, device=y.device) if w is None else w
            return (y * w[:, None]).sum(dim=0) / w.sum()
        return torch.zeros(y.shape[1], dtype=torch.float64, device=y.device)


class LogLossObjective:
    fused = "log_loss"

    def gradient(self, y, pred):
        if pred.shape[1] == 1:
            return pred - y, pred * (1.0 - pred)
        label = y.to(torch.int64).reshape(-1)
        h = pred * (1.0 - pred)
        g = pred.clone()
        g[torch.arange(g.shape[0], device=g.device), label] -= 1.0
        return g, h

    def transform(self, pred):
        if pred.shape[1] == 1:
            return 1.0 / (1.0 + torch.exp(-pred))
        s = pred.max(dim=1).values
        e_x = torch.exp(pred - s[:, None])
        return e_x / e_x.sum(dim=1)[:, None]

    def initialise_prediction(self, y, w, boost_from_average):
        counted = y.is_cuda and y.numel() > 0 and not y.requires_grad
        if counted:
            stats = ops.label_counts(y)
            bad, most, wide = stats[:3].tolist()
            if bad:
                raise ValueError("Expected labels to be non-zero whole numbers")
            if not wide:  # (more classes are counted by the operators below)
                n_targets = most + 1 if most > 1 else 1
                if not boost_from_average:
                    return torch.zeros(n_targets, dtype=torch.float64, device=y.device)
                return ops.label_priors(stats, y.numel(), n_targets)
        if not counted and not bool(((y == torch.floor(y)) & (y >= 0)).all()):
            raise ValueError("Expected labels to be non-zero whole numbers")
        num_class = int(y.max().item() + 1)
        n_targets = num_class if num_class > 2 else 1
        if not boost_from_average:
            return torch.zeros(n_targets, dtype=torch.float64, device=y.device)
        if n_targets == 1:
            prob = y.sum() / y.numel()
            return (-torch.log(1 / prob - 1)).reshape(1)
        prob = torch.bincount(y.reshape(-1).to(torch.int64), minlength=num_class).to(torch.float64) / y.numel()
        return torch.log(prob)


class LBBase:
    def __init__(self, n_estimators=100, objective=None, base_models=(Tree(max_depth=8),), init="average",
                 learning_rate=0.1, subsample=1.0, random_state=None, verbose=0):
        if not 0.0 < subsample <= 1.0:
            raise ValueError("subsample should be in (0, 1]")
        self.subsample = subsample
        self.n_estimators = n_estimators
        self.objective = objective
        self.base_models = base_models
        self.init = init
        self.learning_rate = learning_rate
        self.random_state = random_state
        self.verbose = verbose
        self.models_ = []

    def __getitem__(self, i):
        return self.models_[i]

    def __len__(self):
        return len(self.models_)

    def __iter__(self):
        return iter(self.models_)

    def _prepare(self, X, y):
        X = ops.as_device(X)
        y = ops.as_device(y, torch.float64)
        if y.dim() == 1:
            y = y.reshape(-1, 1)
        return X, y

    def _weights(self, y, sample_weight):
        """The rows' weights; None (all ones) where nothing but this module's own code sees them."""
        if sample_weight is not None:
            return ops.as_device(sample_weight, torch.float64)
        objective = self._objective_instance
        plain = (type(self) in (LBRegressor, LBClassifier) and not self.verbose
                 and _as_defined(self, LBBase, "_get_weighted_gradient")
                 and type(objective) in (SquaredErrorObjective, LogLossObjective) and not vars(objective)
                 and _as_defined(objective, type(objective), "gradient", "transform", "initialise_prediction"))
        return None if plain else torch.ones(y.shape[0], dtype=torch.float64, device=y.device)

    def _get_weighted_gradient(self, y, pred, sample_weight, learning_rate):
        fused = getattr(self._objective_instance, "fused", None)
        if fused is not None and pred.is_cuda:
            g, h = ops.weighted_gradient(fused, y, pred, sample_weight, learning_rate)
        else:
            g, h = self._objective_instance.gradient(y, self._objective_instance.transform(pred))
            if sample_weight is None:
                sample_weight = torch.ones(y.shape[0], dtype=torch.float64, device=y.device)
            g = g * sample_weight[:, None] * learning_rate
            h = torch.clamp(h * sample_weight[:, None], min=1e-8)
        if self.subsample < 1.0:
            # legateboost.py:215-222: one Bernoulli(subsample) draw per row zeroes its gradient and hessian. The
            # seed is taken from the estimator's RandomState at the same place as in the reference, so the tree
            # seeds that follow are the reference's; the draws themselves come from torch's generator, not
            # from cupynumeric's XORWOW stream, so which rows are kept is not comparable with the reference.
            seed = int(self.random_state_.randint(0, 2**32, dtype=np.int64))
            gen = torch.Generator(device=g.device).manual_seed(seed)
            draw = torch.rand(y.shape[0], generator=gen, device=g.device, dtype=torch.float64)
            if fused is not None and g.is_cuda:  # (g and h are this call's own)
                ops.keep_rows(draw, self.subsample, g, h)
                return g, h
            mask = draw < self.subsample
            mask = mask.to(torch.float64)[:, None]
            g = g * mask
            h = h * mask
        return g, h

    def _predict(self, X):
        plain = self.model_init_
        if (self.models_ and _as_defined(self.models_[0], Tree, "batch_predict") and _float64_on_device(plain)
                and plain.dim() == 1 and plain.shape[0] == self.models_[0].leaf_value.shape[1]):
            return Tree.batch_predict_from(plain, self.models_, X)
        init = self.model_init_.reshape(1, -1)
        if self.models_:
            return init + type(self.models_[0]).batch_predict(self.models_, X)
        return init.repeat(X.shape[0], 1).contiguous()

    def fit(self, X, y, sample_weight=None):
        X, y = self._prepare(X, y)
        self.n_features_in_ = X.shape[1]
        if not isinstance(self.base_models, tuple) or len(self.base_models) == 0:
            raise ValueError("base_models should be a tuple")
        self.random_state_ = _check_random_state(self.random_state)
        self._objective_instance = self._make_objective()
        w = self._weights(y, sample_weight)
        self.model_init_ = self._objective_instance.initialise_prediction(y, w, self.init == "average")
        self.models_ = []
        self.train_metric_ = []
        train_pred = self._predict(X)
        # The gradient pass can leave the quantiser's first sums where g and h reach the tree as it wrote them. It then has a
        # workgroup per 4096 entries: below four million of them (several outputs: eight) the pass over g and h that it saves costs
        # less. Fits of 5 rounds of depth 6 with the sums and without, ms: 300,000 x 20 1.21 and
        # 1.18, 1,000,000 x 50 2.14 and 2.10, 2,000,000 x 40 2.95 and 2.92, 4,000,000 x 30 3.71 and 3.72, 6,000,000 x 30 5.28 and
        # 5.29 (two classes 5.37 and 5.40), 10,000,000 x 100 17.98 and 18.08; three classes, 1,500,000 x 20 2.65 and 2.62,
        # 2,000,000 x 30 4.01 and 4.00; two outputs, 4,000,000 x 30 5.42 and 5.50; eight classes, 600,000 x 20 3.12 and 3.13,
        # 2,000,000 x 30 6.65 and 6.85; 16, 3,000,000 x 30 12.7 and 13.3. Rows of more than 128 classes are a thread's work, and a
        # workgroup's entries few of them: never (two rounds of depth 3, ms: 70,000 x 4 with 130 classes 2.88 and 2.66, 20,000 with 500
        # 8.4 and 5.1, 10,000 with 1000 14.9 and 8.8).
        fused = getattr(self._objective_instance, "fused", None)
        plain = (fused is not None and self.subsample == 1.0 and train_pred.is_cuda and train_pred.numel() > 0
                 and _as_defined(self, LBBase, "_get_weighted_gradient"))
        sums = (plain and train_pred.numel() >= (4000000 if train_pred.shape[1] == 1 else 8000000)
                and (fused != "log_loss" or train_pred.shape[1] <= 128))

        def own(model):
            return isinstance(model, Tree) and _as_defined(model, Tree, "fit", "fit_update_predictions", "_fit")

        at_hand = None  # the next round's gradients, formed where the last tree's values were added
        for i in range(self.n_estimators):
            model = _copy_of(self.base_models[i % len(self.base_models)]).set_random_state(self.random_state_)
            if plain and own(model):
                if at_hand is None:
                    at_hand = ops.weighted_gradient(fused, y, train_pred, w, self.learning_rate, sums=sums)
                g, h = at_hand[:2]
                chunks = at_hand[2] if sums else None

                def next_round(pred, leaf_value, row_leaf):
                    ops.next_gradient(fused, leaf_value, row_leaf, pred, y, w, self.learning_rate, g, h, chunks)

                if i + 1 < self.n_estimators and own(self.base_models[(i + 1) % len(self.base_models)]):
                    model._fit(X, g, h, train_pred, chunks, next_round)
                else:
                    at_hand = None
                    model._fit(X, g, h, train_pred, chunks)
            else:
                at_hand = None
                g, h = self._get_weighted_gradient(y, train_pred, w, self.learning_rate)
                if hasattr(model, "fit_update_predictions"):
                    model.fit_update_predictions(X, g, h, train_pred)
                else:
                    train_pred += model.fit(X, g, h).predict(X)
            self.models_.append(model)
            if self.verbose:
                print("i: {} train loss: {:.6f}".format(i, self._loss(y, train_pred, w)))
        self._train_pred = train_pred
        return self

    def update(self, X, y, sample_weight=None):
        X, y = self._prepare(X, y)
        w = self._weights(y, sample_weight)
        if self.models_ and all(type(m).clear is Tree.clear for m in self.models_):
            torch._foreach_zero_([a for m in self.models_ for a in (m.leaf_value, m.hessian)])
        else:
            for m in self.models_:
                m.clear()
        self.model_init_ = self._objective_instance.initialise_prediction(y, w, self.init == "average")
        pred = self.model_init_.reshape(1, -1).repeat(X.shape[0], 1).contiguous()
        fused = getattr(self._objective_instance, "fused", None)
        if (fused is not None and self.subsample == 1.0 and X.shape[0] > 0
                and _as_defined(self, LBBase, "_get_weighted_gradient")
                and Tree.update_rounds(self.models_, X, y, w, fused, self.learning_rate, pred)):
            return self
        for m in self.models_:
            g, h = self._get_weighted_gradient(y, pred, w, self.learning_rate)
            if hasattr(m, "update_and_predict"):
                m.update_and_predict(X, g, h, pred)
            else:
                m.update(X, g, h)
                pred += m.predict(X)
        return self


class LBRegressor(LBBase):
    def _make_objective(self):
        return SquaredErrorObjective()

    def _loss(self, y, pred, w):
        return float((((pred - y) ** 2).sum(dim=1) * w).sum() / w.sum() / y.shape[1])

    def predict(self, X):
        X = ops.as_device(X)
        pred = self._objective_instance.transform(self._predict(X))
        return pred.squeeze(1) if pred.shape[1] == 1 else pred


class LBClassifier(LBBase):
    def _make_objective(self):
        return LogLossObjective()

    def _loss(self, y, pred, w):
        p = self._objective_instance.transform(pred)
        if p.shape[1] == 1:
            p = torch.cat([1.0 - p, p], dim=1)
        label = y.to(torch.int64).reshape(-1)
        picked = p[torch.arange(p.shape[0], device=p.device), label]
        return float((-torch.log(picked) * w).sum() / w.sum())

    def predict_proba(self, X):
        X = ops.as_device(X)
        objective, init = self._objective_instance, self.model_init_
        if (type(objective) is LogLossObjective and _as_defined(objective, LogLossObjective, "transform") and self.models_
                and _as_defined(self, LBBase, "_predict")):
            raw = type(self.models_[0]).batch_predict(self.models_, X)
            if (_float64_on_device(raw) and _float64_on_device(init) and raw.dim() == 2
                    and init.shape == raw.shape[1:] and init.device == raw.device):
                return ops.class_probabilities(raw, init)
            p = objective.transform(init.reshape(1, -1) + raw)
        else:
            p = objective.transform(self._predict(X))
        if p.shape[1] == 1:
            p = torch.cat([1.0 - p, p], dim=1)
        return p

    def predict(self, X):
        return self.predict_proba(X).argmax(dim=1)


# the methods as they stand here, whatever is put in their place later
_DEFINED = {cls: {n: getattr(cls, n) for n in names} for cls, names in (
    (LBBase, ("_get_weighted_gradient", "_predict")),
    (SquaredErrorObjective, ("gradient", "transform", "initialise_prediction")),
    (LogLossObjective, ("gradient", "transform", "initialise_prediction")),
    (Tree, ("fit", "fit_update_predictions", "_fit", "batch_predict")),
)}
