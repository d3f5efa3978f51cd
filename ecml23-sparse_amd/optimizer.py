"""The optimizer of the reference's training loop: ``SparseAdam`` (sparse/optimizer.py:9-23), a Keras
Adam that also resets its moments where a sparse layer rewires.

The update of every float32 parameter is one pass of ``ffi_adam_step_f32`` in libffi_hip.so (Keras'
update rule, with its defaults ``beta_1=0.9, beta_2=0.999, epsilon=1e-7``); torch holds the tensors.
"""
from __future__ import annotations

import ctypes

import torch
from torch.autograd import forward_ad

from . import _lib
from . import metrics as metrics_mod
from .custom_layer import StratifiedRewireLayer, StratifiedRewireLayerV2
from .fixed_fan_in_ops import _backward_bias, _forward_bias, _on, _stream_handle, topk_scores

# What SparseOptWrapper looks for before it takes a step without a graph.
_DIRECT_LAYERS = (StratifiedRewireLayerV2, StratifiedRewireLayer)
_DIRECT_LOSSES = (metrics_mod.SparseHingeLoss, metrics_mod.SparseSquaredHingeLoss, metrics_mod.SparseBinaryCrossEntropyLoss)
_MODULE_HOOKS = ("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")
# (as the classes define them: what replaces one on a class or on the layer is to be called)
_MODULE_CALLS = ("forward", "__call__", "_wrapped_call_impl", "_call_impl")
_OVERRIDABLE = frozenset((*_MODULE_CALLS, "_compiled_call_impl"))
_CALLS = {cls: tuple((name, getattr(cls, name)) for name in names)
          for classes, names in ((_DIRECT_LAYERS, _MODULE_CALLS), (_DIRECT_LOSSES, ("__call__",))) for cls in classes}
# From here on the scores are formed, turned into gradients and ranked in one kernel; below, a kernel each is faster: the one kernel's
# ranks cost more than the scores' way through the caches.  us a step, one kernel and several: 128 x 300 x 300,000 x 4 240 and
# 333, 128 x 1,100 x 200,000 x 20 293 and 318, 31 x 45 x 290,420 x 75 514 and 510, 32 x 768 x 131,072 x 32 179 and 151.
_SCORES_IN_ONE_KERNEL = 1 << 24
_has_global_hook = torch.nn.modules.module._has_any_global_hook
_saved_tensor_hooks = torch._C._autograd._top_saved_tensors_default_hooks


def _as_defined(cls):
    return all(getattr(cls, name) is call for name, call in _CALLS[cls])


_MARK = "ecml23-sparse: held"


def _accumulation_node(variable):
    return variable.view_as(variable).grad_fn.next_functions[0][0]


def _is_held(variable):
    """Whether anybody holds the node of autograd's that adds to ``variable.grad``: libraries that exchange gradients put hooks
    on it.  A node that nobody holds goes away, and with it its hooks and the mark put on it here."""
    _accumulation_node(variable).metadata[_MARK] = True
    return _accumulation_node(variable).metadata.pop(_MARK, False)


def adam_step(variable, m, v, gradient, learning_rate, beta_1, beta_2, epsilon, step):
    """One in-place Adam step on contiguous float32 device tensors of equal size; ``step`` counts from 1."""
    for name, t in (("variable", variable), ("m", m), ("v", v), ("gradient", gradient)):
        if t.dtype != torch.float32 or not t.is_cuda or not t.is_contiguous():
            raise TypeError(f"{name} must be a contiguous float32 device tensor")
        if t.numel() != variable.numel():
            raise ValueError(f"{name} has {t.numel()} elements, variable has {variable.numel()}")
    with _on(variable.device):
        _lib.check(_lib.lib().ffi_adam_step_f32(variable.data_ptr(), m.data_ptr(), v.data_ptr(), gradient.data_ptr(),
                                                variable.numel(), float(learning_rate), float(beta_1), float(beta_2),
                                                float(epsilon), int(step), _stream_handle(variable.device)))


class SparseAdam:
    """``SparseAdam(params, learning_rate, update_moments=True)``; ``step()`` applies the gradients
    held in ``param.grad`` (Keras' ``apply_gradients``), ``update_sparse(layer)`` rewires a layer and
    clears the moments of the rewired connections (sparse/optimizer.py:14-23)."""

    def __init__(self, params, learning_rate=0.001, beta_1=0.9, beta_2=0.999, epsilon=1e-7, update_moments=True):
        self.params = list(params)
        self.learning_rate = float(learning_rate)
        self.beta_1, self.beta_2, self.epsilon = float(beta_1), float(beta_2), float(epsilon)
        self.update_moments = bool(update_moments)
        self.iterations = 0
        self._momentums = [torch.zeros_like(p.data) for p in self.params]
        self._velocities = [torch.zeros_like(p.data) for p in self.params]

    def zero_grad(self):
        for p in self.params:
            p.grad = None

    @torch.no_grad()
    def step(self):
        self.iterations += 1
        for p, m, v in zip(self.params, self._momentums, self._velocities):
            if p.grad is None:
                continue
            adam_step(p.data, m, v, p.grad.contiguous(), self.learning_rate, self.beta_1, self.beta_2, self.epsilon,
                      self.iterations)

    def _index_of(self, variable):
        for i, p in enumerate(self.params):
            if p is variable:
                return i
        raise KeyError("the variable is not one of this optimizer's parameters")

    def update_sparse(self, layer):
        if self.update_moments:
            i = self._index_of(layer.sparse_weights)
            moments = [self._momentums[i], self._velocities[i]]
            if getattr(layer, "rewires_in_place", bool)() and all(m.is_contiguous() for m in moments):
                layer._rewire_in_place(moments)
                return
            new_m, new_v = layer.rewire(moments)
            self._momentums[i].copy_(new_m)
            self._velocities[i].copy_(new_v)
        else:
            layer.rewire(None)


class SparseOptWrapper(torch.nn.Module):
    """The training loop's model wrapper (sparse/optimizer.py:26-74): ``train_step((x, y))`` runs the base
    model, the loss, the backward pass and the optimizer step, then lets the optimizer rewire every sparse layer
    when ``optimizer.iterations % rewire_interval == 1`` (``rewire_interval <= 0``: never).

    ``compile(optimizer, loss, metrics)`` takes an optimizer with ``zero_grad()``, ``step()``, ``iterations`` and
    ``update_sparse(layer)`` (``SparseAdam``), a loss called as ``loss(y_true, y_pred)`` and metrics with
    ``update_state(y_true, y_pred)`` / ``result()``.  Several optimizers may be given as a list: they are stepped
    together and the first one that has ``update_sparse`` does the rewiring (torch models often keep a stock optimizer
    for their dense layers).
    """

    def __init__(self, rewire_interval: int, base_model: torch.nn.Module):
        super().__init__()
        self.rewire_interval = int(rewire_interval)
        self.base_model = base_model
        self.optimizers = []
        self.loss = None
        self.metrics = []

    def forward(self, *args, **kwargs):
        return self.base_model(*args, **kwargs)

    def compile(self, optimizer, loss, metrics=()):
        self.optimizers = list(optimizer) if isinstance(optimizer, (list, tuple)) else [optimizer]
        if not any(hasattr(o, "update_sparse") for o in self.optimizers):
            raise TypeError("one of the optimizers must have update_sparse(layer)")
        self.loss = loss
        self.metrics = list(metrics)

    @property
    def optimizer(self):
        """The optimizer that rewires (the reference's single optimizer)."""
        return next(o for o in self.optimizers if hasattr(o, "update_sparse"))

    def sparse_layers(self):
        return [m for m in self.base_model.modules() if hasattr(m, "sparse_weights")]

    def train_step(self, data):
        x, y = data
        for o in self.optimizers:
            o.zero_grad()
        if self._steps_directly(x):
            return self._direct_step(x, y)
        y_pred = self.base_model(x)
        loss = self.loss(y, y_pred)
        loss.backward(metrics_mod.unit_gradient(loss))
        for o in self.optimizers:
            o.step()
        self.handle_sparse_layers()
        with torch.no_grad():
            loss, y_pred = loss.detach(), y_pred.detach()
            hits, loss_value = self._shared_hits(y, y_pred, loss)
            results = {"loss": float(loss) if loss_value is None else loss_value}
            for m in self.metrics:
                if hits is not None and type(m) is metrics_mod.PrecisionAtK:
                    m._add_hits(hits, y_pred.shape[0])
                else:
                    m.update_state(y, y_pred)
                results[getattr(m, "name", type(m).__name__)] = m.result()
        return results

    def _steps_directly(self, x):
        """Whether the step is the layer, one of the library's losses and their gradients with respect to the layer's two
        variables, with nobody to see the graph in between: ``_direct_step`` then calls the library without one.  Everything a
        caller may have put there -- another model or loss, other calls on their classes, hooks on modules, variables or saved tensors, modes, transforms,
        forward derivatives, anomaly detection, tracing -- and everything that is refused takes the general way."""
        layer = self.base_model
        if (type(layer) not in _DIRECT_LAYERS or type(self.loss) not in _DIRECT_LOSSES or type(x) is not torch.Tensor
                or x.requires_grad or x.dtype != torch.float32 or not x.is_cuda or x.dim() != 2 or x.shape[1] != layer.input_dim
                or not x.shape[0] or not layer.use_bias):
            return False
        if (not torch.is_grad_enabled() or torch.is_inference_mode_enabled() or torch.is_anomaly_enabled()
                or torch.compiler.is_compiling() or torch._C._get_tracing_state() is not None
                or torch._C._are_functorch_transforms_active() or torch._C._len_torch_dispatch_stack()
                or torch._C._len_torch_function_stack() or _saved_tensor_hooks(False) is not None or forward_ad._current_level >= 0):
            return False
        if not _as_defined(type(layer)) or not _as_defined(type(self.loss)):
            return False
        if _has_global_hook() or any(layer.__dict__[name] for name in _MODULE_HOOKS) or not _OVERRIDABLE.isdisjoint(layer.__dict__):
            return False
        for variable in (layer._parameters.get("kernel_weights"), layer._parameters.get("bias")):
            if (type(variable) is not torch.nn.Parameter or not variable.requires_grad or variable.grad is not None
                    or variable._backward_hooks or getattr(variable, "_post_accumulate_grad_hooks", None)
                    or variable.device != x.device or variable.dtype != torch.float32 or not variable.is_contiguous()):
                return False
        return all(type(m) is metrics_mod.PrecisionAtK and 1 <= m._k <= metrics_mod.MAX_TOPK for m in self.metrics) and bool(self.metrics)

    @torch.no_grad()
    def _direct_step(self, x, y):
        """The step through the library's own calls: scores, loss, loss gradient and best labels, gradients of the variables,
        optimizer; then one wait for all that the step reports.  (32 x 768 x 131,072 x 32 on the general way: 243 us, of which
        the GPU works 120 -- the graph, its engine's thread and the calls from it; 151 so.)"""
        layer = self.base_model
        weights, bias, lookup = layer.kernel_weights, layer.bias, layer.kernel_indices.view(-1, layer.fan_in)
        by_label = weights.view(-1, layer.fan_in)
        labels = metrics_mod._labels(y, x.device)
        k = max(m._k for m in self.metrics)
        batch, units = x.shape[0], layer.units
        in_one = batch * units >= _SCORES_IN_ONE_KERNEL
        if in_one:
            _, out_grad, loss_sum, (_, top) = metrics_mod.forward_loss(x, lookup, by_label, bias, labels, self.loss.kind, topk=k)
        else:
            scores = _forward_bias(x, lookup, by_label, bias, False)
            out_grad, loss_sum = metrics_mod.sparse_loss_grad(scores, labels, self.loss.kind)
        _, weight_grad, bias_grad = _backward_bias(x, lookup, by_label, out_grad, False, need_feature_grad=False)
        weight_grad = weight_grad.view(-1)
        # (looked for here, where the GPU has work and the host has time: it takes some 15 us)
        with torch.enable_grad():
            held = _is_held(weights) or _is_held(bias)
        if held:
            torch.autograd.backward((weights, bias), (weight_grad, bias_grad))
        else:
            weights.grad, bias.grad = weight_grad, bias_grad
        for o in self.optimizers:
            o.step()
        self.handle_sparse_layers()
        if not in_one:
            _, top = topk_scores(scores, k)
        hits = metrics_mod.topk_hits(top, k, labels, loss_sum)
        results = {"loss": ctypes.c_float(hits[k] / (batch * units)).value}         # (a float32 mean, as a loss returns it)
        for m in self.metrics:
            m._add_hits(hits[:k], batch)
            results[m.name] = m.result()
        return results

    def _shared_hits(self, y, y_pred, loss):
        """``(hits per rank, loss)`` of the step for all its ``PrecisionAtK``: the best labels of the largest k begin with those
        of every smaller one, so one top-k, one count and one wait serve them all, and the loss comes with them."""
        ks = [m._k for m in self.metrics if type(m) is metrics_mod.PrecisionAtK]
        if not ks or not y_pred.is_cuda or y_pred.dim() != 2 or y_pred.dtype != torch.float32 or not y_pred.shape[0]:
            return None, None
        k = max(ks)
        if min(ks) < 1 or k > metrics_mod.MAX_TOPK:
            return None, None
        _, top = topk_scores(y_pred, k)
        along = loss if loss.device == y_pred.device and loss.dtype == torch.float32 and loss.numel() == 1 else None
        hits = metrics_mod.topk_hits(top, k, y, along)
        return hits[:k], hits[k] if along is not None else None

    def handle_sparse_layers(self):
        if self.rewire_interval > 0 and self.optimizer.iterations % self.rewire_interval == 1:
            for layer in self.sparse_layers():
                self.optimizer.update_sparse(layer)


class RewireCallback:
    """Rewires every sparse layer at the start of each epoch but the first (sparse/optimizer.py:77-86)."""

    def __init__(self, model: "SparseOptWrapper"):
        self.model = model

    def on_epoch_begin(self, epoch, logs=None):
        if epoch != 0:
            for layer in self.model.sparse_layers():
                self.model.optimizer.update_sparse(layer)


def backward_sparse_adam(features, lookup, weights, out_grad, nz_words, weight_m, weight_v, bias, bias_m, bias_v,
                         learning_rate, beta_1, beta_2, epsilon, step, transposed=False, grad_is_partial=False,
                         max_density=None, need_feature_grad=True, decide_from_previous=False):
    """Backward pass of the layer and the Adam step on its weights (and bias, unless ``None``) in one call:
    ``weights``, ``bias`` and their moments are updated in place; the weight/bias gradients stay inside the
    library (gradient rows of labels without a non-zero entry of ``out_grad`` are neither written nor read).  Returns ``(feature_grad or None, sparse_kernels_ran)``;
    ``feature_grad`` is formed from the weights as they were on entry."""
    import ctypes

    from .fixed_fan_in_ops import _check_inputs

    batch, num_features, num_units, fan_in = _check_inputs(features, lookup, weights, transposed, out_grad)
    for name, t in (("weights", weights), ("weight_m", weight_m), ("weight_v", weight_v), ("out_grad", out_grad),
                    ("features", features), ("lookup", lookup)):
        if not t.is_contiguous():
            raise ValueError(f"{name} must be contiguous (it is updated or read in place)")
    for name, t in (("weight_m", weight_m), ("weight_v", weight_v)):
        if t.dtype != torch.float32 or t.numel() != weights.numel() or t.device != weights.device:
            raise TypeError(f"{name} must be a float32 tensor with as many elements as weights, on their device")
    if bias is not None:
        for name, t in (("bias", bias), ("bias_m", bias_m), ("bias_v", bias_v)):
            if t is None or t.dtype != torch.float32 or t.numel() != num_units or not t.is_contiguous() or t.device != weights.device:
                raise TypeError(f"{name} must be a contiguous float32 tensor of {num_units} elements on the weights' device")
    taken = ctypes.c_int(-1)
    with _on(features.device):
        feature_grad = torch.empty_like(features) if need_feature_grad else None
        _lib.check(_lib.lib().ffi_backward_sparse_adam_f32(
            features.data_ptr(), lookup.data_ptr(), weights.data_ptr(), out_grad.data_ptr(),
            nz_words.data_ptr() if nz_words is not None else None,
            int(bool(grad_is_partial)) | (2 if decide_from_previous else 0), float(max_density or 0.0),
            feature_grad.data_ptr() if need_feature_grad else None, weight_m.data_ptr(), weight_v.data_ptr(),
            bias.data_ptr() if bias is not None else None, bias_m.data_ptr() if bias is not None else None,
            bias_v.data_ptr() if bias is not None else None,
            float(learning_rate), float(beta_1), float(beta_2), float(epsilon), int(step), ctypes.byref(taken),
            batch, num_features, num_units, fan_in, int(transposed), _stream_handle(features.device)))
    return feature_grad, bool(taken.value)
