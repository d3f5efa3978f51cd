"""Adam step (`ffi_adam_step_f32`) and the SparseAdam object against the numpy oracle
(oracle.adam_step, pinned in tests/test_oracle.py by the closed form of the first step and by
torch.optim.Adam with Keras' epsilon placement).  Gate: 2e-6 absolute on variables of order one,
1e-6 of the largest magnitude on the moments (float32 arithmetic on both sides; fused multiply-adds
differ in the last bit).
"""
import numpy as np
import pytest
import torch

import oracle
from conftest import load_package, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ffi():
    pkg = load_package()
    assert torch.cuda.is_available(), "these tests need the MI355X"
    return pkg


@pytest.mark.parametrize("count", [1, 3, 4, 1023, 5000 * 32, 1_000_003])
def test_adam_steps_against_oracle(ffi, count):
    rng = np.random.default_rng(count)
    w = rng.normal(size=count).astype(np.float32)
    m, v = np.zeros(count, np.float32), np.zeros(count, np.float32)
    wt, mt, vt = (torch.from_numpy(a.copy()).cuda() for a in (w, m, v))
    for step in range(1, 6):
        g = (rng.normal(size=count) * (rng.random(count) < 0.6)).astype(np.float32)
        w, m, v = oracle.adam_step(w, m, v, g, learning_rate=0.002, step=step)
        ffi.optimizer.adam_step(wt, mt, vt, torch.from_numpy(g).cuda(), 0.002, 0.9, 0.999, 1e-7, step)
        torch.cuda.synchronize()
        np.testing.assert_allclose(wt.cpu().numpy(), w, rtol=0, atol=2e-6)
        assert rel_err(mt.cpu().numpy(), m) <= 1e-6
        assert rel_err(vt.cpu().numpy(), v) <= 1e-6


def test_adam_argument_errors(ffi):
    lib = ffi._lib.lib()
    a = torch.zeros(8, device="cuda")
    p = a.data_ptr()
    sh = torch.cuda.current_stream().cuda_stream
    assert lib.ffi_adam_step_f32(None, p, p, p, 8, 0.1, 0.9, 0.999, 1e-7, 1, sh) == -1
    assert lib.ffi_adam_step_f32(p, p, p, p, 0, 0.1, 0.9, 0.999, 1e-7, 1, sh) == -2
    assert lib.ffi_adam_step_f32(p, p, p, p, 8, 0.1, 0.9, 0.999, 1e-7, 0, sh) == -8       # steps count from 1
    assert lib.ffi_adam_step_f32(p + 4, p, p, p, 4, 0.1, 0.9, 0.999, 1e-7, 1, sh) == -8   # alignment


def test_training_loop_reduces_the_loss_and_rewires(ffi):
    # the reference's train step (sparse/optimizer.py:43-74): forward, loss, gradients, Adam, rewire
    gen = torch.Generator(device="cuda").manual_seed(11)
    B, N, L = 64, 128, 2000
    # arrange=False: positions keep their meaning across a rewire, so the moved ones can be named below
    layer = ffi.StratifiedRewireLayerV2(units=L, input_dim=N, connections=L * 16, generator=gen, arrange=False,
                                        rewire_selector=ffi.FixedFractionSelector(0.05))
    opt = ffi.SparseAdam(list(layer.parameters()), learning_rate=0.01)
    loss_fn = ffi.SparseSquaredHingeLoss()
    x = torch.rand((B, N), device="cuda", generator=gen)
    rows = torch.arange(B, device="cuda").repeat_interleave(3)
    cols = torch.randint(0, L, (B * 3,), device="cuda", generator=gen)
    y = (torch.stack([rows, cols], dim=1), None)
    losses = []
    for it in range(1, 41):
        opt.zero_grad()
        loss, _ = layer.forward_loss(x, y, loss_fn)
        loss.backward()
        opt.step()
        losses.append(float(loss.detach()))
        if it % 10 == 1:
            before = layer.kernel_indices.clone()
            opt.update_sparse(layer)
            moved = (layer.kernel_indices != before)
            i = opt._index_of(layer.kernel_weights)
            if moved.any():
                assert not opt._momentums[i][moved].any() and not opt._velocities[i][moved].any()
    assert losses[-1] < 0.5 * losses[0]
    assert opt.iterations == 40


@pytest.mark.parametrize("force_dense", [False, True])
@pytest.mark.parametrize("shape", [(96, 384, 3000, 32, True), (37, 300, 1001, 7, False), (64, 200, 900, 72, False)])
def test_backward_with_adam_epilogue_matches_backward_then_adam(ffi, shape, force_dense):
    # ffi_backward_sparse_adam_f32 against ffi_backward_sparse_f32 followed by ffi_adam_step_f32 (each of them
    # tested against the oracle on its own), two steps in a row, on the sparse kernels and on the dense ones
    B, N, L, K, tp = shape
    rng = np.random.default_rng(sum(shape[:4]))
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    x = dev(np.maximum(rng.standard_normal((N, B) if tp else (B, N)), 0).astype(np.float32))
    lookup = dev(rng.integers(0, N, size=(L, K)).astype(np.int32))
    state = {}
    for fused in (False, True):
        w = dev(rng.standard_normal((L, K)).astype(np.float32)) if not state else state["w0"].clone()
        bias = dev(rng.standard_normal(L).astype(np.float32)) if not state else state["b0"].clone()
        if not state:
            state["w0"], state["b0"] = w.clone(), bias.clone()
            state["g"] = []
            for _ in range(2):
                g = rng.standard_normal((B, L)).astype(np.float32)
                g[rng.random((B, L)) >= 0.01] = 0.0
                g[:, 3] = rng.standard_normal(B)
                state["g"].append(dev(g))
        mw, vw, mb, vb = torch.zeros_like(w), torch.zeros_like(w), torch.zeros_like(bias), torch.zeros_like(bias)
        gxs = []
        for step, g in enumerate(state["g"], start=1):
            md = 1e-9 if force_dense else 1.0
            if fused:
                gx, sparse = ffi.optimizer.backward_sparse_adam(x, lookup, w, g.clone(), None, mw, vw, bias, mb, vb,
                                                                0.01, 0.9, 0.999, 1e-7, step, transposed=tp, max_density=md)
            else:
                gx, gw, gb, sparse = ffi.backward_sparse(x, lookup, w, g, transposed=tp, max_density=md, need_bias_grad=True)
                ffi.optimizer.adam_step(w, mw, vw, gw, 0.01, 0.9, 0.999, 1e-7, step)
                ffi.optimizer.adam_step(bias, mb, vb, gb, 0.01, 0.9, 0.999, 1e-7, step)
            assert sparse == (not force_dense)
            gxs.append(gx)
        torch.cuda.synchronize()
        state["fused" if fused else "plain"] = [t.cpu().numpy() for t in (w, mw, vw, bias, mb, vb, *gxs)]
    for a, b in zip(state["fused"], state["plain"]):
        assert rel_err(a, b) <= 1e-5


@pytest.mark.parametrize("share", [0.0, 0.02, 1.0])
@pytest.mark.parametrize("shape", [(5, 30, 1, 4), (33, 40, 63, 7), (70, 64, 257, 32), (32, 50, 1300, 40), (3, 9, 5000, 1), (40, 300, 300, 260)])
def test_step_on_rows_with_and_without_gradient(ffi, shape, share):
    # rows of both kinds side by side, none of one kind, labels that the whole wavefront takes (share 1: every sample's bit), mask bits
    # behind the batch, and the count that the next call decides from
    B, N, L, K = shape
    rng = np.random.default_rng(sum(shape) + int(100 * share))
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    x, lookup = rng.standard_normal((B, N)).astype(np.float32), rng.integers(0, N, (L, K)).astype(np.int32)
    g = rng.standard_normal((B, L)).astype(np.float32)
    g[rng.random((B, L)) >= share] = 0.0
    words = np.full(((B + 31) // 32, L), 0, dtype=np.uint32)
    for b in range(B):
        words[b // 32] |= (g[b] != 0).astype(np.uint32) << np.uint32(b % 32)
    if B % 32:
        words[-1] |= np.uint32(0x80000000)
    w0, b0 = rng.standard_normal((L, K)).astype(np.float32), rng.standard_normal(L).astype(np.float32)
    start = [w0, 0.1 * rng.standard_normal((L, K)).astype(np.float32), rng.random((L, K)).astype(np.float32),
             b0, 0.1 * rng.standard_normal(L).astype(np.float32), rng.random(L).astype(np.float32)]
    w, mw, vw, bias, mb, vb = [dev(a) for a in start]
    _, sparse = ffi.optimizer.backward_sparse_adam(dev(x), dev(lookup), w, dev(g), dev(words.view(np.int32)), mw, vw, bias, mb, vb,
                                                   0.01, 0.9, 0.999, 1e-7, 3, max_density=4.0, need_feature_grad=False)
    assert sparse
    gw = np.zeros((L, K))
    for k in range(K):
        gw[:, k] = (g.astype(np.float64) * x.astype(np.float64)[:, lookup[:, k]]).sum(axis=0)
    alpha = 0.01 * np.sqrt(1.0 - 0.999 ** 3) / (1.0 - 0.9 ** 3)
    for got, (var, m, v), grad in (((w, mw, vw), start[:3], gw), ((bias, mb, vb), start[3:], g.astype(np.float64).sum(axis=0))):
        m1 = m + (grad - m) * 0.1
        v1 = v + (grad * grad - v) * 0.001
        for a, ref in zip(got, (var - m1 * alpha / (np.sqrt(v1) + 1e-7), m1, v1)):
            assert rel_err(a.cpu().numpy(), ref.astype(np.float32)) <= 1e-5
    # the density that the call has found decides for the next one of the shape
    found = sum(int(np.unpackbits(words[t].view(np.uint8)).sum()) for t in range(words.shape[0])) - (L if B % 32 else 0)
    for limit, expected in (((found + 0.5) / (B * L), True), ((found - 0.5) / (B * L), False)):
        if limit <= 0.0:
            continue
        _, sparse = ffi.optimizer.backward_sparse_adam(dev(x), dev(lookup), w, dev(g), dev(words.view(np.int32)), mw, vw, bias, mb, vb,
                                                       0.01, 0.9, 0.999, 1e-7, 4, max_density=limit, need_feature_grad=False,
                                                       decide_from_previous=True)
        torch.cuda.synchronize()
        assert sparse == expected


@pytest.mark.parametrize("shape,share", [((64, 30, 259, 5), 0.005), ((33, 20, 130, 6), 0.02), ((32, 40, 193, 13), 0.01), ((20, 30, 67, 4), 0.02),
                                         ((16, 9, 1001, 2), 0.03), ((24, 9, 1001, 3), 0.02), ((8, 9, 900_001, 2), 0.005), ((8, 9, 900_001, 5), 0.005)])
def test_step_on_rows_that_share_sixteen_bytes(ffi, shape, share):
    # some of the rows have a gradient: sixteen bytes that lie in a row of either kind, at the end of a wavefront's 64 labels and of the layer,
    # rows shorter than that, and layers of so many labels that the gradients' workgroups are limited
    test_step_on_rows_with_and_without_gradient(ffi, shape, share)


def test_fused_train_step_follows_the_unfused_loop(ffi):
    # layer.fused_train_step + optimizer.step() against forward_loss / backward / optimizer.step(), three steps
    B, N, L = 64, 128, 2000
    x = torch.rand((B, N), device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    rows = torch.arange(B, device="cuda").repeat_interleave(3)
    cols = torch.randint(0, L, (B * 3,), device="cuda", generator=torch.Generator(device="cuda").manual_seed(4))
    y = (torch.stack([rows, cols], dim=1), None)
    loss_fn = ffi.SparseSquaredHingeLoss()
    runs = []
    for fused in (False, True):
        layer = ffi.StratifiedRewireLayerV2(units=L, input_dim=N, connections=L * 16,
                                            generator=torch.Generator(device="cuda").manual_seed(5))
        with torch.no_grad():
            layer.bias.fill_(-1.05)
        opt = ffi.SparseAdam(list(layer.parameters()), learning_rate=0.01)
        losses = []
        for _ in range(3):
            opt.zero_grad()
            if fused:
                loss, _ = layer.fused_train_step(x, y, loss_fn, opt)
            else:
                loss, _ = layer.forward_loss(x, y, loss_fn)
                loss.backward()
            opt.step()
            losses.append(float(loss.detach()))
        torch.cuda.synchronize()
        runs.append((losses, layer.kernel_weights.detach().cpu().numpy(), layer.bias.detach().cpu().numpy()))
    (l0, w0, b0), (l1, w1, b1) = runs
    assert np.allclose(l0, l1, rtol=1e-5)
    assert rel_err(w1, w0) <= 1e-5 and rel_err(b1, b0) <= 1e-5
    assert l0[2] < l0[0]


def test_moments_are_rewired_in_place_or_through_an_override(ffi):
    # the optimizer edits its moments where they are, unless the layer's rewire is not the library's
    class Overridden(ffi.StratifiedRewireLayerV2):
        def rewire(self, other_vars=None):
            return super().rewire(other_vars)

    results = []
    for kind in (ffi.StratifiedRewireLayerV2, Overridden):
        gen = torch.Generator(device="cuda").manual_seed(3)
        layer = kind(units=300, input_dim=64, connections=300 * 24, generator=gen, rewire_selector=ffi.FixedFractionSelector(0.2))
        opt = ffi.SparseAdam(list(layer.parameters()), learning_rate=0.01)
        i = opt._index_of(layer.kernel_weights)
        m, v = opt._momentums[i], opt._velocities[i]
        m.normal_(generator=gen)
        v.uniform_(generator=gen)
        opt.update_sparse(layer)
        assert opt._momentums[i] is m and int((m == 0).sum()) == 300 * 24 // 5 - 1        # (strictly below the k-th smallest)
        results.append((layer.kernel_indices, layer.kernel_weights.detach(), m, v))
    assert layer.rewires_in_place() is False
    assert all(torch.equal(a, b) for a, b in zip(*results))


def _training(ffi, *, batch=20, features=40, labels=500, fan_in=6, loss=None, values=True, rewire=0, layer_class=None, ks=(1, 3, 5), optimizer=None):
    gen = torch.Generator(device="cuda").manual_seed(batch + labels)
    layer = (layer_class or ffi.StratifiedRewireLayerV2)(labels, features, connections=labels * fan_in, generator=gen,
                                                         rewire_selector=ffi.FixedFractionSelector(0.1))
    wrapper = ffi.SparseOptWrapper(rewire, layer)
    adam = ffi.SparseAdam(layer.parameters(), learning_rate=0.01)
    wrapper.compile(optimizer(layer, adam) if optimizer else adam, loss or ffi.SparseSquaredHingeLoss(), [ffi.PrecisionAtK(k) for k in ks])
    x = torch.rand((batch, features), device="cuda", generator=gen)
    flat = torch.randperm(batch * labels, device="cuda", generator=gen)[:3 * batch]
    y = (torch.stack([flat // labels, flat % labels], dim=1), torch.rand(3 * batch, device="cuda", generator=gen) if values else None)
    return wrapper, layer, adam, x, y


def _after_steps(wrapper, layer, adam, x, y, steps=4):
    results = [wrapper.train_step((x, y)) for _ in range(steps)]
    state = [layer.kernel_weights.data, layer.bias.data, layer.kernel_weights.grad, layer.bias.grad, layer.kernel_indices, *adam._momentums, *adam._velocities]
    return results, [t.clone() for t in state]


@pytest.mark.parametrize("case", [dict(), dict(batch=1, labels=33, fan_in=3), dict(batch=129, features=1300, labels=700, fan_in=33), dict(values=False),
                                  dict(batch=70, features=1217, labels=240_000, fan_in=1),        # (scores, gradients and ranks in one kernel)
                                  dict(batch=64, labels=262_144, fan_in=4), dict(rewire=2), dict(rewire=2, layer_class="StratifiedRewireLayer"),
                                  dict(loss="SparseBinaryCrossEntropyLoss"), dict(loss="SparseHingeLoss", ks=(8,)),
                                  dict(optimizer=lambda layer, adam: [torch.optim.SGD([layer.bias], lr=0.1), adam])])
def test_a_step_without_a_graph_is_the_step_with_one(ffi, case):
    case = {**case, **({"loss": getattr(ffi, case["loss"])()} if "loss" in case else {})}
    case = {**case, **({"layer_class": getattr(ffi, case["layer_class"])} if "layer_class" in case else {})}
    direct, general = _training(ffi, **case), _training(ffi, **case)
    assert direct[0]._steps_directly(direct[3])
    seen = []
    general[1].register_forward_hook(lambda *_: seen.append(1) and None)
    got, want = _after_steps(*direct), _after_steps(*general)
    assert len(seen) == 4
    for a, b in zip(got[0], want[0]):
        assert a.keys() == b.keys() and all(abs(a[key] - b[key]) <= 1e-6 * abs(b[key]) for key in a), (a, b)
    one_kernel = case.get("batch", 20) * case.get("labels", 500) >= 1 << 24
    for a, b in zip(got[1], want[1]):
        assert torch.equal(a, b) or (one_kernel and rel_err(a.cpu().numpy(), b.cpu().numpy()) <= 1e-5)      # (sums in another order)


def test_what_a_caller_put_into_a_step_still_runs(ffi):
    calls = []
    note = lambda *_: calls.append(1) and None

    class OwnLoss(type(ffi.SparseSquaredHingeLoss())):
        def __call__(self, y_true, y_pred):
            calls.append(1)
            return super().__call__(y_true, y_pred) * 2

    class OwnLayer(ffi.StratifiedRewireLayerV2):
        def forward(self, inputs):
            calls.append(1)
            return super().forward(inputs)

    class OwnMetric(ffi.PrecisionAtK):
        def update_state(self, y_true, y_pred, sample_weight=None):
            calls.append(tuple(y_pred.shape))

    def own_forward(wrapper, layer, x):
        plain = layer.forward
        layer.forward = lambda inputs: (calls.append(1), plain(inputs))[1]

    puts = [lambda wrapper, layer, x: layer.register_forward_pre_hook(note), lambda wrapper, layer, x: layer.register_forward_hook(note),
            lambda wrapper, layer, x: layer.register_full_backward_hook(note), lambda wrapper, layer, x: layer.kernel_weights.register_hook(note),
            lambda wrapper, layer, x: layer.bias.register_post_accumulate_grad_hook(note), own_forward,
            lambda wrapper, layer, x: wrapper.metrics.append(OwnMetric(1))]
    for put in puts:
        wrapper, layer, _, x, y = _training(ffi)
        put(wrapper, layer, x)
        calls.clear()
        wrapper.train_step((x, y))
        assert calls, put
    for more in (dict(loss=OwnLoss()), dict(layer_class=OwnLayer)):
        wrapper, _, _, x, y = _training(ffi, **more)
        calls.clear()
        wrapper.train_step((x, y))
        assert calls, more
    wrapper, _, _, x, y = _training(ffi)
    calls.clear()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (calls.append(1), t)[1], lambda t: t):
        wrapper.train_step((x, y))
    assert calls
    hook = torch.nn.modules.module.register_module_forward_hook(note)
    try:
        calls.clear()
        wrapper.train_step((x, y))
        assert calls
    finally:
        hook.remove()
    # the gradient of the input, a variable that is held fixed, gradients that add up; what is refused
    x.requires_grad_(True)
    wrapper.train_step((x, y))
    assert x.grad is not None
    wrapper, layer, _, x, y = _training(ffi)
    layer.bias.requires_grad_(False)
    wrapper.train_step((x, y))
    assert layer.bias.grad is None and not layer.bias.any()
    wrapper, layer, adam, x, y = _training(ffi)
    adam.zero_grad = lambda: None
    wrapper.train_step((x, y))
    first = layer.bias.grad.clone()
    layer.bias.grad.fill_(1.0)
    wrapper.train_step((x, y))
    assert float((layer.bias.grad - 1.0).abs().max()) <= 10 * float(first.abs().max())
    with pytest.raises(ValueError):
        wrapper.train_step((x[:, 1:], y))
    with pytest.raises(RuntimeError), torch.no_grad():
        wrapper.train_step((x, y))


def _accumulation_node(variable):
    return variable.expand_as(variable).grad_fn.next_functions[0][0]


@pytest.mark.parametrize("variable", ["kernel_weights", "bias"])
@pytest.mark.parametrize("before", [False, True])
def test_hooks_on_the_node_that_adds_a_gradient_up_run(ffi, variable, before):
    # where libraries that exchange gradients hang theirs: behind the sum, and ahead of it with a gradient to change
    kept, plain = _training(ffi), _training(ffi)
    node, seen = _accumulation_node(getattr(kept[1], variable)), []
    if before:
        node.register_prehook(lambda grads: (seen.append(1), tuple(2.0 * g for g in grads))[1])
    else:
        node.register_hook(lambda *_: seen.append(1) and None)
    for steps in (1, 2):
        results = [run[0].train_step((run[3], run[4])) for run in (kept, plain)]
        assert len(seen) == steps
        if steps == 1:
            assert results[0] == results[1]
            for name in ("kernel_weights", "bias"):
                a, b = (getattr(run[1], name).grad for run in (kept, plain))
                assert torch.equal(a, 2.0 * b if before and name == variable else b)
    assert not node.metadata                                            # (nothing of the step's is left there)
    del node
    kept[0].train_step((kept[3], kept[4]))                              # (a node that nobody keeps goes, and its hooks with it)
    assert len(seen) == 2


def test_a_forward_derivative_of_a_step_is_refused(ffi):
    # as by the layer's op, which has none
    wrapper, _, _, x, y = _training(ffi)
    with torch.autograd.forward_ad.dual_level():
        with pytest.raises(RuntimeError):
            wrapper.train_step((torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)), y))
    wrapper.train_step((x, y))


def test_calls_replaced_on_a_class_are_made(ffi, monkeypatch):
    calls = []

    def counted(call):
        return lambda *args, **kwargs: (calls.append(1), call(*args, **kwargs))[1]

    for owner, name in ((ffi.StratifiedRewireLayerV2, "forward"), (ffi.StratifiedRewireLayerV2, "__call__"), (torch.nn.Module, "_call_impl"),
                        (ffi.metrics.SparseLossBase, "__call__"), (ffi.SparseSquaredHingeLoss, "__call__")):
        wrapper, _, _, x, y = _training(ffi)
        with monkeypatch.context() as patch:
            patch.setattr(owner, name, counted(getattr(owner, name)))
            calls.clear()
            wrapper.train_step((x, y))
            assert calls, (owner, name)
    wrapper, layer, _, x, y = _training(ffi)
    for name in ("_call_impl", "_compiled_call_impl"):                  # (the second is what Module.compile sets)
        layer.__dict__[name] = counted(layer._call_impl)
        calls.clear()
        wrapper.train_step((x, y))
        assert calls, name
        del layer.__dict__[name]


def test_a_variable_that_is_no_parameter_of_the_layer(ffi):
    # computed from another one: the step trains that
    wrapper, layer, adam, x, y = _training(ffi)
    raw = torch.nn.Parameter(layer.kernel_weights.detach().clone())
    del layer.kernel_weights
    layer.kernel_weights = 1.0 * raw
    wrapper.compile(ffi.SparseAdam([raw, layer.bias]), wrapper.loss, wrapper.metrics)
    before = raw.detach().clone()
    assert wrapper.train_step((x, y))["loss"] > 0.0
    assert raw.grad is not None and not torch.equal(before, raw.detach())
