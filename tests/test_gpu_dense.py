"""Layers of few columns: the kernels that write rows out and multiply on the matrix cores, against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle
from conftest import load_package, reference_law_inputs, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture()
def ffi():
    pkg = load_package()
    lib = pkg._lib.lib()
    assert lib.ffi_set_option(b"dense_rows", 1) == 0 and lib.ffi_set_option(b"small_path", -1) == 0
    yield pkg
    assert lib.ffi_set_option(b"dense_rows", 0) == 0 and lib.ffi_set_option(b"small_path", 0) == 0


# (B, N, L, K): one of everything; blocks of 32 columns and of 32 samples, groups of 128 samples, tiles of 64 labels and eights of
# connections, full and with remainders; more connections than columns; more tiles than wavefronts
SHAPES = [(1, 1, 1, 1), (32, 32, 64, 8), (33, 33, 65, 9), (31, 17, 63, 7), (64, 64, 128, 64), (65, 63, 129, 65), (128, 32, 700, 33), (129, 64, 300, 100),
          (260, 12, 130, 31), (300, 40, 1000, 130), (5, 16, 150_000, 3), (40, 50, 90_001, 4)]


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_few_columns(ffi, shape, transposed):
    B, N, L, K = shape
    x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=B + N)
    xt = np.ascontiguousarray(x.T if transposed else x)
    bias = np.linspace(-1, 1, L).astype(np.float32)
    ref = oracle.forward(x, lookup, w, transposed=False)
    ref_gx, ref_gw = oracle.backward(xt, lookup, w, g, transposed=transposed)
    dx, dl, dw, dg, db = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (xt, lookup, w, g, bias))
    forward, grad = (ffi.fan_in_sparse_matmul_tp, ffi.fan_in_sparse_matmul_grad_tp) if transposed else (ffi.fan_in_sparse_matmul, ffi.fan_in_sparse_matmul_grad)
    with_bias = ffi.fan_in_sparse_matmul_tp_bias if transposed else ffi.fan_in_sparse_matmul_bias
    assert rel_err(forward(dx, dl, dw).cpu().numpy(), ref) <= 1e-6
    first = None
    for _ in range(2):
        gx, gw = grad(dx, dl, dw, dg)
        assert rel_err(gx.cpu().numpy(), ref_gx) <= 1e-5 and rel_err(gw.cpu().numpy(), ref_gw) <= 1e-5
        assert first is None or (torch.equal(first[0], gx) and torch.equal(first[1], gw))
        first = gx, gw
    for need_x in (True, False):
        variables = [dx.clone().requires_grad_(need_x), dw.clone().requires_grad_(True), db.clone().requires_grad_(True)]
        out = with_bias(variables[0], dl, variables[1], variables[2])
        assert rel_err(out.detach().cpu().numpy(), ref + bias) <= 1e-6
        grads = torch.autograd.grad(out, [v for v in variables if v.requires_grad], dg)
        assert rel_err(grads[-2].cpu().numpy(), ref_gw) <= 1e-5 and rel_err(grads[-1].cpu().numpy(), g.astype(np.float64).sum(0)) <= 1e-5
    lib, stream = ffi._lib.lib(), torch.cuda.current_stream().cuda_stream
    gx = torch.full_like(dx, float("nan"))
    ffi._lib.check(lib.ffi_input_grad_f32(dl.data_ptr(), dw.data_ptr(), dg.data_ptr(), gx.data_ptr(), B, N, L, K, int(transposed), stream))
    assert rel_err(gx.cpu().numpy(), ref_gx) <= 1e-5


@pytest.mark.parametrize("transposed", [False, True])
def test_what_is_not_finite_stays_with_its_connections(ffi, transposed):
    # columns 3 and 7 hold an infinity and a NaN, label 70 an infinite gradient, label 5 an infinite weight; a weight of 0 meets an infinity
    B, N, L, K = 40, 20, 200, 4
    x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=3)
    lookup[lookup == 3] = 4
    lookup[lookup == 7] = 8
    lookup[10, 1], lookup[11, 2], w[11, 2], lookup[12, 0] = 3, 3, 0.0, 7
    x[1, 3], x[2, 7] = np.inf, np.nan
    g[6, 70], g[7, 71] = -np.inf, np.nan
    w[5, 0] = np.inf
    ref = np.zeros((B, L), np.float64)
    gx_ref, gw_ref = np.zeros((B, N), np.float64), np.zeros((L, K), np.float64)
    with np.errstate(invalid="ignore"):
        for k in range(K):
            ref += w[:, k].astype(np.float64) * x[:, lookup[:, k]]
            gw_ref[:, k] = (g.astype(np.float64) * x[:, lookup[:, k]]).sum(0)
            for l in range(L):
                gx_ref[:, lookup[l, k]] += g[:, l].astype(np.float64) * w[l, k]
    args = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x.T if transposed else x, lookup, w, g)]
    forward, grad = (ffi.fan_in_sparse_matmul_tp, ffi.fan_in_sparse_matmul_grad_tp) if transposed else (ffi.fan_in_sparse_matmul, ffi.fan_in_sparse_matmul_grad)
    for _ in range(2):
        out = forward(*args[:3]).cpu().numpy()
        gx, gw = (t.cpu().numpy() for t in grad(*args))
        for got, want in ((out, ref), (gx.T if transposed else gx, gx_ref), (gw, gw_ref)):
            np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
            np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
            ok = np.isfinite(want)
            np.testing.assert_allclose(got[ok], want[ok], rtol=1e-5, atol=1e-5)
    clean = [torch.from_numpy(np.ascontiguousarray(np.nan_to_num(a, posinf=1.0, neginf=1.0))).cuda() if a.dtype == np.float32 else torch.from_numpy(a).cuda()
             for a in (np.ascontiguousarray(x.T if transposed else x), lookup, w, g)]
    gx, _ = grad(*clean)                                               # (nothing is left of the call before)
    assert bool(torch.isfinite(gx).all())


@pytest.mark.parametrize("B,N", [(40, 20), (130, 50)])
@pytest.mark.parametrize("transposed", [False, True])
def test_weights_that_add_up_to_no_finite_number(ffi, transposed, B, N):
    # an infinite weight under an infinite gradient; weights of one column whose sum overflows and whose products with what they meet, zeros among
    # that, do not; infinities that cancel; all of it beside other connections of the label, and in the last label
    L, K = 200, 6
    x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=5)
    x *= 0.1
    g *= 0.1
    lookup[70], w[70, 2], g[6, 70], g[7, 70] = np.arange(K), np.inf, -np.inf, np.inf
    for l in (30, L - 1):
        lookup[l] = [4, 9, 4, 9, 11, 12]
        w[l, 0] = w[l, 2] = 3e38
        w[l, 1] = w[l, 3] = -2.5e38
    x[3, 4] = x[5, 9] = g[2, 30] = g[8, L - 1] = 0.0
    lookup[100], w[100, 0], w[100, 3] = [15, 1, 2, 15, 3, 3], np.inf, -np.inf
    g[9, 100] = np.nan
    ref = np.zeros((B, L), np.float64)
    gx_ref, gw_ref = np.zeros((B, N), np.float64), np.zeros((L, K), np.float64)
    with np.errstate(invalid="ignore"):
        for k in range(K):
            ref += w[:, k].astype(np.float64) * x[:, lookup[:, k]]
            gw_ref[:, k] = (g.astype(np.float64) * x[:, lookup[:, k]]).sum(0)
            for l in range(L):
                gx_ref[:, lookup[l, k]] += g[:, l].astype(np.float64) * w[l, k]
    args = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x.T if transposed else x, lookup, w, g)]
    forward, grad = (ffi.fan_in_sparse_matmul_tp, ffi.fan_in_sparse_matmul_grad_tp) if transposed else (ffi.fan_in_sparse_matmul, ffi.fan_in_sparse_matmul_grad)
    for _ in range(2):
        out = forward(*args[:3]).cpu().numpy()
        gx, gw = (t.cpu().numpy() for t in grad(*args))
        for got, want in ((out, ref), (gx.T if transposed else gx, gx_ref), (gw, gw_ref)):
            np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
            np.testing.assert_array_equal(np.isposinf(got), np.isposinf(want))
            np.testing.assert_array_equal(np.isneginf(got), np.isneginf(want))
            ok = np.isfinite(want)
            # (products of 3e38 and 0.1, a few of them, each rounded once: their sums may be off by 2^-22 of the largest)
            np.testing.assert_allclose(got[ok], want[ok], rtol=1e-5, atol=1e-5 if np.abs(want[ok]).max() < 1e30 else 1e32)


def test_nothing_finite(ffi):
    B, N, L, K = 128, 32, 3000, 16
    x, lookup, w, g = (torch.from_numpy(a).cuda() for a in reference_law_inputs(B, N, L, K, seed=9))
    nan = float("nan")
    for xs, ws, gs in ((x, torch.full_like(w, nan), torch.full_like(g, nan)), (x, w, torch.full_like(g, nan)), (x, torch.full_like(w, nan), g)):
        gx, gw = ffi.fan_in_sparse_matmul_grad(xs, lookup, ws, gs)
        assert bool(gx.isnan().all()) and bool(gw.isnan().all()) == bool(gs.isnan().all())
    gx, gw = ffi.fan_in_sparse_matmul_grad(x, lookup, w, g)
    assert bool(gx.isfinite().all()) and bool(gw.isfinite().all())


def test_tiny_numbers_are_not_lost(ffi):
    # products and operands below the smallest normal number
    N, L, K = 8, 64, 2
    lookup = torch.arange(L * K, device="cuda", dtype=torch.int32).reshape(L, K) % N
    x = torch.full((3, N), 1e-39, device="cuda")
    w = torch.full((L, K), 0.5, device="cuda")
    assert torch.equal(ffi.fan_in_sparse_matmul(x, lookup, w), torch.full((3, L), 1e-39, device="cuda"))
    gx, gw = ffi.fan_in_sparse_matmul_grad(torch.ones_like(x), lookup, w, torch.full((3, L), 1e-40, device="cuda"))
    np.testing.assert_allclose(gw.cpu().numpy(), 3e-40, rtol=1e-4)
    np.testing.assert_allclose(gx.cpu().numpy(), L * K / N * 0.5e-40, rtol=1e-4)


def test_an_id_out_of_range_is_reported_by_the_next_call(ffi):
    x, lookup, w, g = (torch.from_numpy(a).cuda() for a in reference_law_inputs(4, 50, 300, 6, seed=1))
    ffi.fan_in_sparse_matmul_grad(x, lookup, w, g)
    lookup[3, 2] = 50
    _, gw = ffi.fan_in_sparse_matmul_grad(x, lookup, w, g)
    torch.cuda.synchronize()
    assert float(gw[3, 2]) == 0.0
    with pytest.raises(ffi._lib.FfiError):
        ffi.fan_in_sparse_matmul_grad(x, lookup, w, g)
    lookup[3, 2] = 49
    ffi.fan_in_sparse_matmul_grad(x, lookup, w, g)


# More than one group of 128 samples: few labels' samples are spread over the CUs by the other kernels
@pytest.mark.parametrize("shape", [(641, 32, 1035, 94), (1433, 32, 852, 126), (391, 32, 16_682, 40), (271, 64, 20_608, 92)])
def test_many_samples_of_few_labels_take_the_other_kernels(shape):
    _default_and_others(shape, True)


@pytest.mark.parametrize("shape", [(20_000, 32, 1300, 14), (3000, 64, 1300, 30), (250, 43, 12_000, 20), (1200, 32, 12_000, 20), (2500, 32, 33_000, 6)])
def test_weight_gradients_of_many_samples_take_the_other_kernels(shape):
    _default_and_others(shape, False)


def _default_and_others(shape, input_gradient):
    # (the same kernels add in the same order)
    B, N, L, K = shape
    lib, stream = load_package()._lib.lib(), torch.cuda.current_stream().cuda_stream
    x, lookup, w, g = (torch.from_numpy(a).cuda() for a in reference_law_inputs(B, N, L, K, seed=L))
    results = []
    try:
        for dense in (0, -1):
            assert lib.ffi_set_option(b"dense_rows", dense) == 0
            gx, gw = torch.zeros_like(x), torch.empty_like(w)
            assert lib.ffi_backward_f32(x.data_ptr(), lookup.data_ptr(), w.data_ptr(), g.data_ptr(), gx.data_ptr() if input_gradient else None, gw.data_ptr(),
                                        B, N, L, K, 0, stream) == 0
            results.append((gx, gw))
    finally:
        assert lib.ffi_set_option(b"dense_rows", 0) == 0
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
