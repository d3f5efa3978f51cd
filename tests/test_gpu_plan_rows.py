"""The rows that a plan's build gives the labels of a tile: whatever the fan-in and however full the halves of a tile are, the input
gradient over the plan is the oracle's."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from conftest import load_package, reference_law_inputs, rel_err

pytestmark = pytest.mark.gpu


# fan-ins around the lanes of a label in either sweep; labels that leave a step of eight, and of two, part empty; columns used by
# every label (their halves fill up), evenly, and in two windows
@pytest.mark.parametrize("fan_in", [1, 2, 7, 8, 9, 31, 32, 33, 63, 64, 65, 127, 128, 129, 200])
@pytest.mark.parametrize("features,labels,skewed", [(300, 1237, False), (768, 701, True), (64, 66, True), (1100, 1309, False), (1024, 1030, False)])
def test_any_fan_in(fan_in, features, labels, skewed):
    ffi = load_package()
    lib = ffi._lib.lib()
    x, lookup, w, g = reference_law_inputs(9, features, labels, fan_in, seed=fan_in + labels)
    if skewed:
        lookup[:, : (fan_in + 1) // 2] = 5
        lookup[::3] = lookup[:1]
    dl, dw, dg = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (lookup, w, g))
    plan = ctypes.c_void_p()
    stream = torch.cuda.current_stream().cuda_stream
    ffi._lib.check(lib.ffi_plan_create(dl.data_ptr(), labels, fan_in, features, 9, stream, ctypes.byref(plan)))
    try:
        gx = torch.full((9, features), float("nan"), device="cuda")
        ffi._lib.check(lib.ffi_input_grad_planned_f32(plan, dw.data_ptr(), dg.data_ptr(), gx.data_ptr(), 9, 0, stream))
        assert rel_err(gx.cpu().numpy(), oracle.input_grad(x, lookup, w, g, transposed=False)) <= 1e-5
    finally:
        ffi._lib.check(lib.ffi_plan_destroy(plan))


@pytest.mark.parametrize("features", [768, 1100, 5000])
def test_a_plan_that_is_being_laid_out_serves_other_streams(features):
    # the call that builds the plan does not wait for it: calls on other streams come right behind, and the next edit too
    ffi = load_package()
    B, L, K = 40, 60_000, 16
    x, lookup, w, g = reference_law_inputs(B, features, L, K, seed=features)
    dx, dw, dg = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, w, g))
    shifted = [((lookup + 11 * turn) % features).astype(np.int32) for turn in range(3)]
    on_device = [torch.from_numpy(a).cuda() for a in shifted]
    dl = torch.empty_like(on_device[0])
    streams = [torch.cuda.Stream() for _ in range(3)]
    ffi._lib.check(ffi._lib.lib().ffi_cache_clear())
    for turn in range(3):
        torch.cuda.synchronize()
        dl.copy_(on_device[turn])
        ffi._lib.check(ffi._lib.lib().ffi_lookup_edited(dl.data_ptr()))
        torch.cuda.synchronize()
        results = []
        for i in range(6):
            with torch.cuda.stream(streams[(turn + i) % 3]):
                results.append(ffi.fan_in_sparse_matmul_grad(dx, dl, dw, dg))
        torch.cuda.synchronize()
        ref_gx, ref_gw = oracle.backward(x, shifted[turn], w, g, transposed=False)
        for gx, gw in results:
            assert rel_err(gx.cpu().numpy(), ref_gx) <= 1e-5 and rel_err(gw.cpu().numpy(), ref_gw) <= 1e-5


@pytest.mark.parametrize("batch,features,labels,fan_in", [(256, 512, 140_001, 40), (300, 900, 33_003, 33), (161, 385, 90_000, 65), (200, 448, 70_001, 100)])
def test_columns_sorted_tile_by_tile_with_weights_in_slot_order(batch, features, labels, fan_in):
    # the sums move with their column from thread to thread between the tiles
    ffi = load_package()
    lib = ffi._lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(labels)
    lookup = torch.randint(0, features, (labels, fan_in), generator=gen, device="cuda", dtype=torch.int32)
    lookup[::7, : fan_in // 2] = 3                             # (a column far longer than the others)
    w = torch.randn((labels, fan_in), generator=gen, device="cuda")
    g = torch.randn((batch, labels), generator=gen, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    results = []
    for value in (1, -1, 0):
        assert lib.ffi_set_option(b"plan_sorted_columns", value) == 0 and lib.ffi_set_option(b"plan_weights_in_lds", -1) == 0
        try:
            plan = ctypes.c_void_p()
            ffi._lib.check(lib.ffi_plan_create(lookup.data_ptr(), labels, fan_in, features, batch, stream, ctypes.byref(plan)))
            gx = torch.full((batch, features), float("nan"), device="cuda")
            ffi._lib.check(lib.ffi_input_grad_planned_f32(plan, w.data_ptr(), g.data_ptr(), gx.data_ptr(), batch, 0, stream))
            torch.cuda.synchronize()
            ffi._lib.check(lib.ffi_plan_destroy(plan))
        finally:
            assert lib.ffi_set_option(b"plan_sorted_columns", 0) == 0 and lib.ffi_set_option(b"plan_weights_in_lds", 0) == 0
        results.append(gx)
    exact = torch.zeros((batch, features), dtype=torch.float64, device="cuda")
    magnitude = torch.zeros_like(exact)
    for k in range(fan_in):
        term = g.double() * w[:, k].double()
        exact.index_add_(1, lookup[:, k].long(), term)
        magnitude.index_add_(1, lookup[:, k].long(), term.abs())
    for gx in results:
        # (sums of some thousand terms a stream, in order: far below 2^-24 times their number and magnitude)
        assert bool(((gx.double() - exact).abs() <= 1e-5 * magnitude + 1e-6).all())
        assert rel_err(gx.cpu().numpy(), exact.cpu().numpy()) <= 1e-5
