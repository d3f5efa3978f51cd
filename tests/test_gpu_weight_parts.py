"""Weight gradients of few labels and many samples, whose sums come from several rows of workgroups, against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle
from conftest import load_package, reference_law_inputs, rel_err

pytestmark = pytest.mark.gpu


# (B, N, L, K): one, two, three and four chunks of connections with full and part-filled last ones; rows whose share of the batch tiles
# is uneven or ends within a tile; sizes off four; inputs with and without room for the streaming kernel's slices
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("shape", [(264, 1042, 1146, 104), (419, 998, 2283, 32), (500, 300, 1301, 61), (512, 1200, 601, 120), (333, 768, 4097, 33), (200, 80, 1500, 70),
                                   (161, 700, 90, 128), (225, 900, 5003, 7)])
def test_gradients_of_few_labels(shape, transposed):
    ffi = load_package()
    lib = ffi._lib.lib()
    B, N, L, K = shape
    x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=L)
    xt = np.ascontiguousarray(x.T if transposed else x)
    ref_gx, ref_gw = oracle.backward(xt, lookup, w, g, transposed=transposed)
    ref_gb = g.astype(np.float64).sum(0)
    dx, dl, dw, dg = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (xt, lookup, w, g))
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.ffi_set_option(b"small_path", -1) == 0
    try:
        for need_x in (True, False):                       # (over a plan and from the lookup itself)
            gx, gb = torch.full_like(dx, float("nan")), torch.full((L,), float("nan"), device="cuda")
            storage = torch.full((L * K + 1,), float("nan"), device="cuda")
            for gw in (storage[:-1], storage[1:]):         # (at sixteen bytes and off them)
                for _ in range(2):
                    ffi._lib.check(lib.ffi_backward_bias_f32(dx.data_ptr(), dl.data_ptr(), dw.data_ptr(), dg.data_ptr(), gx.data_ptr() if need_x else None,
                                                             gw.data_ptr(), gb.data_ptr(), B, N, L, K, int(transposed), stream))
                    assert rel_err(gw.cpu().numpy().reshape(L, K), ref_gw) <= 1e-5 and rel_err(gb.cpu().numpy(), ref_gb) <= 1e-5
            assert not need_x or rel_err(gx.cpu().numpy(), ref_gx) <= 1e-5
    finally:
        assert lib.ffi_set_option(b"small_path", 0) == 0


# every fan-in around the quads and chunks that rows are loaded, walked and stored by, with a label count that leaves wavefronts and
# workgroups part empty: over a plan and from the lookup itself, results at sixteen bytes and off them
@pytest.mark.parametrize("fan_in", [1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 23, 24, 25, 28, 29, 31, 32, 33, 36, 47, 63, 64, 65, 73, 95, 97, 127])
@pytest.mark.parametrize("batch,features,labels", [(33, 300, 1301), (64, 768, 517)])
def test_gradients_of_any_fan_in(batch, features, labels, fan_in):
    ffi = load_package()
    lib = ffi._lib.lib()
    x, lookup, w, g = reference_law_inputs(batch, features, labels, fan_in, seed=fan_in + labels)
    _, ref_gw = oracle.backward(x, lookup, w, g)
    ref_gb = g.astype(np.float64).sum(0)
    dx, dl, dw, dg = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, lookup, w, g))
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.ffi_set_option(b"small_path", -1) == 0
    try:
        for need_x in (True, False):
            storage = torch.full((labels * fan_in + 2,), float("nan"), device="cuda")
            for gw in (storage[:-2], storage[1:-1]):
                storage.fill_(float("nan"))
                gx, gb = torch.empty_like(dx), torch.empty((labels,), device="cuda")
                ffi._lib.check(lib.ffi_backward_bias_f32(dx.data_ptr(), dl.data_ptr(), dw.data_ptr(), dg.data_ptr(), gx.data_ptr() if need_x else None,
                                                         gw.data_ptr(), gb.data_ptr(), batch, features, labels, fan_in, 0, stream))
                assert rel_err(gw.cpu().numpy().reshape(labels, fan_in), ref_gw) <= 1e-5 and rel_err(gb.cpu().numpy(), ref_gb) <= 1e-5
                assert int(torch.isnan(storage).sum()) == 2        # (nothing beside the gradient is written)
    finally:
        assert lib.ffi_set_option(b"small_path", 0) == 0


@pytest.mark.parametrize("fan_in", [72, 81, 89, 95, 96])
def test_gradients_of_three_chunks_and_many_labels(fan_in):
    test_gradients_of_any_fan_in(33, 70, 82_001, fan_in)


# Every sum has one writer.  With features of ones the sums of a unit (32 connections of a label) are the same bits, and those of the next unit, whose
# lane adds the samples up in another order, mostly are not: sums that another unit left show.  Labels for many workgroups, whose first units are
# odd ones too; batch tiles shared between rows of workgroups, and not.
@pytest.mark.parametrize("fan_in", [33, 34, 35, 36, 47, 63, 65, 67, 95, 97, 127, 128])
@pytest.mark.parametrize("batch,features,labels", [(33, 300, 40_003), (419, 998, 2283), (31, 96, 1001)])
def test_sums_of_the_lookup_itself_have_one_writer(batch, features, labels, fan_in):
    ffi = load_package()
    lib = ffi._lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(fan_in)
    lookup = torch.randint(0, features, (labels, fan_in), generator=gen, device="cuda", dtype=torch.int32)
    x = torch.ones((batch, features), device="cuda")
    g = torch.randn((batch, labels), generator=gen, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.ffi_set_option(b"small_path", -1) == 0
    try:
        first = None
        for _ in range(4):
            gw = torch.full((labels, fan_in), float("nan"), device="cuda")
            ffi._lib.check(lib.ffi_weight_grad_f32(x.data_ptr(), lookup.data_ptr(), g.data_ptr(), gw.data_ptr(), batch, features, labels, fan_in, 0, stream))
            first = gw if first is None else first
            assert torch.equal(gw, first)
            for k0 in range(0, fan_in, 32):
                unit = gw[:, k0:k0 + 32]
                assert torch.equal(unit, unit[:, :1].expand_as(unit))
        # (sums of `batch` terms, each rounded to 24 bits, in any order)
        exact, magnitude = g.double().sum(0, keepdim=True).t(), g.double().abs().sum(0, keepdim=True).t()
        assert bool(((first.double() - exact).abs() <= batch * 2.0 ** -24 * magnitude).all())
    finally:
        assert lib.ffi_set_option(b"small_path", 0) == 0
