"""The forward kernels over tiles of 64 and of 32 samples: every fan-in's full and part-filled chunks, rows at any alignment, against each
other and the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle
from conftest import load_package, reference_law_inputs, rel_err

pytestmark = pytest.mark.gpu


# fan-ins around the chunks of 16 and of 32 and the quads behind them; batches that fill, start and end within a tile; the most columns that fit; labels that leave
# a wavefront, a workgroup and a round part empty
@pytest.mark.parametrize("fan_in", [1, 3, 4, 5, 8, 9, 15, 16, 17, 24, 31, 32, 33, 36, 37, 41, 47, 48, 49, 63, 64, 65, 127])
@pytest.mark.parametrize("batch,features,labels", [(192, 608, 1500), (192, 608, 66_001), (255, 77, 70_001), (321, 300, 65)])
def test_tiles_of_64_samples_and_of_32_agree(fan_in, batch, features, labels):
    ffi = load_package()
    lib = ffi._lib.lib()
    x, lookup, w, _ = reference_law_inputs(batch, features, labels, fan_in, seed=fan_in + labels)
    dx = torch.from_numpy(np.ascontiguousarray(x.T)).cuda()
    rows = torch.zeros((labels * fan_in + 1,), dtype=torch.int32, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    some = np.r_[0:300, labels // 2:labels // 2 + 300, labels - 300:labels] if labels > 10_000 else np.arange(labels)
    ref = oracle.forward(x, lookup[some], w[some])
    assert lib.ffi_set_option(b"small_path", -1) == 0
    try:
        for shift in (0, 1):                               # (lookup and weights at sixteen bytes and off them)
            dl, dw = rows[shift:shift + labels * fan_in], torch.empty_like(rows, dtype=torch.float32)[shift:shift + labels * fan_in]
            dl.copy_(torch.from_numpy(lookup).reshape(-1))
            dw.copy_(torch.from_numpy(w).reshape(-1))
            out = {}
            for option in (0, -1):
                assert lib.ffi_set_option(b"fwd_lane64", option) == 0
                out[option] = torch.full((batch, labels), float("nan"), device="cuda")
                ffi._lib.check(lib.ffi_forward_f32(dx.data_ptr(), dl.data_ptr(), dw.data_ptr(), out[option].data_ptr(), batch, features, labels, fan_in,
                                                   1, stream))
            assert torch.equal(out[0], out[-1])            # (the same products in the same order)
            assert rel_err(out[0][:, torch.from_numpy(some).cuda()].cpu().numpy(), ref) <= 1e-5
    finally:
        assert lib.ffi_set_option(b"fwd_lane64", 0) == 0 and lib.ffi_set_option(b"small_path", 0) == 0


# The kernel over tiles of 64 takes a layer whose tiles hold 768 labels a CU between them (above, the shapes of 66,001 and 70,001 labels at the fan-ins of whole
# chunks and up to four connections behind them): one tile and one sample more than 32, a last tile of one sample, of 2, of 32, of 33; the most columns.
# The scores are rows of a larger buffer, of which nothing else may change.
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("batch,features,labels,fan_in", [(33, 40, 200_003, 48), (64, 608, 200_003, 64), (129, 300, 70_001, 48), (130, 256, 70_001, 65), (160, 500, 70_001, 52),
                                                          (161, 608, 70_001, 33), (193, 300, 50_001, 48), (255, 77, 50_001, 16)])
def test_tiles_of_64_samples_where_they_end(batch, features, labels, fan_in, transposed):
    ffi = load_package()
    lib = ffi._lib.lib()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert -(-batch // 64) * labels >= 768 * cus
    x, lookup, w, _ = reference_law_inputs(batch, features, labels, fan_in, seed=fan_in + batch)
    dx = torch.from_numpy(np.ascontiguousarray(x.T if transposed else x)).cuda()
    dl, dw = torch.from_numpy(lookup).cuda(), torch.from_numpy(w).cuda()
    whole = torch.full((batch + 65, labels), 12345.0, device="cuda")
    out = whole[1:batch + 1].fill_(float("nan"))
    ffi._lib.check(lib.ffi_forward_f32(dx.data_ptr(), dl.data_ptr(), dw.data_ptr(), out.data_ptr(), batch, features, labels, fan_in, int(transposed),
                                       torch.cuda.current_stream().cuda_stream))
    assert bool((whole[0] == 12345.0).all()) and bool((whole[batch + 1:] == 12345.0).all()) and not bool(out.isnan().any())
    some = np.r_[0:500, labels // 2:labels // 2 + 500, labels - 500:labels]
    assert rel_err(out[:, torch.from_numpy(some).cuda()].cpu().numpy(), oracle.forward(x, lookup[some], w[some])) <= 1e-5


# Labels for eight rounds of a workgroup and more, the last one part empty: stores with a pause between them, whole chunks with two reads at a time
@pytest.mark.parametrize("fan_in", [7, 31, 32, 40, 64])
@pytest.mark.parametrize("batch", [481, 512])
def test_tiles_of_32_samples_and_many_rounds(batch, fan_in):
    features, labels = 70, 140_001
    ffi = load_package()
    lib = ffi._lib.lib()
    streams = max(1, torch.cuda.get_device_properties(0).multi_processor_count // 16)
    assert labels // streams >= 8 * 1024
    x, lookup, w, _ = reference_law_inputs(batch, features, labels, fan_in, seed=fan_in + batch)
    dx, dl, dw = torch.from_numpy(x).cuda(), torch.from_numpy(lookup).cuda(), torch.from_numpy(w).cuda()
    whole = torch.full((batch + 33, labels), 12345.0, device="cuda")
    out = whole[1:batch + 1].fill_(float("nan"))
    assert lib.ffi_set_option(b"fwd_lane64", -1) == 0 and lib.ffi_set_option(b"dense_rows", -1) == 0
    try:
        ffi._lib.check(lib.ffi_forward_f32(dx.data_ptr(), dl.data_ptr(), dw.data_ptr(), out.data_ptr(), batch, features, labels, fan_in, 0,
                                           torch.cuda.current_stream().cuda_stream))
    finally:
        assert lib.ffi_set_option(b"fwd_lane64", 0) == 0 and lib.ffi_set_option(b"dense_rows", 0) == 0
    assert bool((whole[0] == 12345.0).all()) and bool((whole[batch + 1:] == 12345.0).all()) and not bool(out.isnan().any())
    some = np.r_[0:400, labels // 2:labels // 2 + 400, labels - 400:labels]
    assert rel_err(out[:, torch.from_numpy(some).cuda()].cpu().numpy(), oracle.forward(x, lookup[some], w[some])) <= 1e-5


# Every way a row of connections ends, under every use of the scores: loss gradient alone, beside the scores, stored where it is not zero, beside a top-k; top-k alone
ROW_ENDS = [4, 9, 13, 16, 17, 23, 31, 33, 40, 41, 47, 48, 49, 57, 63, 64, 79, 80, 95]


@pytest.mark.parametrize("fan_in", ROW_ENDS)
@pytest.mark.parametrize("batch,features,labels", [(33, 300, 5003), (64, 1216, 4097)])
def test_loss_of_every_row_end(fan_in, batch, features, labels):
    ffi = load_package()
    lib = ffi._lib.lib()
    x, lookup, w, _ = reference_law_inputs(batch, features, labels, fan_in, seed=fan_in)
    bias = np.full(labels, -1.25, np.float32)
    rng = np.random.default_rng(fan_in)
    keys = np.unique(np.repeat(np.arange(batch), 3) * labels + rng.integers(0, labels, batch * 3))
    indices = np.stack([keys // labels, keys % labels], axis=1).astype(np.int64)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    args = (dev(x), dev(lookup), dev(w), dev(bias), (dev(indices), None), oracle.LOSS_SQUARED_HINGE)
    for option in (b"small_path", b"dense_rows"):
        assert lib.ffi_set_option(option, -1) == 0
    try:
        scores, g, loss, masks = ffi.metrics.forward_loss(*args, want_scores=True, want_masks=True)
        _, g_alone, loss_alone, masks_alone = ffi.metrics.forward_loss(*args, want_masks=True)
        _, g_part, loss_part, masks_part = ffi.metrics.forward_loss(*args, want_masks=True, skip_zero_stores=True)
        _, g_top, loss_top, masks_top, (values, best) = ffi.metrics.forward_loss(*args, want_masks=True, topk=5)
        scores_5, g_5, _, _, (values_5, best_5) = ffi.metrics.forward_loss(*args, want_scores=True, want_masks=True, topk=5)
        v, i = ffi.fan_in_sparse_topk(*args[:4], k=5)
        v2, i2, scores_2 = ffi.fan_in_sparse_topk(*args[:4], k=5, want_scores=True)
    finally:
        for option in (b"small_path", b"dense_rows"):
            assert lib.ffi_set_option(option, 0) == 0
    ref = oracle.forward(x, lookup, w) + bias[None, :]
    assert rel_err(scores.cpu().numpy(), ref) <= 1e-5
    # (the same products in the same order, whatever becomes of them)
    assert torch.equal(scores, scores_5) and torch.equal(scores, scores_2)
    ref_v, ref_i = oracle.topk(scores.cpu().numpy(), 5)
    for got_v, got_i in ((values, best), (values_5, best_5), (v, i), (v2, i2)):
        assert np.array_equal(got_i.cpu().numpy(), ref_i) and np.array_equal(got_v.cpu().numpy(), ref_v)
    for got in (masks_alone, masks_part, masks_top):
        assert torch.equal(got, masks)
    # the gradient of the scores that were written, each formed from its score in a few 32-bit steps: 4 ulp of the largest; where the scores are not written,
    # those of the listed labels are formed again, in another order: K terms of at most one, each rounded to 24 bits, twice
    losses, grad = oracle.sparse_loss(scores.cpu().numpy(), indices, np.ones(len(indices), np.float32), oracle.LOSS_SQUARED_HINGE)
    grad = grad / (batch * labels)
    ulps = 4 * 2.0 ** -23 * np.abs(grad).max()
    assert np.abs(g.cpu().numpy() - grad).max() <= ulps
    listed = torch.zeros_like(g, dtype=torch.bool)
    listed[dev(indices[:, 0]), dev(indices[:, 1])] = True
    again = ulps + 2 * (2 * fan_in * fan_in * 2.0 ** -24) / (batch * labels)
    written = g != 0
    for got, where in ((g_alone, None), (g_top, None), (g_5, None), (g_part, written)):
        same = ~listed if where is None else where & ~listed
        assert torch.equal(got[same], g[same])
        there = listed if where is None else where & listed
        assert float((got[there] - g[there]).abs().max()) <= again
    for total in (loss, loss_alone, loss_part, loss_top):
        assert abs(float(total) - losses.sum()) <= 1e-5 * losses.sum()


# few samples and bf16: rows of any fan-in at any alignment, whose last quads start within the quads before; labels that leave a round part empty
@pytest.mark.parametrize("fan_in", [1, 3, 4, 5, 6, 7, 9, 15, 17, 18, 23, 31, 32, 33, 34, 35, 47, 49, 63, 65, 127])
@pytest.mark.parametrize("batch,features,labels", [(3, 300, 1501), (8, 768, 997), (16, 64, 2050), (100, 500, 1303)])
def test_fan_ins_of_few_samples_and_of_bf16(fan_in, batch, features, labels):
    ffi = load_package()
    lib = ffi._lib.lib()
    x, lookup, w, _ = reference_law_inputs(batch, features, labels, fan_in, seed=fan_in + labels)
    stream = torch.cuda.current_stream().cuda_stream
    dx = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    ids = torch.zeros((labels * fan_in + 1,), dtype=torch.int32, device="cuda")
    weights = torch.zeros((labels * fan_in + 1,), device="cuda")
    assert lib.ffi_set_option(b"small_path", -1) == 0
    try:
        for shift in (0, 1):
            dl, dw = ids[shift:shift + labels * fan_in].view(labels, fan_in), weights[shift:shift + labels * fan_in].view(labels, fan_in)
            dl.copy_(torch.from_numpy(lookup))
            dw.copy_(torch.from_numpy(w))
            if batch <= 16:
                out = torch.full((batch, labels), float("nan"), device="cuda")
                ffi._lib.check(lib.ffi_forward_f32(dx.data_ptr(), dl.data_ptr(), dw.data_ptr(), out.data_ptr(), batch, features, labels, fan_in, 0, stream))
                assert rel_err(out.cpu().numpy(), oracle.forward(x, lookup, w)) <= 1e-5
            xb = dx.bfloat16()
            wb = torch.empty((labels * fan_in + 1,), dtype=torch.bfloat16, device="cuda")[shift:shift + labels * fan_in].view(labels, fan_in)
            wb.copy_(dw)
            out = torch.full((batch, labels), float("nan"), device="cuda")
            ffi._lib.check(lib.ffi_forward_bf16_f32(xb.data_ptr(), dl.data_ptr(), wb.data_ptr(), out.data_ptr(), batch, features, labels, fan_in, 0, stream))
            # (the operands are bf16, products and sums fp32: the same bound against the sums of the rounded operands)
            ref = oracle.forward(xb.float().cpu().numpy(), lookup, wb.float().cpu().numpy())
            assert rel_err(out.cpu().numpy(), ref) <= 1e-5
    finally:
        assert lib.ffi_set_option(b"small_path", 0) == 0
