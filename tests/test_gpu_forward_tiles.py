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
    ref = oracle.forward(x, lookup, w) if labels < 10_000 else None
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
            assert ref is None or rel_err(out[0].cpu().numpy(), ref) <= 1e-5
    finally:
        assert lib.ffi_set_option(b"fwd_lane64", 0) == 0 and lib.ffi_set_option(b"small_path", 0) == 0


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
