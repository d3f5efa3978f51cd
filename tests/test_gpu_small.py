"""Small layers: the two launches that read the caller's arrays directly, and the paths for large layers at the same sizes,
against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle
from conftest import load_package, reference_law_inputs, rel_err

pytestmark = pytest.mark.gpu

# (B, N, L, K): one of everything; sample groups, lane groups of 4 and 16 and splits with remainders; several windows of columns
# with 4 and with 16 wavefronts; several shares of the connections
SHAPES = [(1, 1, 1, 1), (17, 12, 63, 44), (8, 40, 16, 8), (9, 2049, 70, 5), (3, 9000, 33, 7), (65, 40, 300, 64), (2, 500, 9000, 16),
          (8, 5000, 4000, 17), (130, 700, 64, 33)]


@pytest.mark.parametrize("small_path", [1, -1])
@pytest.mark.parametrize("transposed", [False, True])
def test_small_layers(small_path, transposed):
    ffi = load_package()
    lib = ffi._lib.lib()
    assert lib.ffi_set_option(b"small_path", small_path) == 0
    try:
        for B, N, L, K in SHAPES:
            x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=B + N)
            xt = np.ascontiguousarray(x.T if transposed else x)
            bias = np.linspace(-1, 1, L).astype(np.float32)
            ref = oracle.forward(x, lookup, w, transposed=False) + bias
            ref_gx, ref_gw = oracle.backward(xt, lookup, w, g, transposed=transposed)
            dx, dl, dw, dg, db = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (xt, lookup, w, g, bias))
            op = ffi.fan_in_sparse_matmul_tp_bias if transposed else ffi.fan_in_sparse_matmul_bias
            variables = [dx.requires_grad_(True), dw.requires_grad_(True), db.requires_grad_(True)]
            first = None
            for _ in range(3):
                out = op(variables[0], dl, variables[1], variables[2])
                gx, gw, gb = torch.autograd.grad(out, variables, dg)
                assert rel_err(out.detach().cpu().numpy(), ref) <= 1e-5, (B, N, L, K)
                assert rel_err(gx.cpu().numpy(), ref_gx) <= 1e-4 and rel_err(gw.cpu().numpy(), ref_gw) <= 1e-4, (B, N, L, K)
                assert rel_err(gb.cpu().numpy(), g.astype(np.float64).sum(0)) <= 1e-5, (B, N, L, K)
                assert first is None or torch.equal(first, gx), (B, N, L, K)
                first = gx
    finally:
        lib.ffi_set_option(b"small_path", 0)


def test_an_id_out_of_range_is_reported_by_the_next_call():
    ffi = load_package()
    x, lookup, w, g = (torch.from_numpy(a).cuda() for a in reference_law_inputs(4, 50, 30, 6, seed=1))
    ffi.fan_in_sparse_matmul_grad(x, lookup, w, g)
    lookup[3, 2] = 50
    gx, gw = ffi.fan_in_sparse_matmul_grad(x, lookup, w, g)
    torch.cuda.synchronize()
    assert float(gw[3, 2]) == 0.0
    with pytest.raises(ffi._lib.FfiError):
        ffi.fan_in_sparse_matmul_grad(x, lookup, w, g)
    lookup[3, 2] = 49
    ffi.fan_in_sparse_matmul_grad(x, lookup, w, g)


def test_a_lookup_whose_ids_only_were_checked_gets_its_plan_when_a_pass_walks_one():
    # 2 samples read the lookup itself, 700 walk a plan; edits that the library is told of lie between them, at one address
    ffi = load_package()
    lib = ffi._lib.lib()
    N, L, K = 300, 5000, 16
    cases = {B: reference_law_inputs(B, N, L, K, seed=B) for B in (2, 700)}
    lookup = torch.empty((L, K), dtype=torch.int32, device="cuda")
    for turn, B in enumerate((2, 700, 2, 2, 700, 700, 2)):
        x, ids, w, g = cases[B]
        ids = (ids + 7 * turn) % N
        lookup.copy_(torch.from_numpy(ids))
        ffi._lib.check(lib.ffi_lookup_edited(lookup.data_ptr()))
        gx, gw = ffi.fan_in_sparse_matmul_grad(*(torch.from_numpy(a).cuda() for a in (x,)), lookup, *(torch.from_numpy(a).cuda() for a in (w, g)))
        ref_gx, ref_gw = oracle.backward(x, ids, w, g, transposed=False)
        assert rel_err(gx.cpu().numpy(), ref_gx) <= 1e-4 and rel_err(gw.cpu().numpy(), ref_gw) <= 1e-4, (turn, B)
    lookup[3, 2] = N
    ffi._lib.check(lib.ffi_lookup_edited(lookup.data_ptr()))
    x, ids, w, g = (torch.from_numpy(a).cuda() for a in cases[2])
    with pytest.raises(ffi._lib.FfiError):
        ffi.fan_in_sparse_matmul_grad(x, lookup, w, g)
