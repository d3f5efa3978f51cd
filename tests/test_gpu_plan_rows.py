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
