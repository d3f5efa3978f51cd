"""Inputs whose tile does not fit in LDS (more than 1,216 columns): the kernels that gather from sample-sliced tables, at
the sizes where they change form, against the CPU oracle."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from conftest import load_package, reference_law_inputs, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ffi():
    return load_package()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# (B, N, L, K): slices of 4, 8, 16 and 32 samples and their edges; several slices per list and one; label blocks and
# chunks of connections with remainders; rows on and off 16-byte boundaries
FORWARD_SHAPES = [(1, 1217, 300, 1), (4, 2000, 257, 16), (5, 1217, 129, 17), (8, 3000, 128, 40), (9, 1300, 65, 33), (16, 2500, 130, 64),
                  (17, 4000, 63, 3), (33, 1300, 64, 72), (100, 40_000, 200, 65), (130, 1500, 97, 130), (64, 70_000, 150, 36)]


@pytest.mark.parametrize("phases", [0, 1, -1])
def test_forward_of_wide_inputs(ffi, phases):
    lib = ffi._lib.lib()
    assert lib.ffi_set_option(b"wide_phases", phases) == 0
    try:
        for B, N, L, K in FORWARD_SHAPES:
            x, lookup, w, _ = reference_law_inputs(B, N, L, K, seed=B + N)
            ref = oracle.forward(x, lookup, w, transposed=False)
            bias = np.linspace(-1, 1, L).astype(np.float32)
            for tp in (False, True):
                dx = dev(x.T if tp else x)
                fwd = ffi.fan_in_sparse_matmul_tp if tp else ffi.fan_in_sparse_matmul
                assert rel_err(fwd(dx, dev(lookup), dev(w)).cpu().numpy(), ref) <= 1e-5, (B, N, L, K, tp)
            out = ffi.fan_in_sparse_matmul_bias(dev(x), dev(lookup), dev(w), dev(bias)).cpu().numpy()
            assert rel_err(out, ref + bias) <= 1e-5, (B, N, L, K)
            # bf16 operands, whose sums are fp32 ones too
            hx, hw = torch.from_numpy(x).bfloat16(), torch.from_numpy(w).bfloat16()
            ref = oracle.forward(hx.float().numpy(), lookup, hw.float().numpy(), transposed=False)
            for tp in (False, True):
                out = ffi.fan_in_sparse_matmul_bf16((hx.t().contiguous() if tp else hx).cuda(), dev(lookup), hw.cuda(), transposed=tp)
                assert rel_err(out.cpu().numpy(), ref) <= 1e-5, (B, N, L, K, tp, "bf16")
    finally:
        lib.ffi_set_option(b"wide_phases", 0)


# The forward pass in phases: (B, L, K) with label blocks of 352 and (from 90,000 labels on) 704 and their edges, rows shorter
# than an oct, of whole octs and with a remainder, up to the longest; ids spread, all of one range, all of the last column,
# falling: a row's places come from counters of a byte each
PHASED_SHAPES = [(32, 351, 9), (17, 353, 8), (40, 705, 64), (70, 352, 65), (33, 300, 255), (20, 101, 256), (18, 92_000, 9), (64, 91_000, 17)]


@pytest.mark.parametrize("spread", ["uniform", "one_range", "last", "falling"])
def test_forward_in_phases(ffi, spread):
    N = 1301
    lib = ffi._lib.lib()
    assert lib.ffi_set_option(b"wide_phases", 1) == 0
    try:
        for B, L, K in PHASED_SHAPES:
            x, lookup, w, _ = reference_law_inputs(B, N, L, K, seed=B + L + K)
            if spread == "one_range":
                lookup = (lookup % 40 + 600).astype(np.int32)
            elif spread == "last":
                lookup[:] = N - 1
            elif spread == "falling":
                lookup = np.ascontiguousarray(-np.sort(-lookup, axis=1))
            hx, hw = torch.from_numpy(x).bfloat16(), torch.from_numpy(w).bfloat16()
            ref = oracle.forward(x, lookup, w, transposed=False)
            ref16 = oracle.forward(hx.float().numpy(), lookup, hw.float().numpy(), transposed=False)
            out = ffi.fan_in_sparse_matmul(dev(x), dev(lookup), dev(w)).cpu().numpy()
            out16 = ffi.fan_in_sparse_matmul_bf16(hx.cuda(), dev(lookup), hw.cuda(), transposed=False).cpu().numpy()
            # sums of K products in another order: K 2^-24 of the largest, 256 at most
            assert rel_err(out, ref) <= 2e-5, (B, L, K)
            assert rel_err(out16, ref16) <= 2e-5, (B, L, K)
    finally:
        lib.ffi_set_option(b"wide_phases", 0)


# (B, N, L, K): streams that are empty, shorter and longer than a chunk; several segments, streams and slices; one column
BACKWARD_SHAPES = [(1, 1217, 900, 3), (4, 2000, 30_000, 9), (5, 1217, 129, 17), (8, 3000, 3000, 40), (9, 1300, 65, 33), (16, 2500, 5000, 64),
                   (17, 40_000, 63, 3), (33, 1300, 9000, 72), (100, 40_000, 200, 65), (130, 1500, 97, 130), (64, 30_000, 3000, 36)]


@pytest.mark.parametrize("transposed", [False, True])
def test_backward_of_wide_inputs(ffi, transposed):
    for B, N, L, K in BACKWARD_SHAPES:
        x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=B + N)
        if (B, N) == (33, 1300):
            lookup[::3] = 7                                     # one column holds a third of all connections
        ref_gx, ref_gw = oracle.backward(np.ascontiguousarray(x.T) if transposed else x, lookup, w, g, transposed=transposed)
        dx, dl, dw, dg = dev(x.T if transposed else x), dev(lookup), dev(w), dev(g)
        bwd = ffi.fan_in_sparse_matmul_grad_tp if transposed else ffi.fan_in_sparse_matmul_grad
        first = None
        for _ in range(2):                                      # the call that builds the plan, and one behind a check of it
            gx, gw = bwd(dx, dl, dw, dg)
            assert rel_err(gx.cpu().numpy(), ref_gx) <= 1e-4, (B, N, L, K)
            assert rel_err(gw.cpu().numpy(), ref_gw) <= 1e-4, (B, N, L, K)
            assert first is None or torch.equal(first, gx)
            first = gx
        if not transposed:
            bias = torch.zeros(L, device="cuda", requires_grad=True)
            gb, = torch.autograd.grad(ffi.fan_in_sparse_matmul_bias(dx.requires_grad_(True), dl, dw, bias), [bias], dg)
            assert rel_err(gb.cpu().numpy(), g.astype(np.float64).sum(0)) <= 1e-5


# Narrow inputs whose slice of samples lies in LDS: (B, N, L, K) with slices of 4 to 64 samples, label blocks and lists with
# remainders, the largest slice that fits, rows on and off 16-byte boundaries
LDS_SHAPES = [(1, 1, 1, 1), (3, 12, 33, 5), (5, 768, 130, 16), (8, 500, 1025, 24), (16, 1216, 300, 33), (9, 64, 2000, 7),
              (33, 100, 65, 17), (64, 1000, 257, 8), (65, 1144, 100, 130)]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("transposed", [False, True])
def test_forward_from_slices_in_lds(ffi, bf16, transposed):
    for B, N, L, K in LDS_SHAPES:
        x, lookup, w, _ = reference_law_inputs(B, N, L, K, seed=B + N)
        tx, tw = torch.from_numpy(x), torch.from_numpy(w)
        if bf16:
            tx, tw = tx.bfloat16(), tw.bfloat16()
        ref = oracle.forward(tx.float().numpy(), lookup, tw.float().numpy(), transposed=False)
        xd = (tx.t().contiguous() if transposed else tx).cuda()
        if bf16:
            out = ffi.fan_in_sparse_matmul_bf16(xd, dev(lookup), tw.cuda(), transposed=transposed)
        else:
            out = (ffi.fan_in_sparse_matmul_tp if transposed else ffi.fan_in_sparse_matmul)(xd, dev(lookup), tw.cuda())
        assert rel_err(out.cpu().numpy(), ref) <= 1e-5, (B, N, L, K)


# Slices in LDS, what the wavefronts share out: full turns of 32 labels and a last one of one round, a single label or none left for
# most of them, fewer rounds than wavefronts; slices with samples missing; features whose rows start at every alignment
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,N,L,K", [(61, 33, 131_073, 4), (64, 32, 2_049, 24), (250, 31, 33_000, 9), (13, 30, 140_001, 5), (7, 29, 270_000, 3), (3, 2, 7, 2)])
def test_forward_from_slices_in_lds_shares(ffi, bf16, B, N, L, K):
    rng = np.random.default_rng(L + K)
    lookup = rng.integers(0, N, (L, K)).astype(np.int32)
    tx = torch.from_numpy(rng.standard_normal(B * N + 1).astype(np.float32))
    tw = torch.from_numpy(rng.standard_normal((L, K)).astype(np.float32))
    if bf16:
        tx, tw = tx.bfloat16(), tw.bfloat16()
    for transposed in (False, True):
        x = tx[1:].view(N, B) if transposed else tx[1:].view(B, N)
        xn = (x.t() if transposed else x).float().numpy().astype(np.float64)
        ref, size = np.zeros((B, L)), np.zeros((B, L))
        for k in range(K):
            term = xn[:, lookup[:, k]] * tw[:, k].float().numpy().astype(np.float64)
            ref += term
            size += np.abs(term)
        xd = tx.cuda()[1:].view(x.shape)
        if bf16:
            out = ffi.fan_in_sparse_matmul_bf16(xd, dev(lookup), tw.cuda(), transposed=transposed)
        else:
            out = (ffi.fan_in_sparse_matmul_tp if transposed else ffi.fan_in_sparse_matmul)(xd, dev(lookup), tw.cuda())
        # K fused products and at most two more sums of partial ones, each rounded once: (K + 2) 2^-24 of the sum of magnitudes
        assert (np.abs(out.cpu().numpy() - ref) <= (K + 2) * 2.0 ** -24 * size + 1e-30).all()


# Slices of eight samples staged by four columns at a time and, of many columns, by one: samples missing, a second slice, columns off four
@pytest.mark.parametrize("B,N,L,K", [(5, 512, 3000, 44), (5, 513, 3000, 44), (7, 1215, 9001, 13), (9, 700, 9000, 24)])
def test_forward_from_slices_of_eight_samples(ffi, B, N, L, K):
    test_forward_from_slices_in_lds_shares(ffi, False, B, N, L, K)


# Wide inputs with few columns and few labels: columns of few connections, segments whose sums are added
@pytest.mark.parametrize("B,N,L,K", [(5, 1_217, 130, 3), (33, 1_242, 3_201, 95), (64, 5_000, 129, 40), (17, 2_000, 13_331, 8), (3, 20_000, 700, 16)])
@pytest.mark.parametrize("transposed", [False, True])
def test_backward_over_many_label_blocks(ffi, B, N, L, K, transposed):
    x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=N + L)
    o_gx, o_gw = oracle.backward(x, lookup, w, g)
    xd = dev(np.ascontiguousarray(x.T) if transposed else x)
    call = ffi.fan_in_sparse_matmul_grad_tp if transposed else ffi.fan_in_sparse_matmul_grad
    for _ in range(2):
        gx, gw = call(xd, dev(lookup), dev(w), dev(g))
        gx = gx.t() if transposed else gx
        assert rel_err(gx.cpu().numpy(), o_gx) <= 2e-5 and rel_err(gw.cpu().numpy(), o_gw) <= 2e-5


# The walk over streams of 32 columns: (batches of the calls in turn -- the first one's plan has steps of four or eight connections and
# serves the others --, N, L, K).  One column behind whole groups; streams of no, one and several chunks; several segments, several
# slices in a launch and several launches; tiles of exactly their positions and one more; more streams than the build counts at a time, and
# so many that its tiles grow and their counts come in rows
WALK_SHAPES = [((20, 70, 3), 1249, 5000, 7), ((70, 20, 200), 1248, 5000, 7), ((1, 130), 1300, 9000, 72), ((300, 33), 2500, 3001, 33),
               ((64,), 1300, 1024, 1), ((32,), 1300, 1025, 1), ((65, 64), 40_000, 20_011, 12), ((3, 40), 1_000_000, 300, 4),
               ((5,), 2_400_000, 70_001, 15), ((2,), 17_000_000, 522_240, 4)]


@pytest.mark.parametrize("shape", WALK_SHAPES, ids=str)
def test_walk_over_streams(ffi, shape):
    batches, N, L, K = shape
    lib = ffi._lib.lib()
    assert lib.ffi_set_option(b"small_path", -1) == 0
    try:
        _, lookup, w, _ = reference_law_inputs(1, N, L, K, seed=L + K)
        dl, dw = dev(lookup), dev(w)
        for B in batches:
            rng = np.random.default_rng(B)
            x, g = rng.standard_normal((B, N), dtype=np.float32), rng.standard_normal((B, L), dtype=np.float32)
            ref_gx, ref_gw = oracle.backward(x, lookup, w, g, transposed=False)
            for tp in (False, True):
                call = ffi.fan_in_sparse_matmul_grad_tp if tp else ffi.fan_in_sparse_matmul_grad
                gx, gw = call(dev(x.T if tp else x), dl, dw, dev(g))
                gx = gx.t() if tp else gx
                assert rel_err(gx.cpu().numpy(), ref_gx) <= 1e-5 and rel_err(gw.cpu().numpy(), ref_gw) <= 1e-5, (B, tp)
    finally:
        lib.ffi_set_option(b"small_path", 0)


# Behind an outdated plan of the global form: gx is cleared by the kernel that moves the weight gradients, or, without them, by one of its
# own; one segment and several, more and less of gx than workgroups have threads
@pytest.mark.parametrize("shape", [(33, 1300, 3000, 9), (70, 40_000, 2000, 5)], ids=str)
@pytest.mark.parametrize("input_only", [False, True])
def test_wide_gradients_behind_an_outdated_plan(ffi, shape, input_only):
    B, N, L, K = shape
    lib = ffi._lib.lib()
    x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=B + K)
    dx, dl, dw, dg = dev(x), dev(lookup), dev(w), dev(g)

    def call():
        if not input_only:
            return ffi.fan_in_sparse_matmul_grad(dx, dl, dw, dg)
        gx = torch.full((B, N), float("nan"), device="cuda")
        ffi._lib.check(lib.ffi_input_grad_f32(dl.data_ptr(), dw.data_ptr(), dg.data_ptr(), gx.data_ptr(), B, N, L, K, 0,
                                              torch.cuda.current_stream().cuda_stream))
        return gx, None

    assert lib.ffi_set_option(b"small_path", -1) == 0
    try:
        call()
        rng = np.random.default_rng(8)
        for _ in range(2):
            lookup = lookup.copy()
            lookup[rng.integers(0, L, 400), rng.integers(0, K, 400)] = rng.integers(0, N, 400)
            dl.copy_(dev(lookup))
            gx, gw = call()
            ref_gx, ref_gw = oracle.backward(x, lookup, w, g, transposed=False)
            assert rel_err(gx.cpu().numpy(), ref_gx) <= 1e-4
            assert gw is None or rel_err(gw.cpu().numpy(), ref_gw) <= 1e-4
    finally:
        lib.ffi_set_option(b"small_path", 0)


# Up to four samples, scores and answer in one launch: fan-ins of one quad, off the quads and of several passes over a row; fewer
# labels than asked for, a label per lane and four, more workgroups than CUs; features that just fit
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,N,L,K,k", [(1, 12, 3, 4, 5), (2, 768, 70_001, 31, 8), (3, 500, 9_000, 64, 3), (4, 9_216, 40_000, 5, 5), (1, 36_864, 5_000, 257, 8),
                                       (1, 30, 3_000_000, 4, 8), (4, 100, 1_100_003, 9, 1)])
def test_topk_of_few_samples(ffi, bf16, B, N, L, K, k):
    rng = np.random.default_rng(L + K)
    x, w = rng.standard_normal((B, N)).astype(np.float32), rng.standard_normal((L, K)).astype(np.float32)
    lookup, bias = rng.integers(0, N, (L, K)).astype(np.int32), rng.standard_normal(L).astype(np.float32)
    tx, tw = torch.from_numpy(x), torch.from_numpy(w)
    if bf16:
        tx, tw = tx.bfloat16(), tw.bfloat16()
        bias[:] = 0
    ref = oracle.forward(tx.float().numpy(), lookup, tw.float().numpy(), transposed=False) + bias
    want = np.argsort(-ref, axis=1, kind="stable")[:, :k]
    values = np.full((B, k), -np.inf, np.float32)
    values[:, :min(k, L)] = np.take_along_axis(ref, want, 1)
    if bf16:
        v, i = ffi.fan_in_sparse_topk_bf16(tx.cuda(), dev(lookup), tw.cuda(), k=k)
    else:
        v, i = ffi.fan_in_sparse_topk(tx.cuda(), dev(lookup), tw.cuda(), bias=dev(bias), k=k)
    v, i = v.cpu().numpy(), i.cpu().numpy()
    bound = 2e-5 * np.abs(ref).max()                    # sums of K products in another order; labels closer than that may change places
    assert (i[:, min(k, L):] == -1).all() and (v[:, min(k, L):] == -np.inf).all()
    assert np.abs(v[:, :min(k, L)] - values[:, :min(k, L)]).max() <= bound
    assert np.abs(np.take_along_axis(ref, i[:, :min(k, L)].astype(np.int64), 1) - values[:, :min(k, L)]).max() <= bound
    assert all(len(set(row[:min(k, L)])) == min(k, L) for row in i)


def test_topk_of_few_samples_ties_and_specials(ffi):
    N, L, K = 20, 100_000, 4
    lookup = (np.arange(L * K, dtype=np.int64) * 7 % N).astype(np.int32).reshape(L, K)
    w = torch.ones((L, K), device="cuda")
    zeros = torch.zeros((2, N), device="cuda")
    # equal scores go to the lower labels; many labels of few wavefronts above all others (more than the list of candidates holds)
    v, i = ffi.fan_in_sparse_topk(zeros, dev(lookup), w, bias=torch.zeros(L, device="cuda"), k=8)
    assert (i.cpu().numpy() == np.arange(8)).all() and (v == 0).all()
    high = torch.from_numpy((np.arange(L) % 4096 < 1500).astype(np.float32)).cuda()
    high[70_000] = 2.0
    v, i = ffi.fan_in_sparse_topk(zeros, dev(lookup), w, bias=high, k=8)
    assert (i.cpu().numpy() == np.array([70_000, 0, 1, 2, 3, 4, 5, 6])).all() and v[0, 0] == 2 and (v[:, 1:] == 1).all()
    special = torch.full((L,), -float("inf"), device="cuda")
    special[5], special[99_999], special[17] = float("nan"), float("inf"), 3.0
    v, i = ffi.fan_in_sparse_topk(zeros, dev(lookup), w, bias=special, k=4)
    assert (i.cpu().numpy() == np.array([99_999, 17, 0, 1])).all()
    assert (v.cpu().numpy() == np.array([np.inf, 3, -np.inf, -np.inf], np.float32)).all()


# Top-k without the scores: every label in the sample that sets the threshold and a part of them; ties across the whole layer,
# more than a candidate list holds
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,N,L,K", [(1, 768, 40_000, 8), (12, 3000, 9_001, 4), (20, 1300, 17_000, 3), (3, 500, 7, 5), (33, 1217, 16_385, 2)])
@pytest.mark.parametrize("tied", [False, True])
def test_topk_by_threshold(ffi, bf16, B, N, L, K, tied):
    x, lookup, w, _ = reference_law_inputs(B, N, L, K, seed=B + N)
    dx, dw = dev(x), dev(np.zeros_like(w) if tied else w)
    k = min(5, L)
    if bf16:
        dx, dw = dx.bfloat16(), dw.bfloat16()
        scores = ffi.fan_in_sparse_matmul_bf16(dx, dev(lookup), dw)
        val, idx = ffi.fan_in_sparse_topk_bf16(dx, dev(lookup), dw, k=k)
    else:
        scores = ffi.fan_in_sparse_matmul(dx, dev(lookup), dw)
        val, idx = ffi.fan_in_sparse_topk(dx, dev(lookup), dw, k=k)
    best = torch.topk(scores, k, dim=1).values                # (possibly summed in another order)
    assert float((val - best).abs().max()) <= 1e-5 * float(best.abs().max())
    assert float((torch.gather(scores, 1, idx.long()) - val).abs().max()) <= 1e-5 * float(best.abs().max())
    if tied:
        assert torch.equal(idx.cpu().long(), torch.arange(k).expand(B, k))


# Scores that are infinite or no number, in every kernel that collects candidates: samples behind the batch's end and slices
# behind the last (three where a workgroup serves two or four) reach no list.  (B, N, L, K, wide_phases): slices in LDS, gathered
# from L2, in phases; the 32-sample tile
NONFINITE_SHAPES = [(5, 768, 20_000, 8, 0), (96, 4096, 9_001, 5, 0), (33, 1300, 17_000, 6, 0), (160, 4096, 9_001, 12, 0), (70, 5000, 3_000, 20, 1),
                    (130, 2000, 5_000, 16, 1), (40, 768, 20_000, 12, 0)]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("shape", NONFINITE_SHAPES)
@pytest.mark.parametrize("n_inf", [2, 40])
def test_topk_of_scores_that_are_not_finite(ffi, bf16, shape, n_inf):
    B, N, L, K, phases = shape
    k = 5
    x, lookup, w, _ = reference_law_inputs(B, N, L, K, seed=B + N)
    x = np.abs(x) + 0.5                                        # (a weight of +inf gives +inf, and one of -inf gives -inf)
    rng = np.random.default_rng(L)
    special = rng.permutation(L)
    bias = np.zeros(L, np.float32)
    at = w if bf16 else bias                                   # (no bias beside bf16 scores)
    for labels, value in ((special[:n_inf], np.inf), (special[n_inf:n_inf + L // 3], -np.inf), (special[-L // 10:], np.nan)):
        if bf16: at[labels, 0] = value
        else: at[labels] = value
    dx, dl, dw, db = dev(x), dev(lookup), dev(w), dev(bias)
    print(f"case {shape} bf16={bf16} n_inf={n_inf}", flush=True)
    lib = ffi._lib.lib()
    assert lib.ffi_set_option(b"wide_phases", phases) == 0
    try:
        if bf16:
            dx, dw = dx.bfloat16(), dw.bfloat16()
            scores = ffi.fan_in_sparse_matmul_bf16(dx, dl, dw)
            val, idx = ffi.fan_in_sparse_topk_bf16(dx, dl, dw, k=k)
        else:
            scores = ffi.fan_in_sparse_matmul_bias(dx, dl, dw, db)
            val, idx = ffi.fan_in_sparse_topk(dx, dl, dw, db, k=k)
    finally:
        lib.ffi_set_option(b"wide_phases", 0)
    scores, val, idx = scores.cpu().numpy(), val.cpu().numpy(), idx.cpu().numpy()
    infinite = np.sort(special[:n_inf])[:k]
    assert np.isposinf(scores[:, special[:n_inf]]).all() and np.isnan(scores).sum() == B * len(special[-L // 10:])
    n = len(infinite)
    assert np.isposinf(val[:, :n]).all() and (idx[:, :n] == infinite).all()
    # the finite rest: the best of the scores without NaN (possibly summed in another order)
    rest = np.where(np.isfinite(scores), scores, -np.inf)
    best = -np.sort(-rest, axis=1)[:, :k - n]
    assert np.abs(val[:, n:] - best).max(initial=0.0) <= 1e-5 * np.abs(rest[np.isfinite(rest)]).max()
    assert np.abs(np.take_along_axis(scores, idx[:, n:].astype(np.int64), 1) - val[:, n:]).max(initial=0.0) <= 1e-5 * np.abs(rest[np.isfinite(rest)]).max()


# Scores that tie by the thousand -- small whole numbers, samples without features -- and layers whose every label outside the sample
# that sets the threshold beats those in it, so that the lists overflow: the answer is that of the score matrix, ties to the
# lower label.  (B, N, wide_phases): slices in LDS, gathered from L2, in phases; the 32-sample tile
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,N,phases", [(1, 500, 0), (7, 300, 0), (40, 200, 0), (70, 3000, 0), (70, 3000, 1)])
@pytest.mark.parametrize("overflow", [False, True])
def test_topk_of_tied_scores_and_full_lists(ffi, bf16, B, N, phases, overflow):
    L, K, k = 81_920, 6, 8                                      # (samples of every 5th and 20th label)
    rng = np.random.default_rng(B + N)
    x = rng.integers(0, 4, (B, N)).astype(np.float32)
    w = rng.integers(-2, 3, (L, K)).astype(np.float32)
    lookup = rng.integers(0, N, (L, K)).astype(np.int32)
    if overflow:
        x[:, 0], lookup[:, 0], w[:, 0] = 1.0, 0, np.where(np.arange(L) % 5 == 0, 0.0, 100.0)
    x[::3, overflow:] = 0.0
    dx, dl, dw = dev(x), dev(lookup), dev(w)
    print(f"case bf16={bf16} B={B} N={N} phases={phases} overflow={overflow}", flush=True)
    lib = ffi._lib.lib()
    assert lib.ffi_set_option(b"wide_phases", phases) == 0
    try:
        for _ in range(2):                                      # (the counters of the first call are cleared for the second)
            if bf16:
                val, idx = ffi.fan_in_sparse_topk_bf16(dx.bfloat16(), dl, dw.bfloat16(), k=k)
            else:
                val, idx = ffi.fan_in_sparse_topk(dx, dl, dw, k=k)
    finally:
        lib.ffi_set_option(b"wide_phases", 0)
    scores = oracle.forward(x, lookup, w, transposed=False)     # (whole numbers: exact in any order)
    ref_v, ref_i = oracle.topk(scores, k)
    assert np.array_equal(idx.cpu().numpy(), ref_i) and np.array_equal(val.cpu().numpy(), ref_v)
    val, idx = ffi.topk_scores(dev(scores), k)
    assert np.array_equal(idx.cpu().numpy(), ref_i) and np.array_equal(val.cpu().numpy(), ref_v)


def _same_values(got, ref, tol, scale):
    """NaN and infinities where the reference has them, the rest within tol x scale."""
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    special = np.isinf(ref)
    assert np.array_equal(np.isinf(got), special) and np.array_equal(got[special], ref[special])
    finite = np.isfinite(ref)
    assert np.abs(got[finite].astype(np.float64) - ref[finite]).max(initial=0.0) <= tol * scale


# (B, N, wide_phases), the small layers' path off: slices in LDS, the 32-sample tile, gathered from L2, in phases
VALUE_SHAPES = [(3, 300, 0), (40, 700, 0), (5, 1300, 0), (70, 2000, 0), (160, 4096, -1), (40, 1300, 1), (70, 5000, 1)]


# Infinities and NaN go where the sums of the layer's definition take them and nowhere else: padded samples, slots and connections
# add none.  Both gradients too, through the walk over the columns.
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,N,phases", VALUE_SHAPES)
def test_infinities_and_nan_stay_where_they_belong(ffi, bf16, B, N, phases):
    L, K = 1_003, 13
    x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=B + N)
    x[0, ::7], x[1, 3], x[B - 1, 5], x[B - 1, 11] = 0.0, np.inf, -np.inf, np.nan
    w[7, 0], w[8, 2], w[L - 1, K - 1], w[L - 1, 0] = np.inf, np.nan, -np.inf, 0.0
    g[0, 9], g[1, 10], g[B - 1, L - 1] = np.inf, np.nan, -np.inf
    tx, tw = torch.from_numpy(x), torch.from_numpy(w)
    if bf16:
        tx, tw = tx.bfloat16(), tw.bfloat16()
    lib = ffi._lib.lib()
    assert lib.ffi_set_option(b"wide_phases", phases) == 0 and lib.ffi_set_option(b"small_path", -1) == 0
    print(f"case bf16={bf16} B={B} N={N} phases={phases}", flush=True)
    try:
        with np.errstate(invalid="ignore"):
            ref = oracle.forward(tx.float().numpy(), lookup, tw.float().numpy(), transposed=False)
        out = (ffi.fan_in_sparse_matmul_bf16 if bf16 else ffi.fan_in_sparse_matmul)(tx.cuda(), dev(lookup), tw.cuda())
        _same_values(out.cpu().numpy(), ref, 1e-5, np.abs(ref[np.isfinite(ref)]).max())
        if not bf16:
            ref_gx, ref_gw = oracle.backward(x, lookup, w, g, transposed=False)
            for _ in range(2):
                gx, gw = ffi.fan_in_sparse_matmul_grad(dev(x), dev(lookup), dev(w), dev(g))
                _same_values(gx.cpu().numpy(), ref_gx, 1e-4, np.abs(ref_gx[np.isfinite(ref_gx)]).max())
                _same_values(gw.cpu().numpy(), ref_gw, 1e-4, np.abs(ref_gw[np.isfinite(ref_gw)]).max())
    finally:
        lib.ffi_set_option(b"wide_phases", 0)
        lib.ffi_set_option(b"small_path", 0)


# Operands below the smallest normal number count for what they are, and so do sums that are subnormal themselves
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("B,N,phases", VALUE_SHAPES)
def test_subnormal_operands_and_sums(ffi, bf16, B, N, phases):
    L, K = 1_003, 12
    rng = np.random.default_rng(B + N)
    lookup = rng.integers(0, N, (L, K)).astype(np.int32)
    lib = ffi._lib.lib()
    assert lib.ffi_set_option(b"wide_phases", phases) == 0 and lib.ffi_set_option(b"small_path", -1) == 0
    print(f"case bf16={bf16} B={B} N={N} phases={phases}", flush=True)
    try:
        for ex, ew, eg in ((-131, 110, 0), (110, -131, 0), (-70, -65, -65), (-131, 0, 0)):         # (bf16 holds multiples of 2^-133)
            x = (rng.integers(-3, 4, (B, N)) * 2.0 ** ex).astype(np.float32)
            w = (rng.integers(-3, 4, (L, K)) * 2.0 ** ew).astype(np.float32)
            g = (rng.integers(-3, 4, (B, L)) * 2.0 ** eg).astype(np.float32)
            tx, tw = torch.from_numpy(x), torch.from_numpy(w)
            if bf16:
                tx, tw = tx.bfloat16(), tw.bfloat16()
                assert np.array_equal(tx.float().numpy(), x) and np.array_equal(tw.float().numpy(), w)
            # (small whole numbers times a power of two: every sum is exact)
            ref = oracle.forward(x, lookup, w, transposed=False)
            out = (ffi.fan_in_sparse_matmul_bf16 if bf16 else ffi.fan_in_sparse_matmul)(tx.cuda(), dev(lookup), tw.cuda())
            assert np.abs(ref).max() > 0 and np.array_equal(out.cpu().numpy(), ref), (ex, ew)
            if not bf16:
                ref_gx, ref_gw = oracle.backward(x, lookup, w, g, transposed=False)
                gx, gw = ffi.fan_in_sparse_matmul_grad(dev(x), dev(lookup), dev(w), dev(g))
                assert np.array_equal(gw.cpu().numpy(), ref_gw) and np.array_equal(gx.cpu().numpy(), ref_gx), (ex, ew)
    finally:
        lib.ffi_set_option(b"wide_phases", 0)
        lib.ffi_set_option(b"small_path", 0)


# Plans of the global form: few and many streams, columns of fewer connections than a step and of many, ids so uneven that the slots are
# far from what uniform ids would give; narrow layers too uneven for the tiled form
@pytest.mark.parametrize("kind", ["uniform", "one column", "squared", "last column"])
@pytest.mark.parametrize("N,L,K", [(1275, 40, 3), (1276, 2_000, 16), (1530, 9_000, 8), (1531, 30_000, 4), (70_000, 300, 2), (255, 5_000, 8), (256, 6_000, 9)])
def test_plans_of_the_global_form(ffi, kind, N, L, K):
    B = 7
    x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=N + L)
    if kind == "one column":
        lookup[:] = N // 2
        lookup[::97] = 0
    elif kind == "squared":
        lookup = (lookup.astype(np.int64) ** 2 // N).astype(np.int32)
    elif kind == "last column":
        lookup[:, :] = N - 1
    ref_gx, ref_gw = oracle.backward(x, lookup, w, g, transposed=False)
    lib = ffi._lib.lib()
    assert lib.ffi_set_option(b"small_path", -1) == 0
    try:
        dx, dl, dw, dg = dev(x), dev(lookup), dev(w), dev(g)
        for _ in range(2):
            gx, gw = ffi.fan_in_sparse_matmul_grad(dx, dl, dw, dg)
            assert rel_err(gx.cpu().numpy(), ref_gx) <= 1e-4 and rel_err(gw.cpu().numpy(), ref_gw) <= 1e-4
    finally:
        lib.ffi_set_option(b"small_path", 0)


# Plans of one stream to seven, which put several slices of the samples into one workgroup of the walk: one label of more connections than the tiled form
# takes, steps of four and of eight connections; samples for fewer slices than a workgroup has wavefronts, as many and more
@pytest.mark.parametrize("streams", [1, 2, 3, 4, 5, 7])
@pytest.mark.parametrize("hint,B", [(0, 193), (0, 641), (32, 193), (32, 481)])
def test_walks_of_few_streams(ffi, streams, hint, B):
    N, L, K = 32 * streams - 3, 1, 1100
    x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=streams + B)
    ref_gx, ref_gw = oracle.backward(x, lookup, w, g, transposed=False)
    dx, dl, dw, dg = dev(x), dev(lookup), dev(w), dev(g)
    lib, stream = ffi._lib.lib(), torch.cuda.current_stream().cuda_stream
    plan = ctypes.c_void_p()
    ffi._lib.check(lib.ffi_plan_create(dl.data_ptr(), L, K, N, hint, stream, ctypes.byref(plan)))
    try:
        for transposed in (0, 1):
            gx = torch.full((N, B) if transposed else (B, N), float("nan"), device="cuda")
            ffi._lib.check(lib.ffi_input_grad_planned_f32(plan, dw.data_ptr(), dg.data_ptr(), gx.data_ptr(), B, transposed, stream))
            got = gx.cpu().numpy()
            # some K / N products of one gradient and a weight each, at most 128 of them: 128 2^-24 of the largest sum
            assert rel_err(got.T if transposed else got, ref_gx) <= 1e-5
    finally:
        ffi._lib.check(lib.ffi_plan_destroy(plan))
    # both gradients in one walk
    assert lib.ffi_set_option(b"small_path", -1) == 0 and lib.ffi_set_option(b"dense_rows", -1) == 0
    try:
        for _ in range(2):
            gx, gw = ffi.fan_in_sparse_matmul_grad(dx, dl, dw, dg)
            assert rel_err(gx.cpu().numpy(), ref_gx) <= 1e-5 and rel_err(gw.cpu().numpy(), ref_gw) <= 1e-4
    finally:
        assert lib.ffi_set_option(b"small_path", 0) == 0 and lib.ffi_set_option(b"dense_rows", 0) == 0


def test_more_lookups_than_the_cache_holds(ffi):
    # the plan that makes room hands its buffers on, to lookups of any shape and form; a lookup with an id out of range in between is
    # refused and leaves the cache usable
    shapes = [(9, 2000, 3_000, 12), (9, 300, 4_000, 16), (9, 1100, 3_000, 8), (9, 40_000, 900, 20), (9, 64, 50, 4), (9, 2000, 3_100, 12)]
    cases = []
    for n in range(14):
        B, N, L, K = shapes[n % len(shapes)]
        x, lookup, w, g = reference_law_inputs(B, N, L, K, seed=n)
        cases.append((oracle.backward(x, lookup, w, g, transposed=False), [dev(a) for a in (x, lookup, w, g)]))
    lib = ffi._lib.lib()
    ffi._lib.check(lib.ffi_cache_clear())
    held = []
    for turn in range(3):
        for (ref_gx, ref_gw), (x, lookup, w, g) in cases:
            for _ in range(2):
                gx, gw = ffi.fan_in_sparse_matmul_grad(x, lookup, w, g)
                assert rel_err(gx.cpu().numpy(), ref_gx) <= 1e-4 and rel_err(gw.cpu().numpy(), ref_gw) <= 1e-4
        held.append(lib.ffi_cache_bytes())
        x, lookup, w, g = cases[turn][1]
        bad = lookup.clone()
        bad[1, 1] = x.shape[1]
        with pytest.raises(ffi._lib.FfiError):
            ffi.fan_in_sparse_matmul_grad(x, bad, w, g)
    assert held[1] == held[2]                                    # (nothing piles up)
    ffi._lib.check(lib.ffi_cache_clear())
    assert lib.ffi_cache_bytes() == 0


def test_a_batch_that_is_too_large_is_refused_before_anything_is_written(ffi):
    B, N, L, K = 65_535 * 32 + 1, 1217, 4, 2
    lib = ffi._lib.lib()
    x, gx = torch.empty((N, B), device="cuda"), torch.empty((N, B), device="cuda")
    gx[:, :8] = gx[:, -8:] = 7.0
    lookup, w = torch.zeros((L, K), dtype=torch.int32, device="cuda"), torch.zeros((L, K), device="cuda")
    g, gw = torch.zeros((B, L), device="cuda"), torch.full((L, K), 7.0, device="cuda")
    torch.cuda.synchronize()
    status = lib.ffi_backward_f32(x.data_ptr(), lookup.data_ptr(), w.data_ptr(), g.data_ptr(), gx.data_ptr(), gw.data_ptr(), B, N, L, K, 1,
                                  torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert status == -3
    assert bool((gw == 7.0).all()) and bool((gx[:, :8] == 7.0).all()) and bool((gx[:, -8:] == 7.0).all())
    del x, gx
    torch.cuda.empty_cache()
    ffi._lib.check(lib.ffi_cache_clear())
