"""Label values counted at the best-ranked labels, one launch for all ranks, against a lookup in plain Python."""
import pytest
import torch

from conftest import load_package

pytestmark = pytest.mark.gpu


# more samples than the table in LDS holds, more positions than threads, none at all; ranks without a label
@pytest.mark.parametrize("batch,k,nnz", [(1, 1, 0), (3, 5, 7), (33, 8, 1500), (2048, 3, 4000), (2050, 8, 9000)])
@pytest.mark.parametrize("with_values", [False, True])
def test_hits_per_rank(batch, k, nnz, with_values):
    ffi = load_package()
    gen = torch.Generator().manual_seed(batch + k)
    top = torch.stack([torch.randperm(20, generator=gen)[:k] for _ in range(batch)]).to(torch.int32)
    top[::3, k - 1] = -1
    indices = torch.stack([torch.randint(-1, batch + 1, (nnz,), generator=gen), torch.randint(0, 20, (nnz,), generator=gen)], dim=1)
    values = torch.randn(nnz, generator=gen) if with_values else None
    want, seen = [0.0] * k, set()
    for p, (b, j) in enumerate(indices.tolist()):
        if (b, j) in seen or not 0 <= b < batch:
            continue
        seen.add((b, j))
        for r, label in enumerate(top[b].tolist()):
            want[r] += (float(values[p]) if with_values else 1.0) * (label == j)
    along = torch.tensor([0.3], device="cuda")
    y = (indices.cuda(), values.cuda() if with_values else None)
    got = ffi.metrics.topk_hits(top.cuda(), k, y, along)
    assert got[:k] == pytest.approx(want, abs=1e-9) and got[k] == float(along)
    metric = ffi.PrecisionAtK(k)
    metric.update_from_topk(y, top.cuda(), 20)
    assert metric.result() == pytest.approx(sum(want) / (batch * k), abs=1e-9)
