"""The order in which a label's connections are put: every place, against the rule in plain Python."""
import numpy as np
import pytest
import torch

from conftest import load_package

pytestmark = pytest.mark.gpu


def arranged(row, label):
    """Places of a chunk's connections: those of the label's first parity and the others in turn, then what is left."""
    role = (label >> 3) & 1
    first = [k for k, i in enumerate(row) if (i & 1) == role]
    second = [k for k, i in enumerate(row) if (i & 1) != role]
    m = min(len(first), len(second))
    return [k for pair in zip(first[:m], second[:m]) for k in pair] + first[m:] + second[m:]


# lane groups of 8, 16 and 32 with remainders, several chunks with a short last one; labels around whole wavefronts
@pytest.mark.parametrize("K", [1, 2, 7, 8, 9, 16, 17, 31, 32, 33, 70])
@pytest.mark.parametrize("n_arrays", [0, 4])
def test_places(K, n_arrays):
    ops = load_package().fixed_fan_in_ops
    rng = np.random.default_rng(K)
    for L in (1, 63, 130):
        lookup = rng.integers(0, 50, size=(L, K)).astype(np.int32)
        lookup[L // 2] &= ~1                                    # one parity only: nothing to move
        arrays = [rng.standard_normal((L, K)).astype(np.float32) for _ in range(n_arrays)]
        order = np.array([[lo + k for lo in range(0, K, 32) for k in arranged(row[lo:lo + 32], j)] for j, row in enumerate(lookup)])
        device = [torch.from_numpy(a.copy()).cuda() for a in [lookup] + arrays]
        for _ in range(2):                                      # the second call finds everything in place
            ops.arrange_connections(*device)
            for d, a in zip(device, [lookup] + arrays):
                np.testing.assert_array_equal(d.cpu().numpy(), np.take_along_axis(a, order, axis=1))
