"""The combine for every number of choices that has its own number of rows on their way."""
import numpy as np
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("k", [0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 17])
def test_combine_of_k_rows(cuda, k):
    """Weighted rows in pair order, then the gated shared row: the same fma chain in fp32, rounded to bf16."""
    from promoe_amd import ops
    T, H = 5, 260
    rng = np.random.default_rng(k)
    rows = rng.normal(0, 1, (max(T * k, 1), H)).astype(np.float32)
    w = rng.random((T, max(k, 1))).astype(np.float32)
    pos = rng.permutation(max(T * k, 1)).astype(np.int32)
    sh, gate = rng.normal(0, 1, (T, H)).astype(np.float32), rng.normal(0, 1, (T, 3)).astype(np.float32)
    dev = lambda a: torch.from_numpy(a).to(cuda)
    y = ops.combine(dev(rows), dev(sh), dev(w), dev(pos), dev(gate)[:, 1], T, H, k).float().cpu().numpy()
    acc = np.zeros((T, H))
    for t in range(T):
        for j in range(k):
            acc[t] = np.float32(acc[t] + np.float64(w[t, j]) * rows[pos[t * k + j]])
    want = acc + (1.0 / (1.0 + np.exp(-gate[:, 1:2].astype(np.float64)))) * sh
    assert np.abs(y - want).max() <= 2.0 ** -8 * np.abs(want).max() + 1e-6   # (the bf16 of the result)
