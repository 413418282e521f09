"""The combine for every number of choices that has its own number of rows on their way."""
import numpy as np
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("k", [0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 17])
def test_combine_of_k_rows(cuda, k):
    """Weighted rows in pair order, then the gated shared row: a chain of fmas in fp32, rounded to bf16."""
    from promoe_amd import ops
    T, H = 5, 260
    rng = np.random.default_rng(k)
    rows = rng.normal(0, 1, (max(T * k, 1), H)).astype(np.float32)
    w = rng.random((T, max(k, 1))).astype(np.float32)
    pos = rng.permutation(max(T * k, 1)).astype(np.int32)
    sh, gate = rng.normal(0, 1, (T, H)).astype(np.float32), rng.normal(0, 1, (T, 3)).astype(np.float32)
    dev = lambda a: torch.from_numpy(a).to(cuda)
    y = ops.combine(dev(rows), dev(sh), dev(w), dev(pos), dev(gate)[:, 1], T, H, k).float().cpu().numpy()
    terms = np.zeros((k + 1, T, H))
    for t in range(T):
        for j in range(k):
            terms[j, t] = np.float64(w[t, j]) * rows[pos[t * k + j]]
    terms[k] = (1.0 / (1.0 + np.exp(-gate[:, 1:2].astype(np.float64)))) * sh
    want = terms.sum(0)
    # each value: the bf16 of the result (half a unit in the last place, at most 2^-8 of it) and the chain's roundings in fp32,
    # at most 18 of 2^-24 of the terms, the gate's few among them: 2^-19 of the terms
    assert (np.abs(y - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -19 * np.abs(terms).sum(0)).all()
