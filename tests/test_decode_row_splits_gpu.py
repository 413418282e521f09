"""int4 decode batches on the chunked-K kernel: units split at 16 and 32 rows, and a shared expert whose block pairs have more
waves than the routed experts'."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from tests.synth import Int4Layer
from tests.test_kernels_gpu import check_layer

pytestmark = pytest.mark.gpu


# launches of at least 1536 block pairs in the w2 pass (the first; the shared expert's reduction is the longer one) and in the
# w13 pass (the second); Zipf routing: units of 1 to all rows
@pytest.mark.parametrize("H,I,I_sh", [(2048, 128, 256), (256, 1024, 256)])
@pytest.mark.parametrize("T", [12, 16, 17, 32, 33, 48, 49, 64])
def test_batches_at_the_edges_of_the_splits(cuda, T, H, I, I_sh):
    print(f"case decode_row_splits T={T} H={H}", flush=True)
    check_layer(Int4Layer(H=H, I=I, E=24, I_sh=I_sh, seed=31, zipf=1.2), T, 4, 0, cuda)


@pytest.mark.parametrize("T", [20, 40])
def test_units_of_more_than_twice_the_split(cuda, T):
    """An expert listed twice for every token: its second half is longer than the split, units from the device list and by value."""
    from promoe_amd import ops
    print(f"case decode_row_splits repeated T={T}", flush=True)
    H, I, E = 2048, 128, 24
    layer = Int4Layer(H=H, I=I, E=E, I_sh=0, seed=32)
    x = O.synth_acts(T, H, seed=5)
    xd = torch.from_numpy(x).to(torch.bfloat16).to(cuda)
    idx = np.ones((T, 2), np.int32)
    d = ops.dispatch(torch.from_numpy(idx).to(cuda), E)
    slots = [torch.from_numpy(s).to(cuda) for s in layer.slots]
    table = torch.tensor([s.data_ptr() for s in slots], dtype=torch.int64, device=cuda)
    wg, wu, wd = layer.experts_fp32[1]
    g, u = x @ wg.T, x @ wu.T
    want = (g / (1.0 + np.exp(-g)) * u) @ wd.T                    # every row of a token
    tok = d.sorted_tok.cpu().numpy()[: 2 * T]
    for host_units in (False, True):
        part_r, _, err, _, _ = ops.experts_decode_int4(xd, d, table, None, H, I, 0, host_units=host_units)
        torch.cuda.synchronize()
        assert int(err.item()) == 0
        got = part_r.cpu().numpy()
        assert np.isfinite(got).all()
        # h in bf16 between the passes: 2^-9 of each of 128 terms
        assert np.abs(got - want[tok]).max() <= 2e-2 * np.abs(want).max(), host_units


def _swiglu_rows(layer, x, idx, d):
    """Every routed partial row as the oracle's expert gives it, in the order of the dispatch."""
    T, k = idx.shape
    want = np.empty((T * k, layer.H), np.float32)
    pos = d.pos_of_pair.cpu().numpy()[: T * k].reshape(T, k)
    for e in np.unique(idx):
        t, j = np.nonzero(idx == e)
        want[pos[t, j]] = O.swiglu_expert(torch.from_numpy(x[t]), *[torch.from_numpy(w) for w in layer.experts_fp32[e]]).numpy()
    return want


# 24 tokens: units split at 16 rows, 40: at 32.  (60 used experts and 5 of more rows than that: one more half than travels by value)
@pytest.mark.parametrize("T", [24, 40])
@pytest.mark.parametrize("used,heavy", [(59, 5), (60, 5), (64, 0), (64, 1)])
def test_units_by_value_at_the_room_for_their_halves(cuda, T, used, heavy):
    from promoe_amd import ops
    print(f"case decode_row_splits by value T={T} used={used} heavy={heavy}", flush=True)
    H, I, k = 2048, 128, 8
    layer = Int4Layer(H=H, I=I, E=64, I_sh=256, seed=33)
    light = np.arange(T * (k - heavy)).reshape(T, k - heavy) % (used - heavy) + heavy
    idx = np.concatenate([np.tile(np.arange(heavy), (T, 1)), light], axis=1).astype(np.int32)
    counts = np.bincount(idx.reshape(-1), minlength=64)
    assert (counts > 0).sum() == used and (counts > (16 if T <= 32 else 32)).sum() == heavy
    x = O.synth_acts(T, H, seed=6)
    xd = torch.from_numpy(x).to(torch.bfloat16).to(cuda)
    d = ops.dispatch(torch.from_numpy(idx).to(cuda), 64, max_units=used)
    slots = [torch.from_numpy(s).to(cuda) for s in layer.slots]
    table = torch.tensor([s.data_ptr() for s in slots], dtype=torch.int64, device=cuda)
    shared = torch.from_numpy(layer.shared_img).to(cuda)
    want = _swiglu_rows(layer, x, idx, d)
    sh = O.swiglu_expert(torch.from_numpy(x), *[torch.from_numpy(w) for w in layer.shared_fp32]).numpy()
    for host_units in (True, False):
        part_r, part_s, err, _, _ = ops.experts_decode_int4(xd, d, table, shared, H, I, 256, host_units=host_units)
        torch.cuda.synchronize()
        assert int(err.item()) == 0
        # h in bf16 between the passes: 2^-9 of each of 128 and 256 terms
        assert np.abs(part_r.cpu().numpy() - want).max() <= 2e-2 * np.abs(want).max(), host_units
        assert np.abs(part_s.cpu().numpy() - sh).max() <= 2e-2 * np.abs(sh).max(), host_units


@pytest.fixture(scope="module")
def long_shared():
    """24 experts of 11 groups in w2 beside a shared expert of 22: several chunks of every pass width, in launches of at least
    1536 block pairs with all units in use."""
    return Int4Layer(H=2048, I=1408, E=24, I_sh=2816, seed=34)


@pytest.mark.parametrize("T", [9, 12, 16, 17, 32, 33, 40, 48])
def test_shared_expert_with_more_waves_over_several_chunks(cuda, long_shared, T):
    """The shared expert's w2 with two waves a block pair (9 to 16 and 33 to 48 tokens), whose sums each have groups of every
    chunk, and the split at 16 rows; units from the device list and by value."""
    from promoe_amd import ops
    layer, H, k = long_shared, 2048, 6
    print(f"case decode_row_splits long shared T={T}", flush=True)
    x = O.synth_acts(T, H, seed=7)
    xd = torch.from_numpy(x).to(torch.bfloat16).to(cuda)
    rng = np.random.default_rng(T)
    # five popular experts for half of the choices, the others in turn: every expert in use, units of a few and of many rows
    idx = np.stack([np.concatenate([rng.permutation(5)[:3], 5 + (np.arange(3) + 3 * t) % 19]) for t in range(T)]).astype(np.int32)
    d = ops.dispatch(torch.from_numpy(idx).to(cuda), 24)
    assert int(d.n_active.item()) == 24
    slots = [torch.from_numpy(s).to(cuda) for s in layer.slots]
    table = torch.tensor([s.data_ptr() for s in slots], dtype=torch.int64, device=cuda)
    shared = torch.from_numpy(layer.shared_img).to(cuda)
    want = _swiglu_rows(layer, x, idx, d)
    sh = O.swiglu_expert(torch.from_numpy(x), *[torch.from_numpy(w) for w in layer.shared_fp32]).numpy()
    for host_units in (False, True):
        part_r, part_s, err, _, _ = ops.experts_decode_int4(xd, d, table, shared, H, 1408, 2816, host_units=host_units)
        torch.cuda.synchronize()
        assert int(err.item()) == 0
        # h in bf16 between the passes: relative 2^-9 a term, sums of 1408 and 2816 terms of random sign
        assert np.abs(part_r.cpu().numpy() - want).max() <= 2e-2 * np.abs(want).max(), host_units
        assert np.abs(part_s.cpu().numpy() - sh).max() <= 2e-2 * np.abs(sh).max(), host_units
