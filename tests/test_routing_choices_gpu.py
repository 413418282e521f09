"""Top-k of rows without k ordinary logits (NaN, which counts as -inf, and -inf): k different experts of the layer on every
route, and a layer forward that
keeps the other tokens' results and goes on."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from tests.synth import Bf16Layer, Int4Layer, Q4KLayer

pytestmark = pytest.mark.gpu
NAN, INF = float("nan"), float("inf")


def _logits(T, E, k, seed):
    lg = np.random.default_rng(seed).standard_normal((T, E)).astype(np.float32)
    rows = [np.full(E, NAN, np.float32), np.full(E, -INF, np.float32), lg[0].copy(), lg[0].copy(), lg[0].copy()]
    rows[2][: E - k + 1] = NAN            # fewer numbers than choices, the last experts'
    rows[3][k // 2:] = -INF               # the first experts'
    rows[4][::2] = NAN
    rows[4][1::2] = -INF
    for i, r in enumerate(rows[: T]):
        lg[(7 * i) % T] = r
    return lg


def _check(idx, d, lg, k, E):
    want, _ = O.topk_route(np.where(np.isnan(lg), -np.inf, lg), k, 0)      # (a NaN counts as -inf; the lower expert among equals)
    assert np.array_equal(idx.cpu().numpy(), want)
    T = lg.shape[0]
    counts, offsets, sp, pp = O.dispatch(want, E)
    assert np.array_equal(d.counts.cpu().numpy(), counts) and np.array_equal(d.offsets.cpu().numpy(), offsets)
    assert np.array_equal(d.sorted_pair.cpu().numpy()[: T * k], sp) and np.array_equal(d.pos_of_pair.cpu().numpy()[: T * k], pp)


@pytest.mark.filterwarnings("ignore:invalid value")
@pytest.mark.parametrize("E,k", [(8, 2), (8, 8), (60, 4), (64, 6), (65, 6), (100, 8), (128, 8), (200, 32), (256, 32)])
def test_rows_without_k_numbers(cuda, E, k):
    from promoe_amd import ops
    from promoe_amd._lib import lib, ptr, cur_stream, check
    for T in (1, 2, 5, 16, 70):
        print(f"case routing_choices E={E} k={k} T={T}", flush=True)
        lg = _logits(T, E, k, seed=E + T)
        lgd = torch.from_numpy(lg).to(cuda)
        idx, w = ops.topk(lgd, k, 0)
        _check(idx, ops.dispatch(idx, E), lg, k, E)
        if T <= 64 and T * k <= 512:
            idx2, w2, d = ops.topk_dispatch(lgd, k, E)
            _check(idx2, d, lg, k, E)
            assert torch.equal(w.view(torch.int32), w2.view(torch.int32))
        ws = torch.zeros(16 + 64 * E, dtype=torch.int32, device=cuda)
        d = ops.Dispatch(T, k, E, min(E, T * k), cuda)
        check(lib.moe_topk_dispatch_ws(ptr(lgd), T, E, E, k, 0, ptr(idx), ptr(w), ptr(d.counts), ptr(d.offsets), ptr(d.sorted_pair),
                                       ptr(d.pos_of_pair), ptr(d.sorted_tok), ptr(d.units), ptr(d.n_active), ptr(d.active_ids),
                                       d.max_units, ptr(ws), ws.numel() * 4, ptr(d.err), cur_stream()), "moe_topk_dispatch_ws")
        _check(idx, d, lg, k, E)


@pytest.mark.filterwarnings("ignore:invalid value")
@pytest.mark.parametrize("cache_rate", [1.0, 0.5])
@pytest.mark.parametrize("kind", ["int4", "bf16", "q4k"])
def test_layer_forward_with_a_token_of_nan_and_with_masked_experts(cuda, kind, cache_rate):
    from tests.test_engine_gpu import build_engine, ref_forward
    mk = {"int4": Int4Layer, "bf16": Bf16Layer, "q4k": Q4KLayer}[kind]
    for E, k in ((8, 2), (20, 4)):
        layers = [mk(H=256, I=256, E=E, I_sh=256, seed=90 + i) for i in range(2)]
        layers[1].bias = np.full(E, -np.inf, np.float32)      # fewer experts than choices
        layers[1].bias[E - 1] = 0.0
        pm = build_engine(layers, k, cuda, max_tokens=300, cache_rate=cache_rate, cache_policy="lru")
        if cache_rate == 1.0:
            for l in range(2):
                pm.acquire_layer(l, np.arange(E, dtype=np.int64))
                pm.release_layer(l)
            pm.drain()
        for T in (1, 1, 2, 8, 12, 17, 32, 33, 65, 300):
            print(f"case routing_choices_layer kind={kind} cache={cache_rate} E={E} T={T}", flush=True)
            for l, layer in enumerate(layers):
                x = O.synth_acts(T, 256, seed=T + l)
                ref = ref_forward(layer, x, k, 0)
                xd = torch.from_numpy(x).to(torch.bfloat16).to(cuda)
                bad = T // 2 if l == 0 else -1
                if l == 0:
                    xd[bad] = NAN
                y = pm.forward(l, xd).float().cpu().numpy()
                torch.cuda.synchronize()
                good = np.arange(T) != bad
                if l == 0:
                    assert np.isnan(y[bad]).all()
                    assert np.array_equal(pm.last_routing_idx(T, k)[bad], np.arange(k))
                if good.any():
                    err = np.abs(y[good] - ref["out"][good]).max() / np.abs(ref["out"]).max()
                    assert err <= 2e-2, (T, l, err)
                    assert np.array_equal(pm.last_routing_idx(T, k)[good], ref["idx"][good]), (T, l)
        pm.drain()
        pm.close()
