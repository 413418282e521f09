"""The w2 pass of the tile kernels with the reduction cut into windows, and the combine that adds the pieces."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from tests.synth import Bf16Layer, Int4Layer, Q4KLayer

pytestmark = pytest.mark.gpu


def _passes(layer, fmt, T, k, dev, routed, shared):
    """Partial rows of one batch, pieces apart: [routed, T k, H], [shared, T, H]."""
    from promoe_amd import ops, _lib as L
    H, I, I_sh, E = layer.H, layer.I, layer.I_sh, layer.E
    x = torch.from_numpy(O.synth_acts(T, H, seed=3)).to(torch.bfloat16).to(dev)
    idx = torch.from_numpy(np.stack([np.random.default_rng(t).permutation(E)[:k] for t in range(T)]).astype(np.int32)).to(dev)
    d = ops.dispatch(idx, E)
    slots = [torch.from_numpy(s).to(dev) for s in layer.slots]
    table = torch.tensor([s.data_ptr() for s in slots], dtype=torch.int64, device=dev)
    sh = torch.from_numpy(layer.shared_img).to(dev)
    part_r = torch.full((routed, T * k, H), float("nan"), device=dev)
    part_s = torch.full((shared, T, H), float("nan"), device=dev)
    h_r = torch.empty(T * k, I, dtype=torch.float16, device=dev)   # (bf16 layers: bf16 in the same room)
    h_s = torch.empty(T, I_sh, dtype=torch.float16, device=dev)
    err = torch.zeros(1, dtype=torch.int32, device=dev)
    ws = torch.empty(ops.prefill_workspace_bytes(fmt, T, H, k, d.max_units), dtype=torch.uint8, device=dev)
    p, phases = L.ptr, 3 if fmt == L.FMT_BF16 else 3 | 4
    L.check(L.lib.moe_experts_prefill_windows(p(x), T, H, I, I_sh, k, fmt, p(d.units), d.max_units, p(d.sorted_tok), p(table),
                                              p(sh), p(h_r), p(h_s), p(part_r), p(part_s), shared, routed, p(ws), p(err), phases,
                                              None, L.cur_stream()), "moe_experts_prefill_windows")
    torch.cuda.synchronize()
    assert int(err.item()) == 0
    return part_r, part_s, d


@pytest.mark.parametrize("cls,I,I_sh,T,routed,shared", [
    (Int4Layer, 384, 640, 70, 3, 2),      # windows of two and five slabs: shorter than the ring, inside a quantisation group
    (Int4Layer, 1408, 256, 129, 2, 1),     # eleven slabs; second tiles of few rows
    (Int4Layer, 2048, 2816, 97, 8, 2),    # the most windows; the shared expert in two windows of eleven groups
    (Q4KLayer, 768, 512, 65, 3, 1),       # windows of four slabs: whole super-blocks
    (Q4KLayer, 512, 512, 200, 4, 2),      # windows of two slabs: half a super-block
    (Bf16Layer, 128, 512, 65, 1, 4),      # windows of two slabs
    (Bf16Layer, 256, 2816, 129, 1, 2),    # of 22; a second tile of one row
    (Bf16Layer, 128, 1024, 300, 1, 8),
])
def test_pieces_add_up_to_the_whole_rows(cuda, cls, I, I_sh, T, routed, shared):
    from promoe_amd import _lib as L
    print(f"case windows {cls.__name__} I={I} I_sh={I_sh} T={T} routed={routed} shared={shared}", flush=True)
    H, k = 512, 2
    layer = cls(H=H, I=I, E=5, I_sh=I_sh, seed=21)
    fmt = {Q4KLayer: L.FMT_Q4K, Int4Layer: L.FMT_INT4_G128, Bf16Layer: L.FMT_BF16}[cls]
    r1, s1, _ = _passes(layer, fmt, T, k, cuda, 1, 1)
    rn, sn, d = _passes(layer, fmt, T, k, cuda, routed, shared)
    # the same products, added in another order: fp32 sums of up to 2816 terms differ by some units of 2^-24 of their norm
    for one, many in ((r1, rn), (s1, sn)):
        assert torch.isfinite(many).all()
        diff = (many.double().sum(0) - one[0].double()).norm() / one[0].double().norm()
        assert diff <= 1e-5, float(diff)
    # the combine: pieces in order, then weight and sum, as separate fp32 operations would give it
    w = torch.rand(T, k, device=cuda)
    y = torch.empty(T, H, dtype=torch.bfloat16, device=cuda)
    p = L.ptr
    L.check(L.lib.moe_combine_windows(p(rn), p(sn), p(w), p(d.pos_of_pair), None, 0, p(y), T, H, k, routed, shared,
                                      L.cur_stream()), "moe_combine_windows")
    rows = rn.double().sum(0)[d.pos_of_pair[: T * k].long()].view(T, k, H)
    want = (rows * w.double()[:, :, None]).sum(1) + sn.double().sum(0)
    # bf16 out: half a unit in the last place, and fp32 sums of a few terms
    bound = 2.0 ** -8 * want.abs() + 1e-5 * ((rows.abs() * w.double()[:, :, None]).sum(1) + sn.double().abs().sum(0))
    assert ((y.double() - want).abs() <= bound).all()


def test_windows_that_do_not_divide_the_reduction_are_refused(cuda):
    """(Every buffer is real and large enough for the sizes as given, and no unit has rows: a call that was taken after all would
    only fail the assertion.)"""
    from promoe_amd import _lib as L
    T, H, k, p = 70, 256, 2, L.ptr
    x = torch.zeros(T, H, dtype=torch.bfloat16, device=cuda)
    units, tok = torch.zeros(4, 4, dtype=torch.int32, device=cuda), torch.zeros(T * k, dtype=torch.int32, device=cuda)
    table, err = torch.zeros(4, dtype=torch.int64, device=cuda), torch.zeros(1, dtype=torch.int32, device=cuda)
    shared = torch.zeros(3 * 512 * H * 2, dtype=torch.uint8, device=cuda)
    h_r, h_s = torch.zeros(T * k, 1024, dtype=torch.float16, device=cuda), torch.zeros(T, 512, dtype=torch.float16, device=cuda)
    part_r, part_s = torch.zeros(9 * T * k, H, device=cuda), torch.zeros(8 * T, H, device=cuda)
    ws = torch.zeros(1 << 20, dtype=torch.uint8, device=cuda)

    def call(fmt, I, I_sh, pieces, routed):
        sh = I_sh > 0
        return L.lib.moe_experts_prefill_windows(p(x), T, H, I, I_sh, k, fmt, p(units), 4, p(tok), p(table), p(shared) if sh else None,
                                                 p(h_r), p(h_s) if sh else None, p(part_r), p(part_s) if sh else None, pieces, routed,
                                                 p(ws), p(err), 3, None, L.cur_stream())
    for fmt, I, routed in ((L.FMT_INT4_G128, 384, 4), (L.FMT_INT4_G128, 128, 2), (L.FMT_BF16, 512, 2), (L.FMT_INT4_G128, 1024, 9),
                           (L.FMT_INT4_G128, 1024, 0)):
        assert call(fmt, I, 0, 1, routed) != 0 and b"windows" in L.lib.moe_last_error(), (fmt, I, routed)
    for I_sh, pieces in ((384, 2), (512, 8)):    # bf16: windows of three slabs, of one
        assert call(L.FMT_BF16, 128, I_sh, pieces, 1) != 0 and b"windows" in L.lib.moe_last_error(), (I_sh, pieces)
    torch.cuda.synchronize()


@pytest.mark.parametrize("cache_rate", [1.0, 0.5])
def test_layer_of_few_wide_experts(cuda, cache_rate):
    """A layer whose routed reduction the engine cuts into windows, every expert resident and half of them."""
    from promoe_amd import _lib as L
    from tests.test_engine_gpu import build_engine, ref_forward
    print(f"case wide experts cache_rate={cache_rate}", flush=True)
    H, I, E, k = 256, 4096, 4, 2
    assert L.lib.moe_prefill_routed_windows(L.FMT_INT4_G128, 70, k, E, H, I) == 2
    assert L.lib.moe_prefill_routed_windows(L.FMT_INT4_G128, 256, 2, 8, 4096, 14336) == 4   # Mixtral shape
    assert L.lib.moe_prefill_routed_windows(L.FMT_INT4_G128, 4096, 2, 8, 4096, 14336) == 1
    assert L.lib.moe_prefill_routed_windows(L.FMT_INT4_G128, 128, 6, 64, 2048, 1408) == 1   # DeepSeek shape: 22 slabs
    layer = Int4Layer(H=H, I=I, E=E, I_sh=256, seed=5)
    pm = build_engine([layer], k, cuda, max_tokens=70, cache_rate=cache_rate, cache_policy="lru")
    for T in (70, 65, 40, 70):
        x = O.synth_acts(T, H, seed=T)
        y = pm.forward(0, torch.from_numpy(x).to(torch.bfloat16).to(cuda))
        torch.cuda.synchronize()
        ref = ref_forward(layer, x, k, 0)
        err = float(np.abs(y.float().cpu().numpy() - ref["out"]).max() / np.abs(ref["out"]).max())
        assert err <= 2e-2, (T, err)
    pm.close()


@pytest.mark.parametrize("cache_rate", [1.0, 0.5])
def test_layer_with_a_shared_expert_in_two_windows(cuda, cache_rate):
    """An int4 shared expert whose reduction is twice the routed experts' and too short for moe_prefill_shared_splits."""
    from promoe_amd import _lib as L
    from tests.test_engine_gpu import build_engine, ref_forward
    print(f"case shared windows cache_rate={cache_rate}", flush=True)
    H, I_sh, k = 256, 2176, 2
    lib, i4 = L.lib, L.FMT_INT4_G128
    assert lib.moe_prefill_shared_splits(i4, 130, H, I_sh) == 1 and lib.moe_prefill_shared_windows(i4, 130, H, I_sh) == 2
    assert lib.moe_prefill_shared_windows(i4, 512, 2048, 2816) == 2      # DeepSeek shape: 32 tiles
    assert lib.moe_prefill_shared_windows(i4, 513, 2048, 2816) == 1
    assert lib.moe_prefill_shared_windows(i4, 130, H, 1920) == 1         # 30 slabs
    assert lib.moe_prefill_shared_windows(i4, 200, 256, 8192) == 2 and lib.moe_prefill_shared_windows(L.FMT_Q4K, 512, 3584, 20480) == 4
    layer = Int4Layer(H=H, I=1024, E=4, I_sh=I_sh, seed=6)
    pm = build_engine([layer], k, cuda, max_tokens=130, cache_rate=cache_rate, cache_policy="lru")
    for T in (130, 65, 128):
        x = O.synth_acts(T, H, seed=T)
        y = pm.forward(0, torch.from_numpy(x).to(torch.bfloat16).to(cuda))
        torch.cuda.synchronize()
        ref = ref_forward(layer, x, k, 0)
        err = float(np.abs(y.float().cpu().numpy() - ref["out"]).max() / np.abs(ref["out"]).max())
        assert err <= 2e-2, (T, err)
    pm.close()


@pytest.mark.parametrize("T", [65, 128, 129, 257])
def test_bf16_layer_with_a_long_shared_expert(cuda, T):
    from promoe_amd import _lib as L
    from tests.test_engine_gpu import build_engine, ref_forward
    print(f"case bf16 shared windows T={T}", flush=True)
    lib, b16 = L.lib, L.FMT_BF16
    assert [lib.moe_prefill_shared_windows(b16, t, 2048, 5632) for t in (65, 128, 129, 256, 257)] == [4, 4, 2, 2, 1]   # Qwen1.5 shape
    assert lib.moe_prefill_shared_windows(b16, 128, 2048, 1408) == 1 and lib.moe_prefill_shared_windows(b16, 100, 256, 5120) == 4
    layer = Bf16Layer(H=256, I=256, E=4, I_sh=5120, seed=7, shared_gate=True)
    pm = build_engine([layer], 2, cuda, max_tokens=257, cache_rate=1.0, cache_policy="lru")
    for _ in range(2):
        x = O.synth_acts(T, 256, seed=T)
        y = pm.forward(0, torch.from_numpy(x).to(torch.bfloat16).to(cuda))
        torch.cuda.synchronize()
        ref = ref_forward(layer, x, 2, 0)
        err = float(np.abs(y.float().cpu().numpy() - ref["out"]).max() / np.abs(ref["out"]).max())
        assert err <= 2e-2, (T, err)
    pm.close()


@pytest.mark.parametrize("cls,I,I_sh,T", [(Int4Layer, 4096, 2304, 70), (Q4KLayer, 4096, 256, 70), (Bf16Layer, 256, 5120, 100)])
def test_the_operators_with_windows_are_the_layer_forward(cuda, cls, I, I_sh, T):
    """ops.experts_prefill with windows, and combine: the launches of the engine's forward, bit for bit."""
    from promoe_amd import ops, _lib as L
    from tests.test_engine_gpu import build_engine
    print(f"case windows ops {cls.__name__} T={T}", flush=True)
    H, E, k = 256, 4, 2
    fmt = {Q4KLayer: L.FMT_Q4K, Int4Layer: L.FMT_INT4_G128, Bf16Layer: L.FMT_BF16}[cls]
    R, S = ops.prefill_windows(fmt, T, k, E, H, I, I_sh)
    assert R * S > 1
    layer = cls(H=H, I=I, E=E, I_sh=I_sh, seed=8)
    pm = build_engine([layer], k, cuda, max_tokens=T, cache_rate=1.0, cache_policy="lru")
    x = torch.from_numpy(O.synth_acts(T, H, seed=T)).to(torch.bfloat16).to(cuda)
    y = pm.forward(0, x)
    torch.cuda.synchronize()
    lg = ops.gate_logits(x, torch.from_numpy(layer.wg).to(torch.bfloat16).to(cuda), None)
    idx, w = ops.topk(lg, k, 0, E=E)
    d = ops.dispatch(idx, E)
    slots = [torch.from_numpy(s).to(cuda) for s in layer.slots]
    table = torch.tensor([s.data_ptr() for s in slots], dtype=torch.int64, device=cuda)
    ws = ops.experts_prefill(x, d, table, torch.from_numpy(layer.shared_img).to(cuda), H, I, I_sh, fmt, windows=True)
    assert ws[0].shape[0] == R * T * k and ws[1].shape[0] == S * T and int(ws[2].item()) == 0
    y2 = ops.combine(ws[0], ws[1], w, d.pos_of_pair, None, T, H, k, routed_pieces=R)
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))
    pm.close()
