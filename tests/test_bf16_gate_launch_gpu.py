"""bf16 decode batches of 1 to 32 tokens whose w13 launch sums the gate rows and routes by itself."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from tests.synth import Bf16Layer
from tests.test_kernels_gpu import bf16_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,I,E,k,mode,I_sh,zipf,gated", [
    (1, 256, 128, 8, 2, 0, 128, None, False), (1, 2048, 256, 60, 4, 0, 512, None, True),
    (2, 512, 256, 8, 2, 2, 0, None, False), (4, 256, 384, 60, 4, 1, 256, 1.1, True),      # one token a gate workgroup, up to 4
    (5, 512, 128, 200, 8, 0, 0, None, False), (8, 2048, 128, 16, 6, 0, 256, 1.2, False),  # two, up to 8; more than 64 experts
    (9, 256, 256, 60, 4, 1, 512, 1.1, True), (16, 256, 128, 256, 32, 0, 0, None, False),
    (16, 256, 1024, 40, 4, 0, 128, 1.2, True),                                            # 32-row sets
    (17, 512, 128, 8, 2, 0, 128, 1.2, False), (25, 256, 256, 100, 4, 2, 0, None, True),   # eight tokens a wave, units of more than
    (32, 256, 1024, 40, 4, 0, 128, 1.2, True), (32, 2048, 128, 16, 16, 1, 256, 1.2, False)])   # 16 rows, of all 32
def test_gate_rows_and_routing_in_the_w13_launch(cuda, T, H, I, E, k, mode, I_sh, zipf, gated):
    """Logits, routing arrays and h rows equal those of the gate, routing and w13 launches, bit for bit, on successive calls
    over one hand-over workspace: ordinary logits, ties, and (two tokens and more) fewer finite logits than choices."""
    from promoe_amd import ops, _lib as L
    print(f"case bf16_gate T={T} H={H} I={I} E={E} k={k} mode={mode} I_sh={I_sh}", flush=True)
    layer = Bf16Layer(H=H, I=I, E=E, I_sh=I_sh, seed=41, zipf=zipf, shared_gate=gated)
    slots = [torch.from_numpy(s).to(cuda) for s in layer.slots]
    table = torch.tensor([s.data_ptr() for s in slots], dtype=torch.int64, device=cuda)
    shared = torch.from_numpy(layer.shared_img).to(cuda) if I_sh else None
    wg = bf16_dev(layer.wg if not gated else np.concatenate([layer.wg, layer.shared_gate[None, :]], axis=0), cuda)
    rows, P = wg.shape[0], T * k
    bias = torch.zeros(E, device=cuda) if layer.bias is None else torch.from_numpy(layer.bias).to(cuda)
    gws, gws_ref = ops.GateWorkspace(cuda, 32, 257), ops.GateWorkspace(cuda, 32, 257)
    p = L.ptr
    for seed in range(3 if T == 1 else 4):
        x = bf16_dev(O.synth_acts(T, H, seed=seed + 70), cuda)
        if seed == 2:                 # ties
            wg = wg.clone()
            wg[E // 2] = wg[1]; wg[E - 1] = wg[1]
            bias = bias.clone()
            bias[E // 2] = bias[1]; bias[E - 1] = bias[1]
        if seed == 3:
            bias = torch.full((E,), float("-inf"), device=cuda)
            bias[E - 1] = 0.0
        if T == 1:
            lg = ops.gate_logits(x, wg, torch.cat([bias, torch.zeros(rows - E, device=cuda)]))
            idx, w = ops.topk(lg, k, mode, E=E)
            d = ops.dispatch(idx, E)
        else:
            lg, idx, w, d, err0 = ops.gate_topk_dispatch(x, wg, bias, E, k, mode, gws_ref)
        h_r = torch.zeros(P, I, dtype=torch.bfloat16, device=cuda)
        h_s = torch.zeros(T, max(I_sh, 1), dtype=torch.bfloat16, device=cuda)
        part = torch.zeros(P, H, device=cuda)
        part_s = torch.zeros(8 * T, H, device=cuda)
        tiles = torch.empty(ops.prefill_workspace_bytes(L.FMT_BF16, T, H, k, d.max_units), dtype=torch.uint8, device=cuda)
        err = torch.zeros(1, dtype=torch.int32, device=cuda)
        L.check(L.lib.moe_experts_prefill(p(x), T, H, I, I_sh, k, L.FMT_BF16, p(d.units), d.max_units, p(d.sorted_tok), p(table),
                                          p(shared), p(h_r), p(h_s), p(part), p(part_s), p(tiles), p(err), 1, L.cur_stream()), "w13")
        d2 = ops.Dispatch(T, k, E, min(E, P), cuda)
        lg2, idx2 = torch.empty(T, rows, device=cuda), torch.empty(T, k, dtype=torch.int32, device=cuda)
        w2 = torch.empty(T, k, device=cuda)
        h_r2, h_s2 = torch.zeros_like(h_r), torch.zeros_like(h_s)
        L.check(L.lib.moe_decode_batch_bf16_gate(
            p(x), T, p(wg), p(bias), rows, p(gws.buf), gws.next_seq(), p(lg2), rows, E, k, mode, H, I, I_sh, p(table), p(shared),
            p(idx2), p(w2), p(d2.counts), p(d2.offsets), p(d2.sorted_pair), p(d2.pos_of_pair), p(d2.sorted_tok), p(d2.units),
            p(d2.n_active), p(d2.active_ids), d2.max_units, p(h_r2), p(h_s2), p(err), None, None, None, 0, L.cur_stream()),
            "moe_decode_batch_bf16_gate")
        torch.cuda.synchronize()
        assert int(err.item()) == 0
        assert torch.equal(lg[:, :rows].contiguous().view(torch.int32), lg2.view(torch.int32))
        assert torch.equal(idx, idx2) and torch.equal(w.view(torch.int32), w2.view(torch.int32))
        n = int(d.n_active.item())
        assert n == int(d2.n_active.item())
        for name in ("counts", "offsets", "pos_of_pair"):
            assert torch.equal(getattr(d, name), getattr(d2, name)), (seed, name)
        assert torch.equal(d.units[:n, :3], d2.units[:n, :3])
        used = int(d.offsets[E].item())          # (rows of repeated choices exist once)
        assert torch.equal(d.sorted_tok[:used], d2.sorted_tok[:used])
        assert torch.equal(h_r[:used].view(torch.int16), h_r2[:used].view(torch.int16)), seed
        if I_sh:
            assert torch.equal(h_s.view(torch.int16), h_s2.view(torch.int16))


@pytest.mark.parametrize("T", [1, 3, 16, 17, 32, 33])
def test_layer_forward(cuda, T):
    from tests.test_engine_gpu import build_engine, ref_forward
    print(f"case bf16_gate_layer T={T}", flush=True)
    layers = [Bf16Layer(H=256, I=256, E=16, I_sh=512, seed=50 + i, shared_gate=True) for i in range(2)]
    pm = build_engine(layers, 4, cuda, cache_rate=1.0, cache_policy="lru")
    for l in range(2):
        pm.acquire_layer(l, np.arange(16, dtype=np.int64))
        pm.release_layer(l)
    pm.drain()
    for step in range(12):                       # more than there are pending slots
        for l, layer in enumerate(layers):
            x = O.synth_acts(T, 256, seed=10 * step + l)
            y = pm.forward(l, torch.from_numpy(x).to(torch.bfloat16).to(cuda))
            torch.cuda.synchronize()
            ref = ref_forward(layer, x, 4, 0)
            err = float(np.abs(y.float().cpu().numpy() - ref["out"]).max() / np.abs(ref["out"]).max())
            assert err <= 2e-2, (step, l, err)
    pm.drain()
    c = pm.counters()
    assert c["forwards"] == 12 and c["miss"] <= 32 and c["evictions"] == 0, c     # misses: the acquisitions only
    pm.close()
