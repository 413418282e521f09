"""Parity of the MFMA prefill expert kernels (through the C ABI) against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from tests.synth import Bf16Layer, Int4Layer, Q4KLayer

pytestmark = pytest.mark.gpu

TOL = 2e-2  # max |y - ref| / max |ref|


def bf16_dev(a, dev):
    return torch.from_numpy(np.asarray(a, np.float32)).to(torch.bfloat16).to(dev)


def run_prefill_gpu(layer, x, k, mode, dev, resident=None):
    from promoe_amd import ops, _lib as L
    H, I, E, I_sh = layer.H, layer.I, layer.E, layer.I_sh
    T = x.shape[0]
    xd = bf16_dev(x, dev)
    wg = layer.wg
    if layer.shared_gate is not None:
        wg = np.concatenate([wg, layer.shared_gate[None, :]], axis=0)
    bias = None
    if layer.bias is not None:
        bias = torch.from_numpy(np.concatenate([layer.bias, np.zeros(wg.shape[0] - E, np.float32)])).to(dev)
    logits = ops.gate_logits(xd, bf16_dev(wg, dev), bias)
    idx, w = ops.topk(logits, k, mode, E=E)
    d = ops.dispatch(idx, E)
    slots = [torch.from_numpy(s).to(dev) for s in layer.slots]
    table = torch.tensor([0 if (resident is not None and e not in resident) else slots[e].data_ptr()
                          for e in range(E)], dtype=torch.int64, device=dev)
    shared = torch.from_numpy(layer.shared_img).to(dev) if I_sh else None
    fmt = L.FMT_BF16 if isinstance(layer, Bf16Layer) else (L.FMT_Q4K if isinstance(layer, Q4KLayer) else L.FMT_INT4_G128)
    part_r, part_s, err, h_r, h_s, _ = ops.experts_prefill(xd, d, table, shared, H, I, I_sh, fmt)
    sg = logits[:, E] if layer.shared_gate is not None else None
    y = ops.combine(part_r, part_s, w, d.pos_of_pair, sg, T, H, k)
    torch.cuda.synchronize()
    return dict(y=y.float().cpu().numpy(), idx=idx.cpu().numpy(), w=w.cpu().numpy(),
                logits=logits.cpu().numpy(), err=int(err.cpu()[0]), d=d)


def check_prefill(layer, T, k, mode, dev, seed=1):
    x = O.synth_acts(T, layer.H, seed=seed)
    got = run_prefill_gpu(layer, x, k, mode, dev)
    lg = O.gate_logits_ordered(x, layer.wg)
    if layer.bias is not None:
        lg = (lg + layer.bias[None, :]).astype(np.float32)
    ref = O.moe_forward(x, layer.wg, layer.experts_fp32, k, mode, shared=layer.shared_fp32,
                        shared_gate=layer.shared_gate, logits=lg)
    assert got["err"] == 0
    assert np.array_equal(got["idx"], ref["idx"])
    _, _, sp, _ = O.dispatch(ref["idx"], layer.E)
    assert np.array_equal(got["d"].sorted_pair.cpu().numpy()[:T * k], sp)
    err = np.abs(got["y"] - ref["out"]).max() / np.abs(ref["out"]).max()
    print(f"  T={T} k={k} mode={mode} max-rel-err={err:.3e}", flush=True)
    assert err <= TOL
    return err


@pytest.mark.parametrize("T", [1, 17, 128, 129, 300, 700])
def test_prefill_layer_small(cuda, T):
    print(f"case prefill_small T={T}", flush=True)
    check_prefill(Bf16Layer(H=256, I=384, E=8, I_sh=256, seed=3), T, 2, 0, cuda)


def test_prefill_layer_small_variants(cuda):
    print("case prefill_small_variants", flush=True)
    # no shared expert, Mixtral routing
    check_prefill(Bf16Layer(H=512, I=128, E=8, I_sh=0, seed=4), 200, 2, 2, cuda)
    # sigmoid-gated shared expert, renormalised routing, Zipf bias: some experts get no token
    check_prefill(Bf16Layer(H=256, I=256, E=60, I_sh=512, seed=5, shared_gate=True, zipf=1.4), 150, 4, 1, cuda)
    # more units than one scan pass is not needed (E <= 1024), K not a multiple of 128
    check_prefill(Bf16Layer(H=768, I=640, E=4, I_sh=128, seed=6), 260, 2, 0, cuda)


def test_prefill_non_resident_expert_is_reported(cuda):
    print("case prefill_non_resident", flush=True)
    layer = Bf16Layer(H=256, I=128, E=4, I_sh=0, seed=7)
    got = run_prefill_gpu(layer, O.synth_acts(64, 256), 2, 0, cuda, resident={0, 1})
    assert got["err"] == 1


def test_prefill_layer_qwen_shape(cuda):
    print("case prefill_qwen T=2048", flush=True)
    # Qwen1.5-MoE-A2.7B layer: H 2048, 60 experts x I 1408, top-4, sigmoid-gated shared expert I 5632
    layer = Bf16Layer(H=2048, I=1408, E=60, I_sh=5632, seed=0, shared_gate=True)
    check_prefill(layer, 2048, 4, 0, cuda)


# ---- int4-g128 experts through the same entry point ----

@pytest.mark.parametrize("T", [1, 17, 96, 97, 193, 400, 700])
def test_prefill_int4_layer_small(cuda, T):
    print(f"case prefill_int4_small T={T}", flush=True)
    check_prefill(Int4Layer(H=256, I=384, E=8, I_sh=256, seed=3), T, 2, 0, cuda)


def test_prefill_int4_layer_small_variants(cuda):
    print("case prefill_int4_small_variants", flush=True)
    check_prefill(Int4Layer(H=512, I=128, E=8, I_sh=0, seed=4), 200, 2, 2, cuda)
    check_prefill(Int4Layer(H=256, I=256, E=60, I_sh=512, seed=5, shared_gate=True, zipf=1.4), 150, 4, 1, cuda)
    check_prefill(Int4Layer(H=768, I=640, E=4, I_sh=128, seed=6), 260, 2, 0, cuda)


def test_prefill_int4_non_resident_expert_is_reported(cuda):
    print("case prefill_int4_non_resident", flush=True)
    layer = Int4Layer(H=256, I=128, E=4, I_sh=0, seed=7)
    got = run_prefill_gpu(layer, O.synth_acts(64, 256), 2, 0, cuda, resident={0, 1})
    assert got["err"] == 1


def test_prefill_int4_deepseek_shape(cuda):
    print("case prefill_int4_deepseek T=512", flush=True)
    # DeepSeek-MoE-16B layer shape; 16 experts instead of 64 keeps host-side quantisation short
    layer = Int4Layer(H=2048, I=1408, E=16, I_sh=2816, seed=0, zipf=1.2)
    check_prefill(layer, 512, 6, 0, cuda)


# ---- q4_K experts ----

@pytest.mark.parametrize("T", [1, 17, 97, 193, 400])
def test_prefill_q4k_layer_small(cuda, T):
    print(f"case prefill_q4k_small T={T}", flush=True)
    check_prefill(Q4KLayer(H=256, I=512, E=8, I_sh=256, seed=3), T, 2, 0, cuda)


def test_prefill_q4k_variants(cuda):
    print("case prefill_q4k_variants", flush=True)
    check_prefill(Q4KLayer(H=512, I=256, E=8, I_sh=0, seed=4), 200, 2, 2, cuda)
    check_prefill(Q4KLayer(H=256, I=256, E=60, I_sh=512, seed=5, shared_gate=True, zipf=1.1), 515, 8, 0, cuda)


def test_prefill_wide_shared_expert_in_pieces(cuda):
    """A shared expert much wider than the routed ones over few tokens: the w2 pass cuts its reduction into
    windows (moe_prefill_shared_splits) and leaves one piece of partial rows per window for the combine."""
    from promoe_amd import _lib as L
    print("case prefill shared expert in pieces", flush=True)
    assert L.lib.moe_prefill_shared_splits(L.FMT_Q4K, 130, 256, 16384) == 4
    assert L.lib.moe_prefill_shared_splits(L.FMT_INT4_G128, 200, 256, 8192) == 2
    assert L.lib.moe_prefill_shared_splits(L.FMT_BF16, 130, 256, 16384) == 1       # nibble formats only
    assert L.lib.moe_prefill_shared_splits(L.FMT_INT4_G128, 2048, 2048, 2816) == 1  # DeepSeek shape: 22 groups
    assert L.lib.moe_prefill_shared_splits(L.FMT_Q4K, 512, 3584, 20480) == 4        # Qwen2-57B shape
    check_prefill(Q4KLayer(H=256, I=256, E=4, I_sh=16384, seed=6, shared_gate=True), 130, 2, 0, cuda)
    check_prefill(Int4Layer(H=256, I=128, E=4, I_sh=8192, seed=7), 200, 2, 1, cuda)
    check_prefill(Int4Layer(H=512, I=128, E=4, I_sh=8192, seed=8), 70, 2, 0, cuda)   # 1 x 2 tiles: 2 pieces, short last tile


@pytest.mark.parametrize("cls,I", [(Int4Layer, 128), (Q4KLayer, 256)])
@pytest.mark.parametrize("T", [31, 32, 33, 127, 128, 129, 257])
def test_prefill_nibble_tile_edges(cuda, T, cls, I):
    """Every token to one expert: row blocks of 32 and tiles of 128 rows just short, full and just over; reductions of
    two slabs (q4_K: four; shorter than the ring they go through) and of eight."""
    print(f"case prefill_nibble_edges T={T} {cls.__name__}", flush=True)
    check_prefill(cls(H=512, I=I, E=1, I_sh=I, seed=9), T, 1, 0, cuda)


def test_prefill_nibble_without_room_for_the_converted_activations(cuda):
    """A workspace without room for the fp16 copy of x (phase bit 2 not set): the call takes memory of its own, same bits."""
    from promoe_amd import ops, _lib as L
    print("case prefill_no_room", flush=True)
    layer = Int4Layer(H=256, I=128, E=4, I_sh=128, seed=10)
    x = bf16_dev(O.synth_acts(70, 256), cuda)
    idx, _ = ops.topk(ops.gate_logits(x, bf16_dev(layer.wg, cuda), None), 2, 0)
    d = ops.dispatch(idx, 4)
    slots = [torch.from_numpy(s).to(cuda) for s in layer.slots]
    table = torch.tensor([s.data_ptr() for s in slots], dtype=torch.int64, device=cuda)
    shared = torch.from_numpy(layer.shared_img).to(cuda)
    a = ops.experts_prefill(x, d, table, shared, 256, 128, 128, L.FMT_INT4_G128)
    small = torch.empty(int(L.lib.moe_prefill_workspace_bytes(70, 2, d.max_units)), dtype=torch.uint8, device=cuda)
    ws = tuple(torch.zeros_like(t) for t in a[:5]) + (small,)
    b = ops.experts_prefill(x, d, table, shared, 256, 128, 128, L.FMT_INT4_G128, ws=ws)
    torch.cuda.synchronize()
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1]) and int(b[2].item()) == 0


def test_prefill_converts_the_activations_of_every_call(cuda):
    """Two calls that share a workspace with room for the fp16 copy: the second is over its own x, whatever bits above the
    documented ones its phases have."""
    from promoe_amd import ops, _lib as L
    print("case prefill_converts_each_call", flush=True)
    layer = Int4Layer(H=256, I=128, E=2, I_sh=128, seed=20)
    xs = [bf16_dev(O.synth_acts(70, 256, seed=70 + i), cuda) for i in range(2)]
    d = ops.dispatch(torch.zeros(70, 1, dtype=torch.int32, device=cuda), 2)
    slots = [torch.from_numpy(s).to(cuda) for s in layer.slots]
    table = torch.tensor([s.data_ptr() for s in slots], dtype=torch.int64, device=cuda)
    shared = torch.from_numpy(layer.shared_img).to(cuda)
    ref = ops.experts_prefill(xs[1], d, table, shared, 256, 128, 128, L.FMT_INT4_G128)
    ws = ops.experts_prefill(xs[0], d, table, shared, 256, 128, 128, L.FMT_INT4_G128)
    got = ops.experts_prefill(xs[1], d, table, shared, 256, 128, 128, L.FMT_INT4_G128, phases=3 | 8, ws=ws)
    torch.cuda.synchronize()
    assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1]) and int(got[2].item()) == 0


@pytest.mark.parametrize("T", [1, 15, 16, 17, 32, 33, 63, 64, 65])
def test_bf16_decode_batch_edges(cuda, T):
    """Every token to one expert, on the weight-stream kernel up to 64 tokens: passes of 16, 32 and 64 rows just short,
    full and just over; a routed reduction of two slabs (fewer than the waves that share it) and a shared one of 32 in
    two windows."""
    from promoe_amd import _lib as L
    print(f"case bf16_decode_edges T={T}", flush=True)
    assert L.lib.moe_prefill_shared_splits(L.FMT_BF16, T, 256, 2048) == (2 if T <= 64 else 1)
    check_prefill(Bf16Layer(H=256, I=128, E=1, I_sh=2048, seed=11, shared_gate=True), T, 1, 0, cuda)


@pytest.mark.parametrize("H,I,E,I_sh", [(256, 1024, 40, 128), (2048, 128, 40, 0)])
@pytest.mark.parametrize("T", [24, 64])
def test_bf16_decode_batch_row_sets(cuda, T, H, I, E, I_sh):
    """Grids of 1024 workgroups of 32-row sets and more (w13 of the first shape, w2 of the second), 16-row sets in the
    other pass; 64 tokens over 40 experts: units of few rows and units without any."""
    print(f"case bf16_decode_row_sets T={T} H={H}", flush=True)
    check_prefill(Bf16Layer(H=H, I=I, E=E, I_sh=I_sh, seed=12, zipf=1.2), T, 4, 1, cuda)


@pytest.mark.parametrize("T,k", [(1, 2), (16, 1), (16, 2), (13, 5), (16, 4), (17, 3), (32, 2), (33, 2), (40, 2), (64, 1), (64, 2), (65, 2)])
def test_bf16_decode_batch_units_of_more_rows_than_tokens(cuda, T, k):
    """An expert listed several times for one token: its unit has up to T k rows, more than one pass takes (16, 32 or 64 by
    the batch) and just over, a last pass of one row among them.  Every partial row against the oracle's expert."""
    from promoe_amd import ops, _lib as L
    print(f"case bf16_decode_repeated_experts T={T} k={k}", flush=True)
    H, I, E, I_sh = 256, 256, 3, 128
    layer = Bf16Layer(H=H, I=I, E=E, I_sh=I_sh, seed=13)
    x = O.synth_acts(T, H, seed=14)
    idx = np.ones((T, k), np.int32)
    if T == 33:                 # 65 rows of one expert, one of another
        idx[0, 0] = 2
    d = ops.dispatch(torch.from_numpy(idx).to(cuda), E)
    slots = [torch.from_numpy(s).to(cuda) for s in layer.slots]
    table = torch.tensor([s.data_ptr() for s in slots], dtype=torch.int64, device=cuda)
    shared = torch.from_numpy(layer.shared_img).to(cuda)
    part_r = torch.full((T * k, H), float("nan"), device=cuda)
    part_s = torch.full((T, H), float("nan"), device=cuda)
    h_r = torch.empty(T * k, I, dtype=torch.bfloat16, device=cuda)
    h_s = torch.empty(T, I_sh, dtype=torch.bfloat16, device=cuda)
    err = torch.zeros(1, dtype=torch.int32, device=cuda)
    tiles = torch.empty(ops.prefill_workspace_bytes(L.FMT_BF16, T, H, k, d.max_units), dtype=torch.uint8, device=cuda)
    ops.experts_prefill(bf16_dev(x, cuda), d, table, shared, H, I, I_sh, L.FMT_BF16, ws=(part_r, part_s, err, h_r, h_s, tiles))
    torch.cuda.synchronize()
    assert int(err.item()) == 0
    pos = d.pos_of_pair.cpu().numpy()[: T * k]
    assert np.array_equal(np.sort(pos), np.arange(T * k))
    xt = torch.from_numpy(x)
    ref = [O.swiglu_expert(xt, *[torch.from_numpy(w) for w in ws]).numpy() for ws in layer.experts_fp32]
    want = np.stack([ref[idx[p // k, p % k]][p // k] for p in range(T * k)])
    got = part_r.cpu().numpy()[pos]
    assert np.abs(got - want).max() <= TOL * np.abs(want).max()      # (h between the passes in bf16)
    sh = O.swiglu_expert(xt, *[torch.from_numpy(w) for w in layer.shared_fp32]).numpy()
    assert np.abs(part_s.cpu().numpy() - sh).max() <= TOL * np.abs(sh).max()


def _last_columns_image(kind, H, I, dev):
    """Image of an H x I expert whose weights are zero but for the last columns of the intermediate dimension (bf16, int4: 128,
    q4_K: 256), made from a small expert of just these: the image, and the small expert's fp32 weights."""
    from promoe_amd import layout as LY
    small_I = 256 if kind == "q4k" else 128
    cls = {"bf16": Bf16Layer, "int4": Int4Layer, "q4k": Q4KLayer}[kind]
    layer = cls(H=H, I=small_I, E=1, seed=15)
    src = torch.from_numpy(layer.slots[0]).to(dev)
    if kind == "bf16":
        big = torch.zeros(LY.bf16_expert_bytes(H, I), dtype=torch.uint8, device=dev)
        nk, group = H // 64, H // 64 * 16384                       # w13: 128-row groups of nk slabs, rotated by group
        for m in range(2):                                         # gate, up: the last group of each half
            t = src[m * group:(m + 1) * group].view(nk, 16384).roll(-((m * LY.slab_step(nk)) % nk), 0)
            g = (m + 1) * I // 128 - 1
            big[g * group:(g + 1) * group] = t.roll((g * LY.slab_step(nk)) % nk, 0).reshape(-1)
        nk = I // 64
        s2, b2 = src[2 * group:].view(H // 128, 2, 16384), big[2 * I * H * 2:].view(H // 128, nk, 16384)
        for g in range(H // 128):
            for j in range(2):
                b2[g, (nk - 2 + j + g * LY.slab_step(nk)) % nk] = s2[g, (j + g * LY.slab_step(2)) % 2]
        return big, layer.experts_fp32[0]
    mk = LY.int4_layout if kind == "int4" else LY.q4k_layout
    ls, lb = mk(H, small_I), mk(H, I)
    big = torch.zeros(lb["total_bytes"], dtype=torch.uint8, device=dev)
    for sec, per in (("q", 1024), ("s", 32 if kind == "int4" else 128), ("z", 8 if kind == "int4" else 32)):  # bytes per tile
        n13 = 2 * small_I // 16 * (H // 128) * per
        end = lb["off13_" + sec] + 2 * I // 16 * (H // 128) * per
        big[end - n13:end] = src[ls["off13_" + sec]:ls["off13_" + sec] + n13]
        gs, gb = small_I // 128 * per, I // 128 * per
        rows = H // 16
        big[lb["off2_" + sec]:lb["off2_" + sec] + rows * gb].view(rows, gb)[:, gb - gs:] = \
            src[ls["off2_" + sec]:ls["off2_" + sec] + rows * gs].view(rows, gs)
    return big, layer.experts_fp32[0]


@pytest.mark.parametrize("kind,H,I", [("bf16", 256, 2097408), ("int4", 1024, 1400064), ("q4k", 1024, 1400064), ("int4", 256, 1408),
                                      ("q4k", 256, 1536), ("bf16", 256, 1408)])
def test_expert_images_of_two_gib_and_more(cuda, kind, H, I):
    """Offsets inside an expert image past 31 bits (and the same construction on a small expert): only the weights at the far
    end of each matrix are not zero."""
    from promoe_amd import ops, _lib as L
    print(f"case prefill_large_image {kind} H={H} I={I}", flush=True)
    img, ws = _last_columns_image(kind, H, I, cuda)
    assert I < 10000 or img.numel() >= 1 << 31
    T = 3
    x = O.synth_acts(T, H, seed=16)
    d = ops.dispatch(torch.zeros(T, 1, dtype=torch.int32, device=cuda), 1)
    table = torch.tensor([img.data_ptr()], dtype=torch.int64, device=cuda)
    fmt = {"bf16": L.FMT_BF16, "int4": L.FMT_INT4_G128, "q4k": L.FMT_Q4K}[kind]
    part_r, _, err, *_ = ops.experts_prefill(bf16_dev(x, cuda), d, table, None, H, I, 0, fmt)
    torch.cuda.synchronize()
    assert int(err.item()) == 0
    ref = O.swiglu_expert(torch.from_numpy(x), *[torch.from_numpy(np.asarray(w)) for w in ws]).numpy()
    got = part_r.cpu().numpy()
    assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()


@pytest.mark.parametrize("cls", [Int4Layer, Bf16Layer])
@pytest.mark.parametrize("T", [1023, 1024, 1025, 2100])
def test_prefill_tile_list_of_many_units(cuda, T, cls):
    """Unit lists just short of, as long as and longer than one scan of the tile list takes: every token a unit of its own, and
    the rows of every third a unit of 40 or 130 rows; the same partial rows as from one unit of all tokens."""
    from promoe_amd import ops, _lib as L
    print(f"case prefill_many_units T={T} {cls.__name__}", flush=True)
    layer = cls(H=256, I=128, E=1, seed=18)
    fmt = L.FMT_BF16 if cls is Bf16Layer else L.FMT_INT4_G128
    slot = torch.from_numpy(layer.slots[0]).to(cuda)
    table = torch.tensor([slot.data_ptr()], dtype=torch.int64, device=cuda)
    sizes = [(1, 1, 40, 1, 1, 130)[u % 6] for u in range(T)]
    P = sum(sizes)
    x = bf16_dev(O.synth_acts(P, 256, seed=19), cuda)
    d = ops.dispatch(torch.zeros(P, 1, dtype=torch.int32, device=cuda), 1)
    ref = ops.experts_prefill(x, d, table, None, 256, 128, 0, fmt)
    many = ops.Dispatch(P, 1, 1, T, cuda)
    many.sorted_tok = d.sorted_tok
    rows0 = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    u = np.stack([np.zeros(T), sizes, rows0, np.zeros(T)], axis=1).astype(np.int32)
    u[T // 2] = (-1, 0, 0, 0)                     # an unused entry in the middle
    many.units = torch.from_numpy(u).to(cuda)
    got = ops.experts_prefill(x, many, table, None, 256, 128, 0, fmt,
                              ws=(torch.full_like(ref[0], float("nan")), None, ref[2], ref[3], None,
                                  torch.zeros(ops.prefill_workspace_bytes(fmt, P, 256, 1, T), dtype=torch.uint8, device=cuda)))
    torch.cuda.synchronize()
    assert int(got[2].item()) == 0
    live = torch.ones(P, dtype=torch.bool, device=cuda)
    live[rows0[T // 2]: rows0[T // 2] + sizes[T // 2]] = False
    assert torch.equal(got[0][live], ref[0][live]) and bool(torch.isnan(got[0][~live]).all())
