"""int4 prefill on the scaled matrix instructions: the order of the fields on the CPU, the kernel against 64 bits on the GPU."""
import os
import re

import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from promoe_amd import layout as LY
from tests.synth import Int4Layer

_SRC = open(os.path.join(os.path.dirname(LY.__file__), "csrc", "moe_prefill_int4.h")).read()


def test_fields_of_the_spread_hold_the_k_that_the_activations_are_written_in():
    """p6_spread with the masks of the source on every nibble of two dwords in the image's order: field f holds k = p6_k16(f)."""
    masks = [[int(v, 16) for v in re.findall(r"0x([0-9a-f]{8})u", re.search(r"%s = \(int\)\((.*)\);" % d, _SRC).group(1))]
             for d in ("d0", "d1", "d2")]
    order = [int(v) for v in re.search(r"constexpr int t\[16\] = \{([^}]*)\}", _SRC).group(1).split(",")]
    assert sorted(order) == list(range(16))
    for k in range(16):
        for q in (1, 2, 4, 8, 15):
            w = [0, 0]
            w[k // 8] = q << int(LY._NIB_SHIFT[k % 8])
            a, b = w
            a2, b2 = (a << 2) & 0xffffffff, ((b << 2) | (a >> 30)) & 0xffffffff
            d = [(a & masks[0][0]) | (a2 & masks[0][1]), (b & masks[1][0]) | (b2 & masks[1][1]), (a & masks[2][0]) | (b2 & masks[2][1])]
            bits = d[0] | (d[1] << 32) | (d[2] << 64)
            assert bits == q << (6 * order.index(k)), (k, q)


def _ref64(x, ws):
    x = torch.from_numpy(x).double()
    w = [torch.from_numpy(np.ascontiguousarray(a)).double() for a in ws]
    return (torch.nn.functional.silu(x @ w[0].T) * (x @ w[1].T)) @ w[2].T


def _run(layer, x, idx, dev, pieces=1):
    from promoe_amd import ops, _lib as L
    lib, ptr = L.lib, L.ptr
    T, k = idx.shape
    d = ops.dispatch(torch.from_numpy(idx).to(dev), layer.E)
    slots = [torch.from_numpy(s).to(dev) for s in layer.slots]
    table = torch.tensor([s.data_ptr() for s in slots], dtype=torch.int64, device=dev)
    shared = torch.from_numpy(layer.shared_img).to(dev) if layer.I_sh else None
    xd = torch.from_numpy(x).to(torch.bfloat16).to(dev)
    part_r = torch.full((T * k, layer.H), float("nan"), device=dev)
    part_s = torch.full((pieces * T, layer.H), float("nan"), device=dev) if layer.I_sh else None
    h_r = torch.empty(T * k, layer.I, dtype=torch.bfloat16, device=dev)
    h_s = torch.empty(T, layer.I_sh, dtype=torch.bfloat16, device=dev) if layer.I_sh else None
    err = torch.zeros(1, dtype=torch.int32, device=dev)
    ws = torch.empty(ops.prefill_workspace_bytes(L.FMT_INT4_G128, T, layer.H, k, d.max_units), dtype=torch.uint8, device=dev)
    L.check(lib.moe_experts_prefill_pieces(ptr(xd), T, layer.H, layer.I, layer.I_sh, k, L.FMT_INT4_G128, ptr(d.units), d.max_units,
                                           ptr(d.sorted_tok), ptr(table), ptr(shared), ptr(h_r), ptr(h_s), ptr(part_r), ptr(part_s),
                                           pieces, ptr(ws), ptr(err), 3 | 4, L.cur_stream()), "moe_experts_prefill_pieces")
    torch.cuda.synchronize()
    assert int(err.item()) == 0
    pos = d.pos_of_pair.cpu().numpy()[: T * k].reshape(T, k)
    routed = part_r.cpu()[torch.from_numpy(pos).long()]      # [T, k, H]
    return routed, (part_s.cpu().view(pieces, T, layer.H).double().sum(0) if layer.I_sh else None)


# An element of h is off by at most 2^-9 of itself or 2^-11 of its block's largest, x by less, weights not at all: 2^-9 in norm
BOUND = 2.0 ** -9


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,I,I_sh,pieces", [
    (1, 256, 128, 128, 1),       # one row, one group of h, two of x
    (32, 512, 384, 256, 1), (33, 256, 640, 128, 1), (64, 256, 128, 0, 1), (65, 512, 256, 384, 1),
    (97, 256, 1152, 640, 1),     # nine groups: two rounds of four zero-point groups and one
    (128, 768, 128, 128, 1), (129, 256, 384, 512, 1), (300, 1024, 2176, 256, 1),   # 17 groups: past one chunk of zero points
    (70, 256, 128, 2560, 2),     # windows of ten groups: the second one starts in the middle of four
    (130, 256, 256, 5120, 4), (40, 512, 128, 1024, 4),
])
def test_rows_against_64_bits(cuda, T, H, I, I_sh, pieces):
    print(f"case int4 split T={T} H={H} I={I} I_sh={I_sh} pieces={pieces}", flush=True)
    layer = Int4Layer(H=H, I=I, E=2, I_sh=I_sh, seed=T)
    x = O.synth_acts(T, H, seed=T)
    idx = np.zeros((T, 1), np.int32)
    idx[T // 2 + 1:] = 1                       # two experts: rows that are gathered, tiles of several heights
    routed, shared = _run(layer, x, idx, cuda, pieces)
    want = torch.stack([_ref64(x[t:t + 1], layer.experts_fp32[idx[t, 0]])[0] for t in range(T)])
    assert _rel(routed[:, 0], want) <= BOUND
    if I_sh:
        assert _rel(shared, _ref64(x, layer.shared_fp32)) <= BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("scale,outlier", [(1.0, 50.0), (1e-6, 1.0), (3e5, 1.0), (1.0, 3e4)])
def test_rows_of_wide_ranges(cuda, scale, outlier):
    """Columns that stand out, tiny rows, and rows past the fp16 range: a scale per 32 values covers all of bf16."""
    layer = Int4Layer(H=512, I=256, E=2, I_sh=128, seed=3)
    x = O.synth_acts(70, 512, seed=5)
    x[:, ::97] *= outlier
    x = O.round_bf16((x * scale).astype(np.float32))
    idx = np.zeros((70, 1), np.int32)
    routed, shared = _run(layer, x, idx, cuda)
    assert _rel(routed[:, 0], _ref64(x, layer.experts_fp32[0])) <= BOUND
    assert _rel(shared, _ref64(x, layer.shared_fp32)) <= BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_a_row_with_no_number_spoils_only_itself(cuda, bad):
    layer = Int4Layer(H=256, I=256, E=2, I_sh=128, seed=4)
    x = O.synth_acts(40, 256, seed=6)
    clean, clean_s = _run(layer, x, np.zeros((40, 1), np.int32), cuda)
    x[7, 100] = bad
    x[9] = 0
    routed, shared = _run(layer, x, np.zeros((40, 1), np.int32), cuda)
    keep = [t for t in range(40) if t not in (7, 9)]
    assert torch.equal(routed[keep], clean[keep]) and torch.equal(shared[keep], clean_s[keep])
    assert not torch.isfinite(routed[7]).any() and not torch.isfinite(shared[7]).any()
    assert (routed[9] == 0).all() and (shared[9] == 0).all()
