"""Rows of the int4 tile kernel against 64 bits, with weights that every number format in use holds exactly: what is left is
what x, the rows between the two passes and the sums lose."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from promoe_amd import layout as LY

pytestmark = pytest.mark.gpu


def _image(mats, H, I):
    """Slot image and fp32 weights of one expert from (q [N, K], s [N, G], z [N, G]) of gate, up and down."""
    lay = LY.int4_layout(H, I)

    def interleave(a, b):
        nb = a.shape[0] // 16
        return np.stack([a.reshape(nb, 16, -1), b.reshape(nb, 16, -1)], axis=1).reshape(2 * a.shape[0], -1)

    t13 = LY.tile_int4(*[interleave(a, b) for a, b in zip(mats[0], mats[1])])
    img = np.zeros(lay["total_bytes"], np.uint8)
    for off, arr in zip(("off13_q", "off13_s", "off13_z", "off2_q", "off2_s", "off2_z"), t13 + LY.tile_int4(*mats[2])):
        img[lay[off]: lay[off] + arr.size] = arr
    return img, [(q.astype(np.float64) - np.repeat(z, 128, 1)) * np.repeat(s.astype(np.float64), 128, 1) for q, s, z in mats]


def _exact_expert(H, I, rng):
    """Random nibbles and zero points, scales that are powers of two: (q - z) s has four bits."""
    mats = []
    for n, k in ((I, H), (I, H), (H, I)):
        s = 2.0 ** rng.integers(-8, -5, (n, k // 128))
        mats.append((rng.integers(0, 16, (n, k)).astype(np.uint8), s.astype(np.float16),
                     rng.integers(4, 12, (n, k // 128)).astype(np.uint8)))
    return _image(mats, H, I)


def _picking_expert(H, first):
    """128 columns of h: column i is silu(x[0]) * x[first + i]; output n is h[n % 128]."""
    I = 128
    mats = []
    for pick, n, k in ((np.zeros(I, int), I, H), (first + np.arange(I), I, H), (np.arange(H) % 128, H, I)):
        z = (np.arange(n * (k // 128)) % 16).astype(np.uint8).reshape(n, -1)
        z[np.arange(n), pick // 128] %= 15
        q = np.repeat(z, 128, 1)
        q[np.arange(n), pick] += 1
        mats.append((q, np.ones((n, k // 128), np.float16), z))
    return _image(mats, H, I)


def _run(x, idx, experts, shared, H, I, I_sh, dev, pieces=1):
    from promoe_amd import ops, _lib as L
    lib, ptr = L.lib, L.ptr
    T, k = idx.shape
    d = ops.dispatch(torch.from_numpy(idx).to(dev), len(experts))
    slots = [torch.from_numpy(e).to(dev) for e in experts]
    table = torch.tensor([s.data_ptr() for s in slots], dtype=torch.int64, device=dev)
    sh = torch.from_numpy(shared).to(dev) if I_sh else None
    xd = torch.from_numpy(x).to(torch.bfloat16).to(dev)
    part_r = torch.full((T * k, H), float("nan"), device=dev)
    part_s = torch.full((pieces * T, H), float("nan"), device=dev) if I_sh else None
    h_r = torch.empty(T * k, I, dtype=torch.bfloat16, device=dev)
    h_s = torch.empty(T, I_sh, dtype=torch.bfloat16, device=dev) if I_sh else None
    err = torch.zeros(1, dtype=torch.int32, device=dev)
    ws = torch.empty(ops.prefill_workspace_bytes(L.FMT_INT4_G128, T, H, k, d.max_units), dtype=torch.uint8, device=dev)
    L.check(lib.moe_experts_prefill_pieces(ptr(xd), T, H, I, I_sh, k, L.FMT_INT4_G128, ptr(d.units), d.max_units,
                                           ptr(d.sorted_tok), ptr(table), ptr(sh), ptr(h_r), ptr(h_s), ptr(part_r), ptr(part_s),
                                           pieces, ptr(ws), ptr(err), 3 | 4, L.cur_stream()), "moe_experts_prefill_pieces")
    torch.cuda.synchronize()
    assert int(err.item()) == 0
    pos = d.pos_of_pair.cpu().numpy()[: T * k].reshape(T, k)
    routed = part_r.cpu()[torch.from_numpy(pos).long()].double().numpy()      # [T, k, H]
    return routed, (part_s.cpu().view(pieces, T, H).double().sum(0).numpy() if I_sh else None)


def _ref64(x, w):
    g, u = x.astype(np.float64) @ w[0].T, x.astype(np.float64) @ w[1].T
    with np.errstate(over="ignore"):
        return (g / (1.0 + np.exp(-g)) * u) @ w[2].T


@pytest.mark.parametrize("T", [1, 33, 70, 128, 200])
def test_elements_keep_eleven_bits(cuda, T):
    """Each output is one element of x times a constant, through h: x (bf16) is exact, h is rounded to fp16 once, whatever the
    other elements of its block of columns are (every 32nd is 64 times larger)."""
    print(f"case int4 elements T={T}", flush=True)
    H = 256
    rng = np.random.default_rng(T)
    x = rng.choice([-1.0, 1.0], (T, H)) * 2.0 ** rng.uniform(-5, 2, (T, H))
    x[:, 5::32] *= 64.0
    x[:, 9::32] = 4.25 + rng.integers(0, 16, (T, 8)) / 32.0
    x[:, 0] = 4.0
    x = O.round_bf16(x.astype(np.float32))
    (img, w), (simg, sw) = _picking_expert(H, 1), _picking_expert(H, 128)
    routed, shared = _run(x, np.zeros((T, 1), np.int32), [img], simg, H, 128, 128, cuda)
    for got, ws in ((routed[:, 0], w), (shared, sw)):
        want = _ref64(x, ws)
        # half a unit in the last place of fp16 is at most 2^-11 of a value; silu in fp32 adds a few units of 2^-22
        assert (np.abs(got - want) <= (2.0 ** -11 + 2.0 ** -19) * np.abs(want)).all()


@pytest.mark.parametrize("T,H,I,I_sh,pieces", [
    (1, 256, 128, 128, 1), (33, 256, 640, 128, 1), (65, 512, 256, 384, 1), (129, 256, 384, 512, 1),
    (190, 256, 1152, 640, 1),     # tiles of 96 rows, 95 in use
    (251, 768, 2176, 256, 1),     # tiles of 128 rows, 126 and 125 in use; 17 groups
    (70, 256, 128, 2560, 2),      # windows of ten groups
    (121, 512, 256, 5120, 4), (96, 256, 128, 8192, 8),
])
def test_rows_of_exact_weights(cuda, T, H, I, I_sh, pieces):
    """Two experts, so that rows are gathered.  The roundings of h to fp16, at most 2^-11 of a value and evenly spread below that,
    are 2^-11 / sqrt(3) in norm at most; signs of no order leave that of the sums."""
    print(f"case int4 rows T={T} H={H} I={I} I_sh={I_sh} pieces={pieces}", flush=True)
    rng = np.random.default_rng(T)
    experts = [_exact_expert(H, I, rng) for _ in range(2)]
    simg, sw = _exact_expert(H, I_sh, rng)
    x = O.synth_acts(T, H, seed=T)
    idx = (np.arange(T) % 2).astype(np.int32)[:, None]
    routed, shared = _run(x, idx, [e[0] for e in experts], simg, H, I, I_sh, cuda, pieces)
    want = np.stack([_ref64(x[t:t + 1], experts[idx[t, 0]][1])[0] for t in range(T)])
    err = np.linalg.norm(routed[:, 0] - want) / np.linalg.norm(want)
    ref = _ref64(x, sw)
    err_s = np.linalg.norm(shared - ref) / np.linalg.norm(ref)
    print(f"  {err:.3e} {err_s:.3e}", flush=True)
    assert max(err, err_s) <= 2.0 ** -11


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_a_row_with_no_number_spoils_only_itself(cuda, bad):
    print(f"case int4 row of {bad}", flush=True)
    rng = np.random.default_rng(4)
    (img, _), (simg, _) = _exact_expert(256, 256, rng), _exact_expert(256, 128, rng)
    x = O.synth_acts(40, 256, seed=6)
    idx = np.zeros((40, 1), np.int32)
    clean, clean_s = _run(x, idx, [img], simg, 256, 256, 128, cuda)
    x[7, 100] = bad
    x[9] = 0
    routed, shared = _run(x, idx, [img], simg, 256, 256, 128, cuda)
    keep = [t for t in range(40) if t not in (7, 9)]
    assert np.array_equal(routed[keep], clean[keep]) and np.array_equal(shared[keep], clean_s[keep])
    assert not np.isfinite(routed[7]).any() and not np.isfinite(shared[7]).any()
    assert (routed[9] == 0).all() and (shared[9] == 0).all()
