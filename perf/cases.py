"""What a user of this framework has it do: MoE layers run through the expert-cache engine (`PrefetchMngr.forward`).

A state is a short stack of MoE layers of one of the configured model shapes, its expert images in pinned host memory,
an engine on a stream of the program's own and the hidden states that reach the layers.  One pass is one forward of
every layer of the stack (as a model calls its sparse blocks, one after the other), or a run of such decode steps (always
for the stacks whose experts do not all fit the device).

  deepseek-int4   DeepSeek-MoE-16B: 2048 x 1408, 64 experts top-6, shared expert 2816, int4-g128, Zipf(1.2) routing
  mixtral-int4    Mixtral-8x7B: 4096 x 14336, 8 experts top-2 (softmax over the selected logits), int4-g128
  qwen-bf16       Qwen1.5-MoE-A2.7B: 2048 x 1408, 60 experts top-4, gated shared expert 5632, bf16
  qwen2-q4k       Qwen2-57B-A14B: 3584 x 2560, 64 experts top-8, gated shared expert 20480, q4_K, Zipf(1.1) routing
"""
from __future__ import annotations

import numpy as np
import torch

from promoe_amd import _lib as L
from promoe_amd import layout as LY
from promoe_amd import synth
from promoe_amd.engine import ModuleMeta, PinnedBuffer, PrefetchMngr

SHAPES = {
    "deepseek-int4": dict(fmt="int4", H=2048, E=64, I=1408, k=6, I_sh=2816, gated=False, mode=L.ROUTE_SOFTMAX_TOPK, zipf=1.2),
    "mixtral-int4": dict(fmt="int4", H=4096, E=8, I=14336, k=2, I_sh=0, gated=False, mode=L.ROUTE_TOPK_SOFTMAX, zipf=0.0),
    "qwen-bf16": dict(fmt="bf16", H=2048, E=60, I=1408, k=4, I_sh=5632, gated=True, mode=L.ROUTE_SOFTMAX_TOPK, zipf=0.0),
    "qwen2-q4k": dict(fmt="q4k", H=3584, E=64, I=2560, k=8, I_sh=20480, gated=True, mode=L.ROUTE_SOFTMAX_TOPK, zipf=1.1),
}
FORMATS = {"int4": L.FMT_INT4_G128, "bf16": L.FMT_BF16, "q4k": L.FMT_Q4K}
# the largest token group of a forward: a prompt as the configurations prefill it
MOST_TOKENS = {"deepseek-int4": 2048, "mixtral-int4": 4096, "qwen-bf16": 2048, "qwen2-q4k": 1024}


def _case(name, shape, tokens, layers, steps=1, cache_rate=1.0):
    c = dict(shape=shape, tokens=tokens, layers=layers, steps=steps, cache_rate=cache_rate)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one sequence being decoded, four layers of the int4 model: the smallest call, a few launches of 40 MB each
        _case("deepseek int4 decode 1", "deepseek-int4", 1, 4),
        # a small serving batch: about 18 of the 64 experts are in use
        _case("deepseek int4 decode 12", "deepseek-int4", 12, 4),
        # the same model with 24 of 64 experts per layer on the device (LRU): decode steps that wait for the host link
        _case("deepseek int4 cached decode", "deepseek-int4", 1, 2, 24, 0.375),
        # a short prompt of odd length: few rows per expert
        _case("deepseek int4 prefill 379", "deepseek-int4", 379, 2),
        # a full prompt
        _case("deepseek int4 prefill 2048", "deepseek-int4", 2048, 2),
        # wide experts, one sequence: weight streaming
        _case("mixtral int4 decode 1", "mixtral-int4", 1, 1),
        # the largest call: 1024 rows per expert, bound by the matrix cores
        _case("mixtral int4 prefill 4096", "mixtral-int4", 4096, 1),
        # bf16 experts (what inject_model makes by default): one sequence, a serving batch, a prompt of odd length
        _case("qwen bf16 decode 1", "qwen-bf16", 1, 2),
        _case("qwen bf16 decode 20", "qwen-bf16", 20, 2),
        _case("qwen bf16 prefill 1999", "qwen-bf16", 1999, 1),
        # q4_K experts from GGUF files: three sequences, and a prompt
        _case("qwen2 q4k decode 3", "qwen2-q4k", 3, 1),
        _case("qwen2 q4k prefill 512", "qwen2-q4k", 512, 1),
    ]


def draw(rng):
    shape = rng.choice(sorted(SHAPES))
    if shape == "deepseek-int4" and rng.random() < 0.25:
        return _case(None, shape, rng.randint(1, 4), 2, rng.randint(12, 24), rng.choice([0.25, 0.375, 0.5, 0.75]))
    tokens = min(MOST_TOKENS[shape], int(round(2.0 ** rng.uniform(0.0, np.log2(MOST_TOKENS[shape]) + 0.01))))
    if tokens > 64:
        return _case(None, shape, tokens, 2 if shape == "deepseek-int4" else 1)
    # decode: a few steps over a stack
    layers = rng.randint(3, 5) if shape == "deepseek-int4" else rng.randint(1, 2)
    return _case(None, shape, tokens, layers, rng.randint(2, 6))


def _expert_bytes(fmt, H, I):
    if I == 0:
        return 0
    return {"int4": LY.int4_layout, "q4k": LY.q4k_layout}[fmt](H, I)["total_bytes"] if fmt != "bf16" else LY.bf16_expert_bytes(H, I)


def _images(fmt, n, H, I, dev, gen):
    if fmt == "int4":
        return synth.random_int4_images(n, H, I, dev, gen)
    if fmt == "q4k":
        return synth.random_q4k_images(n, H, I, dev, gen)
    w = torch.empty(n, 3 * I * H, dtype=torch.bfloat16, device=dev)
    w.normal_(0.0, 0.02, generator=gen)
    return w.view(torch.uint8)


_program_stream = None


def _stream():
    """The program's stream: torch's current stream from the first preparation on, and every engine's compute stream
    (what inject_model leaves a program with)."""
    global _program_stream
    if _program_stream is None:
        _program_stream = torch.cuda.Stream()
        torch.cuda.set_stream(_program_stream)
    return _program_stream


def prepare(case, seed):
    s = SHAPES[case["shape"]]
    dev = torch.device("cuda:0")
    stream = _stream()
    gen = torch.Generator(device=dev).manual_seed(seed)
    H, E, I, k, I_sh, fmt = s["H"], s["E"], s["I"], s["k"], s["I_sh"], s["fmt"]
    n_layer, T, steps = case["layers"], case["tokens"], case["steps"]
    total = _expert_bytes(fmt, H, I)
    chunks = LY.split_chunks_int4(H, I) if fmt == "int4" else [("w", 0, total)]
    meta = ModuleMeta(n_layer, E)
    meta.init_param_list([c[0] for c in chunks])
    meta.init_from_map({"num_expert_per_token": str(k), "cache_rate": str(case["cache_rate"]), "cache_policy": "lru"})
    meta.handle_uninited_configs()
    pm = PrefetchMngr(meta, backend=L.BACKEND_HIP, compute_stream=stream.cuda_stream)
    stage = PinnedBuffer(total * n_layer * E)
    pm._keep.append(stage)
    host = torch.from_numpy(stage.array).view(n_layer, E, total)
    dense = []
    for l in range(n_layer):
        host[l].copy_(_images(fmt, E, H, I, dev, gen))
        gate = (torch.randn(E + int(s["gated"]), H, device=dev, generator=gen) * 0.02).to(torch.bfloat16)
        bias = torch.from_numpy(synth.zipf_bias(E, s["zipf"], seed * 100 + l)).to(dev) if s["zipf"] else None
        shared = _images(fmt, 1, H, I_sh, dev, gen)[0] if I_sh else None
        dense.append((gate, bias, shared))
        for e in range(E):
            base = (l * E + e) * total
            for name, off, n in chunks:
                pm.add_one_expert_param(stage.array[base + off: base + off + n], l, e, name)
    pm.init_gpu_mem_buffer()
    for l, (gate, bias, shared) in enumerate(dense):
        pm.set_layer(l, H, I, I_sh, k, s["mode"], gate, bias, shared, shared_gated=s["gated"], fmt=FORMATS[fmt])
    pm.forward_prepare(max(64, T))
    pm.launch_thread()
    if case["cache_rate"] >= 1.0:  # every expert into its slot, as after the first tokens of a program
        for l in range(n_layer):
            pm.acquire_layer(l, np.arange(E, dtype=np.int64))
            pm.release_layer(l)
        pm.drain()
    # hidden states as they leave the layer norm in front of a sparse block
    xs = [[torch.randn(T, H, device=dev, generator=gen).to(torch.bfloat16) for _ in range(n_layer)] for _ in range(steps)]
    torch.cuda.synchronize()
    return {"pm": pm, "xs": xs}


def run(state):
    pm = state["pm"]
    return [pm.forward(l, x) for step in state["xs"] for l, x in enumerate(step)]


def _experts_in_use(case):
    """Distinct routed experts of one forward, on average over a few draws of the routing."""
    s = SHAPES[case["shape"]]
    E, k, T = s["E"], s["k"], case["tokens"]
    rng = np.random.default_rng(7)
    sd = 0.02 * np.sqrt(s["H"])
    bias = -s["zipf"] * np.log(np.arange(1, E + 1))
    n = []
    for _ in range(8):
        logits = rng.normal(0.0, sd, (T, E)) + bias
        n.append(np.unique(np.argpartition(-logits, k - 1, axis=1)[:, :k]).size)
    return float(np.mean(n))


def work(case):
    s = SHAPES[case["shape"]]
    H, I, I_sh, k, T = s["H"], s["I"], s["I_sh"], s["k"], case["tokens"]
    rows = s["E"] + int(s["gated"])
    nbytes = (_experts_in_use(case) * _expert_bytes(s["fmt"], H, I) + _expert_bytes(s["fmt"], H, I_sh) + rows * H * 2
              + 2 * T * H * 2)
    flops = 2.0 * T * (3 * H * (k * I + I_sh) + rows * H)
    n = case["layers"] * case["steps"]
    return {"bytes": n * nbytes, "flops": n * flops}


def tolerance(case):
    # operands and the rows between the two expert products in 16 bits, sums in fp32, result in bf16: against the same
    # layers in 64 bits the outputs are off by 1.7e-3 to 2.4e-3 in norm and by at most 1.3e-2 at one value
    return {"rel": 1e-2, "max": 5e-2}
