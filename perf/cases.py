"""The work that programs have this package do, as cases that can be timed: the MoE layer from a single decoded token to a
training step of 32768 tokens, the residual add + RMSNorm on either side of it, and the histogram of expert ids.

A case is a dict of plain values. "op" says which entry point it runs:

  infer   MoE.forward with autograd off (evaluation, prefill, decode), called eagerly
  replay  the same call captured once in a graph and replayed on new tokens, as a serving loop runs its decode steps
  train   MoE.forward and backward: output, router logits, the gradients of the tokens and of every parameter
  norm    fused_residual_add_rmsnorm, forward and backward
  count   continuous_count

tokens T, hidden H, intermediate I, experts E, top_k k, dtype, bias (per-expert biases of both projections), skew (0: every
expert equally likely; towards 1: the tokens share a direction, so that the router prefers some experts as trained routers do).
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "cute-kernels_amd"))  # the package's folder, from the repository's root

from fma import KernelBackend, MoE, continuous_count, fused_residual_add_rmsnorm, swiglu_packed  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}

# layer shapes of this repository's benchmark, tests and measurements: (H, I, E, k)
SHAPES = [
    (4096, 14336, 8, 2),
    (2048, 1408, 64, 8),
    (4096, 1536, 128, 8),
    (2048, 8192, 8, 2),
    (2048, 1024, 64, 8),
    (2880, 2880, 32, 4),
    (2048, 768, 128, 8),
]
# the fp32 layer is for small problems and for checking (the CPU-runnable configuration and sizes around it)
SHAPES_FP32 = [(256, 512, 8, 2), (512, 512, 16, 2), (576, 256, 32, 4)]


def _moe(op, T, shape, dtype="bf16", bias=False, skew=0.0):
    H, I, E, k = shape
    return dict(op=op, T=T, H=H, I=I, E=E, k=k, dtype=dtype, bias=bias, skew=skew)


def listed():
    return [
        # one user, one token: every kernel is small, the launches and the host's work between them count
        dict(_moe("infer", 1, (2048, 1408, 64, 8)), name="decode_1"),
        # a decode step of a few users inside a captured graph: no host work, the kernels' own latency counts
        dict(_moe("replay", 8, (2048, 1024, 64, 8)), name="decode_8_graph"),
        # a small serving batch on few large experts: the weights stream once for a handful of rows each
        dict(_moe("infer", 16, (4096, 14336, 8, 2)), name="decode_16_large_experts"),
        # a larger serving batch on many experts: a few rows each, all experts' weights read
        dict(_moe("infer", 100, (4096, 1536, 128, 8)), name="decode_100_many_experts"),
        # the prompt of one user, ragged length, in fp16 with biases
        dict(_moe("infer", 1021, (2048, 8192, 8, 2), dtype="fp16", bias=True), name="prefill_1021_fp16_bias"),
        # a prefill chunk over many experts: around 256 rows each
        dict(_moe("infer", 4096, (4096, 1536, 128, 8)), name="prefill_4096_many_experts"),
        # the CPU-runnable configuration: a small training step in fp32
        dict(_moe("train", 512, (256, 512, 8, 2), dtype="fp32"), name="train_512_fp32"),
        # the three training steps of the benchmark
        dict(_moe("train", 8192, (4096, 1536, 128, 8)), name="train_8192_many_experts"),
        dict(_moe("train", 32768, (2048, 1408, 64, 8), skew=0.5), name="train_32768_fine_grained"),
        dict(_moe("train", 16384, (4096, 14336, 8, 2)), name="train_16384_large_experts"),
        # the norm before the layer in such a training step
        dict(op="norm", T=16384, H=4096, dtype="bf16", name="norm_16384"),
        # the stand-alone histogram: 16 Mi ids in [0, 64)
        dict(op="count", n=1 << 24, E=64, dtype="int32", skew=0.0, name="count_16Mi"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case of the same ranges."""
    op = rng.choices(
        ["decode", "replay", "prefill", "train", "train_fp32", "norm", "count"], [5, 2, 5, 4, 1, 1.5, 1.5]
    )[0]
    if op == "norm":
        return dict(op="norm", T=_log_int(rng, 64, 32768), H=rng.choice([1024, 2048, 2880, 4096]),
                    dtype=rng.choice(["bf16", "bf16", "fp16"]))  # fmt: skip
    if op == "count":
        return dict(op="count", n=_log_int(rng, 1 << 16, 1 << 26), E=rng.choice([8, 64, 72, 128, 256]),
                    dtype=rng.choice(["int32", "int32", "int64"]), skew=rng.choice([0.0, 1.2]))  # fmt: skip
    if op == "train_fp32":
        return _moe("train", _log_int(rng, 64, 2048), rng.choice(SHAPES_FP32), dtype="fp32")
    shape = rng.choice(SHAPES)
    options = dict(
        dtype=rng.choice(["bf16", "bf16", "bf16", "fp16"]),
        bias=rng.random() < 0.25,
        skew=rng.choice([0.0, 0.0, 0.25, 0.5]),
    )
    if op in ("decode", "replay"):
        return _moe("infer" if op == "decode" else "replay", _log_int(rng, 1, 128), shape, **options)
    largest = work(_moe("train", 16384, SHAPES[0]))["flops"]
    if op == "prefill":
        return _moe("infer", _log_int(rng, 129, 8192), shape, **options)
    most = min(32768, int(largest / work(_moe("train", 1, shape))["flops"]))
    return _moe("train", _log_int(rng, 256, most), shape, **options)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _tokens(case, layer_direction, g):
    """N(0, 1) activations, `skew` of whose standard deviation is common to all tokens."""
    noise = torch.randn(case["T"], case["H"], generator=g, device="cuda")
    skew = case["skew"]
    if skew:
        noise = noise * math.sqrt(1.0 - skew * skew) + skew * layer_direction
    return noise.to(DTYPES[case["dtype"]])


def prepare(case, seed):
    g = _generator(seed)
    op = case["op"]
    if op == "count":
        dtype = torch.int32 if case["dtype"] == "int32" else torch.int64
        if case["skew"] == 0.0:
            ids = torch.randint(0, case["E"], (case["n"],), generator=g, device="cuda", dtype=dtype)
        else:  # Zipf with that exponent
            p = torch.arange(1, case["E"] + 1, device="cuda", dtype=torch.float32) ** -case["skew"]
            cdf = (p / p.sum()).cumsum(0)
            u = torch.rand(case["n"], generator=g, device="cuda")
            ids = torch.searchsorted(cdf, u).clamp_(max=case["E"] - 1).to(dtype)
        return dict(op=op, ids=ids, E=case["E"])
    if op == "norm":
        T, H, dtype = case["T"], case["H"], DTYPES[case["dtype"]]
        x, residual, normed_grad, residual_grad = (
            torch.randn(T, H, generator=g, device="cuda").to(dtype) for _ in range(4)
        )
        weight = (1.0 + 0.1 * torch.randn(H, generator=g, device="cuda")).to(dtype).requires_grad_()
        return dict(op=op, x=x, residual=residual, weight=weight, grads=(normed_grad, residual_grad))

    H, I, E, k = case["H"], case["I"], case["E"], case["k"]
    torch.manual_seed(seed)
    with torch.device("cuda"):
        moe = MoE(E, k, H, I, swiglu_packed, True, case["bias"], 0.02)
        with torch.no_grad():
            moe.gate.weight.normal_(0.0, 0.02)
            if case["bias"]:
                moe.c_fc.bias.normal_(0.0, 0.02)
                moe.c_proj.bias.normal_(0.0, 0.02)
    moe = moe.to(DTYPES[case["dtype"]])
    direction = torch.randn(H, generator=g, device="cuda")
    x = _tokens(case, direction, g)
    if op == "train":
        dy = torch.randn(case["T"], H, generator=g, device="cuda").to(x.dtype)
        return dict(op=op, moe=moe, x=x, dy=dy)
    if op == "infer":
        return dict(op=op, moe=moe, x=x)
    # replay: warm up on a side stream, then capture; every step copies its tokens into the captured input
    static_x = x.clone()
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                moe(static_x, kernel_backend=KernelBackend.cuda)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outputs = moe(static_x, kernel_backend=KernelBackend.cuda)
    return dict(op=op, moe=moe, x=x, static_x=static_x, graph=graph, outputs=outputs)


def run(state):
    op = state["op"]
    if op == "infer":
        with torch.no_grad():
            y, logits = state["moe"](state["x"], kernel_backend=KernelBackend.cuda)
        return dict(y=y, logits=logits)
    if op == "replay":
        state["static_x"].copy_(state["x"])
        state["graph"].replay()
        y, logits = state["outputs"]
        return dict(y=y, logits=logits)
    if op == "train":
        moe = state["moe"]
        moe.zero_grad(set_to_none=True)
        x = state["x"].detach().requires_grad_()
        y, logits = moe(x, kernel_backend=KernelBackend.cuda)
        y.backward(state["dy"])
        grads = {name: p.grad for name, p in moe.named_parameters()}
        return dict(y=y.detach(), logits=logits.detach(), x_grad=x.grad, **grads)
    if op == "norm":
        weight = state["weight"]
        weight.grad = None
        x = state["x"].detach().requires_grad_()
        residual = state["residual"].detach().requires_grad_()
        normed, stream = fused_residual_add_rmsnorm(x, residual, weight, 1e-5, kernel_backend=KernelBackend.cuda)
        torch.autograd.backward((normed, stream), state["grads"])
        return dict(normed=normed.detach(), stream=stream.detach(), x_grad=x.grad, residual_grad=residual.grad,
                    weight_grad=weight.grad)  # fmt: skip
    return continuous_count(state["ids"], state["E"], kernel_backend=KernelBackend.cuda)


def work(case):
    """bytes and operations of one pass: inputs read once, outputs written once. An inference pass needs the weights of the
    experts that some token chose (their expected number at equal odds); a training step writes every weight's gradient."""
    op = case["op"]
    if op == "count":
        return dict(bytes=case["n"] * (4 if case["dtype"] == "int32" else 8) + 4 * case["E"], flops=0)
    s = BYTES[case["dtype"]]
    if op == "norm":
        # forward: x, residual in, normed, stream out; backward: stream and two gradients in, two gradients out
        return dict(bytes=9 * case["T"] * case["H"] * s + 2 * case["H"] * s, flops=0)
    T, H, I, E, k = (case[n] for n in ("T", "H", "I", "E", "k"))
    expert = 3 * H * I + (2 * I + H if case["bias"] else 0)
    flops = 2 * T * k * 3 * H * I + 2 * T * H * E
    if op == "train":
        return dict(bytes=s * (4 * T * H + T * E + 2 * (E * expert + E * H)), flops=3 * flops)
    chosen = E * (1.0 - (1.0 - k / E) ** T)
    return dict(bytes=s * (2 * T * H + T * E + chosen * expert + E * H), flops=flops)


def tolerance(case):
    """Relative error (2-norm) between two correct implementations: two to four times what the package shows against the same
    pass evaluated in 64 bits with the same choice of experts (the largest over outputs and gradients of layers of 8 to 128
    experts and 512 to 4000 tokens: bf16 6e-3, fp16 8e-4, fp32 7e-7; the norm: bf16 3e-3, fp16 4e-4)."""
    op, dtype = case["op"], case["dtype"]
    if op == "count":
        return "exact"
    if op == "norm":
        return {"rel": 1e-2 if dtype == "bf16" else 1.5e-3}
    return {"rel": {"bf16": 1.5e-2, "fp16": 3e-3, "fp32": 3e-6}[dtype]}
