"""GPU parity of a forward pass of one token without a backward: up to eight choices run in three launches (router product, first
projection, second projection with the combine), which choose the experts from the logits. Two copies of the token take the path of
several tokens: the same bits, for every number of choices around the pairs and the limit of eight."""

import pytest
import torch

from fma import KernelBackend, MoE, swiglu_packed

from gpu_util import DEV

pytestmark = pytest.mark.gpu

# hidden, intermediate, experts, choices: odd and even choices; partial column blocks and K steps; up to 64 experts (four keys per lane)
# and more, up to the limit; nine choices: the path of several tokens
SHAPES = [(8, 8, 1, 1), (264, 40, 3, 3), (520, 2048, 256, 6), (2056, 264, 200, 7), (1000, 1000, 65, 5), (2048, 1408, 64, 8),
          (2048, 768, 8, 2), (512, 512, 16, 9), (72, 4104, 64, 4)]  # fmt: skip


def _layer(H, I, E, k, dtype, bias):
    torch.manual_seed(H + I + E + k)
    with torch.device(DEV):
        moe = MoE(E, k, H, I, swiglu_packed, True, bias, 0.02)
        with torch.no_grad():
            moe.gate.weight.normal_(0.0, 0.02)
            if bias:
                moe.c_fc.bias.normal_(0.0, 0.5)
                moe.c_proj.bias.normal_(0.0, 0.5)
    return moe.to(dtype)


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,I,E,k", SHAPES)
@torch.no_grad()
def test_same_bits_as_two_tokens(H, I, E, k, dtype, bias):
    moe = _layer(H, I, E, k, dtype, bias)
    for seed in range(3):
        x = torch.randn(1, H, device=DEV, generator=torch.Generator(device=DEV).manual_seed(seed)).to(dtype)
        y, logits = moe(x, kernel_backend=KernelBackend.cuda)
        y2, logits2 = moe(x.expand(2, H).contiguous(), kernel_backend=KernelBackend.cuda)
        assert torch.equal(logits[0], logits2[0])
        assert torch.equal(y[0], y2[0]) and torch.equal(y2[0], y2[1])


@torch.no_grad()
def test_ties_and_non_finite_tokens():
    """equal logits: the lowest experts, as for several tokens; a token with an infinity or a NaN gives what it gives there"""
    moe = _layer(256, 512, 16, 4, torch.bfloat16, False)
    moe.gate.weight.zero_()
    x = torch.randn(1, 256, device=DEV).bfloat16()
    for value in (None, float("inf"), float("nan")):
        if value is not None:
            x[0, 3] = value
        y, logits = moe(x, kernel_backend=KernelBackend.cuda)
        y2, logits2 = moe(x.expand(2, 256).contiguous(), kernel_backend=KernelBackend.cuda)
        assert torch.equal(logits[0].isnan(), logits2[0].isnan()) and torch.equal(y[0].isnan(), y2[0].isnan())
        assert torch.equal(logits[0].nan_to_num(), logits2[0].nan_to_num()) and torch.equal(y[0].nan_to_num(), y2[0].nan_to_num())
