"""GPU parity of the two tile sizes of the fp32 grouped GEMM (fma_grouped_gemm on fp32): integer operands, whose products are exact in
fp32 (|sum| <= 9 K < 2^24), against a float64 product, in every layout, with reductions that can and cannot be read in 16-byte
pieces."""

import pytest
import torch

from fma import grouped_gemm

from gpu_util import DEV

pytestmark = pytest.mark.gpu

SIZES = [
    # 256 tiles of 128 x 128, one per compute unit: large tiles, none of them full at the far edges
    ([2047], [2041], [36]),
    ([2047], [2041], [35]),
    ([1025, 0, 513, 130], [1664, 200, 1000, 1300], [17, 16, 1, 64]),
    # few tiles: 64 x 64, at the edges of a tile and of a K step, offsets of later groups odd
    ([64, 65, 1, 127], [64, 63, 129, 1], [32, 33, 31, 64]),
    ([3, 128], [5, 192], [7, 100]),
    ([1], [1], [1]),
    # 384 large tiles, 1536 small ones: large over few k, small over many
    ([767] * 16, [511] * 16, [6] * 15 + [1]),
    ([767] * 16, [511] * 16, [300] * 15 + [299]),
]


@pytest.mark.parametrize("tA", [False, True])
@pytest.mark.parametrize("tB", [False, True])
@pytest.mark.parametrize("Ms,Ns,Ks", SIZES)
def test_tiles(Ms, Ns, Ks, tA, tB):
    g = torch.Generator(device=DEV).manual_seed(sum(Ms) + sum(Ks))
    As, Bs, Ds = [], [], []
    for M, N, K in zip(Ms, Ns, Ks):
        a = torch.randint(-3, 4, (K, M) if tA else (M, K), device=DEV, generator=g).float()
        b = torch.randint(-3, 4, (N, K) if tB else (K, N), device=DEV, generator=g).float()
        As.append(a.reshape(-1))
        Bs.append(b.reshape(-1))
        Ds.append(((a.T if tA else a).double() @ (b.T if tB else b).double()).float().reshape(-1))
    sizes = [torch.tensor(v, dtype=torch.int64).to(torch.uint32).to(DEV) for v in (Ms, Ns, Ks)]
    out = grouped_gemm(
        A=torch.cat(As), B=torch.cat(Bs), C=None, M_array=sizes[0], N_array=sizes[1], K_array=sizes[2],
        output_shape=(sum(m * n for m, n in zip(Ms, Ns)),), is_A_transposed=tA, is_B_transposed=tB,
    )  # fmt: skip
    assert torch.equal(out, torch.cat(Ds))
