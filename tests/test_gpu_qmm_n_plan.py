"""[K, N] weights on the tile kernel: widths and K ranges that the plan picks, against
the product of the dequantized weights in 64 bits."""
import pytest
import torch

import mlx_amd
from mlx_amd import _lib

pytestmark = pytest.mark.gpu

# (M, K, N, launches): three ranges of 224 columns with a ragged last tile of rows and
# columns; all of K in 224 columns, two rounds; ranges that are not equally long; 192
# columns in ranges; a single K-step more than ranges divide; M * N not a multiple of 4
CASES = (
    (1000, 14336, 4032, "ksplit=3"),
    (2048, 512, 14336, "ksplit=1"),
    (300, 4096, 4096, "ksplit="),
    (257, 1088, 2048, "ksplit="),
    (129, 2112, 448, "ksplit="),
    (515, 576, 1088, "ksplit=1"),
)


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("bits", (4, 8))
@pytest.mark.parametrize("M,K,N,launch", CASES)
def test_columns_and_ranges(gpu, dtype, bits, M, K, N, launch):
    code = {torch.float16: 1, torch.bfloat16: 2}[dtype]
    rc, plan = _lib.qmm_plan(M, N, K, bits=bits, group_size=64, transpose=False, dtype=code)
    assert rc == _lib.OK and f"qmm_n_tile({launch}" in plan, plan
    g = torch.Generator(device="cuda").manual_seed(M + bits)
    x = torch.randn((M, K), generator=g, device="cuda").to(dtype)
    w = (torch.randn((K, N), generator=g, device="cuda") * K ** -0.5).to(dtype)
    q = mlx_amd.quantize(w, 64, bits)
    y = mlx_amd.quantized_matmul(x, *q, transpose=False, group_size=64, bits=bits)
    exact = mlx_amd.dequantize(q[0], q[1].float(), q[2].float(), 64, bits).double()
    want = x.double() @ exact
    size = x.double().abs() @ exact.abs()
    # weights and result are rounded to the type once each, sums are fp32
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    err = (y.double() - want).abs()
    assert bool((err <= half * want.abs() + (half / 2 + 2e-6) * size).all()), float(
        (err / size).max())
