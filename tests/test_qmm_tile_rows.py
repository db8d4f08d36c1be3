"""The 256-row tile kernel from 65 rows of x on, where the kernel of up to 128 rows per tile
is not taken (K no whole 128 codes, more than 256 rows over a long K): every width and type,
without and with the scale image, whole K and K ranges, each tile width."""
import pytest
import torch

import mlx_amd
from mlx_amd import _lib

# a row past a tile, ragged and whole rows of y, one K-step and more; tiles of 160, 192 and 224
# columns are chosen by N
SHAPES = {
    (65, 129, 64): "[qmm_t_tile]+qmm_t_tile(nt=5)",
    (257, 160, 320): "[qmm_t_tile]+qmm_t_tile(nt=5)",
    (257, 20513, 192): "[qmm_t_tile]+qmm_t_tile(nt=6)",
    (300, 24644, 192): "[qmm_t_tile]+qmm_t_tile(nt=7)",
    (70, 225, 1088): "[qmm_t_tile_k_split]+qmm_t_tile(ksplit=2)+reduce_k_splits(2)",
    (257, 448, 4096): "[qmm_t_tile_k_split]+qmm_t_tile(ksplit=8)+reduce_k_splits(8)",
    (513, 161, 320): "[qmm_t_tile_sb_transposed]+interleave_sb+qmm_t_tile(nt=5,pairs)",
    (514, 13700, 192): "[qmm_t_tile_sb_transposed]+interleave_sb+qmm_t_tile(nt=6,pairs)",
    (513, 16388, 192): "[qmm_t_tile_sb_transposed]+interleave_sb+qmm_t_tile(nt=7,pairs)",
    (520, 232, 2112):
        "[qmm_t_tile_sb_transposed]+interleave_sb+qmm_t_tile(ksplit=4,pairs)+reduce_k_splits(4)",
}
CODE = {torch.float16: _lib.FLOAT16, torch.bfloat16: _lib.BFLOAT16}


@pytest.mark.parametrize("bits,group", ((2, 64), (3, 32), (4, 64), (5, 32), (6, 64), (8, 32)))
@pytest.mark.parametrize("dtype", CODE)
def test_plans(bits, group, dtype):
    for (M, N, K), want in SHAPES.items():
        rc, plan = _lib.qmm_plan(M, N, K, dtype=CODE[dtype], group_size=group, bits=bits,
                                 workspace_bytes=1 << 30)
        assert rc == _lib.OK and plan == want, (M, N, K, plan)


@pytest.mark.gpu
@pytest.mark.parametrize("bits,group", ((2, 64), (3, 32), (4, 64), (5, 32), (6, 64), (8, 32)))
@pytest.mark.parametrize("dtype", CODE)
def test_products(gpu, bits, group, dtype):
    half = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    for M, N, K in SHAPES:
        g = torch.Generator(device="cuda").manual_seed(M + N + K)
        x = torch.randn((M, K), generator=g, device="cuda").to(dtype)
        w = (torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).to(dtype)
        q = mlx_amd.quantize(w, group, bits)
        y = mlx_amd.quantized_matmul(x, *q, group_size=group, bits=bits).double()
        # weights s c + b in float32, rounded once to the type
        w_hat = mlx_amd.dequantize(q[0], q[1].float(), q[2].float(), group_size=group,
                                   bits=bits).double()
        want = x.double() @ w_hat.T
        size = x.double().abs() @ w_hat.abs().T
        # half an ulp of the result and of every weight, fp32 sums over K terms
        err = (y - want).abs()
        assert bool((err <= half * want.abs() + (half + 2e-6) * size).all()), (M, N, K)
