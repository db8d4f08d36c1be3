"""qqmm on the block-scaled matrix instruction: fewer K-steps than LDS stages, one
more, ragged tiles, scale bytes in the caller's layout and as an image,
K ranges --
against the product of the two dequantized operands in 64 bits."""
import pytest
import torch

import mlx_amd

pytestmark = pytest.mark.gpu

# (M, N, K)
SHAPES = ((16, 4, 128), (257, 129, 384), (511, 260, 512), (512, 1000, 640), (769, 132, 896),
          (100, 4096, 4096), (513, 2050, 2176))


@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16, torch.float32))
@pytest.mark.parametrize("mode", ("mxfp8", "mxfp4"))
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_steps_tiles_and_scales(gpu, mode, dtype, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    # operands on the grid of the format (each block's largest code is the format's
    # largest, its scale a power of two), so that quantizing x changes nothing
    table = torch.tensor((6.0, 4.0, 3.0, 1.5, 1.0, 0.5) if mode == "mxfp4" else
                         (448.0, 416.0, 256.0, 96.0, 3.5, 1.0), device="cuda")

    def grid(rows):
        v = table[torch.randint(0, 6, (rows, K // 32, 32), generator=g, device="cuda")]
        v[..., 0] = table[0]
        sign = torch.randint(0, 2, v.shape, generator=g, device="cuda").float() * 2 - 1
        e = torch.randint(-3, 3, (rows, K // 32, 1), generator=g, device="cuda").float()
        return (v * sign * torch.exp2(e - (2 if mode == "mxfp4" else 9))).reshape(rows, K)

    x, w = grid(M).to(dtype), grid(N).to(dtype)
    wq, scales = mlx_amd.quantize(w, mode=mode)
    xq, xs = mlx_amd.quantize(x, mode=mode)
    exact_w = mlx_amd.dequantize(wq, scales, mode=mode, dtype=torch.float32).double()
    exact_x = mlx_amd.dequantize(xq, xs, mode=mode, dtype=torch.float32).double()
    assert torch.equal(exact_w, w.double()) and torch.equal(exact_x, x.double())
    y = mlx_amd.qqmm(x, wq, scales, mode=mode)
    want = exact_x @ exact_w.T
    size = exact_x.abs() @ exact_w.abs().T
    half = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    # the e4m3 instruction keeps about 17 bits below a step's largest product
    sums = 2e-5 if mode == "mxfp8" and dtype != torch.float32 else 2e-6
    err = (y.double() - want).abs()
    assert bool((err <= half * want.abs() + sums * size).all()), float((err / size).max())


@pytest.mark.parametrize("mode", ("mxfp8", "mxfp4"))
@pytest.mark.parametrize("M", (8, 16, 100, 512))
def test_scale_bytes_at_any_address(gpu, mode, M):
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn((M, 1152), generator=g, device="cuda").bfloat16()
    wq, scales = mlx_amd.quantize(
        torch.randn((300, 1152), generator=g, device="cuda").bfloat16(), mode=mode)
    want = mlx_amd.qqmm(x, wq, scales, mode=mode)
    for offset in (1, 2, 4):
        flat = torch.empty(scales.numel() + offset, dtype=torch.uint8, device="cuda")
        flat[offset:] = scales.reshape(-1)
        moved = flat[offset:].view(scales.shape)
        assert torch.equal(mlx_amd.qqmm(x, wq, moved, mode=mode), want)
