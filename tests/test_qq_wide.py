"""Products of two mxfp8 operands in tiles of 256 x 256 (two LDS stages)."""
import pytest
import torch

import mlx_amd

# more 256 x 128 tiles than a round holds (256), no more 256 x 256 tiles than that, so the
# wide tile is chosen; one, two, three, five and nine steps; a row or column past a tile,
# rows of y that are no whole 16-byte pieces, a last tile of one row of W, several rounds
SHAPES = ((4111, 2503, 128), (4096, 2560, 256), (2049, 3841, 384), (300, 32001, 640),
          (257, 18002, 1152), (513, 45060, 512))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
def test_products(gpu, M, N, K, dtype):
    g = torch.Generator(device="cuda").manual_seed(M * N + K)

    def grid(rows):  # small whole numbers that the format holds, whatever their block's scale
        table = torch.tensor((7.0, 4.0, -4.0, 3.0, -2.0, 1.0), device="cuda")
        v = table[torch.randint(0, 6, (rows, K), generator=g, device="cuda")]
        v[:, ::32] = table[0]
        scale = torch.randint(0, 3, (rows, K // 32), generator=g, device="cuda")
        return (v * scale.repeat_interleave(32, 1).float().exp2()).to(dtype)

    x, w = grid(M), grid(N)
    y = mlx_amd.qqmm(x, *mlx_amd.quantize(w, mode="mxfp8"), mode="mxfp8")
    # products are whole numbers up to 784 and sums stay below 2**17: nothing is lost before
    # the one rounding of the result
    want = x.double() @ w.double().T
    assert float(want.abs().max()) < 2.0 ** 17
    assert torch.equal(y, want.to(dtype))
