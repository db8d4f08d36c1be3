"""Products of two mxfp8 operands in tiles of 256 x 256 (two LDS stages)."""
import pytest
import torch

import mlx_amd
from mlx_amd import _lib

# fewer rounds of 256 x 256 tiles than of 256 x 128; one, two, three, five and nine steps; a
# row or column past a tile, rows of y that are no whole 16-byte pieces, a last tile of one
# row of W, one round and (531 tiles) three
SHAPES = ((4111, 2503, 128), (4096, 2560, 256), (2049, 3841, 384), (300, 32001, 640),
          (257, 18002, 1152), (513, 45060, 512))


@pytest.mark.parametrize("M,N,K", SHAPES + ((8192, 14336, 4096), (2861, 11008, 2048), (5530, 6002, 4096)))
def test_wide_tiles(M, N, K):
    for dtype in (_lib.FLOAT16, _lib.BFLOAT16):
        rc, plan = _lib.fp_qqmm_plan(M, N, K, _lib.MXFP8, dtype)
        assert rc == _lib.OK and plan == "fp_quantize_activations+qq_mfma(e4m3)", plan


# one round either way; K ranges fill the chip; a short K, results stored by the element
@pytest.mark.parametrize("M,N,K", ((512, 14336, 4096), (1024, 4096, 14336), (5083, 4096, 256),
                                   (3920, 4099, 1024), (2650, 6002, 768), (5285, 4099, 256)))
def test_narrow_tiles(M, N, K):
    rc, plan = _lib.fp_qqmm_plan(M, N, K, _lib.MXFP8, _lib.BFLOAT16)
    assert rc == _lib.OK and "qq_mfma(e4m3,bn=128)" in plan, plan


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
