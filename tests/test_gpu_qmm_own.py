"""The tiles whose wavefronts own their rows of W against float64 on the dequantized
weights: heights of the last tile of an expert, ragged columns, one and several K-steps,
more tiles than workgroups, every width."""
import pytest
import torch

import mlx_amd
from mlx_amd import _lib, nn

pytestmark = pytest.mark.gpu

BITS = (2, 3, 4, 5, 6, 8)
# every height of a last tile (16 rows each), whole tiles and an expert without rows
ROWS = (1, 16, 17, 63, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 255, 256, 257, 0, 600)


def _indices(tokens, dtype=torch.int64):
    e = torch.cat([torch.full((n,), i) for i, n in enumerate(ROWS)])
    g = torch.Generator().manual_seed(5)
    return e[torch.randperm(len(e), generator=g)].reshape(tokens, -1).to("cuda", dtype)


@pytest.mark.parametrize("bits", BITS)
@pytest.mark.parametrize("D,F", [
    (128, 1664),  # one step of K, 13 tiles of gated columns: more tiles than workgroups
    (2944, 128),  # 23 steps, one of the second product; 11.5 tiles of columns
])
def test_experts(D, F, bits):
    dtype = torch.bfloat16 if (bits + D) % 2 else torch.float16
    group = (32, 64, 128)[bits % 3]
    torch.manual_seed(bits)
    block = nn.SwitchGLU(D, F, len(ROWS), group_size=group, bits=bits, dtype=dtype)
    idx = _indices(sum(ROWS))
    x = torch.randn((idx.shape[0], D), device="cuda").to(dtype)
    assert block._in_one_call(x, idx) is not None
    y = block(x, idx)

    def weight(layer, e):
        # scale * code + bias, rounded once (dequantize rounds the product and the sum)
        s, b = layer.scales[e].double(), layer.biases[e].double()
        codes = mlx_amd.dequantize(layer.weight[e], torch.ones_like(s, dtype=torch.float32),
                                   torch.zeros_like(s, dtype=torch.float32),
                                   group_size=group, bits=bits).double()
        w = codes.unflatten(1, (-1, group)) * s[..., None] + b[..., None]
        return w.flatten(1).to(dtype).double()

    want = torch.empty(y.shape, device="cuda", dtype=torch.float64)
    for e, n in enumerate(ROWS):
        at = idx == e
        assert int(at.sum()) == n
        if n:
            xe = x[at.nonzero()[:, 0]].double()
            gate = (xe @ weight(block.gate_proj, e).T).to(dtype).float()
            up = (xe @ weight(block.up_proj, e).T).to(dtype).float()
            h = (torch.nn.functional.silu(gate).to(dtype).float() * up).to(dtype)
            want[at] = h.double() @ weight(block.down_proj, e).T
    # both sides round gate, up, silu, h and the result to the type; where their sums fall on
    # either side of a tie the values of h differ by an ulp, and the result's own rounding
    # adds up to half of one
    d = (y.double() - want).norm() / want.norm()
    assert float(d) < (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)
    # and row by row: a row of another expert or of another position is no near miss
    r = (y.double() - want).norm(dim=-1) / want.norm(dim=-1)
    assert float(r.max()) < (2.0 ** -6 if dtype == torch.bfloat16 else 2.0 ** -9)
