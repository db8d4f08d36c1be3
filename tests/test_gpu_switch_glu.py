"""The expert-routed gated MLP in one call against its three products: few pairs,
groups of small tiles, 256-row tiles with ragged ends, experts without rows,
indices out of range, index types."""
import pytest
import torch

from mlx_amd import _lib, nn

pytestmark = pytest.mark.gpu


def _block(D, F, E, group, bits, dtype):
    torch.manual_seed(D + F + E)
    block = nn.SwitchGLU(D, F, E, group_size=group, bits=bits, dtype=dtype)
    return block


@pytest.mark.parametrize("tokens,top,E,D,F,group,bits", [
    (1, 2, 4, 256, 384, 64, 4),       # one product per pair
    (24, 2, 4, 1024, 512, 64, 4),     # grouped in small tiles
    (300, 2, 4, 256, 384, 64, 4),     # 256-row tiles, the last ones ragged
    (700, 4, 9, 320, 200 * 8, 32, 8), # ragged columns of the gated tile
    (513, 1, 2, 128, 1152, 64, 3),
    (513, 1, 2, 192, 192, 64, 6),
])
@pytest.mark.parametrize("index_type", (torch.int64, torch.int32))
def test_against_the_three_products(tokens, top, E, D, F, group, bits, index_type):
    dtype = torch.bfloat16 if tokens % 2 else torch.float16
    block = _block(D, F, E, group, bits, dtype)
    g = torch.Generator(device="cuda").manual_seed(tokens)
    x = torch.randn((tokens, D), generator=g, device="cuda").to(dtype)
    # (the last expert gets no rows)
    idx = torch.randint(0, max(1, E - 1), (tokens, top), generator=g, device="cuda").to(index_type)
    if tokens > 1:
        idx[1, 0] = E + 3  # no such expert: a row of zeros
    assert block._in_one_call(x, idx) is not None
    y = block(x, idx)
    block.activation = lambda t: torch.nn.functional.silu(t)
    assert block._in_one_call(x, idx) is None
    want = block(x, idx)
    assert y.shape == want.shape == (tokens, top, D) and y.dtype == dtype
    if tokens > 1:
        assert not y[1, 0].any()
    # the same roundings (weights, products, activation, h), sums in another order:
    # the odd value of h lands on its neighbour, half an ulp of the result each
    d = (y.double() - want.double()).norm() / want.double().norm()
    assert float(d) < (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)


def test_batched_tokens_and_what_is_left_to_the_layers():
    block = _block(256, 512, 4, 64, 4, torch.bfloat16)
    x = torch.randn((3, 50, 256), device="cuda").bfloat16()
    idx = torch.randint(0, 4, (3, 50, 2), device="cuda")
    y = block(x, idx)
    assert torch.equal(y, block(x.reshape(150, 256), idx.reshape(150, 2)).reshape(y.shape))
    assert block._in_one_call(x.float(), idx) is None
    assert block._in_one_call(x, idx[:2]) is None
    assert block._in_one_call(x, idx.to(torch.uint8)) is None
    lib = _lib.load()
    assert lib.mlxrocm_switch_glu_workspace_size(8, 2, 256, 512, 4, 64, 4, 0) == 0  # float32
    assert lib.mlxrocm_switch_glu_workspace_size(8, 2, 250, 512, 4, 64, 4, 2) == 0


@pytest.mark.parametrize("D,dtype,tokens", [(256, torch.float32, 512), (96, torch.bfloat16, 2048)])
def test_pairs_ordered_by_expert_give_the_same_rows(D, dtype, tokens):
    block = _block(D, 192, 8, 32, 4, dtype)
    block.activation = torch.nn.functional.gelu  # (not one call)
    x = torch.randn((tokens, D), device="cuda").to(dtype)
    idx = torch.randint(0, 8, (tokens, 2), device="cuda").to(torch.int32)
    assert block._sorts(x, idx)
    y = block(x, idx)
    block.sort_threshold = 1 << 20
    assert not block._sorts(x, idx)
    assert torch.equal(y, block(x, idx))


@pytest.mark.parametrize("tokens,top,E,D,F,group", [
    (700, 2, 4, 512, 1664, 64),    # the second product in one round of tiles
    (3000, 4, 9, 1280, 640, 32),   # more rounds than one; 11 tiles of up to 256 rows an expert
    (300, 2, 3, 1920, 1024, 128),  # few tiles
])
@pytest.mark.parametrize("bits", (4, 8))
def test_the_bits_of_the_three_products(tokens, top, E, D, F, group, bits):
    """Many rows, no ranges of K: whatever kernel takes a product sums its codes in their order,
    as gather_qmm's tiles do, and the results agree to the bit (bfloat16: in float16 the gate of
    torch and that of the one call round here and there differently)."""
    dtype = torch.bfloat16
    block = _block(D, F, E, group, bits, dtype)
    g = torch.Generator(device="cuda").manual_seed(tokens)
    x = torch.randn((tokens, D), generator=g, device="cuda").to(dtype)
    idx = torch.randint(0, E, (tokens, top), generator=g, device="cuda")
    y = block(x, idx)
    block.activation = lambda t: torch.nn.functional.silu(t)
    assert block._in_one_call(x, idx) is None
    assert torch.equal(y, block(x, idx))


@pytest.mark.parametrize("bits", (4, 8))
@pytest.mark.parametrize("tokens,top,E,D,F,group", [
    (700, 1, 2, 4096, 4352, 64),   # experts of more than 16 MB at 8 bits, the last product in one round
    (900, 2, 8, 2048, 2304, 64),   # the last product in one round of the narrowest tiles
    (1900, 3, 5, 4096, 4224, 32),  # experts of more than 16 MB at 8 bits, two rounds
])
def test_the_bits_of_the_three_products_large_experts(tokens, top, E, D, F, group, bits):
    """The same where the tile kernel takes the last product, or all of them with tiles in the
    order of their experts; an expert without rows, and pairs without an expert."""
    block = _block(D, F, E, group, bits, torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(tokens)
    x = torch.randn((tokens, D), generator=g, device="cuda").bfloat16()
    idx = torch.randint(0, E, (tokens, top), generator=g, device="cuda")
    idx[idx == 1] = 0
    idx[5, 0] = E
    y = block(x, idx)
    assert not y[5, 0].any()
    block.activation = lambda t: torch.nn.functional.silu(t)
    assert block._in_one_call(x, idx) is None
    assert torch.equal(y, block(x, idx))
