"""The layer blocks on the host: which projections a block may pass by and hand to
one call of the library.  No GPU: the operators are stand-ins."""
import pytest
import torch

from mlx_amd import nn, ops

D, F, E = 64, 128, 4


@pytest.fixture
def stubs(monkeypatch):
    """Operators that record their calls; products are ones."""
    calls = []

    def quantize(w, group_size=None, bits=None, mode="affine"):
        g, b = group_size or 64, bits or 4
        s = torch.zeros(w.shape[:-1] + (w.shape[-1] // g,), dtype=w.dtype)
        return torch.zeros(w.shape[:-1] + (w.shape[-1] * b // 32,), dtype=torch.uint32), s, s.clone()

    def gather_qmm(x, w, *args, rhs_indices=None, **kw):
        calls.append("gather_qmm")
        shape = torch.broadcast_shapes(x.shape[:-2], rhs_indices.shape)
        return torch.ones(*shape, x.shape[-2], w.shape[-2], dtype=x.dtype)

    def quantized_matmul(x, w, *args, **kw):
        calls.append("quantized_matmul")
        return torch.ones(*x.shape[:-1], w.shape[-2], dtype=x.dtype)

    def quantized_swiglu(x, gate, up, *args):
        calls.append("quantized_swiglu")
        return torch.ones(*x.shape[:-1], gate[0].shape[0], dtype=x.dtype)

    class Fast:
        def switch_glu(self, x, indices, *args):
            calls.append("switch_glu")
            return torch.zeros(*indices.shape, x.shape[-1], dtype=x.dtype)

    monkeypatch.setattr(ops, "quantize", quantize)
    monkeypatch.setattr(ops, "gather_qmm", gather_qmm)
    monkeypatch.setattr(ops, "quantized_matmul", quantized_matmul)
    monkeypatch.setattr(ops, "quantized_swiglu", quantized_swiglu)
    monkeypatch.setattr(ops, "_fast", Fast())
    return calls


def _switch_glu():
    return nn.SwitchGLU(D, F, E, dtype=torch.bfloat16, device="cpu")


class _Adapter(nn.QuantizedSwitchLinear):
    def forward(self, x, indices, sorted_indices=False):
        return super().forward(x, indices, sorted_indices) + 1


class _LinearAdapter(nn.QuantizedLinear):
    def forward(self, x):
        return super().forward(x) + 1


class _Wrapper(torch.nn.Module):
    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, *args, **kwargs):
        return self.inner(*args, **kwargs) + 1


@pytest.mark.parametrize("name", ("gate_proj", "up_proj", "down_proj"))
@pytest.mark.parametrize("how", ("subclass", "wrapper", "hook", "pre-hook", "forward"))
def test_switch_glu_calls_projections_that_are_more_than_their_buffers(stubs, name, how):
    x, indices = torch.ones(3, D, dtype=torch.bfloat16), torch.zeros(3, 2, dtype=torch.int64)
    block = _switch_glu()
    block(x, indices)
    assert stubs == ["switch_glu"]
    layer = getattr(block, name)
    seen = []
    if how == "subclass":
        layer.__class__ = _Adapter
    elif how == "wrapper":
        setattr(block, name, _Wrapper(layer))
    elif how == "hook":
        layer.register_forward_hook(lambda *args: seen.append(name))
    elif how == "pre-hook":
        layer.register_forward_pre_hook(lambda *args: seen.append(name))
    else:
        inner = layer.forward
        layer.forward = lambda *args, **kwargs: inner(*args, **kwargs) + 1
    y = block(x, indices)
    assert stubs[1:] == ["gather_qmm"] * 3
    assert y.shape == (3, 2, D)
    if "hook" in how:
        assert seen == [name]
    elif name == "down_proj":
        assert bool((y == 2).all())


@pytest.mark.parametrize("dtype,width,pairs,ordered", (
    (torch.float32, D, 1022, False), (torch.float32, D, 1024, True),
    (torch.bfloat16, D, 4096, False), (torch.bfloat16, 96, 4094, False),
    (torch.bfloat16, 96, 4096, True)))
@pytest.mark.parametrize("threshold", (64, 5000))
def test_switch_glu_orders_pairs_that_the_products_do_not_group(
        stubs, monkeypatch, dtype, width, pairs, ordered, threshold):
    seen = []

    def gather_qmm(x, w, *args, rhs_indices=None, sorted_indices=False, **kw):
        """Every result is its expert plus the sum of its row of x."""
        seen.append((sorted_indices, bool((rhs_indices[1:] >= rhs_indices[:-1]).all())))
        y = x.sum(-1, keepdim=True) + rhs_indices[..., None, None]
        return y.expand(*y.shape[:-1], w.shape[-2])

    monkeypatch.setattr(ops, "gather_qmm", gather_qmm)
    block = nn.SwitchGLU(width, F, E, dtype=dtype, device="cpu", group_size=32,
                         activation=lambda t: t, sort_threshold=threshold)
    indices = torch.arange(pairs).reshape(-1, 2) * 7 % E
    tokens = torch.arange(pairs // 2) % 5
    x = torch.zeros(pairs // 2, width, dtype=dtype)
    x[:, 0] = tokens
    y = block(x, indices.int())
    ordered = ordered and threshold == 64
    assert [s for s, _ in seen] == [ordered] * 3 and (not ordered or all(o for _, o in seen))
    want = F * (tokens[:, None] + indices).double() ** 2 + indices
    assert y.shape == (pairs // 2, 2, width)
    assert torch.equal(y.double(), want.to(dtype).double()[..., None].expand(y.shape))


@pytest.mark.parametrize("rows", (1, 8, 9))
@pytest.mark.parametrize("how", ("plain", "subclass", "wrapper", "hook", "other layer"))
def test_swiglu_calls_projections_that_are_more_than_their_buffers(stubs, rows, how):
    block = nn.SwiGLU(D, F, dtype=torch.bfloat16, device="cpu")
    seen = []
    if how == "subclass":
        block.up_proj.__class__ = _LinearAdapter
    elif how == "wrapper":
        block.gate_proj, block.up_proj = _Wrapper(block.gate_proj), _Wrapper(block.up_proj)
    elif how == "hook":
        block.gate_proj.register_forward_hook(lambda *args: seen.append(1))
    elif how == "other layer":  # (no scales)
        block.gate_proj = torch.nn.Linear(D, F, dtype=torch.bfloat16)
    y = block(torch.ones(rows, D, dtype=torch.bfloat16))
    assert y.shape == (rows, D)
    products = 2 if how == "other layer" else 3
    assert stubs == (["quantized_swiglu", "quantized_matmul"] if how == "plain" and rows <= 8
                     else ["quantized_matmul"] * products)
    assert len(seen) == (how == "hook")
