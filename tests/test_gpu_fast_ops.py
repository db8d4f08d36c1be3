"""The operators' native host path against their own Python bodies: the same
results to the bit where it takes a call, and nothing taken that the bodies
have to convert, expand or refuse."""
import pytest
import torch

import mlx_amd
from mlx_amd import _lib, ops

pytestmark = pytest.mark.gpu


class _Nothing:
    def __getattr__(self, name):
        return lambda *args: None


@pytest.fixture
def both(monkeypatch):
    def run(fn):
        monkeypatch.setattr(ops, "_fast", _lib.load_fast())
        fast = fn()
        monkeypatch.setattr(ops, "_fast", _Nothing())
        body = fn()
        fast, body = (t if isinstance(t, tuple) else (t,) for t in (fast, body))
        assert len(fast) == len(body)
        for a, b in zip(fast, body):
            assert a.shape == b.shape and a.dtype == b.dtype and a.requires_grad == b.requires_grad
            assert torch.equal(a.detach().view(torch.uint8), b.detach().view(torch.uint8))

    return run


def _x(*shape, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(sum(shape))
    return torch.randn(shape, generator=g).to(dtype).cuda()


@pytest.mark.parametrize("mode,group,bits", [("affine", 64, 4), ("affine", 32, 3), ("mxfp4", None, None),
                                             ("nvfp4", 16, 4)])
@pytest.mark.parametrize("lead", [(), (1,), (5,), (3, 40)])
@pytest.mark.parametrize("transpose", [True, False])
def test_products(both, mode, group, bits, lead, transpose):
    q = mlx_amd.quantize(_x(192, 256), group, bits, mode)
    kw = dict(transpose=transpose, group_size=group, bits=bits, mode=mode)
    x = _x(*lead, 256 if transpose else 192)
    plain = (x, *q, *(() if mode == "affine" else (None,)), transpose, group, bits, mode, None)
    assert _lib.load_fast().quantized_matmul(*plain) is not None
    both(lambda: mlx_amd.quantized_matmul(x, *q, **kw))
    both(lambda: mlx_amd.quantize(x if lead else x[None], group, bits, mode))
    both(lambda: mlx_amd.dequantize(*q, group_size=group, bits=bits, mode=mode))
    if transpose and mode != "affine":
        both(lambda: mlx_amd.qqmm(x, *q, group_size=group, bits=bits, mode=mode))
    if transpose and mode == "affine" and len(lead) < 2:
        both(lambda: mlx_amd.quantized_swiglu(x, q, q, group, bits))


def test_what_is_left_to_the_bodies(both):
    fast = _lib.load_fast()
    q = mlx_amd.quantize(_x(192, 256))
    x = _x(5, 256)
    rest = (True, None, None, "affine", None)
    strided = _x(5, 512)[:, ::2]
    assert fast.quantized_matmul(strided, *q, *rest) is None
    both(lambda: mlx_amd.quantized_matmul(strided, *q))
    assert fast.quantized_matmul(x.float(), *q, *rest) is None
    both(lambda: mlx_amd.quantized_matmul(x.float(), *q))
    assert fast.quantized_matmul(x[:, :128].contiguous(), *q, *rest) is None
    assert fast.quantized_matmul(x, q[0], q[1], None, *rest) is None
    assert fast.quantized_matmul(x, *q, True, 48, None, "affine", None) is None
    assert fast.quantized_matmul(x, *q, True, None, None, "mxfp5", None) is None
    assert fast.quantized_matmul(x.cpu(), *q, *rest) is None
    assert fast.quantized_matmul(x[:0], *q, *rest) is None
    leaf = x.clone().requires_grad_()
    assert fast.quantized_matmul(leaf, *q, *rest) is None
    both(lambda: mlx_amd.quantized_matmul(leaf, *q))
    with torch.no_grad():
        assert fast.quantized_matmul(leaf, *q, *rest) is not None
    y = mlx_amd.quantized_matmul(leaf, *q)
    (dx,) = torch.autograd.grad(y, leaf, torch.ones_like(y))
    assert dx.shape == leaf.shape


@pytest.mark.parametrize("rows", (1, 3, 16, 48, 600))
def test_an_image_of_scales_and_biases(both, rows):
    """Neither the host path nor an image decides which kernel multiplies."""
    q = mlx_amd.quantize(_x(512, 4096), 64, 8)
    image = mlx_amd.quantized_matmul_sb_image(q[1], q[2], 64)
    x = _x(rows, 4096)
    kw = dict(group_size=64, bits=8)
    both(lambda: mlx_amd.quantized_matmul(x, *q, **kw, sb_image=image))
    strided = torch.stack([x, x], dim=-1)[..., 0]
    assert not strided.is_contiguous()
    want = mlx_amd.quantized_matmul(x, *q, **kw)
    assert torch.equal(mlx_amd.quantized_matmul(x, *q, **kw, sb_image=image), want)
    assert torch.equal(mlx_amd.quantized_matmul(strided, *q, **kw, sb_image=image), want)


def test_on_another_stream_and_thread():
    import threading

    q = mlx_amd.quantize(_x(4096, 4096))
    x = [_x(1, 4096), _x(48, 4096), _x(7, 4096)]
    want = [mlx_amd.quantized_matmul(t, *q) for t in x]
    torch.cuda.synchronize()
    got = [None] * len(x)

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                got[i] = mlx_amd.quantized_matmul(x[i], *q)
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(x))]
    [t.start() for t in threads]
    [t.join() for t in threads]
    for a, b in zip(got, want):
        assert torch.equal(a, b)
