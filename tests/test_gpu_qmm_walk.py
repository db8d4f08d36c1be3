"""The few-row kernel whose x walks through LDS: the edges of its tiles of rows of
W and x, its 128-code chunks and stages, K ranges, every width, group and mode,
against the exact product of the dequantized weights."""
import pytest
import torch

import mlx_amd
from mlx_amd import _lib

pytestmark = pytest.mark.gpu

ROWS = (2, 3, 5, 8, 9, 16, 17, 31, 33, 48, 49, 64)
# N and K: less than a tile, ragged tiles, a ragged last chunk (K % 128), a last
# stage of one chunk, one and several rounds of workgroups, K in ranges
SHAPES = ((4, 1024), (67, 1120), (1000, 2080), (4096, 4096), (5001, 1152), (33000, 1024),
          (512, 14336))


def _check(x, q, group, bits, mode, y):
    # bf16 / f16 products are exact in fp32; sums are fp32 over K terms: the result
    # is within half an ulp of its type of the exact sum, plus the sums' own 2e-6
    if mode == "affine":
        w = mlx_amd.dequantize(q[0], q[1].float(), q[2].float(), group, bits).double()
    else:
        w = mlx_amd.dequantize(q[0], q[1], mode=mode, dtype=torch.float32).double()
    want = x.double() @ w.T
    size = x.double().abs() @ w.abs().T
    # (codes are multiplied with an offset that the biases take back, in fp32: that adds
    # offset / (2^bits - 1) times the size of the product at worst)
    f16 = x.dtype == torch.float16
    offset = {8: 1024 if f16 else 0, 4: 64 if f16 else 128}.get(bits, 2 ** (bits or 0))
    sums = 2e-6 * (1 if mode != "affine" else 1 + offset / (2 ** bits - 1) / 8)
    half = 2.0 ** -8 if x.dtype == torch.bfloat16 else 2.0 ** -11
    err = (y.double() - want).abs()
    ok = bool((err <= half * want.abs() + sums * size).all())
    assert ok, (tuple(x.shape), tuple(q[0].shape), group, bits, mode, float((err / size).max()))


def _inputs(M, N, K, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((M, K), generator=g, device="cuda").to(dtype)
    w = (torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).to(dtype)
    return x, w


@pytest.mark.parametrize("bits", (2, 3, 4, 5, 6, 8))
@pytest.mark.parametrize("group", (32, 64, 128))
def test_affine(bits, group):
    taken = 0
    for i, (N, K) in enumerate(SHAPES):
        K = K // group * group
        dtype = (torch.bfloat16, torch.float16)[(i + bits) % 2]
        for M in ROWS[(i + bits) % 2::2]:
            if not _lib.load().mlxrocm_qmm_rows_supported(
                    M, N, K, 1, group, bits, 2 if dtype == torch.bfloat16 else 1):
                continue  # (kernels that round the weights to the type: another bound)
            taken += 1
            x, w = _inputs(M, N, K, dtype, M + N)
            q = mlx_amd.quantize(w, group, bits)
            y = mlx_amd.quantized_matmul(x, *q, group_size=group, bits=bits)
            _check(x, q, group, bits, "affine", y)
    assert taken >= 18, taken


@pytest.mark.parametrize("bits", (2, 3, 4, 5, 6, 8))
def test_x_of_one_sign(bits):
    """Where every x has one sign the codes' offset weighs most against the result.
    float16 results may lose nothing to it: sums in fp32 within half of what rounding
    the exact result loses (the two add up in squares: sqrt(1 + 1/4))."""
    for group, N, K in ((64, 1024, 2048), (128, 4096, 4096), (64, 4096, 8192)):
        for M in (3, 6, 20, 40):
            if not _lib.load().mlxrocm_qmm_rows_supported(M, N, K, 1, group, bits, 1):
                continue
            x, w = _inputs(M, N, K, torch.float16, M)
            x = x.abs()
            q = mlx_amd.quantize(w, group, bits)
            y = mlx_amd.quantized_matmul(x, *q, group_size=group, bits=bits)
            exact = x.double() @ mlx_amd.dequantize(
                q[0], q[1].float(), q[2].float(), group, bits).double().T
            rounding = (exact.half().double() - exact).norm()
            assert float((y.double() - exact).norm() / rounding) < 1.25 ** 0.5, (group, N, K, M)


def _same_kind(y, want):
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isposinf(), want.isposinf())
    assert torch.equal(y.isneginf(), want.isneginf())


@pytest.mark.parametrize("bits", (2, 3, 4, 5, 6, 8))
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
def test_infinite_and_huge_x(bits, dtype):
    """One x that is infinite, NaN or near the end of bfloat16 decides its row as a
    product with the dequantized weights does, and leaves the other rows alone."""
    taken = 0
    for (N, K), M, group in ((SHAPES[1], 8, 32), (SHAPES[3], 16, 64), (SHAPES[3], 64, 128),
                             (SHAPES[6], 40, 64), (SHAPES[5], 33, 64)):
        if not _lib.load().mlxrocm_qmm_rows_supported(
                M, N, K, 1, group, bits, 2 if dtype == torch.bfloat16 else 1):
            continue
        taken += 1
        x, w = _inputs(M, N, K, dtype, M)
        x[0, K // 3] = float("inf")
        x[1, K - 1] = float("-inf")
        x[2, 7] = float("nan")
        x[3, 5], x[3, K - 3] = float("inf"), float("-inf")
        x[4, K // 2] = torch.finfo(dtype).max  # (bfloat16: its products leave fp32)
        q = mlx_amd.quantize(w, group, bits)
        y = mlx_amd.quantized_matmul(x, *q, group_size=group, bits=bits)
        wd = mlx_amd.dequantize(q[0], q[1].float(), q[2].float(), group, bits).to(dtype).double()
        want = x.double() @ wd.T
        _same_kind(y[:4], want[:4].to(dtype))
        assert bool(y[4:].isfinite().all())
        # against weights rounded to the type: that, the sums and the result
        size = x[4:].double().abs() @ wd.abs().T
        half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        assert bool(((y[4:].double() - want[4:]).abs() <= 2 * half * size).all())
    assert taken >= 3


def test_infinite_x_in_the_gated_form():
    x, gate = _inputs(5, 18944, 3584, torch.bfloat16, 1)
    _, up = _inputs(5, 18944, 3584, torch.bfloat16, 2)
    x[1, 100], x[3, 3583] = float("inf"), float("-inf")
    g, u = mlx_amd.quantize(gate, 128, 8), mlx_amd.quantize(up, 128, 8)
    y = mlx_amd.quantized_swiglu(x, g, u, 128, 8)
    a, b = (mlx_amd.quantized_matmul(x, *q, group_size=128, bits=8) for q in (g, u))
    _same_kind(y, (a.float() * torch.sigmoid(a.float()).bfloat16()).bfloat16() * b)
    assert bool(y[::2].isfinite().all()) and bool(a[1].isinf().any())


@pytest.mark.parametrize("mode", ("mxfp4", "mxfp8", "nvfp4"))
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
def test_fp_modes(mode, dtype):
    taken = 0
    for N, K in SHAPES:
        K = K // 32 * 32
        for M in ROWS:
            x, w = _inputs(M, N, K, dtype, M + N)
            q = mlx_amd.quantize(w, mode=mode)
            taken += _lib.load().mlxrocm_fp_qmm_rows_supported(
                M, N, K, 1, _lib.MXFP4 + ("mxfp4", "mxfp8", "nvfp4").index(mode),
                2 if dtype == torch.bfloat16 else 1)
            _check(x, q, None, None, mode, mlx_amd.quantized_matmul(x, *q, mode=mode))
    assert taken >= 30


def test_fp8_codes_that_no_quantizer_writes():
    # 0x7f and 0xff stand for +-480, not NaN
    x, w = _inputs(8, 96, 1024, torch.bfloat16, 3)
    wq, scales = mlx_amd.quantize(w, mode="mxfp8")
    codes = wq.view(torch.uint8).clone()
    codes[::7, ::97] = 0x7F
    codes[3::11, 5::64] = 0xFF
    q = (codes.view(torch.uint32), scales)
    _check(x, q, None, None, "mxfp8", mlx_amd.quantized_matmul(x, *q, mode="mxfp8"))


def test_stacks_of_weights_and_the_tensor_wide_scale():
    x, w = _inputs(24, 640, 4096, torch.bfloat16, 5)
    q = mlx_amd.quantize(w.reshape(2, 320, 4096), 64, 8)
    y = mlx_amd.quantized_matmul(x.reshape(2, 12, 4096), *q, group_size=64, bits=8)
    for i in range(2):
        _check(x.reshape(2, 12, 4096)[i], [t[i] for t in q], 64, 8, "affine", y[i])
    qf = mlx_amd.quantize(w.reshape(2, 320, 4096), mode="mxfp4")
    y = mlx_amd.quantized_matmul(x.reshape(2, 12, 4096), *qf, mode="mxfp4")
    for i in range(2):
        _check(x.reshape(2, 12, 4096)[i], [t[i] for t in qf], None, None, "mxfp4", y[i])
    # nvfp4 with global scales goes through qqmm: 24 rows against one row at a time
    one = torch.ones((), device="cuda")
    g = w.abs().max().float()
    qn = mlx_amd.quantize(w, mode="nvfp4", global_scale=g)
    kw = dict(mode="nvfp4", global_scale_x=one, global_scale_w=g)
    y = mlx_amd.qqmm(x, *qn, **kw)
    rows = torch.cat([mlx_amd.qqmm(x[i:i + 1], *qn, **kw) for i in range(24)])
    assert float((y.double() - rows.double()).norm() / rows.double().norm()) < 2.0 ** -8


@pytest.mark.parametrize("bits,group,N,K", ((8, 128, 18944, 3584), (8, 64, 4099, 1024),
                                            (4, 32, 5504, 2048), (6, 64, 9000, 2048)))
def test_gated_form(bits, group, N, K):
    for M in (3, 5, 8):
        x, gate = _inputs(M, N, K, torch.bfloat16, 1)
        _, up = _inputs(M, N, K, torch.bfloat16, 2)
        g, u = mlx_amd.quantize(gate, group, bits), mlx_amd.quantize(up, group, bits)
        y = mlx_amd.quantized_swiglu(x, g, u, group, bits).double()
        a, b = (mlx_amd.quantized_matmul(x, *q, group_size=group, bits=bits) for q in (g, u))
        want = ((a.float() * torch.sigmoid(a.float()).bfloat16()).bfloat16() * b).double()
        # same sums in another order, then the same four roundings: a few last places
        assert float((y - want).norm() / want.norm()) < 2.0 ** -7


def _at_byte(t, offset):
    """The same values in memory that starts `offset` bytes past an aligned address."""
    flat = torch.empty(t.numel() * t.element_size() + offset, dtype=torch.uint8, device=t.device)
    flat[offset:] = t.contiguous().view(torch.uint8).reshape(-1)
    return flat[offset:].view(t.dtype).view(t.shape)


@pytest.mark.parametrize("mode", ("mxfp4", "mxfp8", "nvfp4"))
def test_scale_bytes_at_any_address(mode):
    for M in (3, 16, 40):
        x, w = _inputs(2 * M, 640, 4096, torch.bfloat16, M)
        q = mlx_amd.quantize(w, mode=mode)
        stack = mlx_amd.quantize(w.reshape(2, 320, 4096), mode=mode)
        want = mlx_amd.quantized_matmul(x[:M], *q, mode=mode)
        want2 = mlx_amd.quantized_matmul(x.reshape(2, M, 4096), *stack, mode=mode)
        for offset in (1, 2, 4):
            y = mlx_amd.quantized_matmul(x[:M], q[0], _at_byte(q[1], offset), mode=mode)
            assert torch.equal(y, want)
            y = mlx_amd.quantized_matmul(
                x.reshape(2, M, 4096), stack[0], _at_byte(stack[1], offset), mode=mode)
            assert torch.equal(y, want2)


def test_a_stack_whose_scales_lie_at_odd_strides():
    lib = _lib.load()
    M, N, K, group, bits = 16, 320, 4096, 64, 8
    x, w = _inputs(2 * M, 2 * N, K, torch.bfloat16, 7)
    q = [mlx_amd.quantize(t, group, bits) for t in w.reshape(2, N, K)]
    per = N * K // group
    spread = [torch.zeros(2 * per + 8, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    for which in range(2):
        for i in range(2):
            at = i * (per + 3)
            spread[which][at:at + per] = q[i][1 + which].reshape(-1)
    wq = torch.stack([t[0].view(torch.int32) for t in q])
    out = torch.empty((2, M, N), dtype=torch.bfloat16, device="cuda")
    need = lib.mlxrocm_qmm_rows_workspace_size(M, N, K, 2, group, bits, _lib.BFLOAT16)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    _lib.check(lib.mlxrocm_qmm_rows(
        x.data_ptr(), wq.data_ptr(), spread[0].data_ptr(), spread[1].data_ptr(), out.data_ptr(), M,
        N, K, 2, M * K, N * K * bits // 32, per + 3, group, bits, _lib.BFLOAT16, ws.data_ptr(),
        need, torch.cuda.current_stream().cuda_stream))
    for i in range(2):
        _check(x[i * M:(i + 1) * M], q[i], group, bits, "affine", out[i])
