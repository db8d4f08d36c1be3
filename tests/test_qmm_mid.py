"""The 65..256-row kernel: where it is taken, and its products at the edges of its tiles,
K-steps, table segments and ranges."""
import pytest
import torch

import mlx_amd
from mlx_amd import _lib


@pytest.mark.parametrize("M,N,K,taken", (
    (64, 4096, 4096, False), (65, 4096, 4096, True), (256, 4096, 14336, True),
    (257, 4096, 4096, False), (257, 2048, 2048, True), (2049, 1024, 1024, False),
    (128, 32768, 4096, True), (128, 32769, 4096, False),  # one round of 256 workgroups
    (100, 4096, 4160, False),  # K in whole steps
))
def test_rule(M, N, K, taken):
    need = _lib.load().mlxrocm_qmm_workspace_size(M, N, K, 1, 0, 64, 4, _lib.BFLOAT16, 1)
    rc, plan = _lib.qmm_plan(M, N, K, dtype=_lib.BFLOAT16, workspace_bytes=need)
    assert rc == _lib.OK and ("qmm_mid(" in plan) == taken, plan


# by the accounts of both kernels: three tiles of 96 rows at 8 bits and codes that are dear to
# unpack leave the tile kernel ahead
@pytest.mark.parametrize("bits,group,M,N,K,taken", (
    (8, 32, 193, 4096, 14336, False), (8, 64, 224, 4096, 14336, False),
    (8, 32, 193, 8192, 8192, False), (8, 64, 256, 8192, 8192, False),
    (6, 128, 129, 11008, 4096, False), (6, 32, 193, 14336, 4096, False),
    (3, 64, 129, 11008, 4096, False), (2, 32, 129, 11008, 4096, False),
    (8, 32, 96, 4096, 4096, True), (8, 64, 256, 4096, 4096, True), (6, 64, 192, 4096, 4096, True),
    (6, 32, 96, 4096, 14336, True), (4, 32, 128, 4096, 14336, True), (3, 32, 700, 2048, 2048, True),
))
def test_rule_of_every_width(bits, group, M, N, K, taken):
    need = _lib.load().mlxrocm_qmm_workspace_size(M, N, K, 1, 0, group, bits, _lib.BFLOAT16, 1)
    rc, plan = _lib.qmm_plan(M, N, K, group_size=group, bits=bits, dtype=_lib.BFLOAT16,
                             workspace_bytes=need)
    assert rc == _lib.OK and ("qmm_mid(" in plan) == taken, plan


def test_less_scratch_keeps_the_other_plan():
    M, N, K = 97, 222, 4096
    need = _lib.load().mlxrocm_qmm_workspace_size(M, N, K, 1, 0, 64, 4, _lib.BFLOAT16, 1)
    assert need > 0
    rc, plan = _lib.qmm_plan(M, N, K, dtype=_lib.BFLOAT16, workspace_bytes=0)
    assert rc == _lib.OK and "qmm_mid(" not in plan, plan


@pytest.mark.parametrize("bits,group", ((4, 64), (8, 32), (3, 128)))
def test_workspace_counts_the_scale_image(bits, group):
    """mlxrocm_qmm_prepacked takes a workspace that is smaller by the image: what is left
    holds the planes of the same plan."""
    lib = _lib.load()
    for M in (512, 513, 700, 1024, 1500, 2048):
        for N in (64, 222, 1024, 1401, 2048, 4096):
            for K in (128, 640, 1024, 2048):
                need = lib.mlxrocm_qmm_workspace_size(M, N, K, 1, 0, group, bits, _lib.BFLOAT16, 1)
                image = lib.mlxrocm_qmm_sb_image_size(N, K, 1, group, _lib.BFLOAT16)
                rc, plan = _lib.qmm_plan(M, N, K, group_size=group, bits=bits,
                                         dtype=_lib.BFLOAT16, workspace_bytes=need)
                planes = int(plan.split("reduce_k_splits(")[1][:-1]) if "reduce" in plan else 0
                rest = planes * M * ((N + 3) // 4 * 4) * 4
                assert rc == _lib.OK and need >= (image + 255) // 256 * 256 + rest, (M, N, K, plan)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", ((512, 1024, 2048), (2048, 1024, 2048), (600, 1024, 4096),
                                   (600, 803, 4096)))
def test_prepacked_with_the_smaller_workspace(gpu, M, N, K):
    lib = _lib.load()
    x = torch.randn((M, K), device="cuda").to(torch.bfloat16)
    wq, s, b = mlx_amd.quantize((torch.randn((N, K), device="cuda") / 64).to(torch.bfloat16))
    image = mlx_amd.quantized_matmul_sb_image(s, b, 64)
    room = lib.mlxrocm_qmm_workspace_size(M, N, K, 1, 0, 64, 4, _lib.BFLOAT16, 1)
    room -= (lib.mlxrocm_qmm_sb_image_size(N, K, 1, 64, _lib.BFLOAT16) + 255) // 256 * 256
    ws = torch.empty(max(room, 1), dtype=torch.uint8, device="cuda")
    y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    _lib.check(lib.mlxrocm_qmm_prepacked(
        x.data_ptr(), wq.data_ptr(), s.data_ptr(), b.data_ptr(), image.data_ptr(), y.data_ptr(),
        M, N, K, 1, M * K, 0, 0, 64, 4, _lib.BFLOAT16, 1, ws.data_ptr(), room,
        torch.cuda.current_stream().cuda_stream))
    assert torch.equal(y, mlx_amd.quantized_matmul(x, wq, s, b))


# (rows: one tile of 64, 96 and 128, several with a short last one; N: one row of W past a
# tile, no whole 16-byte rows of y, less than a tile; K: one step, fewer steps than stages,
# more than a table segment holds (2048 codes at groups of 32), many ranges)
SHAPES = ((65, 129, 128), (97, 100, 256), (128, 257, 384), (129, 1027, 512), (256, 128, 4096),
          (200, 4099, 2176), (66, 32640, 2304), (700, 640, 640))


@pytest.mark.gpu
@pytest.mark.parametrize("bits", (2, 3, 4, 5, 6, 8))
@pytest.mark.parametrize("group", (32, 64, 128))
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
def test_products(gpu, bits, group, dtype):
    half = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    code = {torch.float16: _lib.FLOAT16, torch.bfloat16: _lib.BFLOAT16}[dtype]
    for M, N, K in SHAPES:
        g = torch.Generator(device="cuda").manual_seed(M + N + K)
        x = torch.randn((M, K), generator=g, device="cuda").to(dtype)
        w = (torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).to(dtype)
        q = mlx_amd.quantize(w, group, bits)
        assert "qmm_mid(" in _lib.qmm_plan(
            M, N, K, dtype=code, group_size=group, bits=bits, workspace_bytes=1 << 30)[1]
        y = mlx_amd.quantized_matmul(x, *q, group_size=group, bits=bits).double()
        # weights s c + b in float32, rounded once to the type
        w_hat = mlx_amd.dequantize(q[0], q[1].float(), q[2].float(), group_size=group,
                                   bits=bits).double()
        want = x.double() @ w_hat.T
        size = x.double().abs() @ w_hat.abs().T
        # half an ulp of the result and of every weight, fp32 sums over K terms
        err = (y - want).abs()
        assert bool((err <= half * want.abs() + (half + 2e-6) * size).all()), (M, N, K)


@pytest.mark.gpu
def test_values_that_are_not_finite_stay_in_their_row(gpu):
    M, N, K = 130, 300, 1024
    x = torch.randn((M, K), device="cuda").to(torch.bfloat16)
    q = mlx_amd.quantize((torch.randn((N, K), device="cuda") / 32).to(torch.bfloat16))
    clean = mlx_amd.quantized_matmul(x, *q)
    x[M - 1, 5] = float("nan")
    y = mlx_amd.quantized_matmul(x, *q)
    assert bool(y[M - 1].isnan().all()) and torch.equal(y[: M - 1], clean[: M - 1])


@pytest.mark.gpu
def test_replays_and_streams(gpu):
    x = torch.randn((100, 4096), device="cuda").to(torch.bfloat16)
    q = mlx_amd.quantize((torch.randn((1030, 4096), device="cuda") / 64).to(torch.bfloat16))
    want = mlx_amd.quantized_matmul(x, *q)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = []
    for _ in range(4):
        for s in streams:
            with torch.cuda.stream(s):
                got.append(mlx_amd.quantized_matmul(x, *q))
    torch.cuda.synchronize()
    assert all(torch.equal(y, want) for y in got)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = mlx_amd.quantized_matmul(x, *q)
    for i in range(4):
        x.copy_(torch.randn((100, 4096), device="cuda"))
        want = mlx_amd.quantized_matmul(x, *q)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), i
