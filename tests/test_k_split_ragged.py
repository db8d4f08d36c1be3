"""K ranges where rows of y do not fill whole 16-byte pieces: the fp32 planes are
padded, the sum of the planes is not."""
import pytest
import torch

import mlx_amd
from mlx_amd import _lib

# N % 4 of 1, 2, 3 and 0; one and several tiles, rows past a tile, M * N odd and even; the
# rule that the 16-bit types take in affine mode
RULES = {(255, 775, 4096): "qmm_mid", (66, 1001, 2048): "qmm_mid", (97, 222, 1536): "qmm_mid",
         (513, 803, 2048): "qmm_mid", (70, 449, 1024): "qmm_mid", (130, 640, 1024): "qmm_mid",
         (300, 803, 4096): "qmm_t_tile_k_split", (265, 1002, 3520): "qmm_t_tile_k_split",
         (600, 803, 4096): "qmm_t_tile_sb_transposed", (514, 229, 2112): "qmm_t_tile_sb_transposed"}
SHAPES = tuple(RULES)
FP = {"mxfp4": _lib.MXFP4, "mxfp8": _lib.MXFP8, "nvfp4": _lib.NVFP4}


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dtype", (_lib.FLOAT32, _lib.BFLOAT16))
def test_split_with_scratch_and_plain_without(M, N, K, dtype):
    need = _lib.load().mlxrocm_qmm_workspace_size(M, N, K, 1, 0, 64, 4, dtype, 1)
    rc, plan = _lib.qmm_plan(M, N, K, dtype=dtype, workspace_bytes=need)
    assert rc == _lib.OK and "reduce_k_splits" in plan, plan
    rule = RULES[M, N, K] if dtype != _lib.FLOAT32 else "qmm_t_split_fp32"
    assert plan.startswith(f"[{rule}]"), plan
    if N % 4 and dtype != _lib.FLOAT32 and M < 512:  # (these took no workspace before)
        rc, plan = _lib.qmm_plan(M, N, K, dtype=dtype, workspace_bytes=0)
        assert rc == _lib.OK and "reduce_k_splits" not in plan, plan


@pytest.mark.parametrize("M,N,K,split", (
    (1495, 4099, 1024, False), (6334, 1001, 1344, False), (2195, 3001, 1344, False),
    (990, 3001, 1344, True), (700, 6002, 2048, True), (1501, 1502, 4096, True),
))
def test_ranges_where_planes_cost_less_than_they_save(M, N, K, split):
    need = _lib.load().mlxrocm_qmm_workspace_size(M, N, K, 1, 0, 64, 4, _lib.BFLOAT16, 1)
    rc, plan = _lib.qmm_plan(M, N, K, dtype=_lib.BFLOAT16, workspace_bytes=need)
    assert rc == _lib.OK and "qmm_t_tile" in plan and ("reduce_k_splits" in plan) == split, plan
    rc, plan = _lib.fp_qmm_plan(M, N, K)
    assert rc == _lib.OK and ("reduce_k_splits" in plan) == split, plan


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("mode", ("affine", "mxfp4", "mxfp8", "nvfp4"))
@pytest.mark.parametrize("dtype", (torch.float32, torch.float16, torch.bfloat16))
def test_products(gpu, M, N, K, mode, dtype):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn((M, K), generator=g, device="cuda").to(dtype)
    w = (torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).to(dtype)
    q = mlx_amd.quantize(w, mode=mode)
    if mode == "affine":
        w_hat = mlx_amd.dequantize(q[0], q[1].float(), q[2].float()).double()
    else:
        w_hat = mlx_amd.dequantize(*q, mode=mode, dtype=torch.float32).double()
    y = mlx_amd.quantized_matmul(x, *q, mode=mode)
    want = x.double() @ w_hat.T
    size = x.double().abs() @ w_hat.abs().T
    # half an ulp of the result; weights rounded to the type (16-bit affine) or products
    # formed from bf16 halves (float32, 2**-16); fp32 sums over K terms
    half = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    terms = 2.0 ** -16 if dtype == torch.float32 else (half if mode == "affine" else 0.0) + 2e-6
    err = (y.double() - want).abs()
    assert bool((err <= half * want.abs() + terms * size).all()), float((err / size).max())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("mode", ("mxfp4", "mxfp8"))
def test_both_operands_quantized(gpu, M, N, K, mode):
    g = torch.Generator(device="cuda").manual_seed(M * N)

    def grid(rows):  # numbers of the format, so that quantizing x changes nothing
        table = torch.tensor((6.0, 3.0, 1.5, -0.5) if mode == "mxfp4" else (448.0, -256.0, 96.0, 3.5),
                             device="cuda")
        v = table[torch.randint(0, 4, (rows, K), generator=g, device="cuda")]
        v[:, ::32] = table[0]
        return (v / table[0].log2().floor().exp2()).bfloat16()

    x, q = grid(M), mlx_amd.quantize(grid(N), mode=mode)
    y = mlx_amd.qqmm(x, *q, mode=mode)
    x_hat, w_hat = x.double(), mlx_amd.dequantize(*q, mode=mode, dtype=torch.float32).double()
    want, size = x_hat @ w_hat.T, x_hat.abs() @ w_hat.abs().T
    # (the e4m3 instruction keeps about 17 bits below a step's largest product)
    err = (y.double() - want).abs()
    assert bool((err <= 2.0 ** -8 * want.abs() + 2e-5 * size).all()), float((err / size).max())


@pytest.mark.parametrize("dtype", (_lib.FLOAT32, _lib.BFLOAT16))
def test_built_in_scratch_takes_the_same_plan(dtype):
    """mlxrocm_qmm_static has 64 MiB and the results of mlxrocm_qmm: what fits there without
    planes is planned alike with any scratch."""
    lib = _lib.load()
    for M in (66, 255, 300, 513, 1023, 2000):
        for N in (449, 5119, 10762, 14333, 32001):
            for K in (2048, 4096, 14336, 18944, 28672):
                need = lib.mlxrocm_qmm_workspace_size(M, N, K, 1, 0, 64, 4, dtype, 1)
                rc, plan = _lib.qmm_plan(M, N, K, dtype=dtype, workspace_bytes=need)
                assert rc == _lib.OK
                rc, built_in = _lib.qmm_plan(M, N, K, dtype=dtype, workspace_bytes=64 << 20)
                # (the same kernels and ranges, with less scratch for some rows of x at a time)
                if rc == _lib.OK:
                    assert set(built_in.split("+")) == set(plan.split("+")), (M, N, K, built_in)
                    assert built_in == plan or need > 64 << 20
                else:
                    assert need > 64 << 20


# (M, N, K), both modes of qqmm's own kernel and, at K % 128 != 0 or in nvfp4, the others
QQ = ((96, 775, 4096), (300, 1001, 4096), (511, 222, 2048), (130, 803, 4160))


def qqmm_bytes_without_planes(M, N, K, mode, dtype_size=2):
    up = lambda n: (n + 255) // 256 * 256
    if mode != _lib.NVFP4 and K % 128 == 0:  # codes and scales of x, scales of W
        return up(M * K * (8 if mode == _lib.MXFP8 else 4) // 8) + up(M * K // 32) + up(N * K // 32)
    return up(M * K * dtype_size) + up(N * (K // 32) * 4)  # x again, the scale image


@pytest.mark.parametrize("M,N,K", QQ)
@pytest.mark.parametrize("mode", FP.values(), ids=FP)
def test_qqmm_without_room_for_planes(M, N, K, mode):
    least = qqmm_bytes_without_planes(M, N, K, mode)
    need = _lib.load().mlxrocm_fp_qqmm_workspace_size(M, N, K, mode, _lib.BFLOAT16)
    rc, plan = _lib.fp_qqmm_plan(M, N, K, mode, _lib.BFLOAT16, need)
    assert rc == _lib.OK and ("reduce_k_splits" in plan) == (need > least), plan
    rc, plan = _lib.fp_qqmm_plan(M, N, K, mode, _lib.BFLOAT16, least)
    assert rc == _lib.OK and "reduce_k_splits" not in plan, plan
    rc, plan = _lib.fp_qqmm_plan(M, N, K, mode, _lib.BFLOAT16, least - 1)
    assert rc == _lib.INVALID_ARGUMENT


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", QQ)
@pytest.mark.parametrize("mode", FP)
def test_qqmm_with_and_without_planes(gpu, M, N, K, mode):
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(M * N)
    x = torch.randn((M, K), generator=g, device="cuda").bfloat16()
    wq, s = mlx_amd.quantize(torch.randn((N, K), generator=g, device="cuda") * K ** -0.5, mode=mode)
    ws = torch.empty(qqmm_bytes_without_planes(M, N, K, FP[mode]), dtype=torch.uint8, device="cuda")
    y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    _lib.check(lib.mlxrocm_fp_qqmm(
        x.data_ptr(), wq.data_ptr(), s.data_ptr(), y.data_ptr(), M, N, K, FP[mode], _lib.BFLOAT16,
        ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
    want = mlx_amd.qqmm(x, wq, s, mode=mode)
    # the same products in another order: an ulp of some results
    assert float((y.double() - want.double()).norm() / want.double().norm()) < 2.0 ** -9


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", ((300, 803, 4096), (265, 1002, 3520), (600, 803, 4096)))
@pytest.mark.parametrize("dtype", (torch.float32, torch.bfloat16))
def test_scratch_for_some_rows_gives_the_same_bits(gpu, M, N, K, dtype):
    lib = _lib.load()
    code = {torch.float32: _lib.FLOAT32, torch.bfloat16: _lib.BFLOAT16}[dtype]
    x = torch.randn((M, K), device="cuda").to(dtype)
    wq, s, b = mlx_amd.quantize((torch.randn((N, K), device="cuda") / 64).to(dtype))
    want = mlx_amd.quantized_matmul(x, wq, s, b)
    need = lib.mlxrocm_qmm_workspace_size(M, N, K, 1, 0, 64, 4, code, 1)
    for room in (need * 7 // 8, need * 2 // 3):
        plan = _lib.qmm_plan(M, N, K, dtype=code, workspace_bytes=room)[1]
        assert plan.count("reduce_k_splits") > 1, plan
        ws = torch.empty(room, dtype=torch.uint8, device="cuda")
        y = torch.full((M, N), -1.0, dtype=dtype, device="cuda")
        _lib.check(lib.mlxrocm_qmm(
            x.data_ptr(), wq.data_ptr(), s.data_ptr(), b.data_ptr(), y.data_ptr(), M, N, K, 1,
            M * K, 0, 0, 64, 4, code, 1, ws.data_ptr(), room,
            torch.cuda.current_stream().cuda_stream))
        assert torch.equal(y, want)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", ((255, 14333, 18944), (600, 2735, 14336)))
def test_built_in_scratch_takes_what_it_took(gpu, M, N, K):
    """mlxrocm_qmm_static plans within its 64 MiB: the rows of x in blocks, where planes for
    all of them do not fit beside the split x."""
    lib = _lib.load()
    assert lib.mlxrocm_qmm_workspace_size(M, N, K, 1, 0, 64, 4, _lib.FLOAT32, 1) > 64 << 20
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn((M, K), generator=g, device="cuda")
    wq, s, b = mlx_amd.quantize(torch.randn((N, K), generator=g, device="cuda") * K ** -0.5)
    y = torch.empty((M, N), device="cuda")
    _lib.check(lib.mlxrocm_qmm_static(
        x.data_ptr(), wq.data_ptr(), s.data_ptr(), b.data_ptr(), y.data_ptr(), M, N, K, 1, M * K,
        0, 0, 64, 4, _lib.FLOAT32, 1, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(y, mlx_amd.quantized_matmul(x, wq, s, b))
