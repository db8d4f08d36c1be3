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


def _indices(rows):
    e = torch.cat([torch.full((n,), i) for i, n in enumerate(rows)])
    g = torch.Generator().manual_seed(5)
    return e[torch.randperm(len(e), generator=g)].reshape(-1, 1).to("cuda")


@pytest.mark.parametrize("bits", BITS)
@pytest.mark.parametrize("D,F,rows,group", [
    (128, 1664, ROWS, 64),  # one step of K, 13 tiles of gated columns: more tiles than workgroups
    (2944, 128, ROWS, 128), # 23 steps, one of the second product; 11.5 tiles of columns
    (384, 2432, (1, 0, 97, 182), 32),  # the second product in ranges of 9 and 10 steps
    (128, 5248, (2, 65, 0, 199), 32),  # the same, in four
])
def test_experts(D, F, rows, group, bits):
    dtype = torch.bfloat16 if (bits + D) % 2 else torch.float16
    torch.manual_seed(bits)
    block = nn.SwitchGLU(D, F, len(rows), group_size=group, bits=bits, dtype=dtype)
    idx = _indices(rows)
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
    for e, n in enumerate(rows):
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


# heights of a tile from 64 to 256 rows with a short last one, one and several rounds of tiles,
# ranges of K (the odd step among them), rows of y of any number of elements
SHAPES = ((321, 8191, 2176), (300, 2736, 8192), (257, 14337, 4096), (511, 4098, 4224),
          (1537, 4099, 4096), (3000, 1023, 1024), (4097, 2050, 256),
          (66, 18944, 3584), (2048, 4096, 14336))
FP = {"mxfp4": (_lib.MXFP4, 32, 4), "mxfp8": (_lib.MXFP8, 32, 8), "nvfp4": (_lib.NVFP4, 16, 4)}
CODE = {torch.float16: _lib.FLOAT16, torch.bfloat16: _lib.BFLOAT16}


def _relative(y, want, dtype):
    # results rounded once (half an ulp of 2**-7 / 2**-10 of the value), sums in 32 bits of
    # another order (2**-24 each, some tens of roundings)
    half = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    d = y.double() - want
    rms = want.pow(2).mean().sqrt()
    assert float(d.norm() / want.norm()) < half
    assert bool((d.abs() <= half * want.abs() * 1.001 + 2.0 ** -17 * rms).all())


@pytest.mark.parametrize("bits", BITS)
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
def test_products(bits, dtype):
    taken = 0
    for M, N, K in SHAPES:
        group = (32, 64, 128)[(M + bits) % 3]
        if not _lib.load().mlxrocm_qmm_rows_supported(M, N, K, 1, group, bits, CODE[dtype]):
            continue
        taken += 1
        g = torch.Generator(device="cuda").manual_seed(M)
        x = torch.randn((M, K), generator=g, device="cuda").to(dtype)
        w = (torch.randn((N, K), generator=g, device="cuda") / K ** 0.5).to(dtype)
        wq, s, b = mlx_amd.quantize(w, group, bits)
        y = mlx_amd.quantized_matmul(x, wq, s, b, group_size=group, bits=bits)
        codes = mlx_amd.dequantize(wq, torch.ones_like(s, dtype=torch.float32),
                                   torch.zeros_like(s, dtype=torch.float32), group, bits).double()
        w_hat = codes.unflatten(1, (-1, group)) * s.double()[..., None] + b.double()[..., None]
        w_hat = w_hat.flatten(1).to(dtype).double()
        _relative(y, x.double() @ w_hat.T, dtype)
        # the image made beforehand, and rows that are no numbers stay by themselves
        image = mlx_amd.quantized_matmul_sb_image(s, b, group)
        assert torch.equal(y, mlx_amd.quantized_matmul(x, wq, s, b, group_size=group, bits=bits,
                                                       sb_image=image))
        x[M - 1] = float("nan")
        z = mlx_amd.quantized_matmul(x, wq, s, b, group_size=group, bits=bits)
        assert torch.equal(z[:-1], y[:-1]) and bool(z[-1].isnan().all())
    assert taken >= 5


@pytest.mark.parametrize("mode", FP)
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
def test_floating_point_codes(mode, dtype):
    code, group, bits = FP[mode]
    taken = 0
    for M, N, K in SHAPES:
        if not _lib.load().mlxrocm_fp_qmm_rows_supported(M, N, K, 1, code, CODE[dtype]):
            continue
        taken += 1
        g = torch.Generator(device="cuda").manual_seed(M)
        x = torch.randn((M, K), generator=g, device="cuda").to(dtype)
        w = (torch.randn((N, K), generator=g, device="cuda")).to(dtype)
        wq, s = mlx_amd.quantize(w, mode=mode)[:2]
        y = mlx_amd.quantized_matmul(x, wq, s, None, mode=mode)
        w_hat = mlx_amd.dequantize(wq, s, None, mode=mode, dtype=dtype).double()
        _relative(y, x.double() @ w_hat.T, dtype)
    assert taken >= 4


def test_replayed_from_a_graph():
    M, N, K = 300, 2736, 8192
    wq, s, b = mlx_amd.quantize((torch.randn((N, K), device="cuda") / 64).bfloat16())
    x = torch.randn((M, K), device="cuda").bfloat16()
    assert _lib.load().mlxrocm_qmm_rows_supported(M, N, K, 1, 64, 4, _lib.BFLOAT16)
    mlx_amd.quantized_matmul(x, wq, s, b)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = mlx_amd.quantized_matmul(x, wq, s, b)
    for seed in range(4):
        torch.manual_seed(seed)
        x.copy_(torch.randn((M, K), device="cuda"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, mlx_amd.quantized_matmul(x, wq, s, b)), seed


@pytest.mark.parametrize("N,K,bits", ((1024, 4096, 8), (1024, 4096, 4), (2048, 1024, 2)))
def test_a_kept_image_is_read(N, K, bits):
    """The caller's image of scales and biases takes the place of one made in the call, with
    and without K ranges, on the host path and beside it."""
    lib = _lib.load()
    wq, s, b = mlx_amd.quantize((torch.randn((N, K), device="cuda") / 64).bfloat16(), 64, bits)
    taken = [M for M in (200, 640, 1500, 4096)
             if lib.mlxrocm_qmm_rows_supported(M, N, K, 1, 64, bits, _lib.BFLOAT16)]
    assert taken
    kw = dict(group_size=64, bits=bits)
    image = mlx_amd.quantized_matmul_sb_image(s, b, 64)
    for M in taken:
        x = torch.randn((M, K), device="cuda").bfloat16()
        strided = torch.stack([x, x], dim=-1)[..., 0]
        want = mlx_amd.quantized_matmul(x, wq, s, b, **kw)
        for rows in (x, strided):
            assert torch.equal(mlx_amd.quantized_matmul(rows, wq, s, b, **kw, sb_image=image), want)
            # (doubling is exact: a call that makes its own image gives `want` here as well)
            twice = mlx_amd.quantized_matmul(rows, wq, s, b, **kw, sb_image=2 * image)
            assert torch.equal(twice, 2 * want), M


@pytest.mark.parametrize("bits", (3, 8))
@pytest.mark.parametrize("E,D,F,tokens", ((8, 512, 384, 70), (4, 2176, 256, 70)))
def test_few_pairs_of_an_expert(bits, E, D, F, tokens):
    """Tiles of 17 and 33 pairs per expert and more, with the scratch the call names, and the
    products one by one with less: the same roundings."""
    lib = _lib.load()
    torch.manual_seed(bits)
    block = nn.SwitchGLU(D, F, E, group_size=64, bits=bits, dtype=torch.bfloat16)
    x = torch.randn((tokens, D), device="cuda").bfloat16()
    idx = torch.randint(0, E, (tokens, 2), device="cuda")
    idx[3, 1] = E + 2  # no such expert: a row of zeros
    y = block(x, idx)
    assert not y[3, 1].any()
    need = lib.mlxrocm_switch_glu_workspace_size(tokens, 2, D, F, E, 64, bits, _lib.BFLOAT16)
    ops = [t for layer in (block.gate_proj, block.up_proj, block.down_proj)
           for t in (layer.weight, layer.scales, layer.biases)]
    plain = tokens * 2 * F * 2 * 2 + 3 * 4 * tokens * 2  # h, up and the pairs
    got = {}
    for room in (need, need - 1):
        ws = torch.empty(room, dtype=torch.uint8, device="cuda")
        out = torch.empty((tokens, 2, D), dtype=torch.bfloat16, device="cuda")
        _lib.check(lib.mlxrocm_switch_glu(
            x.data_ptr(), idx.data_ptr(), 8, *[t.data_ptr() for t in ops], out.data_ptr(), tokens,
            2, D, F, E, 64, bits, _lib.BFLOAT16, ws.data_ptr(), room,
            torch.cuda.current_stream().cuda_stream))
        got[room] = out
    assert need > plain and torch.equal(got[need], y)
    d = (got[need - 1].double() - y.double()).norm() / y.double().norm()
    assert float(d) < 2.0 ** -8


def _weights(N, K, bits, dtype, group=64):
    g = torch.Generator(device="cuda").manual_seed(N + K + bits)
    w = (torch.randn((N, K), generator=g, device="cuda") / K ** 0.5).to(dtype)
    return mlx_amd.quantize(w, group, bits)


def _c_call(entry, x, q, image, N, bits, code, transpose, workspace_bytes, group=64):
    """A call at the C boundary on one product; image: None, or a 1-tuple with it or None."""
    (M, K), (wq, s, b) = x.shape, q
    out = torch.full((M, N), 7.0, dtype=x.dtype, device="cuda")
    ws = torch.full((workspace_bytes,), 0x7f, dtype=torch.uint8, device="cuda")
    between = [] if image is None else [image[0].data_ptr() if image[0] is not None else None]
    _lib.check(entry(
        x.data_ptr(), wq.data_ptr(), s.data_ptr(), b.data_ptr(), *between, out.data_ptr(), M, N, K,
        1, M * K, 0, 0, group, bits, code, *transpose,
        ws.data_ptr() if workspace_bytes else None, workspace_bytes,
        torch.cuda.current_stream().cuda_stream))
    return out


# shapes that the tiles of this file take (the first three in mlxrocm_qmm too; then fewer than 512
# rows, and planes of more than 64 MB) and shapes that they leave to the tile kernel
TABLE = ((2048, 4096, 4096, 8), (1024, 4096, 4096, 4), (5000, 1024, 4096, 4), (300, 14336, 4096, 2),
         (2048, 4096, 14336, 4), (600, 803, 4096, 4), (1024, 14336, 4096, 8), (1792, 7168, 4096, 4))


@pytest.mark.parametrize("M,N,K,bits", TABLE)
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
def test_prepacked_calls_have_the_bits_of_plain_ones(M, N, K, bits, dtype):
    """mlxrocm_qmm_prepacked those of mlxrocm_qmm and mlxrocm_qmm_rows_prepacked those of
    mlxrocm_qmm_rows, with the scratch of the plain call and without the image's share of it;
    quantized_matmul those of the entry that it takes, with an image and without."""
    lib, code = _lib.load(), CODE[dtype]
    q = _weights(N, K, bits, dtype)
    x = torch.randn((M, K), device="cuda").to(dtype)
    image = mlx_amd.quantized_matmul_sb_image(q[1], q[2], 64)
    share = -(-lib.mlxrocm_qmm_sb_image_size(N, K, 1, 64, code) // 256) * 256
    rows = bool(lib.mlxrocm_qmm_rows_supported(M, N, K, 1, 64, bits, code))
    assert rows == ((M, N, K, bits) in TABLE[:5])

    need = lib.mlxrocm_qmm_workspace_size(M, N, K, 1, 0, 64, bits, code, 1)
    plan = _lib.qmm_plan(M, N, K, bits=bits, dtype=code)[1]
    assert ("qmm_own" in plan) == ((M, N, K, bits) in TABLE[:3])
    share = share if "interleave_sb" in plan else 0
    plain = _c_call(lib.mlxrocm_qmm, x, q, None, N, bits, code, (1,), need)
    for room in (need, need - share):
        for kept in (image, None) if room == need else (image,):
            y = _c_call(lib.mlxrocm_qmm_prepacked, x, q, (kept,), N, bits, code, (1,), room)
            assert torch.equal(y, plain), (room, kept is None)
    if rows:
        need = lib.mlxrocm_qmm_rows_workspace_size(M, N, K, 1, 64, bits, code)
        share = -(-lib.mlxrocm_qmm_sb_image_size(N, K, 1, 64, code) // 256) * 256
        table, plain = plain, _c_call(lib.mlxrocm_qmm_rows, x, q, None, N, bits, code, (), need)
        assert torch.equal(table, plain) or "qmm_own" not in plan
        for room in (need, need - share):
            for kept in (image, None) if room == need else (image,):
                y = _c_call(lib.mlxrocm_qmm_rows_prepacked, x, q, (kept,), N, bits, code, (), room)
                assert torch.equal(y, plain), (room, kept is None)
    # (native host path, then the Python one)
    strided = torch.stack([x, x], dim=-1)[..., 0]
    for t in (x, strided):
        for kept in (image, None):
            y = mlx_amd.quantized_matmul(t, *q, group_size=64, bits=bits, sb_image=kept)
            assert torch.equal(y, plain), kept is None


# the smallest calls found of every height of the tiles, in one range of K and in several:
# (rows of a tile, M, N, K, ranges)
HEIGHTS = {
    3: ((64, 327, 1314, 128, 1), (64, 314, 476, 2176, 6), (96, 197, 17868, 128, 1),
        (96, 2123, 404, 2048, 4), (128, 295, 16506, 256, 1), (128, 678, 528, 8192, 13),
        (160, 706, 10790, 128, 1), (160, 262, 7404, 3072, 4), (192, 650, 13474, 256, 1),
        (192, 518, 2096, 8192, 8), (224, 770, 15378, 256, 1), (224, 1292, 1184, 8192, 8),
        (256, 1573, 8292, 384, 1), (256, 1154, 2748, 8192, 4)),
    4: ((64, 2125, 424, 128, 1), (64, 279, 552, 2176, 6), (96, 195, 16420, 128, 1),
        (96, 1888, 524, 2176, 4), (128, 300, 17312, 256, 1), (128, 2252, 532, 4096, 4),
        (160, 515, 14652, 256, 1), (160, 2945, 524, 4096, 4), (192, 515, 19196, 256, 1),
        (192, 331, 8228, 4224, 3), (224, 582, 19046, 384, 1), (224, 398, 9600, 4224, 3),
        (256, 680, 19184, 640, 1), (256, 2776, 1136, 8192, 4)),
    8: ((64, 2614, 404, 128, 1), (64, 316, 500, 2176, 6), (96, 199, 16414, 128, 1),
        (96, 1241, 532, 2176, 6), (128, 2748, 2050, 128, 1), (128, 1156, 540, 4096, 8),
        (160, 546, 13156, 256, 1), (160, 2819, 604, 2048, 4), (192, 523, 19880, 256, 1),
        (192, 526, 4492, 3072, 4), (224, 578, 19098, 256, 1), (224, 587, 6436, 3072, 3),
        (256, 1360, 9476, 384, 1), (256, 2320, 1824, 4224, 3)),
    "mxfp8": ((64, 103, 462, 128, 1), (64, 208, 412, 1024, 4), (96, 257, 13206, 128, 1),
              (96, 596, 516, 4224, 11), (128, 674, 8400, 128, 1), (128, 1169, 456, 8192, 11),
              (160, 514, 13456, 256, 1), (160, 534, 1824, 6144, 8), (192, 515, 19906, 256, 1),
              (192, 322, 9960, 3072, 3), (224, 590, 19148, 384, 1), (224, 769, 4712, 4096, 3),
              (256, 1384, 9598, 640, 1), (256, 1806, 2412, 6144, 3)),
}


@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
@pytest.mark.parametrize("codes", HEIGHTS)
def test_every_height(codes, dtype):
    """Every height of the tiles with and without K ranges, named by the plan of the call: no
    constant of the rule drops one from the tests unseen."""
    for rows, M, N, K, ranges in HEIGHTS[codes]:
        kernel = f"qmm_own(rows={rows},ksplit={ranges})"
        g = torch.Generator(device="cuda").manual_seed(M)
        x = torch.randn((M, K), generator=g, device="cuda").to(dtype)
        if codes == "mxfp8":
            assert kernel in _lib.fp_qmm_rows_plan(M, N, K, 1, _lib.MXFP8, CODE[dtype])[1]
            w = torch.randn((N, K), generator=g, device="cuda").to(dtype)
            wq, s = mlx_amd.quantize(w, mode=codes)[:2]
            y = mlx_amd.quantized_matmul(x, wq, s, None, mode=codes)
            w_hat = mlx_amd.dequantize(wq, s, None, mode=codes, dtype=dtype).double()
        else:
            assert kernel in _lib.qmm_rows_plan(M, N, K, 1, 64, codes, CODE[dtype])[1]
            wq, s, b = _weights(N, K, codes, dtype)
            y = mlx_amd.quantized_matmul(x, wq, s, b, group_size=64, bits=codes)
            w_hat = mlx_amd.dequantize(wq, torch.ones_like(s, dtype=torch.float32),
                                       torch.zeros_like(s, dtype=torch.float32), 64, codes).double()
            w_hat = w_hat.unflatten(1, (-1, 64)) * s.double()[..., None] + b.double()[..., None]
            w_hat = w_hat.flatten(1).to(dtype).double()
        _relative(y, x.double() @ w_hat.T, dtype)
