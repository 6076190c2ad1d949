"""The direct-to-LDS GEMM tiles that fill ragged grids (128x192, 256x160, and
256x256 for fp16 rows), the tile choice's own routes, and the MX-int8 linear
whose activation is quantized straight to fp16 rows."""
import pytest
import torch

import voyager_amd.library  # noqa: F401  (defines quantized_ops)
from helpers import assert_same_bits
from oracle import tables as T
from voyager_amd import gemm, packed

pytestmark = pytest.mark.gpu

# edges of the tiles and tile counts of every remainder by 8 (the XCD ranges)
SIZES = [(65, 200, 1040), (129, 1928, 144), (257, 328, 528), (300, 2600, 272), (513, 1160, 96), (385, 968, 2064)]


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("fmt", ["fp8", "bf16"])
def test_ragged_tiles(fmt, M, N, K):
    """Every tile adds a result's products in the same order, so the new ones
    and the chosen one give the bits of tile 33 (checked against the oracle
    elsewhere), with alpha and bias, bf16 and float32."""
    g = torch.Generator().manual_seed(M + N + K)
    a, b = torch.randn(M, K, generator=g).cuda(), (torch.randn(N, K, generator=g) * 0.1).cuda()
    bias = torch.randn(N, generator=g).bfloat16().cuda()
    alpha = torch.tensor(0.75, device="cuda")
    if fmt == "fp8":
        a, b = (t.to(torch.float8_e4m3fn).view(torch.uint8) for t in (a, b))
    else:
        a, b = a.bfloat16(), b.bfloat16()
    for dt in (torch.bfloat16, torch.float32):
        outs = []
        for hint in (33, 25, 26, 0):
            out = torch.empty(M, N, dtype=dt, device="cuda")
            d = gemm.GemmDesc()
            d.A, d.B, d.C = a.data_ptr(), b.data_ptr(), out.data_ptr()
            d.M, d.N, d.K = M, N, K
            d.lda, d.ldb, d.ldc = K * a.element_size(), K * a.element_size(), N
            d.a_fmt = d.b_fmt = gemm.OP_FP8 if fmt == "fp8" else gemm.OP_BF16
            d.tile_hint = hint
            d.epi = gemm._epilogue(gemm.EPI_PLAIN, dt, alpha, bias)
            gemm.run(d, a.device)
            outs.append(out)
        assert all(torch.equal(outs[0], o) for o in outs[1:])


@pytest.mark.parametrize("M,N,K", SIZES)
def test_mx8_f16_ragged_tiles(M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    w = (torch.randn(N, K, generator=g) * 0.1).bfloat16().cuda()
    tab = T.quantization_map("int8").cuda()
    pw = packed.quantize_mx_packed(w, tab, [-1], 16, 127.0, True)
    bw = gemm.bake_mx8_f16(pw.codes.view(torch.int8), pw.scale, pw.bias)
    x16, ex = gemm.quantize_mx8_f16(x)
    ref = gemm.linear_mx8_f16(x16, ex, bw, tile=0, splits=1)
    for tile in (5, 6, 7):
        assert torch.equal(gemm.linear_mx8_f16(x16, ex, bw, tile=tile, splits=1), ref)


@pytest.mark.parametrize("M,N,K", [(1024, 4096, 8192), (1111, 2064, 16384), (1500, 4096, 6160)])
def test_lowered_mxint8_two_pass(M, N, K):
    """The lowered linear's fp16 rows are the values its packed codes rebase
    to (blocks of zeros, tiny, huge, infinite and NaN values; a code has no
    negative zero, and a zero's sign does not enter a sum), and its result is
    theirs bit for bit."""
    from voyager_amd import lower

    assert gemm.mxint8_two_pass_pays(M, N, K)
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).bfloat16()
    x[3, :32] = 0
    x[5] *= 2.0**-120
    x[7, 16:32] *= 2.0**100
    x[9, 5] = float("inf")
    x[11, 40] = float("nan")
    x[13, :16] *= 2.0**-30
    x = x.cuda()
    w = (torch.randn(N, K, generator=g) * 0.1).bfloat16().cuda()
    bias = torch.randn(N, generator=g).bfloat16().cuda()
    tab = T.quantization_map("int8").cuda()
    pw = packed.quantize_mx_packed(w, tab, [-1], 16, 127.0, True)
    px = packed.quantize_mx_packed(x, tab, [-1], 16, 127.0, True)
    bx = gemm.bake_mx8_f16(px.codes.view(torch.int8), px.scale, px.bias)
    x16, ex = gemm.quantize_mx8_f16(x, as_codes=True)
    assert ((x16 == bx.w) | (x16.isnan() & bx.w.isnan())).all() and torch.equal(ex, bx.e)
    got = lower.lowered_mxint8_linear(x, tab, pw.codes, pw.scale, pw.bias, 16, bias)
    exp = gemm.linear_mxint8(px.codes, px.scale, pw.codes, pw.scale, 16, px.bias, pw.bias, bias=bias)
    assert_same_bits(got, exp)
