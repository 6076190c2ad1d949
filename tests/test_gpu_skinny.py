"""GEMMs of at most 64 rows (``k_skinny``) and the lowered linears that
quantize at most 8 rows in the same launch: at the edges of the row tiles
(16, 32, 64), of the weight tiles (16 rows; 1, 2 or 4 of them a workgroup) and
of K (one chunk, part of a group, fewer groups than waves, several groups a
wave and part of one), against the exact product of the decoded operands and,
bit for bit, one launch against two."""

import pytest
import torch

import voyager_amd.library  # noqa: F401  (defines quantized_ops)
from helpers import assert_same_bits, max_rel_err
from voyager_amd import formats, gemm, lower, packed

pytestmark = pytest.mark.gpu

# (M, N, K): N around 16 and past one and two rounds of 256 tiles
SHAPES = [(1, 16, 16), (3, 40, 528), (4, 1000, 4096), (8, 4104, 272), (16, 8200, 1040), (17, 100, 4096),
          (32, 4112, 64), (33, 1048, 2064), (64, 8192, 512), (5, 14336, 320)]
# MX-int8 decodes in the kernel and holds scales beside the codes: every row
# tile and weight tile with several groups a wave and part of one at the end
MX_SHAPES = [s for s in SHAPES if s[2] % 64 == 0] + [
    (3, 4112, 4160), (7, 1000, 4160), (8, 4104, 4160), (16, 4112, 4160), (16, 8200, 4160), (17, 1000, 4160),
    (32, 4112, 4160), (32, 8208, 4160), (33, 1048, 4032), (64, 4096, 4032)]


def _inputs(M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g)
    x[M // 2, : K // 2] = 0.0                # blocks of zeros
    x[M - 1, 0] = 1e30                       # saturates E4M3, a huge block
    if M > 1:
        x[0, -16:] = 1e-39                   # a subnormal block
    w = torch.randn(N, K, generator=g) * 0.02
    return x.bfloat16().cuda(), w.bfloat16().cuda()


def _log(call):
    gemm.plan_log = log = []
    try:
        return call(), log
    finally:
        gemm.plan_log = None


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_skinny_fp8(M, N, K):
    x, w = _inputs(M, N, K)
    tab = formats.quantization_map("fp8_e4m3")
    sx = torch.tensor(0.013, dtype=torch.bfloat16, device="cuda")
    xq, wq = packed.quantize_packed(x, sx, tab), packed.quantize_packed(w, sx, tab)
    y, log = _log(lambda: gemm.linear_fp8(xq, wq, sx, tile_hint=gemm.TILE_SKINNY))
    assert [p[0] for p in log] == [gemm.FAMILY_SKINNY]
    vx, vw = packed.unpack_codes(xq, tab).double(), packed.unpack_codes(wq, tab).double()
    # the FP8 MFMA rounds the products it adds at once to a common grid (3.2e-4
    # of the sum of their magnitudes at worst, the same as the tiled kernels');
    # then bf16(bf16(acc) * s), two roundings of half an ulp (2**-8) each
    exp = vx @ vw.T * sx.double()
    room = vx.abs() @ vw.abs().T * sx.double() * 2.0**-11 + exp.abs() * 2.0**-7
    assert ((y.double() - exp).abs() <= room).all()
    one = lower.lowered_fp8_linear(x, sx, tab, wq, sx)
    assert torch.equal(one, y if M <= 8 else gemm.linear_fp8(xq, wq, sx))


@pytest.mark.parametrize("M,N,K", MX_SHAPES)
def test_skinny_mxint8(M, N, K):
    x, w = _inputs(M, N, K)
    tab = formats.quantization_map("int8")
    px, pw = (packed.quantize_mx_packed(t, tab, [-1], 16, 127.0, True) for t in (x, w))

    def value(p):
        s = torch.ldexp(torch.ones_like(p.scale, dtype=torch.float64), p.scale.to(torch.int32) - p.bias)
        return p.codes.view(torch.int8).double() * s.repeat_interleave(16, 1)

    args = (px.codes, px.scale, pw.codes, pw.scale, 16, px.bias, pw.bias)
    alpha, bias = torch.tensor(0.75, device="cuda"), torch.randn(N, device="cuda").bfloat16()
    y, log = _log(lambda: gemm.linear_mxint8(*args, out_dtype=torch.float32, bias=bias, alpha=alpha,
                                             tile_hint=gemm.TILE_SKINNY))
    assert [p[0] for p in log] == [gemm.FAMILY_SKINNY]
    ref = value(px) @ value(pw).T * 0.75 + bias.double()
    # exact products; float32 sums of K terms, each rounded
    room = value(px).abs() @ value(pw).abs().T * 0.75 * K * 2.0**-24 + ref.abs() * 2.0**-22
    assert ((y.double() - ref).abs() <= room).all()
    assert torch.equal(lower.lowered_mxint8_linear(x, tab, pw.codes, pw.scale, pw.bias, 16, bias),
                       gemm.linear_mxint8(*args, bias=bias, tile_hint=gemm.TILE_SKINNY if M <= 8 else 0))


@pytest.mark.parametrize("M,N,K", [(3, 40, 528), (8, 4104, 4160), (20, 100, 4112), (33, 56, 1040)])
def test_skinny_mxint8_padded_rows(M, N, K):
    """Codes and scale bytes as columns of wider tensors, the scale views
    ending where their storage does (or one to three bytes before, as their
    rows are 4-byte aligned): the contiguous operands' bits, also where a
    group's scales go past the row's end and hold the next row's."""
    x, w = _inputs(M, N, K)
    tab = formats.quantization_map("int8")
    px, pw = (packed.quantize_mx_packed(t, tab, [-1], 16, 127.0, True) for t in (x, w))

    def padded(t, at, unit):
        pitch = -(-(at + t.shape[1]) // unit) * unit
        wide = torch.full((t.shape[0], pitch), 0x7f, dtype=t.dtype, device="cuda")
        view = wide[:, at:at + t.shape[1]]
        view.copy_(t)
        return view

    flat = gemm.linear_mxint8(px.codes, px.scale, pw.codes, pw.scale, 16, px.bias, pw.bias)
    args = [f(p) for p in (px, pw) for f in (lambda p: padded(p.codes, 16, 16), lambda p: padded(p.scale, 4, 4))]
    y, log = _log(lambda: gemm.linear_mxint8(*args, 16, px.bias, pw.bias))
    assert [p[0] for p in log] == [gemm.FAMILY_SKINNY]
    assert_same_bits(y, flat)
    if M <= 8:
        one = lower.lowered_mxint8_linear(x, tab, args[2], args[3], pw.bias, 16)
        assert_same_bits(one, flat)


@pytest.mark.parametrize("M,N,K", [s for s in SHAPES if s[2] % 8 == 0] + [(2, 7, 24)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_skinny_bf16(M, N, K, out_dtype):
    x, w = _inputs(M, N, K)
    x = x.clamp(-10, 10)
    y, log = _log(lambda: gemm.gemm_bf16(x, w, out_dtype, tile_hint=gemm.TILE_SKINNY))
    assert [p[0] for p in log] == [gemm.FAMILY_SKINNY]
    ref = x.double() @ w.double().T
    room = 2.0**-8 if out_dtype == torch.bfloat16 else 1e-5
    assert max_rel_err(y, ref) < room
    assert max_rel_err(torch.ops.quantized_ops.linear(x, w, out_dtype=out_dtype), ref) < room
    # a batch of products, the rows' tiles of each its own
    xb, wb = torch.stack([x, 2 * x]), torch.stack([w, w * 0.5])
    yb, log = _log(lambda: gemm.gemm_bf16(xb, wb, out_dtype, tile_hint=gemm.TILE_SKINNY))
    assert [p[0] for p in log] == [gemm.FAMILY_SKINNY]
    assert max_rel_err(yb, torch.stack([ref, ref])) < room
    yb = torch.ops.quantized_ops.matmul(xb, wb, layout="xc,kc->xk", out_dtype=out_dtype)
    assert max_rel_err(yb, torch.stack([ref, ref])) < room


def test_skinny_hint_past_its_rows():
    """A hint for the few-row kernel runs the tiles where it cannot."""
    x, w = _inputs(65, 136, 320)
    x = x.clamp(-8, 8)
    y, log = _log(lambda: gemm.gemm_bf16(x, w, torch.float32, tile_hint=gemm.TILE_SKINNY))
    assert [p[0] for p in log] == [gemm.FAMILY_STAGED]
    assert max_rel_err(y, x.double() @ w.double().T) < 1e-5


def test_rows8_nan_and_infinity():
    """Values the fast quotients do not decide: NaN, infinities, quotients on
    a bf16 rounding midpoint, in one launch as in two."""
    x, w = _inputs(8, 64, 512)
    x[0, 5], x[1, 7], x[2, 9] = float("nan"), float("inf"), float("-inf")
    x[3] = torch.arange(512, device="cuda").bfloat16()
    tab8, tabf = formats.quantization_map("int8"), formats.quantization_map("fp8_e4m3")
    pw = packed.quantize_mx_packed(w, tab8, [-1], 16, 127.0, True)
    px = packed.quantize_mx_packed(x, tab8, [-1], 16, 127.0, True)
    two = gemm.linear_mxint8(px.codes, px.scale, pw.codes, pw.scale, 16, px.bias, pw.bias)
    assert torch.equal(lower.lowered_mxint8_linear(x, tab8, pw.codes, pw.scale, pw.bias, 16), two)
    for s in (0.013, 3.0, 2.0**-130):
        sx = torch.tensor(s, dtype=torch.bfloat16, device="cuda")
        wq = packed.quantize_packed(w, torch.tensor(0.013, dtype=torch.bfloat16, device="cuda"), tabf)
        two = gemm.linear_fp8(packed.quantize_packed(x, sx, tabf), wq, sx)
        one = lower.lowered_fp8_linear(x, sx, tabf, wq, sx)
        assert torch.equal(one.nan_to_num(12345.0), two.nan_to_num(12345.0)) and one.isnan().any()


@pytest.mark.parametrize("rows", [4, 16])
def test_fp8_scale_of_more_dims_is_refused(rows):
    """A scale with more dimensions than the activation's rows does not
    broadcast to them, however many rows there are."""
    x, w = torch.zeros(rows, 64).bfloat16().cuda(), torch.zeros(32, 64, dtype=torch.uint8, device="cuda")
    scale = torch.ones(1, 1, 1, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ValueError, match="more dims"):
        lower.lowered_fp8_linear(x, scale, formats.quantization_map("fp8_e4m3"), w, scale.reshape(()))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_rows8_scale_dtypes(dtype):
    """The E4M3 linear of at most 8 rows under a scale of its own precision:
    the codes of ``quantize``, whose quotient takes the scale as it is."""
    x, w = _inputs(7, 48, 1040)
    tab = formats.quantization_map("fp8_e4m3")
    sx, one = torch.tensor(0.0137, dtype=dtype, device="cuda"), torch.ones((), dtype=torch.bfloat16, device="cuda")
    wq = packed.quantize_packed(w, torch.tensor(0.013, dtype=torch.bfloat16, device="cuda"), tab)
    two = gemm.linear_fp8(packed.quantize_packed(x, sx, tab), wq, one, tile_hint=gemm.TILE_SKINNY)
    assert torch.equal(gemm.linear_fp8_rows8(x, sx, wq, one), two)
