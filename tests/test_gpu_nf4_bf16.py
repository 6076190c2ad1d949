"""The MXNF4 linear of an activation decoded to bf16 (``vh_gemm_nf4_bf16``)
and the quantize that writes it (``vh_nf4_quantize_bf16``)."""
import pytest
import torch

import voyager_amd.library  # noqa: F401  (defines quantized_ops)
from helpers import assert_same_bits
from oracle import tables as T

pytestmark = pytest.mark.gpu


def _maps():
    vt = T.quantization_map("lut4_to_int6")
    index, entries, _ = T.codebook_index_table(vt)
    return index.cuda(), entries.cuda(), T.quantization_map("fp8_e5m3").cuda()


@pytest.mark.parametrize("M,K,N,splits", [
    (1, 64, 16, 0), (17, 64, 16, 0), (32, 192, 80, 0), (33, 4160, 48, 7), (64, 4096, 1024, 0), (65, 640, 208, 3),
    (96, 128, 112, 0), (97, 576, 1040, 0), (128, 320, 64, 0), (129, 4160, 48, 0), (160, 256, 272, 1),
    (161, 64, 144, 0), (193, 448, 528, 2), (201, 4096, 2064, 0), (225, 704, 64, 11), (256, 16448, 32, 1),
    (257, 384, 336, 0), (511, 1088, 96, 0)])
def test_gemm_nf4_bf16(M, K, N, splits):
    """Every row tile's edges, ragged columns, odd block counts and K ranges,
    against the float64 product of the operands ``nf4_decode_bf16`` gives:
    products of two bf16 are exact in float32, so a sum of K of them in any
    order is within K 2^-24 of their magnitudes' sum (and a bf16 result
    within half an ulp more)."""
    from voyager_amd import gemm, packed

    index, entries, stab = _maps()
    g = torch.Generator().manual_seed(M * 7 + K + N)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    w = (torch.randn(N, K, generator=g) * 0.02).bfloat16().cuda()
    wb = gemm.bake_nf4_weight(w, index, stab, entries)
    px = packed.quantize_mx_packed(x, index, [-1], 64, 31.0, False, stab)
    xo, wo = gemm.nf4_decode_bf16(px, wb)
    xd, wd = xo.cpu().double(), wo.cpu().double()
    bias = torch.randn(N, generator=g).bfloat16()
    ref = (xd @ wd.T) * 0.75 + bias.double()
    bound = K * 2.0**-24 * (xd.abs() @ wd.abs().T) + 2.0**-22 * ref.abs() + 2.0**-23 * bias.double().abs()
    alpha = torch.tensor(0.75, device="cuda")
    for dt, ulp in ((torch.float32, 0.0), (torch.bfloat16, 2.0**-8)):
        y = gemm.gemm_nf4_bf16(xo, wb, dt, bias.cuda(), alpha, splits).cpu().double()
        assert ((y - ref).abs() <= bound + ulp * ref.abs()).all()


@pytest.mark.parametrize("M,K", [(1, 64), (19, 192), (130, 4160), (1, 14336)])
def test_nf4_quantize_bf16(M, K):
    """Bit for bit quantize_mx to codes and their decode, with blocks of
    zeros, tiny, huge, infinite and NaN values."""
    from voyager_amd import formats, gemm, packed

    index, entries, stab = _maps()
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn(M, K, generator=g).bfloat16()
    x *= (2.0 ** torch.randint(-60, 60, (M, K // 64, 1), generator=g)).bfloat16().expand(M, K // 64, 64).reshape(M, K)
    x[0, :64] = 0
    x[-1, 3] = float("nan")
    x[M // 2, K - 1] = float("inf")
    x[M // 2, K - 64] = -float("inf")
    x = x.cuda()
    wb = gemm.bake_nf4_weight(torch.randn(16, K, generator=g).bfloat16().cuda(), index, stab, entries)
    px = packed.quantize_mx_packed(x, index, [-1], 64, 31.0, False, stab)
    xo, _ = gemm.nf4_decode_bf16(px, wb, decode_w=False)
    got = gemm.nf4_quantize_bf16(x, wb, formats.classify(index), formats.classify(stab))
    assert_same_bits(got, xo)


@pytest.mark.parametrize("form", ["plain", "misaligned", "strided", "transposed", "float32", "float16"])
@pytest.mark.parametrize("M,K,N", [(17, 4096, 2064), (190, 1088, 4112), (320, 640, 2048), (300, 704, 2064)])
def test_linear_nf4_routes(form, M, K, N):
    """Every form of activation ``linear_nf4`` takes above 16 rows, on the
    route it chooses, against the fused kernel (the bound of
    ``test_gemm_nf4_bf16`` for each of the two sums), eagerly and from a
    replayed graph."""
    from voyager_amd import gemm, packed

    index, entries, stab = _maps()
    g = torch.Generator().manual_seed(M + K + N)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    w = (torch.randn(N, K, generator=g) * 0.02).bfloat16().cuda()
    if form == "misaligned":
        x = torch.cat([x.new_zeros(1), x.reshape(-1)])[1:].view(M, K)
        assert x.data_ptr() % 16
    elif form == "strided":
        x = torch.stack([x, x], 2).reshape(M, 2 * K)[:, ::2]
    elif form == "transposed":
        x = x.t().contiguous().t()
    elif form != "plain":
        x = x.to(getattr(torch, form))
    wb = gemm.bake_nf4_weight(w, index, stab, entries)
    px = packed.quantize_mx_packed(x.contiguous(), index, [-1], 64, 31.0, False, stab)
    xo, wo = gemm.nf4_decode_bf16(px, wb)
    bound = 2 * K * 2.0**-24 * (xo.double().abs() @ wo.double().abs().T)
    ref = gemm.linear_nf4_prefill(x, wb, index, stab, torch.float32, tile=1, two_pass=False)

    def call():
        return gemm.linear_nf4(x, wb, index, stab, torch.float32)

    got = call()
    assert ((got - ref).double().abs() <= bound).all()
    assert torch.equal(gemm.gemm_nf4_packed(px, wb, torch.float32), got)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, call())


@pytest.mark.parametrize("M,K,N", [(201, 256, 1040), (600, 512, 272)])
def test_given_tile_runs_the_fused_kernel(M, K, N):
    """Where two passes are the choice, a given tile or split still runs
    ``vh_gemm_nf4`` at it."""
    from voyager_amd import gemm, packed

    index, entries, stab = _maps()
    g = torch.Generator().manual_seed(M + K + N)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    wb = gemm.bake_nf4_weight((torch.randn(N, K, generator=g) * 0.02).bfloat16().cuda(), index, stab, entries)
    assert gemm.nf4_two_pass_pays(M, N, K)
    px = packed.quantize_mx_packed(x, index, [-1], 64, 31.0, False, stab)
    for tile, splits in ((1, 1), (2, 0), (0, 2)):
        ref = gemm.linear_nf4_prefill(x, wb, index, stab, torch.float32, tile=tile, splits=splits, two_pass=False)
        assert torch.equal(gemm.gemm_nf4_packed(px, wb, torch.float32, tile=tile, splits=splits), ref)
        assert torch.equal(gemm.linear_nf4_prefill(x, wb, index, stab, torch.float32, tile=tile, splits=splits), ref)
