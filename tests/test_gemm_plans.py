"""The kernels and tiles the GEMM dispatch picks, evaluated on the host: the
sizes its rules were measured at, either side of each line they draw."""

import pytest

from voyager_amd import gemm


def _plan(fmt, M, N, K, batch=1, hint=0):
    """(family, tile) of ``vh_gemm`` on 16-byte aligned contiguous operands."""
    d = gemm.GemmDesc()
    size = 2 if fmt == gemm.OP_BF16 else 1
    d.A, d.B, d.C = 1 << 12, 1 << 13, 1 << 14
    d.M, d.N, d.K, d.batch = M, N, K, batch
    d.lda = d.ldb = K * size
    d.ldc = N
    d.a_fmt = d.b_fmt = fmt
    if fmt == gemm.OP_MXI8:
        d.a_scale, d.b_scale = 1 << 15, 1 << 16
        d.a_scale_ld = d.b_scale_ld = -(-K // 64) * 4
        d.a_block = d.b_block = 16
        d.a_bias = d.b_bias = 133
    d.tile_hint = hint
    d.epi.out_dtype = gemm.VH_BF16
    return gemm.plan(d)[:2]


@pytest.mark.parametrize("fmt,M,N,K,tile", [
    # a tile's own time below K = 4096 is mostly fill and store: few large tiles
    (gemm.OP_FP8, 4096, 2816, 512, 41), (gemm.OP_FP8, 3000, 8960, 256, 41), (gemm.OP_FP8, 1111, 8960, 512, 41),
    (gemm.OP_FP8, 4096, 14336, 512, 41), (gemm.OP_BF16, 1024, 14336, 256, 41), (gemm.OP_BF16, 2500, 8960, 256, 41),
    (gemm.OP_BF16, 1500, 8960, 512, 41),
    # from K = 4096 on
    (gemm.OP_FP8, 513, 4096, 4096, 33), (gemm.OP_FP8, 1111, 4096, 14336, 25), (gemm.OP_FP8, 2048, 14336, 4096, 44),
    (gemm.OP_BF16, 300, 14336, 4096, 25), (gemm.OP_BF16, 2048, 4096, 14336, 31)])
def test_direct_tiles(fmt, M, N, K, tile):
    family = gemm.FAMILY_DIRECT_FP8 if fmt == gemm.OP_FP8 else gemm.FAMILY_DIRECT_BF16
    assert _plan(fmt, M, N, K) == (family, tile)


@pytest.mark.parametrize("M,N,K,tile", [(2500, 14336, 256, 7), (8192, 8960, 512, 7), (4096, 8960, 256, 7),
                                        (1111, 4096, 14336, 5), (2048, 4096, 4096, 3), (2048, 14336, 4096, 7)])
def test_fp16_row_tiles(M, N, K, tile):
    assert gemm.mx8_f16_plan(M, N, K) == (tile, 1)
