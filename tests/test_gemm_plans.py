"""The kernels and tiles the GEMM dispatch picks, evaluated on the host: the
sizes its rules were measured at, either side of each line they draw."""

import ctypes

import pytest

from voyager_amd import gemm, lower
from voyager_amd._lib import load


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
    (gemm.OP_BF16, 300, 14336, 4096, 25), (gemm.OP_BF16, 2048, 4096, 14336, 31),
    # many tiles of 256 x 256 are not the fastest
    (gemm.OP_BF16, 2048, 14336, 4096, 26), (gemm.OP_BF16, 3000, 8192, 3072, 31), (gemm.OP_BF16, 4096, 8960, 14336, 26)])
def test_direct_tiles(fmt, M, N, K, tile):
    family = gemm.FAMILY_DIRECT_FP8 if fmt == gemm.OP_FP8 else gemm.FAMILY_DIRECT_BF16
    assert _plan(fmt, M, N, K) == (family, tile)


@pytest.mark.parametrize("batch,M,N,K", [(256, 17, 1024, 128), (256, 65, 1024, 64), (32, 17, 4096, 64),
                                         (256, 128, 512, 128)])
def test_direct_tiles_short_batches(batch, M, N, K):
    assert _plan(gemm.OP_BF16, M, N, K, batch)[1] == 41


@pytest.mark.parametrize("M,N,K,tile", [(2500, 14336, 256, 7), (8192, 8960, 512, 7), (4096, 8960, 256, 7),
                                        (1111, 4096, 14336, 5), (2048, 4096, 4096, 3), (2048, 14336, 4096, 7)])
def test_fp16_row_tiles(M, N, K, tile):
    assert gemm.mx8_f16_plan(M, N, K) == (tile, 1)


# (rows, N, K, batch): the few-row kernel or the tiles
FEW_ROWS = {
    gemm.OP_BF16: {True: [(1, 4096, 64, 1), (64, 4096, 64, 1), (16, 8192, 128, 1), (32, 8192, 2048, 1),
                          (64, 8192, 2048, 1), (16, 14336, 2048, 1), (32, 14336, 4096, 1), (16, 32768, 4096, 1), (16, 512, 512, 8),
                          (17, 256, 128, 8), (64, 128, 128, 8), (32, 1024, 4096, 32), (33, 1024, 2048, 4)],
                   False: [(32, 8192, 128, 1), (64, 8192, 512, 1), (1, 14336, 512, 1), (64, 14336, 4096, 1),
                           (1, 32768, 1024, 1), (16, 20480, 4096, 1), (65, 4096, 4096, 1), (1, 4096, 128, 256),
                           (16, 1024, 128, 256), (32, 1024, 512, 32), (32, 512, 128, 8), (64, 64, 2048, 64)]},
    gemm.OP_FP8: {True: [(1, 4096, 64, 1), (64, 4096, 512, 1), (16, 8192, 512, 1), (32, 14336, 4096, 1)],
                  False: [(32, 8192, 512, 1), (1, 14336, 1024, 1), (64, 14336, 4096, 1), (1, 20480, 4096, 1),
                          (16, 32768, 14336, 1)]},
    gemm.OP_MXI8: {True: [(16, 4096, 128, 1), (32, 14336, 256, 1), (64, 4096, 4096, 1), (1, 65536, 256, 1),
                          (1, 28672, 1024, 1)],
                   False: [(16, 4096, 64, 1), (17, 4096, 128, 1), (64, 4112, 4096, 1), (1, 28672, 576, 1)]},
}


@pytest.mark.parametrize("fmt,few,M,N,K,batch", [(f, few) + c for f, d in FEW_ROWS.items() for few, cs in d.items()
                                                 for c in cs])
def test_few_rows(fmt, few, M, N, K, batch):
    assert (_plan(fmt, M, N, K, batch)[0] == gemm.FAMILY_SKINNY) == few
    if M <= 64:
        assert _plan(fmt, M, N, K, batch, gemm.TILE_SKINNY)[0] == gemm.FAMILY_SKINNY
    else:  # as any hint that names no tile of its own
        assert _plan(fmt, M, N, K, batch, gemm.TILE_SKINNY) == (gemm.FAMILY_STAGED, 4)


@pytest.mark.parametrize("fmt", [gemm.OP_BF16, gemm.OP_FP8, gemm.OP_MXI8])
@pytest.mark.parametrize("M,N", [(0, 64), (4, 0), (0, 0)])
def test_empty_products(fmt, M, N):
    _plan(fmt, M, N, 64)
    _plan(fmt, M, N, 64, 3)


@pytest.mark.parametrize("M,N,K", [(17, 1536, 8960), (256, 1536, 8960), (201, 1280, 4096), (300, 3072, 4096),
                                   (512, 2816, 4096), (64, 8960, 512), (400, 4608, 2048), (256, 4096, 4096)])
def test_nf4_splits_fill_one_round(M, N, K):
    """As many K ranges as one round of 256 workgroups takes, and no more."""
    sp = ctypes.c_int32(0)
    assert load().vh_gemm_nf4_bf16_plan(M, N, K, ctypes.byref(sp)) == 0
    tiles, blocks = -(-M // 256) * -(-N // 64), K // 64
    most = max(1, min(256 // tiles, blocks // 4))
    assert tiles * sp.value <= 256
    assert sp.value == -(-blocks // -(-blocks // most))  # ranges of whole blocks


# (M, N, K): two passes, or the weight decoded in the GEMM
TWO_PASS = {True: [(512, 4096, 1024), (511, 4096, 4096), (700, 4096, 4096), (400, 14336, 4096), (1000, 1024, 4096),
                   (1025, 512, 14336), (300, 8960, 2048)],
            False: [(17, 14336, 4096), (256, 4096, 14336), (300, 4096, 4096), (300, 14336, 4096), (511, 4096, 14336),
                    (512, 1024, 4096), (700, 1024, 14336), (300, 8192, 1024), (300, 14336, 512), (300, 1024, 64)]}


@pytest.mark.parametrize("two,M,N,K", [(t,) + c for t, cs in TWO_PASS.items() for c in cs])
def test_nf4_two_pass(two, M, N, K):
    assert gemm.nf4_two_pass_pays(M, N, K) == two


# (M, N, K) of few blocks of K: the fastest of the three forms
SHORT = {gemm.NF4_TWO_PASS: [(600, 4608, 64), (256, 256, 256), (201, 4096, 512), (769, 4096, 128), (288, 16400, 1024)],
         gemm.NF4_FUSED: [(256, 4096, 64), (64, 32768, 256), (201, 32768, 512), (256, 24576, 1024), (400, 7168, 256)],
         gemm.NF4_BF16: [(160, 11008, 512), (17, 32768, 512), (64, 24576, 1024), (201, 14336, 4096)]}


@pytest.mark.parametrize("route,M,N,K", [(r,) + c for r, cs in SHORT.items() for c in cs])
def test_nf4_route(route, M, N, K):
    assert load().vh_gemm_nf4_route(M, N, K) == route


@pytest.mark.parametrize("N,full", [(64, True), (16384, True), (16400, False), (20480, False), (28672, False),
                                    (32768, True), (32832, False), (65536, True), (128256, True)])
def test_one_launch_rounds(N, full):
    """The E4M3 linear that quantizes its rows in the launch: not where a
    round of its workgroups would be mostly empty."""
    assert lower._full_rounds(N) == full
