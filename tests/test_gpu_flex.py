"""The register-staged tiles (csrc/flex_tile.hpp): int8 and bf16 GEMM and conv for every shape,
stride and alignment the pipelined kernels do not take, with K split over
workgroups where tiles are few.  Sizes at the edges of the tiles (16 x 128,
64 x 64, 128 x 128), of the 16-byte chunks and of the 256-byte stages; each call
is repeated, since a split leaves its arrival counters for the next launch."""
import numpy as np
import pytest

import aiehlc_amd as mi
import oracle
from aiehlc_amd import synth
from hip_capture import Capture

pytestmark = pytest.mark.gpu


def _i8(rng, *shape):
    return rng.integers(-128, 128, size=shape, dtype=np.int8)


# K at the edges of the short tile's 64-byte stages, of which it takes three
SHORT_K = [(M, N, K) for K in (16, 31, 63, 64, 65, 127, 128, 129, 191, 192, 193)
           for M, N in ((1, 17), (65, 63), (64, 130), (700, 40))]

GEMM_SHAPES = [
    # M, N, K
    (1, 16, 16),      # the smallest that runs here: one chunk of one row
    (1, 17, 17),      # one byte past a chunk in k and in columns
    (3, 127, 31),     # a skinny tile one column short
    (16, 129, 255),   # ... and one column over, one byte short of a stage
    (17, 64, 256),    # one row past the skinny tile, whole stages
    (63, 65, 257),    # the 64 x 64 tile, one short and one over
    (64, 64, 100),
    (130, 70, 515),   # three stages, the last of 3 bytes
    (5, 40, 4099),    # one tile, 17 stages: split over many workgroups
    (70, 300, 2050),  # ten tiles, split
    (300, 700, 200),
    (1100, 1030, 330),  # more tiles than CUs
    (2500, 2300, 70),   # large enough for the 128 x 128 tile
    (60, 2100, 520),  # one row of 64 x 64 tiles, 33: two paired groups of 16 and one alone
    (9, 33, 65600),   # K >= 2^16: the requant form without the rounding add
]


@pytest.mark.parametrize("M,N,K", GEMM_SHAPES + SHORT_K)
@pytest.mark.parametrize("layout", [mi.B_NN, mi.B_NT])
def test_gemm_i8_flex(ctx, M, N, K, layout):
    print(f"[case] flex gemm {M}x{N}x{K} layout {layout} plan {ctx.plan_gemm_i8(M, N, K)}", flush=True)
    rng = np.random.default_rng(M + 3 * N + 5 * K + layout)
    A = _i8(rng, M, K)
    B = _i8(rng, N, K) if layout == mi.B_NT else _i8(rng, K, N)
    Co = oracle.gemm_i8(A, B, b_nt=layout == mi.B_NT)
    shift = 10
    dA, dB = ctx.upload(A), ctx.upload(B)
    dY, dC, dY2 = ctx.empty((M, N), np.int8), ctx.empty((M, N), np.int32), ctx.empty((M, N), np.int8)
    for rep in range(3):
        ctx.copy_h2d(dY, np.full((M, N), 77, np.int8))
        ctx.copy_h2d(dC, np.full((M, N), 77, np.int32))
        ctx.gemm_i8_rq(dA, dB, dY, M, N, K, shift, rep == 1, dC, layout)
        ctx.gemm_i8_rq(dA, dB, dY2, M, N, K, 0, False, None, layout)
        ctx.wait(60_000)
        assert np.array_equal(ctx.download(dC), Co), rep
        assert np.array_equal(ctx.download(dY), oracle.requant(Co, shift, relu=rep == 1)), rep
        assert np.array_equal(ctx.download(dY2), oracle.requant(Co, 0)), rep
    for b in (dA, dB, dY, dC, dY2):
        b.free()


@pytest.mark.parametrize("M,N,K,layout", [(128, 128, 8192, mi.B_NT), (130, 256, 5120, mi.B_NN)])
def test_gemm_i8_flex_in_place_of_few_pipelined_tiles(ctx, M, N, K, layout):
    """Shapes the 128x128 pipelined kernel takes, over a K long enough that
    the split is the plan (in one part they would be a quarter of the CUs)."""
    plan = ctx.plan_gemm_i8(M, N, K)
    assert plan["kernel"] == mi.KERNEL_TILE64 and plan["workgroups"] > -(-M // 64) * -(-N // 64), plan
    test_gemm_i8_flex(ctx, M, N, K, layout)


# Splits of each tile (they differ in the size of a tile's slot and in how many
# partial sums are in flight): M, N, K, CUs planned for (0: the device's), tile,
# least splits.  bf16 has the same plan at half the K.
SPLITS = [
    (70, 300, 2050, 0, (16, 128), 2),
    (67, 111, 1414, 8, (64, 64), 2),
    (260, 1300, 2600, 0, (64, 64), 4),
    (300, 400, 4100, 0, (64, 64), 6),
    (70, 513, 2326, 8, (128, 128), 3),
    (195, 4201, 3415, 0, (128, 128), 3),
]


def _planned_split(ctx, M, N, K, cus, tile, splits):
    plan = ctx.plan_gemm_i8(M, N, K)
    tiles = -(-M // tile[0]) * -(-N // tile[1])
    assert (plan["tile_m"], plan["tile_n"]) == tile and plan["workgroups"] >= splits * tiles, plan


@pytest.mark.parametrize("M,N,K,cus,tile,splits", SPLITS)
@pytest.mark.parametrize("layout", [mi.B_NN, mi.B_NT])
def test_gemm_i8_flex_splits_of_each_tile(ctx, M, N, K, cus, tile, splits, layout):
    prev = ctx.plan_set_cus(cus or 256)
    try:
        _planned_split(ctx, M, N, K, cus, tile, splits)
        test_gemm_i8_flex(ctx, M, N, K, layout)
    finally:
        ctx.plan_set_cus(prev)


@pytest.mark.parametrize("M,N,K,layout", [(5, 40, 1000, mi.B_NN), (70, 90, 300, mi.B_NT), (130, 150, 48, mi.B_NN),
                                          (33, 100, 2100, mi.B_NT)])
@pytest.mark.parametrize("off", [1, 3, 8])
def test_gemm_i8_flex_strided_unaligned(ctx, M, N, K, layout, off):
    """Operands at byte offset `off` with padded rows, exactly as long as the
    entry point says (the last row has no padding), results strided too and
    the padding between result rows left alone."""
    lda, ldb, ldc = K + off, (K if layout == mi.B_NT else N) + 2 * off, N + off
    rows_b = N if layout == mi.B_NT else K
    cols_b = K if layout == mi.B_NT else N
    rng = np.random.default_rng(M + N + K + off)
    A, B = _i8(rng, M, K), _i8(rng, rows_b, cols_b)
    bufA = _i8(rng, off + (M - 1) * lda + K)
    bufB = _i8(rng, off + (rows_b - 1) * ldb + cols_b)
    for m in range(M):
        bufA[off + m * lda: off + m * lda + K] = A[m]
    for r in range(rows_b):
        bufB[off + r * ldb: off + r * ldb + cols_b] = B[r]
    dA, dB = ctx.upload(bufA), ctx.upload(bufB)
    sentinel = np.full(1 + (M - 1) * ldc + N, -5, np.int32)  # C at a 4-byte offset
    dC = ctx.upload(sentinel)
    ctx.gemm_i8_i32(dA.ptr + off, dB.ptr + off, dC.ptr + 4, M, N, K, lda, ldb, ldc, layout)
    ctx.wait(60_000)
    got = ctx.download(dC)
    want = sentinel.copy()
    Co = oracle.gemm_i8(A, B, b_nt=layout == mi.B_NT)
    for m in range(M):
        want[1 + m * ldc: 1 + m * ldc + N] = Co[m]
    assert np.array_equal(got, want)
    for b in (dA, dB, dC):
        b.free()


def test_gemm_i8_flex_recorded(ctx):
    """Split products in a recorded chain (they share the context's workspace
    and counters), replayed with eager calls between the replays."""
    M, N, K, K2 = 7, 300, 3000, 1111
    rng = np.random.default_rng(5)
    A, B, B2 = _i8(rng, M, K), _i8(rng, K, K2), _i8(rng, K2, N)
    dA, dB, dB2 = ctx.upload(A), ctx.upload(B), ctx.upload(B2)
    dH, dY, dE = ctx.empty((M, K2), np.int8), ctx.empty((M, N), np.int8), ctx.empty((M, K2), np.int8)
    with ctx.record() as g:
        ctx.gemm_i8_rq(dA, dB, dH, M, K2, K, 11, True)
        ctx.gemm_i8_rq(dH, dB2, dY, M, N, K2, 10)
    for rep in range(4):
        A = _i8(rng, M, K)
        ctx.copy_h2d(dA, A)
        g.launch()
        ctx.gemm_i8_rq(dA, dB, dE, M, K2, K, 9)
        ctx.wait(60_000)
        H = oracle.gemm_i8_rq(A, B, 11, True)
        assert np.array_equal(ctx.download(dH), H), rep
        assert np.array_equal(ctx.download(dY), oracle.gemm_i8_rq(H, B2, 10)), rep
        assert np.array_equal(ctx.download(dE), oracle.gemm_i8_rq(A, B, 9)), rep
    g.destroy()
    for b in (dA, dB, dB2, dH, dY, dE):
        b.free()


@pytest.mark.parametrize("N", [1, 2, 7, 10, 15])
@pytest.mark.parametrize("M,K", [(1, 16), (1, 31), (70, 17), (64, 256), (300, 1000), (5, 4099)])
@pytest.mark.parametrize("off", [0, 3])
def test_gemm_i8_flex_narrow_b(ctx, M, N, K, off):
    """B row-major with rows below one 16-byte load (a classifier's head),
    operands exactly as long as the entry points say: dense, then with padded
    rows at an odd address."""
    print(f"[case] flex gemm {M}x{N}x{K} off {off} plan {ctx.plan_gemm_i8(M, N, K)}", flush=True)
    rng = np.random.default_rng(M + 3 * N + 5 * K + off)
    A, B = _i8(rng, M, K), _i8(rng, K, N)
    Co = oracle.gemm_i8(A, B)
    lda, ldb = K + off, N + off
    bufA, bufB = _i8(rng, off + (M - 1) * lda + K), _i8(rng, off + (K - 1) * ldb + N)
    for m in range(M):
        bufA[off + m * lda: off + m * lda + K] = A[m]
    for k in range(K):
        bufB[off + k * ldb: off + k * ldb + N] = B[k]
    dA, dB, dC, dY = ctx.upload(bufA), ctx.upload(bufB), ctx.empty((M, N), np.int32), ctx.empty((M, N), np.int8)
    for rep in range(2):
        ctx.copy_h2d(dC, np.full((M, N), 77, np.int32))
        ctx.gemm_i8_i32(dA.ptr + off, dB.ptr + off, dC, M, N, K, lda, ldb, N)
        if off == 0:
            ctx.gemm_i8_rq(dA, dB, dY, M, N, K, 9, True)
        ctx.wait(60_000)
        assert np.array_equal(ctx.download(dC), Co), rep
        assert off or np.array_equal(ctx.download(dY), oracle.requant(Co, 9, relu=True)), rep
    for b in (dA, dB, dC, dY):
        b.free()


@pytest.mark.parametrize("layout", [mi.B_NN, mi.B_NT])
@pytest.mark.parametrize("M,N,K,which", [(5, 33, 100, "A"), (5, 20, 19, "B"), (3, 3, 19, "B")])
def test_gemm_i8_flex_long_rows(ctx, M, N, K, which, layout):
    """A pitch of 2^25 bytes or more: offsets within a tile pass 32 bits'
    range for larger tiles."""
    rows_b, cols_b = (N, K) if layout == mi.B_NT else (K, N)
    lda = (1 << 25) + 3 if which == "A" else K
    ldb = (1 << 25) + 1 if which == "B" else cols_b
    print(f"[case] flex gemm {M}x{N}x{K} lda {lda} ldb {ldb} layout {layout}", flush=True)
    rng = np.random.default_rng(M + N + K + layout)
    A, B = _i8(rng, M, K), _i8(rng, rows_b, cols_b)
    dA, dB = ctx.empty(((M - 1) * lda + K,), np.int8), ctx.empty(((rows_b - 1) * ldb + cols_b,), np.int8)
    for d, ld, mat in ((dA, lda, A), (dB, ldb, B)):
        for r in range(mat.shape[0]):
            row = np.ascontiguousarray(mat[r])
            ctx._call("miaie_copy_h2d", d.ptr + r * ld, row.ctypes.data, mi._sz(row.nbytes))
    dC = ctx.empty((M, N), np.int32)
    ctx.gemm_i8_i32(dA, dB, dC, M, N, K, lda, ldb, N, layout)
    ctx.wait(60_000)
    assert np.array_equal(ctx.download(dC), oracle.gemm_i8(A, B, b_nt=layout == mi.B_NT))
    for b in (dA, dB, dC):
        b.free()


# bf16 products are exact in fp32; each of the K additions is off by at most
# 2^-24 / 2 of a partial sum, whose size stays below 6 times the results' rms
# (partial sums of N(0, 1) terms scaled to it, over at most 6e6 results)
def _bf16_bar(K):
    return 6 * max(K, 32) * 2.0**-25


BF16_SHAPES = [
    (1, 8, 8),        # the smallest dense rows: one chunk of one row
    (1, 1, 8),        # rows of B below one load, down to a column
    (70, 3, 9),
    (300, 7, 130),
    (17, 5, 4100),    # ... split
    (1, 9, 9),        # a value past a chunk
    (16, 127, 127),   # skinny tile, one column short, a value short of a stage
    (17, 129, 128),
    (63, 65, 129),
    (64, 64, 33),
    (4, 40, 4100),    # one tile, 33 stages: split
    (130, 270, 1030),  # split, ragged
    (1024, 512, 512),  # whole 256x256 tiles, but few
    (1000, 1000, 100),
    (2500, 2300, 40),  # large enough for the 128x128 tile
]


@pytest.mark.parametrize("M,N,K", BF16_SHAPES + [(M, N, (K + 1) // 2) for M, N, K in SHORT_K])
def test_gemm_bf16_flex(ctx, M, N, K):
    print(f"[case] flex bf16 {M}x{N}x{K}", flush=True)
    A = synth.bf16_normal((M, K), 1, 1.0 / np.sqrt(K))
    B = synth.bf16_normal((K, N), 2, 1.0)
    # what lies past the operands' ends must not matter: they sit between NaNs
    nan = np.full(64, 0x7FC0, np.uint16)
    dA, dB = ctx.upload(np.concatenate([nan, A.ravel(), nan])), ctx.upload(np.concatenate([nan, B.ravel(), nan]))
    R = oracle.gemm_bf16(A, B, f64=True)
    dC = ctx.empty((M, N), np.float32)
    first = None
    for rep in range(3):
        ctx.copy_h2d(dC, np.full((M, N), np.nan, np.float32))
        ctx.gemm_bf16_f32(dA.ptr + 128, dB.ptr + 128, dC, M, N, K)
        ctx.wait(60_000)
        C = ctx.download(dC)
        err = np.abs(C.astype(np.float64) - R).max() / np.sqrt(np.mean(R * R))
        assert err <= _bf16_bar(K), (rep, err)
        # the order of arrival of the splits does not matter
        assert first is None or np.array_equal(C, first), rep
        first = C
    for b in (dA, dB, dC):
        b.free()


@pytest.mark.parametrize("M,N,K,cus,tile,splits", [s for s in SPLITS if s[2] % 2 == 0])
def test_gemm_bf16_flex_splits_of_each_tile(ctx, M, N, K, cus, tile, splits):
    prev = ctx.plan_set_cus(cus or 256)
    try:
        _planned_split(ctx, M, N, K, cus, tile, splits)
        test_gemm_bf16_flex(ctx, M, N, K // 2)
    finally:
        ctx.plan_set_cus(prev)


@pytest.mark.parametrize("M,N,K", [(2, 3, (1 << 24) + 8), (2, (1 << 24) + 5, 8)])
def test_gemm_bf16_flex_long_rows(ctx, M, N, K):
    """Rows of 2^24 values or more, few of them not 0 and whole numbers: the
    sums are exact in any order."""
    print(f"[case] flex bf16 {M}x{N}x{K}", flush=True)
    rng = np.random.default_rng(1)
    A, B = np.zeros((M, K), np.float32), np.zeros((K, N), np.float32)
    ks = np.unique(np.concatenate([[0, K - 1], rng.integers(0, K, 500)]))
    ns = np.unique(np.concatenate([[0, N - 1], rng.integers(0, N, 500)]))
    A[:, ks] = rng.integers(-8, 9, (M, len(ks)))
    B[np.ix_(ks, ns)] = rng.integers(-8, 9, (len(ks), len(ns)))
    bits = lambda x: (x.view(np.uint32) >> 16).astype(np.uint16)  # exact: small whole numbers
    dA, dB, dC = ctx.upload(bits(A)), ctx.upload(bits(B)), ctx.empty((M, N), np.float32)
    ctx.gemm_bf16_f32(dA, dB, dC, M, N, K)
    ctx.wait(60_000)
    want = np.zeros((M, N), np.float32)
    want[:, ns] = A[:, ks] @ B[np.ix_(ks, ns)]
    assert np.array_equal(ctx.download(dC), want)
    for b in (dA, dB, dC):
        b.free()


def test_gemm_bf16_flex_nan_stays_in_its_row_and_column(ctx):
    """A NaN or infinity in one row of A (column of B) reaches that row
    (column) of C alone, K and N ragged."""
    M, N, K = 70, 75, 150
    A, B = synth.bf16_normal((M, K), 3, 0.1), synth.bf16_normal((K, N), 4, 1.0)
    A[11, K - 1] = 0x7FC0  # NaN
    B[K - 1, 66] = 0x7F80  # inf
    dA, dB, dC = ctx.upload(A), ctx.upload(B), ctx.empty((M, N), np.float32)
    ctx.gemm_bf16_f32(dA, dB, dC, M, N, K)
    ctx.wait(60_000)
    bad = ~np.isfinite(ctx.download(dC))
    want = np.zeros((M, N), bool)
    want[11, :] = True
    want[:, 66] = True
    assert np.array_equal(bad, want)
    for b in (dA, dB, dC):
        b.free()


@pytest.mark.parametrize("K", [32, 64, 96, 128, 192, 256, 320, 384, 448, 512, 576, 1088, 2112])
def test_gemm_bf16_256_tiles_k_sweep(ctx, K):
    """Every k-tile count of the 256x256 kernels' prologue and tail, planned
    for one CU so that they are the choice."""
    M, N = 512, 256
    A, B = synth.bf16_normal((M, K), 5, 1.0 / np.sqrt(K)), synth.bf16_normal((K, N), 6, 1.0)
    dA, dB, dC = ctx.upload(A), ctx.upload(B), ctx.empty((M, N), np.float32)
    prev = ctx.plan_set_cus(1)
    try:
        ctx.gemm_bf16_f32(dA, dB, dC, M, N, K)
        ctx.wait(60_000)
    finally:
        ctx.plan_set_cus(prev)
    R = oracle.gemm_bf16(A, B, f64=True)
    err = np.abs(ctx.download(dC).astype(np.float64) - R).max() / np.sqrt(np.mean(R * R))
    assert err <= _bf16_bar(K), err
    for b in (dA, dB, dC):
        b.free()


CONV_SHAPES = [
    # N, H, W, Cin, Cout, R, S, stride, pad
    (1, 4, 4, 1, 1, 1, 1, 1, 0),      # 16 bytes of X; W (1 byte) too small: one thread per output
    (1, 4, 4, 1, 16, 1, 1, 1, 0),     # 16 bytes of each, k of one value: one thread per output
    (1, 4, 4, 1, 16, 5, 5, 1, 2),     # about the smallest that runs on tiles
    (2, 9, 11, 3, 64, 7, 7, 2, 3),    # a stem: runs of 21 bytes, pads on every side
    (1, 5, 5, 5, 3, 3, 3, 1, 1),      # pixels fewer than a tile, 3 channels
    (3, 7, 1, 16, 65, 3, 1, 1, 1),    # one column, R != S, one channel past a tile
    (2, 1, 30, 6, 20, 1, 5, 1, 2),    # padding rows only above and below a single row
    (1, 3, 3, 30, 40, 3, 3, 1, 4),    # padding wider than the filter: runs wholly outside
    (5, 6, 7, 33, 17, 3, 3, 3, 1),    # stride 3
    (1, 70, 130, 17, 66, 3, 3, 1, 1),  # rows longer than a pixel tile
    (40, 3, 2, 8, 24, 2, 2, 1, 0),    # many images within one pixel tile (two output columns, one row... 2 x 1)
    (1, 13, 13, 130, 70, 5, 5, 1, 2),  # k of 5 runs of 650 bytes: stages across runs, split
    (2, 20, 20, 130, 200, 3, 3, 1, 1),  # 64 x 64 tiles, split
    (1, 3, 3, 7300, 5, 3, 3, 1, 1),   # k >= 2^16: the requant form without the rounding add
    (4, 64, 64, 3, 130, 3, 3, 1, 1),  # 256 x 2 tiles: 128 x 128
    (8, 96, 96, 32, 192, 1, 1, 1, 0),  # a large grid of the implicit-GEMM shapes
    # one stage of k and more pixel tiles than fit at once: walked over
    (1, 520, 262, 3, 20, 3, 3, 1, 1),   # rows longer than a tile; k of 48 bytes
    (4100, 6, 7, 3, 10, 3, 3, 1, 1),    # images smaller than a tile
    (1, 260, 262, 3, 20, 7, 7, 1, 3),   # k of 224 bytes: 256-byte stages
    (8, 160, 160, 100, 128, 1, 1, 1, 0),  # 128 x 128
    # (fewer tiles than fit with 64-byte stages)
    (1, 260, 262, 3, 20, 3, 3, 1, 1),   # rows longer than a tile
    (2100, 6, 7, 3, 10, 3, 3, 1, 1),    # images smaller than a tile
    (70000, 2, 1, 16, 70, 1, 1, 1, 0),  # one column, two channel tiles, the last partial
]


@pytest.mark.parametrize("shape", CONV_SHAPES)
@pytest.mark.parametrize("off", [0, 5])
def test_conv2d_i8_flex(ctx, shape, off):
    """Bit-exact against the oracle, shifts over [0, 31], operands at byte
    offset `off` of their buffers, three calls in a row (split sums leave their
    counters for the next launch)."""
    N, H, W, Cin, Cout, R, S, stride, pad = shape
    print(f"[case] flex conv {shape} off {off}", flush=True)
    rng = np.random.default_rng(sum(shape) + off)
    X, Wt = _i8(rng, N, H, W, Cin), _i8(rng, Cout, R, S, Cin)
    if Cin == 7300:
        X[:], Wt[:] = -128, -128
    sh = rng.integers(0, 32, size=Cout, dtype=np.uint8) if sum(shape) % 2 else rng.integers(8, 13, size=Cout, dtype=np.uint8)
    Ho, Wo = (H + 2 * pad - R) // stride + 1, (W + 2 * pad - S) // stride + 1
    lead = _i8(rng, off)  # exactly as long as the operands: nothing behind them
    dX = ctx.upload(np.concatenate([lead, X.ravel()]))
    dW = ctx.upload(np.concatenate([lead, Wt.ravel()]))
    dS = ctx.upload(sh)
    dY = ctx.empty((off + N * Ho * Wo * Cout + 16,), np.int8)
    want = oracle.conv2d_nhwc_i8(X, Wt, sh, stride, pad).ravel()
    for rep in range(3):
        ctx.copy_h2d(dY, np.full(dY.nbytes, 77, np.int8))
        ctx.conv2d_i8_nhwc(dX.ptr + off, dW.ptr + off, dS, dY.ptr + off, N, H, W, Cin, Cout, R, S, stride, pad)
        ctx.wait(60_000)
        got = ctx.download(dY)
        assert np.array_equal(got[off:-16], want), rep
        assert (got[:off] == 77).all() and (got[-16:] == 77).all(), rep
    for b in (dX, dW, dS, dY):
        b.free()


@pytest.mark.parametrize("off", [0, 5])
def test_conv2d_i8_flex_128_split(ctx, off):
    """128 x 128 tiles split over k, planned for 8 CUs."""
    prev = ctx.plan_set_cus(8)
    try:
        test_conv2d_i8_flex(ctx, (1, 12, 12, 400, 520, 3, 3, 1, 1), off)
    finally:
        ctx.plan_set_cus(prev)


@pytest.mark.parametrize("R,Cout", [(17, 1), (2, 5)])
def test_conv2d_i8_flex_of_2_30_pixels(ctx, R, Cout):
    """2^30 output pixels: of one channel over two stages of k, 2^24 workgroups
    with a 64 x 64 tile, one more than a launch takes; of five channels and a k of
    four values, more outputs than a launch has threads.  Strips of rows at the
    image's top, middle and end against the oracle."""
    H = W = 32768
    pad, rows = R // 2, 24
    print(f"[case] flex conv {H}x{W} -> {Cout}, {R}x{R}", flush=True)
    rng = np.random.default_rng(3)
    Wt, sh = _i8(rng, Cout, R, R, 1), np.full(Cout, 12 if R > 2 else 7, np.uint8)
    Ho = Wo = H + 2 * pad - R + 1
    dX, dY = ctx.empty((H, W), np.int8), ctx.empty((Ho, Wo, Cout), np.int8)
    dW, dS = ctx.upload(Wt), ctx.upload(sh)
    ctx.fill_i8(dX, H * W, 9)
    ctx.conv2d_i8_nhwc(dX, dW, dS, dY, 1, H, W, 1, Cout, R, R, 1, pad)
    ctx.wait(60_000)
    for first in (0, 16380, Ho - rows):
        lo, hi = max(first - pad, 0), min(first + rows + pad, H)
        x, y = np.empty((hi - lo, W), np.int8), np.empty((rows, Wo, Cout), np.int8)
        ctx._call("miaie_copy_d2h", x.ctypes.data, dX.ptr + lo * W, mi._sz(x.nbytes))
        ctx._call("miaie_copy_d2h", y.ctypes.data, dY.ptr + first * Wo * Cout, mi._sz(y.nbytes))
        want = oracle.conv2d_nhwc_i8(x.reshape(1, hi - lo, W, 1), Wt, sh, 1, pad)
        assert np.array_equal(y, want[0, first - lo:first - lo + rows]), first
    for b in (dX, dY, dW, dS):
        b.free()


@pytest.mark.parametrize("shape,direct", [
    ((8, 224, 224, 2, 1, 3, 3, 1, 1), True), ((4, 112, 112, 4, 4, 1, 1, 1, 0), True), ((1, 14, 14, 1, 20, 1, 1, 1, 0), True),
    ((4, 112, 112, 16, 1, 1, 1, 1, 0), True), ((8, 112, 112, 1, 1, 5, 5, 1, 2), True), ((4, 112, 112, 8, 16, 1, 1, 1, 0), False),
    ((8, 224, 224, 3, 16, 3, 3, 1, 1), False), ((4, 112, 112, 17, 1, 1, 1, 1, 0), False), ((1, 30, 30, 1, 2, 9, 9, 1, 4), False)])
def test_conv2d_i8_of_a_tiny_k(shape, direct):
    """A k of a few values: one thread per output where a tile's stage would be
    mostly empty, at 256 CUs, tiles on the other side of the line."""
    N, H, W, Cin, Cout, R, S, stride, pad = shape
    print(f"[case] conv of a tiny k {shape}", flush=True)
    rng = np.random.default_rng(sum(shape))
    X, Wt = _i8(rng, N, H, W, Cin), _i8(rng, Cout, R, S, Cin)
    sh = rng.integers(0, 13, size=Cout, dtype=np.uint8)
    want = oracle.conv2d_nhwc_i8(X, Wt, sh, stride, pad)
    cap = Capture()
    c = cap.ctx
    dX, dW, dS, dY = c.upload(X), c.upload(Wt), c.upload(sh), c.empty(want.shape, np.int8)
    exe, grids = cap.record(lambda: c.conv2d_i8_nhwc(dX, dW, dS, dY, N, H, W, Cin, Cout, R, S, stride, pad))
    assert (grids == [(-(-want.size // 256), 1, 1)]) == direct, grids
    cap.replay(exe)
    cap.sync()
    assert np.array_equal(c.download(dY), want)
    cap.ok(cap.hip.hipGraphExecDestroy(exe))
    cap.close()


@pytest.mark.parametrize("shape,tiles", [
    ((4, 28, 28, 96, 128, 5, 5, 1, 2), False), ((4, 28, 28, 96, 256, 5, 5, 1, 2), True), ((4, 56, 56, 96, 128, 3, 3, 2, 1), True),
    ((4, 56, 56, 32, 128, 3, 3, 2, 1), False), ((8, 28, 28, 32, 192, 5, 5, 1, 2), False), ((4, 28, 28, 64, 128, 1, 1, 1, 0), True),
    ((2, 28, 28, 64, 128, 1, 1, 1, 0), False)])
def test_conv2d_i8_implicit_gemm_grids(ctx, shape, tiles):
    """Layers of the implicit-GEMM shapes, planned for 32 CUs: three to six (and
    nine) 64 x 64 tiles per CU on register-staged tiles (all in x) or on
    fragments from memory (channel tiles in y)."""
    N, H, W, Cin, Cout, R, S, stride, pad = shape
    print(f"[case] implicit GEMM conv {shape}", flush=True)
    rng = np.random.default_rng(sum(shape))
    X, Wt = _i8(rng, N, H, W, Cin), _i8(rng, Cout, R, S, Cin)
    sh = rng.integers(8, 13, size=Cout, dtype=np.uint8)
    want = oracle.conv2d_nhwc_i8(X, Wt, sh, stride, pad)
    cap = Capture()
    c = cap.ctx
    c.plan_set_cus(32)
    dX, dW, dS, dY = c.upload(X), c.upload(Wt), c.upload(sh), c.empty(want.shape, np.int8)
    exe, grids = cap.record(lambda: c.conv2d_i8_nhwc(dX, dW, dS, dY, N, H, W, Cin, Cout, R, S, stride, pad))
    assert len(grids) == 1 and (grids[0][1] == 1) == tiles, grids
    cap.replay(exe)
    cap.sync()
    assert np.array_equal(c.download(dY), want)
    cap.ok(cap.hip.hipGraphExecDestroy(exe))
    cap.close()
