"""Entry points recorded by the caller's own HIP capture of the context's
stream (not miaie_graph_begin).  Such a graph may be replayed on any stream,
beside other work of the context, so what it holds must not touch the
context's workspace: no split of K."""
import ctypes as C
import threading

import numpy as np
import pytest

import aiehlc_amd as mi
import oracle
from aiehlc_amd import synth
from hip_capture import NON_BLOCKING, RELAXED, THREAD_LOCAL, Capture

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cap():
    c = Capture()
    yield c
    c.close()


def _beside_eager_splits(cap, exe, fill_out, check_out):
    """Replays on the second stream while the context runs products that
    are split over K through its workspace."""
    ctx = cap.ctx
    M, N, K = 16, 512, 8192
    assert ctx.plan_gemm_i8(M, N, K)["workgroups"] > -(-M // 16) * -(-N // 128)  # split
    A, B = synth.int8((M, K), 1), synth.int8((K, N), 2)
    dA, dB, dY = ctx.upload(A), ctx.upload(B), ctx.empty((M, N), np.int8)
    want = oracle.gemm_i8_rq(A, B, 11)
    for rep in range(4):
        fill_out()
        ctx.copy_h2d(dY, np.full((M, N), 77, np.int8))
        cap.sync()
        for _ in range(6):
            cap.replay(exe)
            ctx.gemm_i8_rq(dA, dB, dY, M, N, K, 11)
        cap.sync()
        check_out(rep)
        assert np.array_equal(ctx.download(dY), want), rep
    for b in (dA, dB, dY):
        b.free()
    cap.ok(cap.hip.hipGraphExecDestroy(exe))


CONV_SHAPES = [
    # N, H, W, Cin, Cout, R, stride, pad
    (8, 7, 7, 512, 512, 3, 2, 1),    # taps kernel, split when run directly
    (8, 7, 7, 512, 512, 3, 1, 1),    # taps against the chunked row-block kernel
    (1, 7, 7, 96, 64, 5, 1, 2),      # implicit GEMM on fragments from memory
    (1, 13, 13, 130, 70, 5, 1, 2),   # register-staged tiles
]


@pytest.mark.parametrize("shape", CONV_SHAPES)
def test_captured_conv_leaves_the_workspace_alone(cap, shape):
    N, H, W, Cin, Cout, R, stride, pad = shape
    print(f"[case] captured conv {shape}", flush=True)
    ctx = cap.ctx
    rng = np.random.default_rng(sum(shape))
    X, Wt = (rng.integers(-128, 128, size=s, dtype=np.int8) for s in ((N, H, W, Cin), (Cout, R, R, Cin)))
    sh = rng.integers(8, 13, size=Cout, dtype=np.uint8)
    want = oracle.conv2d_nhwc_i8(X, Wt, sh, stride, pad)
    dX, dW, dS, dY = ctx.upload(X), ctx.upload(Wt), ctx.upload(sh), ctx.empty(want.shape, np.int8)
    exe, grids = cap.record(lambda: ctx.conv2d_i8_nhwc(dX, dW, dS, dY, N, H, W, Cin, Cout, R, R, stride, pad))
    # one kernel (a split taps or implicit-GEMM launch is followed by its sum),
    # and one workgroup per 64 x 64 tile at most (splits are in y or z)
    P = want.size // Cout
    assert len(grids) == 1 and np.prod(grids[0]) <= -(-P // 16) * -(-Cout // 32), grids

    def check(rep):
        assert np.array_equal(ctx.download(dY), want), rep

    _beside_eager_splits(cap, exe, lambda: ctx.copy_h2d(dY, np.full(want.shape, 77, np.int8)), check)
    for b in (dX, dW, dS, dY):
        b.free()


GEMM_SHAPES = [
    # M, N, K, workgroups of the plan without a split, at 256 CUs
    (16, 512, 8192, 8),              # register-staged 64 x 64
    (512, 512, 8192, 16),            # the pipelined 128 x 128 kernel: faster than register-staged tiles unsplit
    (130, 300, 2049, 15),            # register-staged, ragged
]


@pytest.mark.parametrize("M,N,K,workgroups", GEMM_SHAPES)
@pytest.mark.parametrize("layout", [mi.B_NN, mi.B_NT])
def test_captured_int8_gemm_is_planned_without_a_split(cap, M, N, K, workgroups, layout):
    print(f"[case] captured int8 gemm {M}x{N}x{K} layout {layout}", flush=True)
    ctx = cap.ctx
    assert ctx.plan_gemm_i8(M, N, K)["workgroups"] > workgroups  # run directly, it is split
    A, B = synth.int8((M, K), 3), synth.int8((N, K) if layout == mi.B_NT else (K, N), 4)
    want = oracle.gemm_i8_rq(A, B, 11, b_nt=layout == mi.B_NT)
    dA, dB, dY = ctx.upload(A), ctx.upload(B), ctx.empty((M, N), np.int8)
    exe, grids = cap.record(lambda: ctx.gemm_i8_rq(dA, dB, dY, M, N, K, 11, False, None, layout))
    assert len(grids) == 1 and np.prod(grids[0]) == workgroups, grids

    def check(rep):
        assert np.array_equal(ctx.download(dY), want), rep

    _beside_eager_splits(cap, exe, lambda: ctx.copy_h2d(dY, np.full((M, N), 77, np.int8)), check)
    for b in (dA, dB, dY):
        b.free()


def test_captured_bf16_gemm_is_not_split(cap):
    M, N, K = 130, 270, 1030
    print(f"[case] captured bf16 gemm {M}x{N}x{K}", flush=True)
    ctx = cap.ctx
    A, B = synth.bf16_normal((M, K), 1, 1.0 / np.sqrt(K)), synth.bf16_normal((K, N), 2, 1.0)
    R = oracle.gemm_bf16(A, B, f64=True)
    dA, dB, dC = ctx.upload(A), ctx.upload(B), ctx.empty((M, N), np.float32)
    exe, grids = cap.record(lambda: ctx.gemm_bf16_f32(dA, dB, dC, M, N, K))
    assert len(grids) == 1 and grids[0][1] == 1, grids  # (the splits are in y)

    def check(rep):
        # K additions, each off by at most half an ulp of a partial sum, which
        # stays below 6 times the results' rms
        err = np.abs(ctx.download(dC).astype(np.float64) - R).max() / np.sqrt(np.mean(R * R))
        assert err <= 6 * K * 2.0**-25, (rep, err)

    _beside_eager_splits(cap, exe, lambda: ctx.copy_h2d(dC, np.full((M, N), np.nan, np.float32)), check)
    for b in (dA, dB, dC):
        b.free()


@pytest.mark.parametrize("flags", [0, NON_BLOCKING])
@pytest.mark.parametrize("mode", [THREAD_LOCAL, RELAXED])
def test_a_context_is_created_while_another_thread_captures(cap, flags, mode):
    """... on a stream of its own and on a caller's, neither of them nor the
    capture fails, and they work (a split product uses the arrival counters)."""
    print(f"[case] context created during a capture, stream flags {flags} mode {mode}", flush=True)
    hip, begun, created, rcs = cap.hip, threading.Event(), threading.Event(), {}

    def capture():
        s, graph = C.c_void_p(), C.c_void_p()
        rcs["device"] = hip.hipSetDevice(0)
        rcs["stream"] = hip.hipStreamCreateWithFlags(C.byref(s), flags)
        rcs["begin"] = hip.hipStreamBeginCapture(s, mode)
        begun.set()
        created.wait(60)
        rcs["end"] = hip.hipStreamEndCapture(s, C.byref(graph))
        hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(s)

    t = threading.Thread(target=capture)
    t.start()
    begun.wait(60)
    made = []
    try:
        made = [mi.Context(0), mi.Context(0, stream=cap.streams[1].value)]
    finally:
        created.set()
        t.join()
    assert set(rcs.values()) == {0}, rcs
    M, N, K = 16, 512, 8192
    A, B = synth.int8((M, K), 1), synth.int8((K, N), 2)
    for ctx in made:
        dA, dB, dY = ctx.upload(A), ctx.upload(B), ctx.empty((M, N), np.int8)
        ctx.gemm_i8_rq(dA, dB, dY, M, N, K, 11)
        ctx.wait(60_000)
        assert np.array_equal(ctx.download(dY), oracle.gemm_i8_rq(A, B, 11))
        ctx.close()


def test_a_context_is_created_by_the_capturing_thread(cap):
    """In relaxed mode."""
    hip, s, graph = cap.hip, C.c_void_p(), C.c_void_p()
    cap.ok(hip.hipStreamCreateWithFlags(C.byref(s), NON_BLOCKING))
    cap.ok(hip.hipStreamBeginCapture(s, RELAXED))
    try:
        mi.Context(0).close()
        mi.Context(0, stream=cap.streams[1].value).close()
    finally:
        rc = hip.hipStreamEndCapture(s, C.byref(graph))
    cap.ok(rc)
    hip.hipGraphDestroy(graph)
    cap.ok(hip.hipStreamDestroy(s))
