"""Calls that need library scratch under HIP graph capture: captured with no call before them (nothing allocated yet), and
replayed after later calls that need more. Every replay gives the bits of the eager call."""
import numpy as np
import pytest

from metaltile_amd import DType, GpuBuffer, _lib, ops, unpack_f32
from metaltile_amd.runtime import _ensure_init
from metaltile_amd.synth import make_case
from tests.hip_graph import Graph

pytestmark = pytest.mark.gpu


def _operands(seed, dt, bits, M, N, K, E=1):
    c = make_case(seed, dt, bits, 64, M, N, K, E=E)
    return [GpuBuffer.from_bytes(v) for v in (c.w.tobytes(), c.scales_bytes, c.biases_bytes)], GpuBuffer.from_bytes(c.x_bytes)


def _gather(dt):
    """Two experts with rows of more than one K slice: f32 partial rows."""
    T, N, K, E = 16, 4096, 14336, 2
    assert ops.plan("gather_csr", dt, 4, 64, 1, N, K, E, T)[2] >= 2 * T * N * 4
    wsb, x = _operands(5, dt, 4, T, N, K, E)
    offsets = GpuBuffer.from_bytes(np.array([0, 7, T], dtype="<u4").tobytes())
    out = GpuBuffer(T * N * 2)
    return [x, *wsb, offsets], out, T * N * 2, lambda: ops.gather_qmv_csr(dt, 4, 64, x, *wsb, offsets, out, T, N, K, E)


def _bit_stream(dt):
    """6-bit codes at 77 rows, K split."""
    M, N, K = 77, 3584, 9472
    assert ops.plan("qmm", dt, 6, 64, M, N, K)[2] >= 2 * M * N * 4
    wsb, x = _operands(6, dt, 6, M, N, K)
    out = GpuBuffer(M * N * 2)
    return [x, *wsb], out, M * N * 2, lambda: ops.qmm(dt, 6, 64, *wsb, x, out, M, N, K)


def _batch(dt):
    """Split matrices of one launch: the partial tiles of all at once."""
    M, N, K = 130, 512, 4096
    assert ops.plan("qmm", dt, 4, 64, M, N, K)[2] >= 2 * M * N * 4
    ops_of = [_operands(7 + j, dt, 4, M, N, K) for j in range(2)]
    out = GpuBuffer(2 * M * N * 2)
    outs = [out.ptr, out.ptr + M * N * 2]
    ws, ss, bs = ([o[0][i] for o in ops_of] for i in range(3))
    x = ops_of[0][1]
    return [b for o in ops_of for b in (*o[0], o[1])], out, 2 * M * N * 2, lambda: ops.qmm_batched(dt, 4, 64, ws, ss, bs, x, outs, [N, N], M, K)


def _slices(dt):
    """Four rows of more than 18432 codes: f32 sums of slices of K."""
    M, N, K = 4, 1024, 18688
    assert "qmv_slices_kernel" in ops.plan("qmm", dt, 4, 64, M, N, K)[1][0][0]
    wsb, x = _operands(8, dt, 4, M, N, K)
    out = GpuBuffer(M * N * 2)
    return [x, *wsb], out, M * N * 2, lambda: ops.qmm(dt, 4, 64, *wsb, x, out, M, N, K)


@pytest.mark.parametrize("make", [_gather, _bit_stream, _batch, _slices], ids=lambda f: f.__name__[1:])
def test_captured_first_and_replayed_after_growth(make):
    dt = DType.BF16
    print(f"[case] scratch under capture, {make.__name__}", flush=True)
    lib = _ensure_init()
    _lib.check(lib.mtq_shutdown())   # nothing is held: the captured call is the first that needs scratch
    _lib.check(lib.mtq_init(0))
    bufs, out, nbytes, call = make(dt)
    big = _operands(9, dt, 4, 512, 4096, 14336)
    big_out = GpuBuffer(512 * 4096 * 2)
    g = Graph()
    try:
        with g:
            call()
        g.replay()
        first = out.read_bytes(nbytes)
        out.upload(np.full(nbytes, 0xFF, np.uint8))
        call()
        assert out.read_bytes(nbytes) == first and any(first)
        # needs more (16 MB of partial tiles): a new buffer, while the graph goes on with the one that it was captured with
        assert ops.plan("qmm", dt, 4, 64, 512, 4096, 14336)[2] == 16 << 20
        for _ in range(3):
            ops.qmm(dt, 4, 64, *big[0], big[1], big_out, 512, 4096, 14336)
            out.upload(np.full(nbytes, 0xFF, np.uint8))
            g.replay()
            assert out.read_bytes(nbytes) == first
            out.upload(np.full(nbytes, 0xFF, np.uint8))
            call()
            assert out.read_bytes(nbytes) == first
    finally:
        g.close()
        for b in bufs + [out, big_out, big[1], *big[0]]:
            b.free()


@pytest.mark.parametrize("bits,G,M,N,K", [(4, 64, 4, 1024, 18688), (8, 64, 3, 272, 18944), (4, 128, 16, 4096, 9344), (8, 64, 8, 8192, 10240)])
def test_slices_without_memory(oracle, bits, G, M, N, K):
    """Where the K slices' sums find no memory the call is served by the kernels that need none, alone and in a batch. Bound,
    2-norm over 2-norm: the roundings to bf16 of the result and, on the tiles, of the weights, each up to 2^-9 of a value: 4e-3."""
    dt = DType.BF16
    print(f"[case] K-sliced qmv without memory b{bits} g{G} M{M} N{N} K{K}", flush=True)
    lib = _ensure_init()
    c = make_case(890 + M, dt, bits, G, M, N, K, bias_rule="midpoint")
    bufs = [GpuBuffer.from_bytes(v) for v in (c.w.tobytes(), c.scales_bytes, c.biases_bytes, c.x_bytes)]
    outs = [GpuBuffer.from_bytes(b"\xff" * (M * N * 2)) for _ in range(2)]
    try:
        assert lib.mtq_set_option(b"scratch.most_kb", 1) == 0
        ops.qmm(dt, bits, G, *bufs, outs[0], M, N, K)
        ops.qmm_batched(dt, bits, G, [bufs[0]], [bufs[1]], [bufs[2]], bufs[3], [outs[1]], [N], M, K)
        got = [o.read_bytes(M * N * 2) for o in outs]
    finally:
        lib.mtq_set_option(b"scratch.most_kb", 0)
    exp = oracle.qmm_f64(c.w, c.scales_f, c.biases_f, c.x_f, M, N, K, bits, G, threads=8).reshape(-1)
    assert got[0] == got[1]
    assert np.linalg.norm(unpack_f32(got[0], dt) - exp) <= 4e-3 * np.linalg.norm(exp)
    for b in bufs + outs:
        b.free()
