"""The K-run kernel in slices of K (mtq_qmm at 3..16 rows of more than 5120 codes): slices of unequal length, runs without a step,
ragged blocks of weight rows, more blocks than a slice's workgroups keep in flight, against the f64-accumulated oracle.

Bound: as for the K-run kernel (rounding of the result, f32 sums, the conversion's offset of up to 1024, which for K = 28672 and
|x| up to 5 leaves about 2^-24 * 1024 * sqrt(K) * scale (0.1) = 1e-3 absolute): max |a-e| / max(|e|, 1) <= 1e-2 (bf16), 4e-3 (f16)."""
import numpy as np
import pytest

from metaltile_amd import DType, GpuBuffer, ops, pack_f32, unpack_f32
from metaltile_amd.runtime import _ensure_init
from metaltile_amd.synth import make_case
from tests.parity import rel_err

pytestmark = pytest.mark.gpu
TOL = {DType.F16: 4e-3, DType.BF16: 1e-2}


@pytest.mark.parametrize("dt", [DType.F16, DType.BF16], ids=lambda d: d.name)
@pytest.mark.parametrize("bits,G,M,K,N", [
    (4, 128, 16, 13824, 272), (4, 64, 5, 5248, 33), (4, 32, 13, 9344, 8211), (4, 64, 16, 28672, 18), (4, 128, 1, 10240, 16),
    (8, 64, 4, 18944, 3584), (8, 32, 16, 5248, 15), (8, 128, 9, 10368, 6500), (8, 64, 3, 81920, 17),
])
def test_slices(oracle, dt, bits, G, M, K, N):
    print(f"[case] K-sliced qmv {dt.name} b{bits} g{G} M{M} K{K} N={N}", flush=True)
    lib = _ensure_init()
    c = make_case(880 + M, dt, bits, G, M, N, K, bias_rule="midpoint")
    bufs = [GpuBuffer.from_bytes(v) for v in (c.w.tobytes(), c.scales_bytes, c.biases_bytes, c.x_bytes)]
    guard = b"\xcd" * 64
    out = GpuBuffer.from_bytes(b"\xff" * (M * N * 2) + guard)
    try:
        assert lib.mtq_set_option(b"qmv.runs", 3) == 0
        rc, launches, _, scratch = ops.plan("qmm", dt, bits, G, M, N, K)
        assert rc == 0 and "qmv_slices_kernel" in launches[0][0] and len(launches) == 2
        ops.qmm(dt, bits, G, *bufs, out, M, N, K)
        raw = out.read_bytes(M * N * 2 + 64)
        assert raw[-64:] == guard
        exp = oracle.qmm_f64(c.w, c.scales_f, c.biases_f, c.x_f, M, N, K, bits, G, threads=8).reshape(-1)
        assert rel_err(unpack_f32(raw[:-64], dt), exp) <= TOL[dt]
        batch = GpuBuffer(M * N * 2)   # alone and in a batch a matrix gives the same bits
        ops.qmm_batched(dt, bits, G, [bufs[0]], [bufs[1]], [bufs[2]], bufs[3], [batch], [N], M, K)
        assert batch.read_bytes(M * N * 2) == raw[:-64]
        batch.free()
    finally:
        lib.mtq_set_option(b"qmv.runs", 0)
        for b in bufs + [out]:
            b.free()


@pytest.mark.parametrize("bits,G,M,N,K,slices", [
    (8, 64, 4, 3584, 18944, True), (4, 64, 3, 1024, 18688, True), (4, 64, 4, 4096, 18432, False), (4, 64, 2, 3584, 18944, False),
    (4, 128, 16, 5120, 13824, True), (4, 128, 8, 5120, 13824, False), (4, 64, 16, 5120, 13824, False), (4, 128, 16, 2048, 8960, False),
    (4, 128, 5, 2048, 9344, True), (4, 64, 17, 4096, 9344, False), (8, 64, 8, 8192, 10240, True), (8, 64, 9, 8192, 10240, False), (8, 64, 16, 8192, 28672, True),
    (8, 128, 16, 8192, 28672, False), (8, 64, 9, 16384, 14336, False), (8, 64, 8, 16384, 14336, True), (8, 32, 5, 28672, 8448, False), (8, 32, 16, 6144, 40960, True),
    (8, 128, 16, 4096, 9344, True),
])
def test_lines(bits, G, M, N, K, slices):
    """Which matrices the K-sliced form is for, on both sides of each line."""
    rc, launches, _, _ = ops.plan("qmm", DType.BF16, bits, G, M, N, K)
    assert rc == 0 and ("qmv_slices_kernel" in launches[0][0]) == slices, launches[0][0]


def test_infinite_activation():
    """Infinite activations give infinities of the weight's sign in every slice's sum, finite rows keep their bits."""
    dt, bits, G, M, N, K = DType.BF16, 4, 64, 4, 32, 18944
    lib = _ensure_init()
    c = make_case(871, dt, bits, G, M, N, K, bias_rule="midpoint")
    plain = c.x_f.reshape(M, K).astype(np.float32)
    x = plain.copy()
    x[1, K // 3] = np.inf
    codes = ((c.w.reshape(N, -1, 1) >> np.arange(0, 32, bits, dtype=np.uint32)) & 15).reshape(N, K).astype(np.float32)
    s, b = (np.repeat(v.reshape(N, K // G), G, axis=1).astype(np.float32) for v in (c.scales_f, c.biases_f))
    w = unpack_f32(pack_f32((codes * s + b).reshape(-1), dt), dt).reshape(N, K)
    bufs = [GpuBuffer.from_bytes(v) for v in (c.w.tobytes(), c.scales_bytes, c.biases_bytes)]
    got = []
    for v in (x, plain):
        xb, out = GpuBuffer.from_bytes(pack_f32(v.reshape(-1), dt)), GpuBuffer(M * N * 2)
        ops.qmm(dt, bits, G, *bufs, xb, out, M, N, K)
        got.append(unpack_f32(out.read_bytes(M * N * 2), dt).reshape(M, N))
        xb.free()
        out.free()
    for v in bufs:
        v.free()
    np.testing.assert_array_equal(got[0][1], w[:, K // 3] * np.float32(np.inf))
    rest = [0, 2, 3]
    np.testing.assert_array_equal(got[0][rest], got[1][rest])
