"""The K-run matrix-core GEMV (mtq_qmm and mtq_qmm_batched at 2..16 rows): the edges of its blocks of 16 weight rows, of its
steps of 128 (64) codes over sixteen waves, of its groups and of the batch, against the f64-accumulated oracle.

Bound: exact-dequant arithmetic, so what is left is the rounding of the result (2^-9 of it in bf16, 2^-12 in f16) and f32
sums; the conversion adds up to 1024 to a code and takes it out again, which for K = 8192 and |x| up to 5 leaves at most
about 2^-24 * 1024 * sqrt(K) * scale (0.1) = 6e-4 absolute. max |a-e| / max(|e|, 1) <= 1e-2 (bf16), 3e-3 (f16)."""
import numpy as np
import pytest

from metaltile_amd import DType, GpuBuffer, ops, unpack_f32
from metaltile_amd.runtime import _ensure_init
from metaltile_amd.synth import make_case
from tests.parity import rel_err

pytestmark = pytest.mark.gpu
TOL = {DType.F16: 3e-3, DType.BF16: 1e-2}


@pytest.mark.parametrize("dt", [DType.F16, DType.BF16], ids=lambda d: d.name)
@pytest.mark.parametrize("bits,G,M,K,Ns", [
    (4, 64, 16, 4096, (272, 1, 40)), (4, 64, 5, 128, (16, 33)), (4, 128, 13, 5120, (4112, 15, 17, 100)), (4, 32, 9, 2048, (130, 4096)),
    (4, 64, 2, 8192, (48,)), (4, 32, 16, 8192, (20, 31)), (4, 128, 16, 7936, (64,)), (4, 32, 3, 3712, (18, 16)),
    (8, 64, 16, 4096, (272, 1, 40)), (8, 32, 7, 5120, (33,)), (8, 128, 4, 3584, (16, 100)), (8, 64, 16, 1152, (4130, 3)), (8, 32, 16, 128, (5, 6)),
])
def test_edges(oracle, dt, bits, G, M, K, Ns):
    print(f"[case] K-run qmv {dt.name} b{bits} g{G} M{M} K{K} N={Ns}", flush=True)
    lib = _ensure_init()
    cases = [make_case(900 + j + M, dt, bits, G, M, N, K, bias_rule="midpoint") for j, N in enumerate(Ns)]
    x = GpuBuffer.from_bytes(cases[0].x_bytes)
    ws, ss, bs = ([GpuBuffer.from_bytes(v) for v in part] for part in zip(*((c.w.tobytes(), c.scales_bytes, c.biases_bytes) for c in cases)))
    guard = b"\xcd" * 64
    outs = [GpuBuffer.from_bytes(b"\xff" * (M * N * 2) + guard) for N in Ns]
    try:
        assert lib.mtq_set_option(b"qmv.runs", 2) == 0
        rc, launches, _, _ = ops.plan("qmm", dt, bits, G, M, Ns[0], K)
        assert rc == 0 and "qmv_runs_kernel" in launches[0][0]
        ops.qmm_batched(dt, bits, G, ws, ss, bs, x, outs, list(Ns), M, K)
        for j, (c, N) in enumerate(zip(cases, Ns)):
            raw = outs[j].read_bytes(M * N * 2 + 64)
            assert raw[-64:] == guard
            exp = oracle.qmm_f64(c.w, c.scales_f, c.biases_f, cases[0].x_f, M, N, K, bits, G).reshape(-1)
            assert rel_err(unpack_f32(raw[:-64], dt), exp) <= TOL[dt], j
            single = GpuBuffer(M * N * 2)
            ops.qmm(dt, bits, G, ws[j], ss[j], bs[j], x, single, M, N, K)
            assert single.read_bytes(M * N * 2) == raw[:-64], j
            single.free()
    finally:
        lib.mtq_set_option(b"qmv.runs", 0)
        for b in [x] + ws + ss + bs + outs:
            b.free()


def test_mixed_batch_keeps_bits():
    """Three rows: the short matrices share a launch, the long one goes its own way; the bits are those of single calls."""
    dt, M, K, Ns = DType.BF16, 3, 2048, (4096, 256, 256)
    cases = [make_case(950 + j, dt, 4, 64, M, N, K) for j, N in enumerate(Ns)]
    x = GpuBuffer.from_bytes(cases[0].x_bytes)
    ws, ss, bs = ([GpuBuffer.from_bytes(v) for v in part] for part in zip(*((c.w.tobytes(), c.scales_bytes, c.biases_bytes) for c in cases)))
    outs, singles = ([GpuBuffer(M * N * 2) for N in Ns] for _ in range(2))
    kernels = [ops.plan("qmm", dt, 4, 64, M, N, K)[1][0][0] for N in Ns]
    assert "qmv_runs" not in kernels[0] and all("qmv_runs" in k for k in kernels[1:])
    ops.qmm_batched(dt, 4, 64, ws, ss, bs, x, outs, list(Ns), M, K)
    for j, N in enumerate(Ns):
        ops.qmm(dt, 4, 64, ws[j], ss[j], bs[j], x, singles[j], M, N, K)
        got = outs[j].read_bytes(M * N * 2)
        assert got == singles[j].read_bytes(M * N * 2) and np.any(unpack_f32(got, dt) != 0.0), j
    for b in [x] + ws + ss + bs + outs + singles:
        b.free()
