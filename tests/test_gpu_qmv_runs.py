"""The K-run matrix-core GEMV (mtq_qmm and mtq_qmm_batched at 2..16 rows): the edges of its blocks of 16 weight rows, of its
steps of 128 (64) codes over sixteen waves, of its groups and of the batch, against the f64-accumulated oracle.

Bound: exact-dequant arithmetic, so what is left is the rounding of the result (half a unit in its last place: at
most 2^-8 of it in bf16, 2^-11 in f16) and f32 sums; the conversion adds up to 1024 to a code and takes it out again, which
for K = 8192 and |x| up to 5 leaves at most about 2^-24 * 1024 * sqrt(K) * scale (0.1) = 6e-4 absolute. max |a-e| / max(|e|, 1) <= 1e-2 (bf16), 3e-3 (f16)."""
import numpy as np
import pytest

from metaltile_amd import DType, GpuBuffer, ops, pack_f32, unpack_f32
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


@pytest.mark.parametrize("dt,bits,G,M,K,Ns,instance", [
    (DType.BF16, 4, 64, 16, 1024, (14000, 9001, 1600), "1, 3"), (DType.F16, 4, 32, 6, 384, (24601,), "1, 3"),
    (DType.F16, 4, 128, 9, 2176, (9001, 7600), "2, 2"), (DType.BF16, 8, 64, 16, 1152, (9001, 8000), "2, 2"),
    (DType.BF16, 4, 64, 5, 5120, (7001, 6000), "3, 1"), (DType.F16, 4, 32, 16, 6272, (7001, 5400), "4, 1"),
    (DType.BF16, 8, 128, 7, 3072, (7001, 6000), "4, 1"), (DType.F16, 8, 32, 3, 4224, (12401,), "5, 1"),
    (DType.BF16, 8, 64, 16, 1024, (14000, 9001), "1, 3"), (DType.F16, 8, 32, 2, 384, (24601,), "1, 3"), (DType.BF16, 8, 128, 5, 640, (24601,), "1, 3"),
    (DType.BF16, 4, 64, 8, 4096, (9001, 7600), "2, 2"), (DType.F16, 4, 32, 3, 2176, (16601,), "2, 2"),   # up to 8 rows: no order between the waves' loads
])
def test_many_blocks_per_workgroup(oracle, dt, bits, G, M, K, Ns, instance):
    """The walk: with PF blocks in flight ahead, every workgroup of the 256 has PF + 2 blocks of 16 weight rows or more, so
    every slot of the ring and both halves of the sums' buffer are used again. A matrix begins inside the wrap, and the last block
    of each is ragged. (The instances' last two numbers are the steps of a run and PF.)"""
    print(f"[case] K-run qmv walk {dt.name} b{bits} g{G} M{M} K{K} N={Ns}", flush=True)
    assert sum(-(-N // 16) for N in Ns) >= 256 * (int(instance[-1]) + 2)
    lib = _ensure_init()
    cases = [make_case(930 + j + M, dt, bits, G, M, N, K, bias_rule="midpoint") for j, N in enumerate(Ns)]
    x = GpuBuffer.from_bytes(cases[0].x_bytes)
    ws, ss, bs = ([GpuBuffer.from_bytes(v) for v in part] for part in zip(*((c.w.tobytes(), c.scales_bytes, c.biases_bytes) for c in cases)))
    guard = b"\xcd" * 64
    outs = [GpuBuffer.from_bytes(b"\xff" * (M * N * 2) + guard) for N in Ns]
    try:
        assert lib.mtq_set_option(b"qmv.runs", 2) == 0
        assert f"{bits}, {G}, {instance}>" in ops.plan("qmm", dt, bits, G, M, Ns[0], K)[1][0][0]
        ops.qmm_batched(dt, bits, G, ws, ss, bs, x, outs, list(Ns), M, K)
        for j, (c, N) in enumerate(zip(cases, Ns)):
            raw = outs[j].read_bytes(M * N * 2 + 64)
            assert raw[-64:] == guard
            exp = oracle.qmm_f64(c.w, c.scales_f, c.biases_f, cases[0].x_f, M, N, K, bits, G, threads=8).reshape(-1)
            assert rel_err(unpack_f32(raw[:-64], dt), exp) <= TOL[dt], j
    finally:
        lib.mtq_set_option(b"qmv.runs", 0)
        for b in [x] + ws + ss + bs + outs:
            b.free()


@pytest.mark.parametrize("dt,bits,G,M,K,Ns", [
    (DType.BF16, 4, 64, 3, 4096, (4096, 1024, 1024)), (DType.F16, 4, 128, 4, 5120, (5120, 5120, 5120)), (DType.BF16, 4, 32, 3, 6144, (6144, 50)),
    (DType.F16, 4, 64, 4, 1024, (1000, 12288)), (DType.BF16, 8, 64, 4, 3584, (3584, 512, 512)), (DType.F16, 8, 32, 3, 5120, (6144, 8192)), (DType.BF16, 4, 64, 4, 4480, (16384, 9001)),
])
def test_layers_of_three_and_four_rows(oracle, dt, bits, G, M, K, Ns):
    """The projections of dense layers by the rule of sizes, no option set: one launch, exact results, the bits of single calls."""
    print(f"[case] K-run qmv layer {dt.name} b{bits} g{G} M{M} K{K} N={Ns}", flush=True)
    cases = [make_case(970 + j + M, dt, bits, G, M, N, K, bias_rule="midpoint") for j, N in enumerate(Ns)]
    x = GpuBuffer.from_bytes(cases[0].x_bytes)
    ws, ss, bs = ([GpuBuffer.from_bytes(v) for v in part] for part in zip(*((c.w.tobytes(), c.scales_bytes, c.biases_bytes) for c in cases)))
    guard = b"\xcd" * 64
    outs = [GpuBuffer.from_bytes(b"\xff" * (M * N * 2) + guard) for N in Ns]
    assert all("qmv_runs_kernel" in ops.plan("qmm", dt, bits, G, M, N, K)[1][0][0] for N in Ns)
    ops.qmm_batched(dt, bits, G, ws, ss, bs, x, outs, list(Ns), M, K)
    for j, (c, N) in enumerate(zip(cases, Ns)):
        raw = outs[j].read_bytes(M * N * 2 + 64)
        assert raw[-64:] == guard
        exp = oracle.qmm_f64(c.w, c.scales_f, c.biases_f, cases[0].x_f, M, N, K, bits, G, threads=8).reshape(-1)
        assert rel_err(unpack_f32(raw[:-64], dt), exp) <= TOL[dt], j
        single = GpuBuffer(M * N * 2)
        ops.qmm(dt, bits, G, ws[j], ss[j], bs[j], x, single, M, N, K)
        assert single.read_bytes(M * N * 2) == raw[:-64], j
        single.free()
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


@pytest.mark.parametrize("dt", [DType.F16, DType.BF16], ids=lambda d: d.name)
@pytest.mark.parametrize("bits,G,M,N,K", [(4, 64, 16, 272, 4096), (4, 128, 9, 33, 5120), (4, 32, 3, 48, 2048), (8, 64, 12, 100, 3584), (8, 32, 5, 20, 1152)])
def test_infinite_and_huge_activations(dt, bits, G, M, N, K):
    """One infinite activation in a row makes its results infinities of the weight's sign, as a product with the weights does, and
    a bf16 one of 1e37 (which the conversion's offset would carry past the f32 range) stays a number: the roundings of the weights
    (2^-9 |w|, |w| about 0.08: 6e-3 rms on a sum of 4096) and of the result, to 3e-2. A NaN stays one. Rows without such a value
    keep their bits."""
    print(f"[case] K-run qmv, infinities {dt.name} b{bits} g{G} M{M} N{N} K{K}", flush=True)
    lib = _ensure_init()
    c = make_case(970 + M, dt, bits, G, M, N, K, bias_rule="midpoint")
    plain = c.x_f.reshape(M, K).astype(np.float32)
    x = plain.copy()
    if dt == DType.BF16:
        x[0, K - 1] = 1e37
    x[1, K // 3] = np.inf
    x[2, 5] = -np.inf
    if M > 3:
        x[M - 1, K // 2] = np.nan
    codes = ((c.w.reshape(N, -1, 1) >> np.arange(0, 32, bits, dtype=np.uint32)) & ((1 << bits) - 1)).reshape(N, K).astype(np.float32)
    s, b = (np.repeat(v.reshape(N, K // G), G, axis=1).astype(np.float32) for v in (c.scales_f, c.biases_f))
    w = unpack_f32(pack_f32((codes * s + b).reshape(-1), dt), dt).reshape(N, K).astype(np.float64)
    bufs = [GpuBuffer.from_bytes(v) for v in (c.w.tobytes(), c.scales_bytes, c.biases_bytes)]
    got = []
    try:
        assert lib.mtq_set_option(b"qmv.runs", 2) == 0
        assert "qmv_runs_kernel" in ops.plan("qmm", dt, bits, G, M, N, K)[1][0][0]
        for v in (x, plain):
            xb, out = GpuBuffer.from_bytes(pack_f32(v.reshape(-1), dt)), GpuBuffer(M * N * 2)
            ops.qmm(dt, bits, G, *bufs, xb, out, M, N, K)
            got.append(np.frombuffer(out.read_bytes(M * N * 2), dtype="<u2").reshape(M, N).copy())
            xb.free()
            out.free()
    finally:
        lib.mtq_set_option(b"qmv.runs", 0)
        for v in bufs:
            v.free()
    values = unpack_f32(got[0].tobytes(), dt).reshape(M, N)
    assert rel_err(values[0], w @ unpack_f32(pack_f32(x[0], dt), dt).astype(np.float64)) <= 3e-2
    with np.errstate(invalid="ignore"):
        for row, k in ((1, K // 3), (2, 5)):
            np.testing.assert_array_equal(values[row], (w[:, k] * np.float64(x[row, k])).astype(np.float32))
    rest = [m for m in range(M) if np.array_equal(x[m], plain[m])]
    np.testing.assert_array_equal(got[0][rest], got[1][rest])
    if M > 3:
        assert np.all(np.isnan(values[M - 1]))


@pytest.mark.parametrize("which", ["w", "scales", "biases", "x", "out"])
def test_operands_off_16_bytes(oracle, which):
    """An operand at 8 bytes past a multiple of 16 (a slice of a larger buffer): the loads of 16 bytes are not for it, so another
    kernel takes the call (the K-run kernel's stores are of single elements: `out` may lie anywhere). f16, K = 512: those that round the weight to
    the element type first add about 2^-12 * |w| (0.1 rms) * sqrt(K) * |x| = 6e-4 rms; 1e-2."""
    dt, bits, G, M, N, K = DType.F16, 4, 64, 16, 72, 512
    print(f"[case] K-run qmv, {which} off 16 bytes", flush=True)
    c = make_case(990, dt, bits, G, M, N, K, bias_rule="midpoint")
    off = {n: 8 if n == which else 0 for n in ("w", "scales", "biases", "x", "out")}
    data = dict(w=c.w.tobytes(), scales=c.scales_bytes, biases=c.biases_bytes, x=c.x_bytes, out=b"\xff" * (M * N * 2))
    bufs = {n: GpuBuffer.from_bytes(b"\xcd" * off[n] + v + b"\xcd" * 64) for n, v in data.items()}
    at = {n: bufs[n].ptr + off[n] for n in bufs}
    exp = oracle.qmm_f64(c.w, c.scales_f, c.biases_f, c.x_f, M, N, K, bits, G).reshape(-1)
    for batch in (False, True):
        bufs["out"].upload(np.full(off["out"] + M * N * 2 + 64, 0xCD, np.uint8))
        if batch:
            ops.qmm_batched(dt, bits, G, [at["w"]], [at["scales"]], [at["biases"]], at["x"], [at["out"]], [N], M, K)
        else:
            ops.qmm(dt, bits, G, at["w"], at["scales"], at["biases"], at["x"], at["out"], M, N, K)
        raw = bufs["out"].read_bytes(off["out"] + M * N * 2 + 64)
        assert raw[:off["out"]] == b"\xcd" * off["out"] and raw[-64:] == b"\xcd" * 64
        assert rel_err(unpack_f32(raw[off["out"]:-64], dt), exp) <= 1e-2, batch
    for b in bufs.values():
        b.free()


@pytest.mark.parametrize("dt", [DType.F16, DType.BF16], ids=lambda d: d.name)
@pytest.mark.parametrize("option,bits,G,M,N,K", [
    (2, 4, 64, 16, 40, 256), (2, 4, 128, 9, 24, 768), (2, 4, 64, 5, 33, 5376), (2, 4, 32, 16, 20, 5888), (2, 4, 64, 3, 17, 6400),
    (2, 8, 64, 16, 40, 128), (2, 8, 32, 7, 24, 2176), (2, 8, 128, 16, 33, 4224), (2, 8, 64, 4, 17, 4992),
    (3, 4, 64, 16, 40, 8448), (3, 4, 128, 5, 33, 13824), (3, 8, 64, 9, 24, 5248), (3, 8, 128, 3, 40, 15232),
])
def test_pairs_of_steps(oracle, dt, option, bits, G, M, N, K):
    """Rows of whole 128-byte lines, whose steps are dealt to the waves in pairs: fewer pairs than waves, pairs that leave some waves
    one round less, single steps behind the pairs, slices of an odd number of pairs."""
    print(f"[case] K-run qmv, pairs {dt.name} b{bits} g{G} M{M} N{N} K{K}", flush=True)
    lib = _ensure_init()
    c = make_case(970 + M, dt, bits, G, M, N, K, bias_rule="midpoint")
    bufs = [GpuBuffer.from_bytes(v) for v in (c.w.tobytes(), c.scales_bytes, c.biases_bytes, c.x_bytes)]
    guard = b"\xcd" * 64
    out = GpuBuffer.from_bytes(b"\xff" * (M * N * 2) + guard)
    try:
        assert lib.mtq_set_option(b"qmv.runs", option) == 0
        name = ops.plan("qmm", dt, bits, G, M, N, K)[1][0][0]
        assert ("qmv_runs_kernel<true" if option == 2 else "qmv_slices_kernel<true") in name
        ops.qmm(dt, bits, G, *bufs, out, M, N, K)
        raw = out.read_bytes(M * N * 2 + 64)
        assert raw[-64:] == guard
        exp = oracle.qmm_f64(c.w, c.scales_f, c.biases_f, c.x_f, M, N, K, bits, G).reshape(-1)
        assert rel_err(unpack_f32(raw[:-64], dt), exp) <= TOL[dt]
    finally:
        lib.mtq_set_option(b"qmv.runs", 0)
        for b in bufs + [out]:
            b.free()
