"""The GEMV on codes (mtq_qmm and mtq_qmm_batched, batches of up to 128 rows where the tile kernels cannot split the rows): the edges
of its tiles of 32 weight rows, of its 16-row operand tiles and its tiles of 48 activation rows, of its steps of 128 codes over the waves
and workgroups that share them and of its groups, against the f64-accumulated oracle.

Bound: exact-dequant arithmetic, so what is left is the rounding of the result (2^-8 of it in bf16, 2^-11 in f16), f32 sums, and the
offset of up to 256 that the conversion adds to a code and takes out again (2^-24 * 256 * sqrt(K) * scale (0.1) * |x| (5) = 5e-4 absolute at
K = 4736). max |a-e| / max(|e|, 1) <= 1e-2 (bf16), 3e-3 (f16)."""
import numpy as np
import pytest

from metaltile_amd import DType, GpuBuffer, ops, pack_f32, unpack_f32
from metaltile_amd.runtime import _ensure_init
from metaltile_amd.synth import make_case
from tests.parity import rel_err

pytestmark = pytest.mark.gpu
TOL = {DType.F16: 3e-3, DType.BF16: 1e-2}
GUARD = b"\xcd" * 64


@pytest.fixture
def codes():
    lib = _ensure_init()
    assert lib.mtq_set_option(b"qmv.codes", 2) == 0
    yield lib
    for name in (b"qmv.codes", b"qmv.codes_kw", b"qmv.codes_nw", b"qmv.codes_stage", b"qmv.codes_slices", b"scratch.most_kb"):
        lib.mtq_set_option(name, 0)


def run(oracle, dt, bits, G, M, K, Ns, more=0.0):
    """Batched and single results against the oracle, to `more` than the bound above; their bytes."""
    cases = [make_case(800 + j + M, dt, bits, G, M, N, K, bias_rule="midpoint") for j, N in enumerate(Ns)]
    x = GpuBuffer.from_bytes(cases[0].x_bytes)
    mats = [[GpuBuffer.from_bytes(v) for v in (c.w.tobytes(), c.scales_bytes, c.biases_bytes)] for c in cases]
    outs = [GpuBuffer.from_bytes(b"\xff" * (M * N * 2) + GUARD) for N in Ns]
    ops.qmm_batched(dt, bits, G, *[list(v) for v in zip(*mats)], x, outs, list(Ns), M, K)
    got = []
    for j, (c, N) in enumerate(zip(cases, Ns)):
        raw = outs[j].read_bytes(M * N * 2 + 64)
        assert raw[-64:] == GUARD, j
        exp = oracle.qmm_f64(c.w, c.scales_f, c.biases_f, cases[0].x_f, M, N, K, bits, G).reshape(-1)
        assert rel_err(unpack_f32(raw[:-64], dt), exp) <= TOL[dt] + more, j
        single = GpuBuffer(M * N * 2)
        ops.qmm(dt, bits, G, *mats[j], x, single, M, N, K)
        assert single.read_bytes(M * N * 2) == raw[:-64], j
        single.free()
        got.append(raw[:-64])
    for b in [x] + outs + sum(mats, []):
        b.free()
    return got


@pytest.mark.parametrize("dt", [DType.F16, DType.BF16], ids=lambda d: d.name)
@pytest.mark.parametrize("bits,G,M,K,Ns,kw,stage,slices", [
    (3, 64, 1, 128, (1, 40), 0, 0, 0), (5, 32, 16, 384, (33, 16), 0, 1, 0), (6, 128, 17, 1152, (129, 7, 50), 4, 0, 2), (2, 64, 32, 1280, (272, 15), 0, 2, 0),
    (4, 128, 33, 4736, (100,), 0, 0, 7), (8, 32, 48, 640, (48, 17, 1, 100), 2, 0, 0), (3, 128, 49, 2176, (37,), 1, 0, 3), (5, 64, 77, 4096, (300, 9), 0, 0, 0),
    (6, 32, 97, 896, (257, 40), 1, 1, 0), (2, 32, 128, 256, (24,), 2, 0, 1), (8, 128, 24, 3712, (20,), 0, 0, 0), (4, 64, 145, 512, (65, 32), 1, 2, 2),
])
def test_edges(oracle, codes, dt, bits, G, M, K, Ns, kw, stage, slices):
    print(f"[case] codes qmm {dt.name} b{bits} g{G} M{M} K{K} N={Ns} kw{kw} stage{stage} slices{slices}", flush=True)
    for name, v in ((b"qmv.codes_kw", kw), (b"qmv.codes_stage", stage), (b"qmv.codes_slices", slices)):
        assert codes.mtq_set_option(name, v) == 0
    assert "qmv_codes_kernel" in ops.plan("qmm", dt, bits, G, M, Ns[0], K)[1][0][0]
    run(oracle, dt, bits, G, M, K, Ns)


@pytest.mark.parametrize("kb", [0, 24, 1])
def test_without_memory_for_the_sums(oracle, codes, kb):
    """With memory for the slices' sums of one matrix at a time (14 and 20 KB) or of none: the same bits alone and in a batch.
    With none they come from the tile kernels, whose weights are rounded to 2^-9 of themselves: six deviations of a sum of K such errors,
    6 * 2^-9 / sqrt(3) * rms w (0.19: scale 0.021, code less midpoint 9.2) * sqrt(K), are 0.045."""
    print(f"[case] codes qmm, {kb} KB of scratch", flush=True)
    assert codes.mtq_set_option(b"qmv.codes_slices", 3) == 0 and codes.mtq_set_option(b"scratch.most_kb", kb) == 0
    run(oracle, DType.BF16, 5, 64, 20, 1152, (58, 83), more=0.045 if kb == 1 else 0.0)


@pytest.mark.parametrize("bits,G,M,N,K", [(5, 64, 24, 1664, 1664), (3, 32, 32, 2944, 1408), (4, 64, 33, 1152, 1152), (6, 128, 24, 4096, 8448), (8, 64, 60, 1920, 1920), (6, 128, 45, 18944, 1024), (8, 64, 40, 72, 16640)])
def test_chosen(oracle, bits, G, M, N, K):
    print(f"[case] chosen codes qmm b{bits} g{G} M{M} N{N} K{K}", flush=True)
    assert "qmv_codes_kernel" in ops.plan("qmm", DType.BF16, bits, G, M, N, K)[1][0][0]
    run(oracle, DType.BF16, bits, G, M, K, (N,))


@pytest.mark.parametrize("dt", [DType.F16, DType.BF16], ids=lambda d: d.name)
@pytest.mark.parametrize("bits,G,M,N,K,slices", [(3, 64, 20, 40, 1152, 0), (6, 32, 48, 100, 768, 0), (8, 128, 8, 33, 1280, 0), (2, 64, 60, 20, 512, 0), (5, 64, 24, 70, 1664, 3), (4, 32, 50, 33, 2176, 7)])
def test_infinite_activations(oracle, codes, dt, bits, G, M, N, K, slices):
    """One infinite activation in a row makes its results infinities of the weight's sign, as a product with the weights does;
    the other rows keep their bits."""
    print(f"[case] codes qmm, infinities {dt.name} b{bits} g{G} M{M} N{N} K{K} slices{slices}", flush=True)
    assert codes.mtq_set_option(b"qmv.codes_slices", slices) == 0
    c = make_case(880 + M, dt, bits, G, M, N, K, bias_rule="midpoint")
    x = c.x_f.reshape(M, K).copy()
    plain = x.copy()
    x[1, K // 3] = np.inf
    bufs = [GpuBuffer.from_bytes(v) for v in (c.w.tobytes(), c.scales_bytes, c.biases_bytes)]
    got = []
    for v in (x, plain):
        xb, out = GpuBuffer.from_bytes(pack_f32(v.reshape(-1), dt)), GpuBuffer(M * N * 2)
        ops.qmm(dt, bits, G, *bufs, xb, out, M, N, K)
        got.append(unpack_f32(out.read_bytes(M * N * 2), dt).reshape(M, N))
        xb.free()
        out.free()
    one = np.zeros((1, K), np.float32)
    one[0, K // 3] = 1.0
    w = oracle.qmm_f64(c.w, c.scales_f, c.biases_f, one, 1, N, K, bits, G).reshape(-1)
    with np.errstate(invalid="ignore"):
        np.testing.assert_array_equal(got[0][1], (w * np.inf).astype(np.float32))
    rest = [m for m in range(M) if m != 1]
    np.testing.assert_array_equal(got[0][rest], got[1][rest])
    for v in bufs:
        v.free()
