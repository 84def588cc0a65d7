"""The GEMV that holds its activations in LDS (mtq_rms_norm_qmv, mtq_gated_rms_norm_qmv, mtq_qmv_batched on row lengths the other fused
kernels do not take, batches of 2..16 rows of 2-, 3-, 5- and 6-bit codes): the edges of its blocks of 16 weight rows, of its pairs of
steps of 128 codes over the waves that share them, of its groups and of its stream over several blocks, against the f64-accumulated oracle.

Bound: exact-dequant arithmetic, so what is left is the rounding of the result (2^-8 of it in bf16, 2^-11 in f16), f32 sums, and the
offset of up to 256 that the conversion adds to a code and takes out again (2^-24 * 256 * sqrt(K) * scale (0.1) * |x| (5) = 5e-4 absolute at
K = 4736). A normalised row keeps 16 significant bits. max |a-e| / max(|e|, 1) <= 1e-2 (bf16), 3e-3 (f16)."""
import numpy as np
import pytest

from metaltile_amd import DType, GpuBuffer, ops, pack_f32, unpack_f32
from metaltile_amd.dtypes import round_through
from metaltile_amd.runtime import _ensure_init
from metaltile_amd.synth import make_case, pack_codes
from tests.parity import rel_err

pytestmark = pytest.mark.gpu
TOL = {DType.F16: 3e-3, DType.BF16: 1e-2}
ODT = {DType.F16: 1, DType.BF16: 2}
GUARD = b"\xcd" * 64


@pytest.fixture
def held():
    lib = _ensure_init()
    assert lib.mtq_set_option(b"qmv.held", 2) == 0
    yield lib
    for name in (b"qmv.held", b"qmv.held_kp", b"qmv.held_nb"):
        lib.mtq_set_option(name, 0)


def upload(c):
    return [GpuBuffer.from_bytes(v) for v in (c.w.tobytes(), c.scales_bytes, c.biases_bytes)]


def check(oracle, c, x_f, buf, dt, M, N, K, bits, G):
    raw = buf.read_bytes(M * N * 2 + 64)
    assert raw[-64:] == GUARD
    exp = oracle.qmm_f64(c.w, c.scales_f, c.biases_f, x_f, M, N, K, bits, G).reshape(-1)
    assert rel_err(unpack_f32(raw[:-64], dt), exp) <= TOL[dt]
    return raw[:-64]


@pytest.mark.parametrize("dt", [DType.F16, DType.BF16], ids=lambda d: d.name)
@pytest.mark.parametrize("bits,G,M,K,Ns,kp,nb", [
    (3, 64, 1, 128, (1, 40), 0, 0), (5, 32, 2, 384, (33, 16), 0, 0), (6, 128, 3, 1152, (129, 7, 50), 4, 1), (2, 64, 16, 1280, (272, 15), 0, 0),
    (4, 128, 1, 4736, (2050,), 8, 0), (8, 32, 4, 640, (48, 17, 1, 100), 2, 2), (3, 128, 9, 2176, (37,), 1, 3), (5, 64, 8, 4096, (1000,), 0, 0),
    (6, 64, 5, 896, (5000, 40), 1, 1), (2, 32, 1, 8192, (24,), 16, 1), (8, 128, 2, 3712, (20,), 0, 0), (4, 32, 1, 256, (30000, 5000), 1, 2),
])
def test_edges(oracle, held, dt, bits, G, M, K, Ns, kp, nb):
    print(f"[case] held qmv {dt.name} b{bits} g{G} M{M} K{K} N={Ns} kp{kp} nb{nb}", flush=True)
    assert held.mtq_set_option(b"qmv.held_kp", kp) == 0 and held.mtq_set_option(b"qmv.held_nb", nb) == 0
    cases = [make_case(700 + j + M, dt, bits, G, M, N, K, bias_rule="midpoint") for j, N in enumerate(Ns)]
    x = GpuBuffer.from_bytes(cases[0].x_bytes)
    mats = [upload(c) for c in cases]
    outs = [GpuBuffer.from_bytes(b"\xff" * (M * N * 2) + GUARD) for N in Ns]
    lists = [list(v) for v in zip(*mats)]
    if M == 1:
        assert "qmv_held_kernel" in ops.plan("qmv", dt, bits, G, 1, Ns[0], K)[1][0][0]
        ops.qmv_batched(dt, bits, G, *lists, x, outs, list(Ns), K)
    else:
        assert "qmv_held_kernel" in ops.plan("qmm", dt, bits, G, M, Ns[0], K)[1][0][0]
        ops.qmm_batched(dt, bits, G, *lists, x, outs, list(Ns), M, K)
    for j, (c, N) in enumerate(zip(cases, Ns)):
        raw = check(oracle, c, cases[0].x_f, outs[j], dt, M, N, K, bits, G)
        if M > 1:   # a matrix gives the same bits alone and in a batch
            single = GpuBuffer(M * N * 2)
            ops.qmm(dt, bits, G, *mats[j], x, single, M, N, K)
            assert single.read_bytes(M * N * 2) == raw, j
            single.free()
    for b in [x] + outs + sum(mats, []):
        b.free()


@pytest.mark.parametrize("dt", [DType.F16, DType.BF16], ids=lambda d: d.name)
@pytest.mark.parametrize("bits,G,N,K", [(4, 64, 40, 128), (4, 128, 129, 1152), (3, 32, 2050, 1280), (5, 64, 1, 2304), (6, 128, 300, 4736), (8, 64, 37, 1664), (2, 64, 500, 7808)])
def test_rms_norm(oracle, held, dt, bits, G, N, K):
    print(f"[case] held rms_norm_qmv {dt.name} b{bits} g{G} N{N} K{K}", flush=True)
    c = make_case(740 + bits, dt, bits, G, 1, N, K, bias_rule="midpoint")
    rng = np.random.default_rng(K)
    nw = oracle.round_through((1.0 + 0.1 * rng.standard_normal(K)).astype(np.float32), ODT[dt])
    eps = np.float32(1e-5)
    x = c.x_f.reshape(-1).astype(np.float64)
    normed = (x / np.sqrt(np.mean(x * x) + float(eps)) * nw).astype(np.float64).reshape(1, K)
    bufs = upload(c) + [GpuBuffer.from_bytes(c.x_bytes), GpuBuffer.from_bytes(pack_f32(nw, dt)), GpuBuffer.from_bytes(eps.tobytes()), GpuBuffer.from_bytes(b"\xff" * (N * 2) + GUARD)]
    w, s, b, xb, nb, eb, out = bufs
    assert "qmv_held_kernel" in ops.plan("rms_norm_qmv", dt, bits, G, 1, N, K)[1][0][0]
    ops.rms_norm_qmv(dt, bits, G, xb, nb, w, s, b, out, eb, N, K)
    check(oracle, c, normed.astype(np.float32), out, dt, 1, N, K, bits, G)
    for v in bufs:
        v.free()


@pytest.mark.parametrize("dt", [DType.F16, DType.BF16], ids=lambda d: d.name)
@pytest.mark.parametrize("G,N,hv,dv", [(64, 40, 1, 128), (128, 129, 9, 128), (32, 2050, 12, 128), (64, 1, 24, 16), (128, 300, 3, 1024), (64, 500, 40, 128)])
def test_gated_norm(oracle, held, dt, G, N, hv, dv):
    K = hv * dv
    print(f"[case] held gated_rms_norm_qmv {dt.name} g{G} N{N} hv{hv} dv{dv}", flush=True)
    c = make_case(760 + hv, dt, 4, G, 1, N, K, bias_rule="midpoint")
    rng = np.random.default_rng(K)
    y = rng.standard_normal((hv, dv)).astype(np.float32)
    z = oracle.round_through(rng.standard_normal((hv, dv)).astype(np.float32), ODT[dt])
    nw = oracle.round_through((1.0 + 0.1 * rng.standard_normal(dv)).astype(np.float32), ODT[dt])
    eps = np.float32(1e-5)
    yd, zd = y.astype(np.float64), z.astype(np.float64)
    row = yd / np.sqrt(np.mean(yd * yd, axis=1, keepdims=True) + float(eps)) * nw * zd / (1.0 + np.exp(-zd))
    bufs = upload(c) + [GpuBuffer.from_bytes(v) for v in (y.tobytes(), pack_f32(z.reshape(-1), dt), pack_f32(nw, dt), eps.tobytes(), b"\xff" * (N * 2) + GUARD)]
    w, s, b, yb, zb, nb, eb, out = bufs
    ops.gated_rms_norm_qmv(dt, G, yb, zb, nb, eb, w, s, b, out, hv, dv, N)
    check(oracle, c, row.reshape(1, K).astype(np.float32), out, dt, 1, N, K, 4, G)
    for v in bufs:
        v.free()


@pytest.mark.parametrize("dt", [DType.F16, DType.BF16], ids=lambda d: d.name)
@pytest.mark.parametrize("bits,G,M,N,K", [(3, 64, 3, 40, 1152), (6, 32, 8, 300, 768), (8, 128, 2, 33, 1280), (2, 64, 16, 20, 512),
                                          (5, 64, 2, 30000, 384), (2, 32, 4, 20000, 1280)])   # (several blocks to a wave: the next one's weights are asked for again)
def test_infinite_activations(oracle, held, dt, bits, G, M, N, K):
    """One infinite activation in a row makes its results infinities of the weight's sign, as a product with the weights does;
    the other rows keep their bits."""
    print(f"[case] held qmv, infinities {dt.name} b{bits} g{G} M{M} N{N} K{K}", flush=True)
    c = make_case(780 + M, dt, bits, G, M, N, K, bias_rule="midpoint")
    x = c.x_f.reshape(M, K).copy()
    plain = x.copy()
    x[1, K // 3] = np.inf
    bufs = upload(c)
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


@pytest.mark.parametrize("dt", [DType.F16, DType.BF16], ids=lambda d: d.name)
@pytest.mark.parametrize("bits,G,N,K,what", [(3, 64, 300, 1152, "row"), (5, 32, 9000, 640, "weight"), (4, 128, 40, 2304, "weight")])
def test_infinities_in_the_norm(dt, bits, G, N, K, what):
    """An infinite element of the row leaves no finite result, an infinite norm weight one where the matrix's element is 0 at most: the
    same elements are finite as without this kernel."""
    print(f"[case] held rms_norm_qmv, infinite {what} {dt.name} b{bits} g{G} N{N} K{K}", flush=True)
    c = make_case(790 + bits, dt, bits, G, 1, N, K, bias_rule="midpoint")
    x, nw = c.x_f.reshape(-1).copy(), np.ones(K, np.float32)
    (x if what == "row" else nw)[K // 3] = np.inf
    bufs = upload(c) + [GpuBuffer.from_bytes(v) for v in (pack_f32(x, dt), pack_f32(nw, dt), np.float32(1e-5).tobytes())]
    w, s, b, xb, nb, eb = bufs
    out, lib, got = GpuBuffer(N * 2), _ensure_init(), []
    for option in (2, 1):
        assert lib.mtq_set_option(b"qmv.held", option) == 0
        try:
            assert ("qmv_held_kernel" in ops.plan("rms_norm_qmv", dt, bits, G, 1, N, K)[1][0][0]) == (option == 2)
            ops.rms_norm_qmv(dt, bits, G, xb, nb, w, s, b, out, eb, N, K)
            got.append(np.isfinite(unpack_f32(out.read_bytes(N * 2), dt)))
        finally:
            lib.mtq_set_option(b"qmv.held", 0)
    assert not got[0].any()
    np.testing.assert_array_equal(got[0], got[1])
    for v in bufs + [out]:
        v.free()


@pytest.mark.parametrize("op,dt,bits,N,K", [
    ("norm", DType.F16, 4, 512, 2304), ("norm", DType.F16, 2, 512, 4096), ("norm", DType.BF16, 4, 512, 2304), ("norm", DType.F16, 5, 512, 2304), ("norm", DType.F16, 8, 512, 1152),
    ("batch", DType.F16, 4, 512, 1024), ("batch", DType.F16, 8, 512, 512), ("batch", DType.BF16, 8, 512, 512), ("batch", DType.F16, 3, 512, 1152),
])
def test_no_more_of_the_codes_offset_than_before(op, dt, bits, N, K):
    """The error of the f32 sums, bare of the result's rounding: the biases of a row's last two groups are set so that its exact
    result is all but 0. The root of its mean square over N rows is no larger than that of the kernels that take these calls without this
    one (half as much again: both are estimates, and the orders of their sums differ), or 2^-20 of what a row's result is without
    those biases: a hundredth of an f16 rounding, and what sums of some hundred f32 terms leave in any order."""
    G, n = 64, K // 64
    rng = np.random.default_rng(K + bits)
    codes = rng.integers(0, 1 << bits, size=(N, n, G), dtype=np.uint8)
    scale = round_through((0.02 * np.abs(rng.standard_normal((N, n))) + 1e-3).astype(np.float32).reshape(-1), dt).reshape(N, n)
    bias = round_through((-(1 << (bits - 1)) * scale + 1e-3 * rng.standard_normal((N, n))).astype(np.float32).reshape(-1), dt).reshape(N, n)
    x = rng.standard_normal((n, G)).astype(np.float32)
    x[-2:] = np.abs(x[-2:])
    x = round_through(x.reshape(-1), dt).reshape(n, G)
    v = x.astype(np.float64) / (np.sqrt(np.mean(x.astype(np.float64) ** 2) + float(np.float32(1e-5))) if op == "norm" else 1.0)
    plain = np.sqrt(np.mean((scale[:, :, None] * codes + bias[:, :, None]) ** 2) * (v * v).sum())
    part = scale * np.einsum("rgk,gk->rg", codes.astype(np.float64), v)
    for g in (-2, -1):
        rest = part.sum(1) + (np.delete(bias, n + g, 1).astype(np.float64) * np.delete(v, n + g, 0).sum(1)).sum(1)
        bias[:, g] = round_through((-rest / v[g].sum()).astype(np.float32), dt)
    exact = part.sum(1) + (bias.astype(np.float64) * v.sum(1)).sum(1)
    bufs = [GpuBuffer.from_bytes(t) for t in (pack_codes(codes.reshape(N, K), bits).tobytes(), pack_f32(scale.reshape(-1), dt), pack_f32(bias.reshape(-1), dt),
                                              pack_f32(x.reshape(-1), dt), pack_f32(np.ones(K, np.float32), dt), np.float32(1e-5).tobytes())]
    w, s, b, xb, nw, eps = bufs
    out = GpuBuffer(2 * N * 2)
    lib = _ensure_init()
    rms = []
    for held in (1, 0):
        assert lib.mtq_set_option(b"qmv.held", held) == 0
        try:
            if op == "norm":
                assert ("qmv_held_kernel" in ops.plan("rms_norm_qmv", dt, bits, G, 1, N, K)[1][0][0]) == (held == 0)
                ops.rms_norm_qmv(dt, bits, G, xb, nw, w, s, b, out, eps, N, K)
            else:
                ops.qmv_batched(dt, bits, G, [w, w], [s, s], [b, b], xb, [out.ptr, out.ptr + N * 2], [N, N], K)
            got = unpack_f32(out.read_bytes(N * 2), dt).astype(np.float64)
        finally:
            lib.mtq_set_option(b"qmv.held", 0)
        rms.append(np.sqrt(np.mean((got - exact) ** 2)))
    print(f"[case] {op} {dt.name} b{bits} {N} x {K}: {rms[0]:.2e} without, {rms[1]:.2e} with, of {plain:.2f}", flush=True)
    assert rms[1] <= max(1.5 * rms[0], 2.0 ** -20 * plain)
    for v in bufs + [out]:
        v.free()
