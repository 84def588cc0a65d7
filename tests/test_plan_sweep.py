"""Routing and launch geometry without a GPU: mtq_plan runs the same code as the typed entry points and records
what they would launch. A sweep over a few thousand shapes checks every recorded launch against the limits of the
part (1024 threads per workgroup, 160 KB of LDS, grid dimensions), that every valid shape is served (the generic
kernel stands behind every specialised one), that argument validation is reached without a device, and pins the
kernels the benchmark configurations are routed to.

Counterpart of the reference's host-side checks before a dispatch is encoded
(crates/metaltile-runtime/src/dispatch/single_dispatch.rs:142-158, buffer_plan.rs:62-77).
"""
import itertools

import pytest

from metaltile_amd import DType, _lib, ops

OK, BAD_ARG, SHAPE, UNSUPPORTED = 0, -2, -3, -7
LDS_MAX = 160 * 1024


def check_launches(tag, launches, n_launches, rows=1):
    # exact-dequant batches run as passes of up to 4 (f32 dot kernels) or 8 / 16 rows over the weights
    assert 1 <= n_launches <= max(8, rows // 4 + 2), f"{tag}: {n_launches} launches"
    assert len(launches) == min(n_launches, 8)
    for kernel, grid, block, lds in launches:
        threads = block[0] * block[1] * block[2]
        assert kernel.startswith(("void mtq::", "mtq::")), f"{tag}: kernel name {kernel!r}"
        assert 1 <= threads <= 1024 and threads % 64 == 0, f"{tag}: {kernel} block {block}"
        assert 1 <= grid[0] < 2 ** 31 and 1 <= grid[1] <= 65535 and 1 <= grid[2] <= 65535, f"{tag}: {kernel} grid {grid}"
        assert grid[0] * grid[1] * grid[2] < 2 ** 32, f"{tag}: {kernel} grid {grid}"
        assert lds <= LDS_MAX, f"{tag}: {kernel} asks for {lds} B of LDS"


def valid(bits, G, N, K):
    return N > 0 and K > 0 and G > 0 and K % G == 0 and (K * bits) % 32 == 0


# row lengths of the models named in the benchmark configurations and their neighbours, and awkward ones
KS = [64, 96, 128, 320, 576, 768, 1024, 1152, 1408, 2048, 2816, 3584, 4096, 5120, 6144, 8192, 11008, 13824, 14336, 18944, 28672]
NS = [1, 7, 64, 100, 131, 333, 768, 1000, 2048, 4096, 5120, 14336, 28672, 128256]
MS = [1, 2, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 64, 65, 100, 128, 256, 300, 512, 640, 1024, 1536, 2048, 3000, 4096]


def test_qmv_qmm_sweep():
    """Every valid (dtype, bits, group, M, N, K) is served by some kernel within the part's limits."""
    n = 0
    for dt in (DType.F32, DType.F16, DType.BF16):
        for bits, G in itertools.product((2, 3, 4, 5, 6, 8), (32, 64, 128)):
            for K in KS:
                if not valid(bits, G, 1, K):
                    continue
                for N in (NS if K in (4096, 14336, 576, 11008) else (100, 4096, 14336)):
                    for M in (MS if (K, N) in ((4096, 4096), (14336, 4096), (4096, 14336), (11008, 4096)) else (1, 4, 16, 300)):
                        if M * K * 4 >= 2 ** 32 or M * N * 4 >= 2 ** 32:
                            continue
                        for op in ("qmv", "qmm", "qmm_mma") if M > 1 else ("qmv",):
                            if op == "qmv" and M > 8:
                                continue
                            tag = f"{op} {dt.name} b{bits} g{G} M{M} N{N} K{K}"
                            rc, launches, scratch, nl = ops.plan(op, dt, bits, G, M, N, K)
                            assert rc == OK, f"{tag}: rc {rc}"
                            check_launches(tag, launches, nl, M)
                            assert scratch < 2 ** 34, tag
                            n += 1
    assert n > 3000


def test_gather_and_fused_sweep():
    n = 0
    for dt in (DType.F16, DType.BF16, DType.F32):
        for bits, G in ((4, 64), (8, 64), (2, 32), (3, 64), (6, 128)):
            for N, K in ((14336, 4096), (4096, 14336), (768, 2048), (2048, 768), (1408, 2048), (100, 576)):
                if not valid(bits, G, N, K):
                    continue
                for E, T in ((8, 32), (8, 2048), (128, 8192), (64, 1), (2047, 4096), (2048, 64), (1, 300), (8, 0)):
                    for op in ("gather_csr", "gather_indices"):
                        tag = f"{op} {dt.name} b{bits} g{G} N{N} K{K} E{E} T{T}"
                        rc, launches, scratch, nl = ops.plan(op, dt, bits, G, 1, N, K, E, T)
                        assert rc == OK, f"{tag}: rc {rc}"
                        if T:
                            check_launches(tag, launches, nl)
                        else:
                            assert nl == 0
                        n += 1
                rc, launches, _, nl = ops.plan("gather_single", dt, bits, G, 1, N, K, 8)
                assert rc == OK
                check_launches(f"gather_single {dt.name} b{bits} N{N} K{K}", launches, nl)
                rc, launches, _, nl = ops.plan("rms_norm_qmv", dt, bits, G, 1, N, K)
                assert rc == OK
                check_launches(f"rms_norm_qmv {dt.name} b{bits} N{N} K{K}", launches, nl)
                if (N * bits) % 32 == 0:
                    for M in (1, 2, 8):
                        rc, launches, scratch, nl = ops.plan("qvm", dt, bits, G, M, N, K)
                        assert rc == OK
                        check_launches(f"qvm {dt.name} b{bits} M{M} N{N} K{K}", launches, nl)
                n += 3
    assert n > 500


def test_validation_without_a_device():
    P = lambda op, *a, **k: ops.plan(op, *a, **k)[0]
    assert P("qmv", 7, 4, 64, 1, 4096, 4096) == BAD_ARG          # no such dtype
    assert P("qmv", DType.BF16, 9, 64, 1, 4096, 4096) == BAD_ARG  # bits
    assert P("qmv", DType.BF16, 1, 64, 1, 4096, 4096) == BAD_ARG
    assert P("qmv", DType.BF16, 4, 64, 1, 0, 4096) == SHAPE       # N == 0
    assert P("qmv", DType.BF16, 4, 64, 1, 4096, 0) == SHAPE
    assert P("qmv", DType.BF16, 4, 0, 1, 4096, 4096) == SHAPE     # group size
    assert P("qmv", DType.BF16, 4, 96, 1, 4096, 4096) == SHAPE    # K % G
    assert P("qmm", DType.BF16, 3, 4, 16, 64, 4) == SHAPE         # K * bits % 32
    assert P("gather_csr", DType.BF16, 4, 64, 1, 4096, 4096, 0, 8) == SHAPE   # no experts
    assert P("qvm", DType.BF16, 3, 64, 1, 100, 4096) == SHAPE     # N * bits % 32
    assert P("qmv", DType.BF16, 4, 64, 0, 4096, 4096) == OK       # no rows: nothing to do
    assert ops.plan("qmv", DType.BF16, 4, 64, 0, 4096, 4096)[3] == 0


def test_benchmark_configurations_are_routed_as_documented():
    def kernels(op, *a, **k):
        rc, launches, _, _ = ops.plan(op, *a, **k)
        assert rc == OK
        return [l[0] for l in launches], launches

    ks, ls = kernels("qmv", DType.BF16, 4, 64, 1, 14336, 4096)
    assert "qmv_rows_walk_kernel<2, 2, 6, 8>" in ks[0] and ls[0][1][0] == 512 and ls[0][2][0] == 512   # two workgroups of eight waves per compute unit walk the rows
    ks, ls = kernels("qmv", DType.F16, 4, 32, 1, 4096, 4096)
    assert "qmv_rows_walk_kernel<1, 2, 5, 16>" in ks[0] and ls[0][1][0] == 256 and ls[0][2][0] == 1024   # up to 4096 rows: sixteen rows per workgroup
    ks, _ = kernels("qmv", DType.BF16, 4, 64, 1, 128256, 4096)
    assert "qmv_rows_walk_kernel<2, 2, 6, 8>" in ks[0]
    ks, _ = kernels("qmv", DType.BF16, 4, 64, 1, 57344, 4096)      # the sizes between stay on the streaming kernel
    assert "qmv_stream_kernel" in ks[0]
    ks, ls = kernels("qmv", DType.BF16, 4, 64, 1, 28672, 8192)
    assert "qmv_rows_walk_kernel<2, 4, 6, 8>" in ks[0] and ls[0][1][0] == 512
    ks, _ = kernels("qmv", DType.F16, 4, 64, 1, 1100, 4096)        # below the walk's sizes: the wave-per-four-rows kernel
    assert "qmv_rows_kernel<1, 0, false>" in ks[0]
    for args in ((DType.BF16, 4, 64, 1, 1026, 4096), (DType.BF16, 4, 32, 1, 1024, 4096), (DType.BF16, 4, 64, 2, 4096, 4096),
                 (DType.BF16, 8, 64, 1, 4096, 4096), (DType.BF16, 4, 64, 1, 512, 4096)):
        assert "qmv_rows_kernel" not in kernels("qmv", *args)[0][0]          # what that kernel does not take
    for args in ((DType.BF16, 4, 64, 2, 14336, 4096), (DType.BF16, 8, 64, 1, 14336, 4096), (DType.BF16, 2, 64, 1, 14336, 8192),
                 (DType.F32, 4, 64, 1, 14336, 4096), (DType.BF16, 4, 64, 1, 14336, 2560), (DType.BF16, 4, 16, 1, 14336, 4096), (DType.BF16, 4, 64, 1, 24576, 2048)):
        assert "qmv_rows_walk_kernel" not in kernels("qmv", *args)[0][0]     # nor the walk: one row, 4-bit, 2048 ... 8192 codes in steps of 1024 or 3584 (2048: up to 20480 rows), groups of 32 / 64 / 128
    ks, ls = kernels("qmv", DType.BF16, 4, 64, 1, 8192, 2048)
    assert "qmv_rows_walk_kernel<2, 1, 6, 8>" in ks[0] and ls[0][1][0] == 512 and ls[0][2][0] == 512
    ks, ls = kernels("qmv", DType.BF16, 4, 64, 1, 18944, 3584)      # rows that end inside a group of 64 chunks
    assert "qmv_rows_walk_ragged_kernel<2, 2, 6, 8, 48>" in ks[0] and ls[0][1][0] == 512 and ls[0][2][0] == 512
    ks, ls = kernels("qmv", DType.F16, 4, 128, 1, 4096, 6144)
    assert "qmv_rows_walk_kernel<1, 3, 7, 16>" in ks[0] and ls[0][1][0] == 256 and ls[0][2][0] == 1024
    ks, ls = kernels("qmv", DType.BF16, 4, 64, 1, 4096, 14336)
    assert "qmv_rows_long_kernel<2, 4, 7, 6>" in ks[0] and ls[0][1][0] == 512 and ls[0][2][0] == 512   # workgroups of eight rows
    ks, ls = kernels("qmv", DType.BF16, 4, 64, 1, 4096, 11008)      # a long row that ends inside a group of 64 chunks
    assert "qmv_rows_long_ragged_kernel<2, 6, 6, 24>" in ks[0] and ls[0][1][0] == 512 and ls[0][2][0] == 512
    ks, ls = kernels("qmv", DType.F16, 4, 128, 1, 3584, 18944)
    assert "qmv_rows_long_ragged_kernel<1, 10, 7, 16>" in ks[0] and ls[0][1][0] == 224 and ls[0][2][0] == 1024
    ks, _ = kernels("qmv", DType.BF16, 4, 64, 1, 5120, 27648)       # built, level with the kernel that serves it, not routed
    assert "qmv_rows" not in ks[0]
    for bits, G, name in ((2, 32, "qmv_rows_walk2_kernel<1, 2, 5, 8>"), (2, 128, "qmv_rows_walk2_kernel<1, 2, 7, 8>"), (4, 64, "qmv_rows_long_kernel<1, 4, 4, 6>")):   # the one-row cells of the width / group sweep
        ks, ls = kernels("qmv", DType.F16, bits, G, 1, 8192, 8192)
        assert name in ks[0] and ls[0][1][0] == 512, ks
    ks, ls = kernels("qmv", DType.F16, 2, 64, 1, 4096, 8192)      # fewer rows of 2-bit codes: the one-row-per-wave kernel
    assert "qmv_rows_long_kernel<1, 2, 2, 6>" in ks[0], ks
    ks, _ = kernels("qmv", DType.F16, 8, 64, 1, 8192, 8192)
    assert "qmv_rows" not in ks[0]
    # the four-row cells of the sweep: one wave per four weight rows where that is ahead (2-bit codes, 4-bit in groups of 32,
    # three or four rows of 4-bit codes); two rows of 4-bit g64 / g128, fewer weight rows and 8-bit codes stay on the matrix-core GEMV
    for bits, G, M, name in ((2, 32, 4, "<1, 2, 8, 5, false>"), (2, 64, 2, "<1, 2, 8, 6, false>"), (4, 32, 2, "<1, 4, 16, 5, false>"), (4, 64, 4, "<1, 4, 16, 6, false>"),
                             (4, 128, 3, "<1, 4, 16, 7, false>")):
        ks, ls = kernels("qmv", DType.F16, bits, G, M, 8192, 8192)
        assert "qmv_rows_few_kernel" + name in ks[0] and ls[0][1][0] == 256 and ls[0][2][0] == 1024, ks
    for args in ((DType.F16, 4, 64, 2, 8192, 8192), (DType.F16, 4, 64, 4, 4096, 8192), (DType.F16, 8, 64, 4, 8192, 8192), (DType.BF16, 4, 64, 4, 14336, 4096),
                 (DType.F16, 2, 64, 5, 8192, 8192)):
        assert "qmv_mfma_kernel" in kernels("qmv", *args)[0][0]
    ks, _ = kernels("qmv", DType.F32, 4, 64, 1, 4096, 4096)
    assert "qmv_stream_kernel<0, 4" in ks[0] or "qmv_kernel<0, 4" in ks[0]
    for M, mb in ((512, 2), (1024, 4), (2048, 8)):     # 64-, 128-, 256-row load-to-LDS tiles
        ks, ls = kernels("qmm_mma", DType.BF16, 4, 64, M, 4096, 4096)
        assert f"qmm_dma_kernel<2, {mb}, 2, 8," in ks[0], ks
        assert ls[0][1][0] == 256 and ls[0][2][0] == 512
    ks, ls = kernels("qmm_mma", DType.BF16, 4, 64, 32, 4096, 4096)
    assert "qmm_dma_kernel<2, 1, 4, 8," in ks[0]       # 32-row tiles on 4 K-groups, K split: a reduce kernel follows
    assert "qmm_split_reduce_kernel" in ks[1]
    ks, _ = kernels("qmm_mma", DType.BF16, 8, 64, 512, 4096, 4096)
    assert "qmm_dma_kernel<2, 2, 2, 8," in ks[0] and ks[0].rstrip(">(mtq::QmmDArgs)").endswith(", 8")   # 8-bit codes: the same tiles
    for bits in (4, 8):     # a down projection at 512 rows: 128 tall tiles, K split in two so that every compute unit has one
        ks, ls = kernels("qmm_mma", DType.BF16, bits, 64, 512, 4096, 14336)
        assert "qmm_dma_kernel<2, 4, 2, 8, 0, false, true, false" in ks[0] and ls[0][1][:2] == (128, 2) and "qmm_split_reduce_kernel" in ks[1]
    ks, _ = kernels("qmm_mma", DType.BF16, 6, 64, 512, 4096, 4096)
    assert "qmm_direct_kernel<2, 6," in ks[0]          # other code widths stay on the register-staged tiles
    ks, ls = kernels("gather_indices", DType.BF16, 4, 64, 1, 14336, 4096, 8, 32)   # 4 rows per expert: the routed 16-row GEMV
    assert "qmv_wide_kernel<2, 64, 2, 2, 2>" in ks[0] and ls[0][1][:2] == (28, 8) and ls[0][2][0] == 1024
    for T in (1, 2, 4):   # the down projection's experts: up to four rows on the routed one-row-per-wave kernel, eight-row workgroups
        ks, ls = kernels("gather_csr", DType.BF16, 4, 64, 1, 4096, 14336, 8, T)
        assert "qmv_rows_long_routed_kernel<2, 4, 7, 6, 1>" in ks[0] and ls[0][1][:2] == (512, T) and ls[0][2][0] == 512, ls
    ks, _ = kernels("gather_csr", DType.BF16, 4, 64, 1, 4096, 14336, 8, 5)
    assert "qmv_mfma_kernel<2, 4," in ks[0]
    ks, ls = kernels("gather_indices", DType.BF16, 4, 64, 1, 2048, 2048, 8, 1)           # the expert widths of other models walk too
    assert "qmv_rows_walk_routed_kernel<2, 1, 6, 2>" in ks[0]
    ks, ls = kernels("gather_csr", DType.BF16, 4, 64, 1, 2048, 7168, 8, 4)
    assert "qmv_rows_walk_routed_ragged_kernel<2, 4, 6, 1, 32>" in ks[0] and ls[0][1][:2] == (128, 4), ls
    ks, ls = kernels("gather_indices", DType.BF16, 4, 64, 1, 2048, 3072, 8, 1)           # other row lengths: the kernels that served them before
    assert "qmv_rows" not in ks[0]
    ks, _ = kernels("gather_indices", DType.BF16, 4, 64, 1, 14336, 4096, 8, 16)           # 2 rows per expert: 8-row passes
    assert "qmv_mfma_kernel<2, 4," in ks[0]
    for view in ("gather_csr", "gather_indices"):      # fewer rows than experts: a grid row per row, not per expert
        for T, E in ((1, 8), (2, 8), (4, 8), (7, 8), (8, 128), (32, 128)):
            ks, ls = kernels(view, DType.BF16, 4, 64, 1, 14336, 4096, E, T)
            # up to eight rows on experts of 14336 x 4096: the routed walk, about 512 workgroups over the grid rows
            kernel = "qmv_rows_walk_routed_kernel<2, 2, 6, " if T <= 8 else "qmv_mfma_kernel<2, 4,"
            assert kernel in ks[0] and ls[0][1][1] == T, (view, T, E, ls)
            if T <= 8 and E <= 64:
                assert ls[0][1][0] == 512 // T and ls[0][2][0] == 512, ls
        ks, ls = kernels("gather_single", DType.BF16, 4, 64, 1, 14336, 4096, 8, 1)
        assert "qmv_rows_walk_routed_kernel<2, 2, 6, 3>" in ks[0] and ls[0][1][:2] == (512, 1)
        ks, ls = kernels(view, DType.BF16, 4, 64, 1, 4096, 14336, 8, 2)     # rows of 14336 codes: the routed one-row-per-wave kernel
        assert "qmv_rows_long_routed_kernel<2, 4, 7, 6, " in ks[0] and ls[0][1][1] == 2, ls
        ks, ls = kernels(view, DType.BF16, 4, 64, 1, 2048, 768, 128, 33)   # (more than 32 rows: a grid row per expert)
        assert ls[0][1][1] == 128
    ks, _ = kernels("gather_indices", DType.BF16, 4, 64, 1, 4096, 4096, 8, 2048)
    assert "moe_count_sort_kernel" in ks[0] and "gather_tiles_kernel<true>" in ks[1] and "qmm_dma_routed_kernel<2, false, 4>" in ks[2]
    for bits, M in itertools.product((2, 4, 8), (1, 4)):   # the sweep configuration's cells
        for G in (32, 64, 128):
            ks, _ = kernels("qmv", DType.F16, bits, G, M, 8192, 8192)
            assert "generic" not in ks[0], (bits, G, M, ks)


@pytest.mark.parametrize("bits,M,N,K,G,tile,ksplit", [
    (6, 77, 16512, 3584, 64, 128, 3), (7, 128, 21760, 3072, 64, 128, 3),       # 129 and 170 of 256 compute units: three splits are one round
    (6, 77, 21888, 3584, 64, 128, 1), (3, 128, 28672, 8128, 64, 128, 1),       # 171 tiles and more: unsplit
    (5, 100, 18944, 2048, 64, 128, 1), (6, 66, 16384, 3584, 64, 64, 1),        # short rows; no more than half the chip
    (6, 100, 3584, 18944, 64, 128, 8), (7, 66, 4096, 9216, 64, 128, 8),        # long rows: tall tiles
    (6, 100, 8192, 9216, 64, 64, 1), (3, 66, 5120, 14336, 128, 64, 1),         # ... but not for one round of 64 x 64 tiles with staged scales
    (6, 100, 8192, 11008, 64, 128, 8), (6, 100, 8192, 8256, 64, 128, 8), (6, 100, 2048, 18944, 64, 64, 4),
])
def test_bit_stream_tiles_at_65_to_128_rows(bits, M, N, K, G, tile, ksplit):
    """The tile height and the K split of the 3-, 5-, 6- and 7-bit codes, on both sides of each line."""
    rc, launches, _, _ = ops.plan("qmm", DType.F16, bits, G, M, N, K)
    assert rc == 0
    args = launches[0][0].split("<")[1].split(", ")
    assert int(args[3]) * 32 == tile and launches[0][1][1] == ksplit, launches


@pytest.mark.parametrize("bits,M,N,K,runs", [
    (4, 2, 1024, 4096, True), (8, 2, 1024, 4096, False), (8, 3, 1024, 4096, True), (4, 4, 512, 2048, True), (4, 2, 2048, 2048, False),
    (4, 3, 512, 8192, False), (4, 2, 4096, 1024, False), (4, 5, 8192, 8192, True), (4, 9, 8192, 8192, False), (4, 16, 1024, 8192, True), (4, 9, 1025, 8192, False),
    (4, 9, 1040, 6144, True), (4, 16, 8192, 512, True), (4, 16, 8208, 512, False), (4, 8, 16384, 512, True), (8, 16, 16384, 2048, True), (4, 16, 13824, 5120, True),
    (4, 16, 16384, 5120, False), (8, 16, 14336, 4096, True), (8, 16, 16384, 4096, False), (4, 1, 1024, 4096, False), (4, 17, 1024, 4096, False),
])
def test_k_run_lines(bits, M, N, K, runs):
    """Which matrices the K-run kernel is for, on both sides of each line."""
    rc, launches, _, _ = ops.plan("qmm", DType.BF16, bits, 64, M, N, K)
    assert rc == 0 and ("qmv_runs_kernel" in launches[0][0]) == runs, launches[0][0]


@pytest.mark.parametrize("bits,G,N,K,rows", [
    (4, 64, 16384, 3584, ()), (4, 64, 16400, 3584, (2, 3, 4)), (4, 128, 24576, 2048, (2, 3, 4)), (4, 64, 24592, 2048, ()), (4, 32, 18944, 3584, ()),
    (8, 64, 16400, 3584, (3, 4)), (8, 128, 24576, 2048, (3, 4)), (4, 64, 18944, 1920, ()), (4, 64, 18304, 4096, (2, 3, 4)), (4, 64, 18320, 4096, ()),
    # up to 6144 weight rows of three steps a run (8 bits: five)
    (4, 64, 4096, 4096, (3, 4)), (8, 32, 3584, 3584, (3, 4)), (4, 128, 6144, 6144, (3, 4)), (4, 64, 6144, 6272, ()), (8, 64, 6144, 5120, (3, 4)), (8, 64, 4096, 5248, ()),
    (4, 64, 6160, 4096, ()), (4, 64, 512, 1024, (3, 4)), (4, 64, 512, 896, ()), (4, 64, 2048, 2048, (3, 4)), (4, 64, 2064, 2048, ()), (4, 32, 2064, 2176, (3, 4)), (8, 64, 2064, 2048, (3, 4)),
    # rows of more than 2048 bytes, but 4096
    (4, 64, 8192, 4096, ()), (4, 64, 8192, 4224, (3, 4)), (4, 64, 13824, 5120, (3, 4)), (4, 64, 16384, 4480, (3, 4)), (4, 64, 16400, 4480, ()), (4, 32, 8192, 5120, (3, 4)),
    (4, 32, 8208, 5120, ()), (8, 64, 16384, 3584, (3, 4)), (8, 64, 13824, 4096, ()), (8, 64, 8192, 2048, ()), (8, 64, 8192, 2176, (3, 4)), (8, 32, 8192, 2560, (3, 4)),
    # 8193 to 12288 rows
    (4, 64, 8208, 4096, (3, 4)), (4, 64, 12288, 1024, (3, 4)), (4, 64, 12304, 4096, ()), (8, 128, 12288, 4096, (3, 4)), (8, 32, 10240, 4096, (3, 4)), (4, 32, 12288, 2048, (3, 4)),
])
def test_k_run_lines_of_few_rows(bits, G, N, K, rows):
    """2, 3 and 4 rows: one rule of sizes, the same at 3 and 4, on both sides of each line."""
    on = tuple(M for M in (2, 3, 4) if "qmv_runs_kernel" in ops.plan("qmm", DType.BF16, bits, G, M, N, K)[1][0][0])
    assert on == rows


@pytest.mark.parametrize("bits", [4, 5, 8])
@pytest.mark.parametrize("M,K", [(17, 2176), (24, 2432), (20, 2944), (64, 2944)])
def test_gemv_on_codes_of_a_layer_is_one_launch(bits, M, K):
    """Matrices of an eighth, a quarter and all of the rows that a square one has: as many waves that share rows, and no slices."""
    for N in (K // 8, K // 4, K):
        _, launches, _, n = ops.plan("qmm", DType.BF16, bits, 64, M, N, K)
        assert n == 1 and "qmv_codes_kernel" in launches[0][0] and launches[0][2][0] == 512


@pytest.mark.parametrize("bits,K,paired", [(4, 1536, False), (4, 1792, True), (4, 1920, False), (4, 2048, True), (4, 2304, False), (4, 2560, True), (4, 4096, True), (4, 4352, False),
                                           (4, 5120, False), (4, 6144, False), (4, 6400, True), (4, 8192, True), (8, 1152, True), (8, 5120, True)])
def test_k_run_steps_in_pairs(bits, K, paired):
    """Which row lengths have their steps dealt to the waves in pairs, on both sides of each line."""
    for M in (5, 8) + ((9, 16) if K <= 6144 else ()):
        name = ops.plan("qmm", DType.BF16, bits, 64, M, 2048, K)[1][0][0]
        assert ("qmv_runs_kernel<true" if paired else "qmv_runs_kernel<false") in name


@pytest.mark.parametrize("bits,G,N,K,held", [
    (4, 64, 256, 2048, False), (4, 64, 1000, 4096, False), (4, 64, 1500, 8192, False), (4, 64, 512, 18432, False), (4, 64, 500, 2304, True), (4, 64, 256, 3072, True), (4, 64, 6000, 3840, True), (4, 64, 6400, 3840, False),
    (4, 64, 70000, 3200, False), (4, 64, 7000, 4224, True), (4, 64, 7000, 4736, True), (4, 64, 7000, 4864, False), (4, 64, 7000, 5248, False), (4, 32, 30000, 1408, True), (4, 32, 70000, 1664, False),
    (2, 64, 16384, 4096, True), (2, 64, 65536, 4096, True), (2, 64, 65537, 4096, False), (2, 64, 70000, 3200, False), (2, 64, 70000, 6400, True), (2, 64, 70000, 6656, False), (2, 64, 70000, 8192, True),
    (3, 64, 100000, 3456, True), (3, 64, 100000, 3584, False), (3, 64, 100000, 4224, True), (3, 64, 100000, 7936, False), (5, 64, 100000, 3968, True), (5, 64, 100000, 4096, False), (6, 64, 100000, 4096, True),
    (5, 64, 4096, 18944, True), (5, 64, 5120, 18944, False), (6, 64, 8192, 18944, True), (2, 64, 8192, 28672, False), (2, 64, 16384, 28672, True), (8, 64, 4096, 4992, True), (8, 64, 4096, 5248, False),
    (4, 64, 65537, 1792, False), (4, 64, 78643, 1792, False), (4, 64, 78644, 1792, True), (4, 64, 98304, 1792, True), (4, 64, 98305, 1792, False), (4, 64, 68000, 1664, True),
    (4, 128, 68000, 1792, True), (4, 128, 68000, 1920, False), (4, 64, 68000, 2432, True), (4, 64, 68000, 2688, False), (4, 64, 68000, 2816, True), (4, 64, 34000, 2944, True), (4, 64, 68000, 4224, True),
    (4, 32, 68000, 1024, True), (4, 32, 68000, 1152, False), (4, 32, 60000, 1152, True), (4, 32, 34000, 1408, False), (2, 64, 100651, 2944, True), (2, 32, 100651, 2944, False), (2, 32, 68000, 1792, True),
    (3, 32, 100651, 2688, True), (3, 32, 100651, 3200, False), (3, 64, 100651, 3200, True), (5, 32, 100651, 3200, False), (5, 32, 131072, 3200, True), (5, 64, 100651, 3200, True), (6, 32, 100651, 3200, True),
    (6, 32, 100651, 3712, False), (8, 32, 100651, 3200, True), (8, 32, 100651, 3712, False), (8, 32, 131072, 3712, True), (8, 64, 100651, 3712, True), (4, 32, 14000, 1664, True), (4, 32, 14500, 1664, False),
    (4, 32, 14080, 2176, True), (4, 32, 14080, 2432, False), (4, 32, 5600, 4224, True), (4, 32, 5700, 4224, False),
])
def test_held_norm_lines(bits, G, N, K, held):
    """Which RMS-normalised rows the GEMV with its activations in LDS is for, on both sides of each line."""
    rc, launches, _, _ = ops.plan("rms_norm_qmv", DType.BF16, bits, G, 1, N, K)
    assert rc == 0 and ("qmv_held_kernel" in launches[0][0]) == held, launches[0][0]


@pytest.mark.parametrize("N,K,waves", [(16384, 3584, 2048), (16000, 3584, 2000), (8192, 3584, 2048), (8000, 3584, 2000), (8208, 3584, 1028), (4096, 3584, 1024), (4096, 9216, 2048), (2048, 9216, 1024), (2048, 18944, 2048)])
def test_held_gemv_waves_of_a_matrix(N, K, waves):
    """More than 1024 waves, or 1024 where four and more share rows and have a few steps each."""
    _, launches, _, _ = ops.plan("rms_norm_qmv", DType.BF16, 3, 64, 1, N, K)
    kernel, grid, block, _ = launches[0]
    assert "qmv_held_kernel" in kernel and grid[0] * (block[0] // 64) == waves


@pytest.mark.parametrize("bits,M,N,K,held", [
    (3, 1, 2048, 2048, False), (3, 2, 2048, 2048, True), (4, 8, 2304, 2304, False), (8, 4, 2304, 2304, False), (6, 8, 8192, 8192, True), (6, 8, 8192, 8320, False), (6, 9, 4096, 4096, True), (6, 9, 4096, 4352, False),
    (5, 4, 8192, 4096, False), (5, 5, 8192, 4096, True), (5, 4, 8064, 4096, True), (5, 4, 10240, 5120, True), (5, 2, 21504, 6144, False), (6, 2, 21504, 6144, True), (5, 4, 4096, 4096, True),
    (3, 4, 28672, 8192, False), (3, 2, 28672, 8192, True), (3, 5, 28672, 8192, True), (3, 4, 16384, 8192, True), (2, 2, 8192, 8192, False), (2, 3, 8192, 8192, True), (2, 2, 28672, 8192, True), (2, 2, 6144, 6144, True),
    (2, 16, 14336, 4096, False), (2, 12, 14336, 4096, True), (2, 16, 13312, 3328, True), (5, 16, 8192, 2048, True), (5, 16, 8200, 2048, False),
    (3, 16, 8192, 1024, False), (3, 16, 4096, 1024, True), (6, 16, 8192, 1024, True), (3, 8, 8192, 1024, True),
])
def test_held_gemv_lines(bits, M, N, K, held):
    """Which batches the GEMV with its activations in LDS is for, on both sides of each line."""
    op = "qmm" if M > 1 else "qmv"
    rc, launches, _, _ = ops.plan(op, DType.BF16, bits, 64, M, N, K)
    assert rc == 0 and ("qmv_held_kernel" in launches[0][0]) == held, launches[0][0]


@pytest.mark.parametrize("bits,G,M,N,K,held", [
    # groups of 32, long rows of tall matrices
    (2, 32, 2, 8960, 6016, True), (2, 32, 2, 9040, 6016, False), (2, 32, 4, 12032, 6016, False), (2, 32, 8, 12032, 6016, True), (2, 64, 4, 12032, 6016, True), (2, 32, 2, 16384, 5120, True), (2, 32, 2, 20480, 5120, False),
    (2, 32, 4, 20480, 5120, True), (2, 32, 4, 16384, 8192, True), (3, 32, 2, 16384, 8192, False), (3, 32, 4, 16384, 8192, True), (6, 32, 2, 16384, 8192, True), (6, 32, 2, 28672, 8192, False),
    (6, 32, 4, 16384, 8192, False), (5, 32, 4, 20480, 5120, False), (5, 32, 4, 20481, 5120, True), (6, 32, 2, 20480, 5120, True), (5, 64, 4, 18432, 6016, False), (5, 64, 4, 18432, 5632, True), (5, 64, 2, 18432, 6016, True),
    # heads
    (2, 64, 2, 65536, 4096, True), (2, 64, 2, 65537, 4096, False), (2, 64, 4, 68000, 3072, True), (2, 64, 4, 68000, 3328, False), (2, 64, 4, 68000, 4224, True), (2, 64, 4, 68000, 7168, False),
    (2, 64, 8, 68000, 4096, True), (2, 32, 4, 34000, 2048, True), (2, 32, 4, 34000, 2944, False), (2, 32, 4, 68000, 1536, False), (3, 64, 2, 68000, 5120, True), (3, 64, 2, 68000, 5248, False),
    (3, 64, 3, 68000, 5248, True), (3, 64, 2, 98304, 4096, True), (3, 64, 2, 98305, 4096, False), (3, 32, 2, 68000, 2048, False), (3, 32, 2, 68000, 2944, True), (3, 32, 2, 65536, 2048, True),
    (3, 64, 8, 68000, 8192, False), (3, 64, 8, 65536, 8192, True), (5, 64, 8, 32768, 4096, True), (5, 64, 8, 32769, 4096, False), (5, 64, 8, 34000, 3840, True), (5, 32, 8, 34000, 2048, False), (5, 32, 8, 34000, 1664, True),
    (6, 64, 4, 100651, 4096, True),
])
def test_held_gemv_lines_of_heads_and_groups_of_32(bits, G, M, N, K, held):
    """Heads, which come alone, and groups of 32, on both sides of each line."""
    rc, launches, _, _ = ops.plan("qmm", DType.BF16, bits, G, M, N, K)
    assert rc == 0 and ("qmv_held_kernel" in launches[0][0]) == held, launches[0][0]


@pytest.mark.parametrize("bits,G,M,N,K,codes", [
    # rows that the tiles cannot split
    (5, 64, 16, 4736, 4736, True), (4, 64, 16, 4736, 4736, False), (4, 64, 17, 4736, 4736, True), (4, 64, 64, 5504, 5504, True), (4, 64, 64, 5760, 5760, True), (4, 64, 64, 8064, 8064, True), (4, 64, 65, 8064, 8064, False), (4, 64, 64, 8320, 8320, False),
    (5, 64, 128, 8064, 8064, True), (5, 64, 65, 8320, 8320, False), (5, 64, 64, 8320, 8320, True), (8, 64, 128, 6784, 6784, True),
    (4, 64, 48, 5760, 5760, True), (8, 64, 96, 4736, 4736, True), (5, 64, 128, 4736, 4736, True), (4, 64, 65, 4736, 4736, False), (5, 64, 129, 4736, 4736, False),
    (4, 64, 96, 2304, 8320, True), (4, 64, 97, 2304, 8320, False), (5, 64, 126, 2304, 8320, True), (5, 64, 126, 3584, 12928, False), (5, 64, 96, 3584, 12928, True),   # (split)
    (4, 64, 32, 9472, 2176, True), (4, 64, 33, 9472, 2176, False), (8, 64, 48, 9472, 2176, True), (5, 64, 64, 9472, 2176, True), (5, 64, 65, 9472, 2176, False),
    (4, 64, 60, 768, 6528, True), (4, 64, 60, 768, 4736, True), (2, 128, 72, 512, 1152, False), (4, 32, 20, 1152, 1152, False), (4, 64, 20, 1152, 1152, True),
    # few weight rows, past 64 activation rows
    (4, 64, 60, 1792, 7040, True), (4, 64, 96, 1792, 7040, True), (8, 64, 96, 1792, 7040, True), (4, 64, 64, 512, 1664, True), (4, 64, 65, 512, 1664, False),
    (4, 64, 65, 1120, 4480, False), (4, 64, 65, 1184, 4736, False), (4, 64, 65, 1185, 4736, True), (4, 64, 71, 896, 7296, False), (4, 64, 65, 2176, 8320, True), (4, 64, 65, 2048, 8320, True), (4, 64, 65, 1664, 8320, False), (8, 64, 65, 512, 1920, False), (8, 64, 65, 512, 2176, True), (5, 64, 128, 1792, 7040, True), (5, 64, 65, 256, 1664, False),
    (8, 64, 128, 1024, 6528, True), (4, 64, 97, 1792, 7040, False),
    # rows that they can
    (5, 64, 32, 4096, 4096, False), (6, 64, 20, 8192, 2048, False), (6, 64, 20, 16384, 4096, False), (6, 64, 17, 18944, 3584, True), (6, 64, 48, 18944, 3584, True),
    (4, 64, 20, 28672, 8192, False), (8, 64, 20, 28672, 8192, True), (8, 64, 48, 28672, 4096, False), (8, 64, 48, 18944, 3584, False), (8, 64, 17, 128256, 4096, True),
    (6, 64, 49, 28672, 8192, False), (6, 64, 48, 128256, 4096, True), (6, 64, 20, 40960, 4096, False),
    (5, 64, 48, 4096, 14336, True), (5, 64, 49, 4096, 14336, False), (6, 64, 77, 5120, 20480, True), (6, 64, 77, 3584, 18944, False), (8, 64, 33, 5120, 20480, True), (8, 64, 32, 5120, 20480, False),
    (4, 64, 49, 3584, 18944, True), (4, 64, 77, 8192, 28672, False), (3, 32, 30, 2560, 10496, False), (7, 64, 24, 4736, 4736, False), (4, 64, 24, 4736, 4672, False),
])
def test_gemv_on_codes_lines(bits, G, M, N, K, codes):
    """Which matrices the GEMV on codes is for, on both sides of each line."""
    rc, launches, _, _ = ops.plan("qmm", DType.BF16, bits, G, M, N, K)
    assert rc == 0 and ("qmv_codes_kernel" in launches[0][0]) == codes, launches[0][0]


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("kw,nw,slices", [(4, 0, 0), (4, 3, 0), (0, 2, 0), (1, 8, 16), (2, 8, 0), (0, 0, 11)])
def test_geometries_that_do_not_fit(mode, kw, nw, slices):
    """A geometry of the GEMV on codes that is asked for and fits a call is used; calls that it does not fit are served all the same."""
    lib = _lib.load()
    names = (b"qmv.codes", b"qmv.codes_kw", b"qmv.codes_nw", b"qmv.codes_slices")
    assert all(lib.mtq_set_option(n, v) == OK for n, v in zip(names, (mode, kw, nw, slices)))
    try:
        for M, K in ((9, 8320), (20, 1152), (33, 1152), (48, 1664), (60, 4736), (128, 1152)):
            rc, launches, _, n = ops.plan("qmm", DType.BF16, 5, 64, M, 1664, K)
            assert rc == OK and n >= 1
            mt = -(-(-(-M // -(-M // 48))) // 16)   # operand tiles of 16 rows
            waves = [w for w in range(max(2, mt), 9) for k in (1, 2, 4) if (not nw or w == nw) and (not kw or k == kw) and w * k <= 8]
            fits = bool(waves) and slices <= K // 128
            assert ("qmv_codes_kernel" in launches[0][0]) == fits, (M, K, launches[0][0])
    finally:
        for n in names:
            lib.mtq_set_option(n, 0)
    for n, v in ((b"qmv.codes_kw", 8), (b"qmv.codes_nw", 1), (b"qmv.codes_nw", 9), (b"qmv.codes_slices", 17)):
        assert lib.mtq_set_option(n, v) == BAD_ARG


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("K", [128, 256, 1152, 1664, 4736])
def test_activations_in_lds_end_on_16_bytes(bits, K):
    """The GEMV that holds its activations in LDS has 16-byte accesses behind the rows and their sums (264 bytes per 128 codes of one
    row); all else in its LDS is a multiple of 16."""
    lib = _lib.load()
    assert lib.mtq_set_option(b"qmv.held", 2) == OK
    try:
        _, launches, _, _ = ops.plan("qmv", DType.BF16, bits, 64, 1, 1000, K)
    finally:
        lib.mtq_set_option(b"qmv.held", 0)
    assert "qmv_held_kernel" in launches[0][0] and launches[0][3] % 16 == 0


@pytest.mark.parametrize("dt,bits,G,M,N,K,first", [
    (DType.BF16, 4, 64, 4, 1024, 18688, "qmv_mfma_kernel"),          # K slices; two passes of two rows
    (DType.BF16, 8, 64, 3, 3584, 18944, "qmv_mfma_kernel"),
    (DType.F16, 4, 128, 16, 4096, 9344, "qmm_d"),                    # K slices; K no multiple of 256: the tiles
    (DType.BF16, 8, 64, 8, 8192, 10240, "qmv_mfma_kernel"),
    (DType.BF16, 4, 64, 8, 4096, 14336, "qmm_d"),                    # the 16-row GEMV with K split, or split tiles
    (DType.BF16, 4, 64, 512, 4096, 14336, "qmm_d"),                  # split tiles
    (DType.F32, 4, 64, 32, 4096, 4096, "qmm_f32_kernel"),
])
def test_products_without_scratch_memory(dt, bits, G, M, N, K, first):
    """A product that writes partial results into the library's buffer runs on a kernel that needs none where the buffer cannot
    be allocated."""
    lib = _lib.load()
    rc, launches, scratch, _ = ops.plan("qmm", dt, bits, G, M, N, K)
    assert rc == OK and scratch > 1024
    try:
        assert lib.mtq_set_option(b"scratch.most_kb", 1) == OK
        rc, launches, scratch, n = ops.plan("qmm", dt, bits, G, M, N, K)
        assert rc == OK and scratch == 0 and first in launches[0][0], (rc, launches)
        assert not any("reduce" in l[0] for l in launches)
    finally:
        lib.mtq_set_option(b"scratch.most_kb", 0)


@pytest.mark.parametrize("bits,E,N,K,per,tall", [
    (4, 128, 768, 2048, 64, True), (4, 128, 768, 2048, 63, False), (8, 128, 768, 2048, 64, True), (8, 128, 768, 2048, 63, False),
    (4, 128, 2048, 768, 96, True), (4, 128, 2048, 768, 95, False), (8, 128, 2048, 768, 64, True), (4, 128, 2048, 768, 192, True),   # short rows
    (4, 8, 4096, 14336, 128, True), (4, 8, 4096, 14336, 127, False), (8, 8, 4096, 14336, 64, True),   # fewer than two tiles a compute unit
    (4, 8, 8192, 4096, 64, True), (4, 8, 8064, 4096, 64, False),
    (8, 2, 8192, 4096, 64, True), (8, 2, 8064, 4096, 64, False),     # tiles for half the chip
    (6, 128, 768, 2048, 128, False), (4, 128, 768, 2080, 128, False),
])
def test_tall_routed_lines(bits, E, N, K, per, tall):
    """Where expert-routed rows run on tiles of up to 160 rows, on both sides of each line; the scratch holds their four tables."""
    rc, launches, scratch, _ = ops.plan("gather_csr", DType.BF16, bits, 32 if K % 64 else 64, 1, N, K, E, per * E)
    assert rc == OK and ("qmm_dma_routed_kernel" in launches[-1][0]) == tall, launches
    rows = 160 if tall else 64
    if bits != 6:
        assert scratch == 16 + (-(-per * E // rows) + E + 1) * 16 * (4 if tall else 1)
