// Host side of the K-run matrix-core GEMV (kernel in qmv_runs_impl.h): which shapes it takes and its geometry.
#include "qmv_runs_impl.h"

namespace mtq {

// Steps of a wave's run, rounded up: K / 16 codes in steps of 128 (64 of 8-bit codes).
static uint32_t runs_steps(int bits, uint32_t K) {
    const uint32_t per = 16u * (bits == 4 ? 128u : 64u);
    return (K + per - 1u) / per;
}

// The activations of a run stay in registers: 16 per step of 4-bit codes and 16 activation rows, 8 per step of 8-bit codes.
static bool runs_shape(int dtype, int bits, uint32_t G, uint32_t M, uint32_t N, uint32_t K) {
    if ((dtype != DT_F16 && dtype != DT_BF16) || (bits != 4 && bits != 8) || (G != 32 && G != 64 && G != 128)) return false;
    if (M == 0 || M > 16 || N == 0 || K == 0 || K % 128 || K % G) return false;
    if (runs_steps(bits, K) > (bits == 4 ? 4u : 5u)) return false;
    return (uint64_t)N * K * bits / 8 < (1ull << 31) && (uint64_t)M * K * 2 < (1ull << 31) && (uint64_t)N * (K / G) * 2 < (1ull << 31);
}
static bool runs_aligned(const void* w, const void* s, const void* b, const void* x) {
    return (uintptr_t)w % 16 == 0 && (uintptr_t)s % 16 == 0 && (uintptr_t)b % 16 == 0 && (uintptr_t)x % 16 == 0;
}

// (instances: qmv_runs_pick.h, one translation unit per element type)
const void* qmv_runs_pick_f16(int bits, uint32_t G, bool sliced, uint32_t xs);
const void* qmv_runs_pick_bf16(int bits, uint32_t G, bool sliced, uint32_t xs);
static const void* runs_pick(int dtype, int bits, uint32_t G, bool sliced, uint32_t xs) {
    return dtype == DT_BF16 ? qmv_runs_pick_bf16(bits, G, sliced, xs) : qmv_runs_pick_f16(bits, G, sliced, xs);
}

bool qmv_runs_takes(const QmvParams& p, const QmvBatch& b) {
    if (b.n < 1 || b.n > 4) return false;
    for (int j = 0; j < b.n; j++)
        if (!runs_shape(p.dtype, p.bits, p.group_size, p.M, b.N[j], p.K) || !runs_aligned(b.w[j], b.scales[j], b.biases[j], p.x)) return false;
    return true;
}

// Where the kernel stands against the others. A matrix's route cannot depend on whether it comes in a batch (it would not have
// the same bits), so a call of one matrix pays for what the projections of a layer gain in one call. The lines lie where two
// matrices of a size together gain more than one alone loses. us, bf16, groups of 64, weights from memory, others -> this, one
// matrix | two in a batch, 5, 9 and 16 rows:
//   2048 x 2048     5.6  8.1  8.1 ->  5.3  5.5  6.1 | 11.4 16.0 16.1 ->  5.6  5.6  6.2
//   4096 x 4096     7.9 10.0 10.0 ->  7.0  7.6  8.8 | 15.4 19.6 20.1 ->  9.9 10.4 11.7     8 bits 17.1 21.9 22.7 -> 12.7 13.2 14.5
//   5120 x 5120    11.4 11.1 11.5 -> 11.3 12.1 13.8 | 22.7 22.1 22.8 -> 14.2 15.0 16.7     8 bits 33.1 28.1 29.1 -> 20.7 21.4 23.3
//   16384 x 2048    8.8  9.2  9.3 -> 10.0 10.4 11.1 | 17.7 18.4 18.5 -> 14.3 14.7 15.4     8 bits 23.3 22.3 22.8 -> 19.2 19.3 20.0
//   14336 x 4096   12.3 13.5 13.6 -> 13.8 14.4 15.8 | 24.8 26.9 27.1 -> 19.7 20.1 21.5     8 bits 37.8 36.9 37.5 -> 31.6 32.0 33.9
//   13824 x 5120   16.3 16.0 16.6 -> 17.0 17.8 19.5 | 32.6 32.1 32.9 -> 25.6 26.3 28.3     (70.8 M codes; 16384 x 5120, 84 M, 16 rows 17.0 -> 19.9 | 34.1 -> 31.5;
//   28672 x 4096, 117 M, 5 rows 19.3 -> 19.9 | 35.9 -> 34.4; 8 bits 16384 x 5120, 16 rows 24.3 -> 28.6 | 48.7 -> 48.9)
//   7168 x 7168    13.9 14.8 15.0 -> 15.6 16.6 18.9 | 27.9 29.6 29.9 -> 23.6 24.5 27.0
//   1024 x 8192     9.9  9.8 10.2 -> 10.2 11.4 13.8 | 19.6 19.7 20.7 -> 10.8 12.0 14.5
//   2048 x 8192     9.4  9.4  9.5 -> 10.8 11.8 14.4 | 18.7 18.7 18.9 -> 11.7 12.7 15.3
//   16384 x 512     7.9  5.8  5.8 ->  8.4  8.2  8.3 | 15.7 11.6 11.6 -> 12.2 12.3 12.4
// and 2, 3 and 4 rows:
//   512 x 3584      5.9  7.1  7.6 ->  5.9  6.0  6.1 | 11.7 14.2 15.2 ->  6.1  6.1  6.3
//   1024 x 4096     5.9  7.2  8.2 ->  6.2  6.3  6.5 | 12.2 14.7 16.8 ->  6.4  6.6  6.9     8 bits 12.7 14.9 16.8 -> 7.8 8.2 8.4
//   768 x 3072      5.3  6.5  7.1 ->  5.9  6.0  6.1 | 10.7 13.2 14.2 ->  6.1  6.2  6.3     8 bits 4.4 5.1 5.6 -> 6.7 6.9 7.0 | 8.7 10.1 11.1 -> 6.9 7.1 7.3
//   1280 x 5120     5.1  5.5  5.7 ->  7.5  7.7  8.0 | 10.0 10.9 11.1 ->  7.7  7.9  8.0
//   512 x 8192      6.3  7.6  8.8 ->  9.5  9.9 10.3 | 13.0 15.5 17.9 ->  9.8 10.2 10.6
//   4096 x 1024     3.6  3.8  3.8 ->  5.3  5.3  5.4 |  7.1  7.4  7.4 ->  6.4  6.4  6.5
// 2 to 4 rows on more than 16384 weight rows: the GEMV's 256 workgroups of sixteen waves hold four rows a wave at once, past that
// every one walks a second block of them (bf16, 2 | 3 | 4 rows alone, then a pair at 4 rows; groups of 64):
//   16384 x 3584    9.7 | 10.0 | 10.0 -> 13.3 | 13.4 | 13.4, 20.0 -> 19.4        8 bits 14.8 | 15.5 | 15.9 -> 16.7 | 16.7 | 16.7, 32.0 -> 28.7
//   16512 x 3584   13.5 | 13.9 | 13.9 -> 14.0 | 14.1 | 14.0, 27.9 -> 20.3        8 bits 17.9 | 18.8 | 19.1 -> 19.2 | 19.1 | 19.2, 38.0 -> 31.1
//   18944 x 3584   13.7 | 14.1 | 14.0 -> 14.5 | 14.6 | 14.4, 28.2 -> 23.0        8 bits 18.4 | 19.2 | 19.6 -> 19.9 | 20.0 | 20.0, 39.2 -> 34.1
//   16512 x 2048    9.6 | 10.2 | 10.3 -> 10.3 | 10.3 | 10.5, 20.5 -> 15.0        8 bits 13.5 | 14.2 | 14.2 -> 12.7 | 12.7 | 12.6, 28.5 -> 18.7
//   24576 x 3072   13.9 | 14.4 | 14.4 -> 14.7 | 14.8 | 14.8, 28.8 -> 24.0        8 bits 17.7 | 19.8 | 19.9 -> 20.7 | 21.0 | 20.8, 39.9 -> 37.3
//   28672 x 2560   13.8 | 14.3 | 14.3 -> 16.3 | 16.4 | 16.4, 28.4 -> 26.3 (seven blocks of 4096 rows each on a workgroup: past six, no)
//   16512 x 4096   15.0 | 15.2 | 15.0 -> 14.5 | 14.7 | 14.6, 30.4 -> 21.3        8 bits 20.2 | 21.0 | 21.2 -> 23.4 | 22.7 | 23.2, 42.5 -> 38.4
// Not in groups of 32, whose scales weigh more here (18944 x 3584, 4 rows 13.7 -> 16.9 | 27.5 -> 27.9), and not with 8 bits at 2 rows
// (24576 x 3072 17.7 -> 20.7 | a pair 35.3 -> 37.4). Fewer weight rows lose more alone than they are sure to gain: 4096 x 4096, 4 rows
// 6.0 -> 7.3 | 12.0 -> 9.3, 8192 x 4096 7.4 -> 9.2 | 14.9 -> 14.2; 5120 x 5120, 3 rows 8.5 -> 9.7 | 17.1 -> 13.1.
// So: below 5 rows the gate and up projections of more than 16384 (to 24576) rows of 2048 to 4096 codes, and short matrices against such rows (the
// K and V projections of grouped-query attention), both with 8-bit codes from 3 rows; from 5 rows up to 75 M codes (60 M of 8 bits), and from 9 rows, where the others take tiles, no more than
// 1024 weight rows of more than 6144 codes (four steps a run, whose registers leave one block in flight) and no more than 8192 of
// fewer than 2048 (some of the sixteen waves have no step, and a workgroup has more than two blocks to walk).
bool qmv_runs_preferred(int bits, uint32_t G, uint32_t M, uint32_t N, uint32_t K) {
    if (M < 2 || M > 16) return false;
    const uint64_t codes = (uint64_t)N * K;
    if (M < 5) {
        if (K < 2048 || K > 4096 || (bits == 8 && M == 2)) return false;
        const bool tall = N > 16384 && N <= 24576 && codes <= 75000000ull && G >= 64;
        return tall || ((uint64_t)N * 2 <= K && codes <= 4500000ull);
    }
    if (M > 8 && ((K > 6144 && N > 1024) || (K < 2048 && N > 8192))) return false;
    return codes <= (bits == 4 ? 75000000ull : 60000000ull);
}

// The K-sliced form against the others; it pays a second launch (about 5 us with its gap), so it is for what they are slow at.
// us, groups of 64 where nothing else is said, others -> this:
//   3, 4 rows of more than 18432 codes (four rows do not fit the LDS of the matrix-core GEMV, which reads the weights twice):
//     3584 x 18944 24.4 -> 19.8, 8 bits 34.3 -> 23.2; 8192 x 28672 53.9 -> 42.9, 8 bits 88.8 -> 60.4; 1024 x 18688 16.0 -> 12.6
//     (at 14336 codes 12.8 -> 19.1)
//   K no multiple of 256 (no K split on the tiles): 4096 x 9344 in groups of 128, 5 / 16 rows 79.7 / 80.2 -> 13.6 / 14.0; 7168 x
//     18560 165 -> 25
//   4-bit rows whose scales are not whole 16-byte vectors (register-staged tiles): 5120 x 13824 in groups of 128, 9 / 16 rows
//     24.4 / 24.8 -> 17.8 / 18.0; 4096 x 11008, 5 / 16 rows 18.1 / 19.0 -> 17.8 / 17.9; but 2048 x 8960 in groups of 128 10.9 -> 11.4, and
//     up to 8 rows, where the 16-row kernel takes it, 5120 x 13824 15.6 -> 17.9
//   8 bits, 5..8 rows on less than twice as many codes as weight rows (two passes of the GEMV): 8192 x 10240 36.2 -> 24.9; and from
//     230 M codes: 8192 x 28672, 16 rows 96.8 -> 64.5 (16384 x 12288, 201 M: 51.9 -> 55.0)
bool qmv_slices_preferred(int bits, uint32_t G, uint32_t M, uint32_t N, uint32_t K) {
    if (M < 3 || M > 16 || K <= 8192) return false;
    if (M <= 4) return K > 18432;
    if (K % 256) return true;
    const uint64_t codes = (uint64_t)N * K;
    if (bits == 8) return codes >= 230000000ull || (M <= 8 && K < 2 * (uint64_t)N);
    return K / G % 8u != 0 && N >= 4096 && !(M <= 8 && codes >= 50000000ull && K % 512 == 0);
}

static uint32_t runs_cus() {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    return (uint32_t)cus;
}

int launch_qmv_runs(const QmvParams& p, const QmvBatch& b, const LaunchCtx& lc) {
    if (!qmv_runs_takes(p, b)) return fail(ERR_UNSUPPORTED, "K-run qmv: shape not taken");
    QmvRunsArgs a{};
    for (int j = 0; j < 4; j++) {
        a.block0[j] = 0x7FFFFFFFu;
        if (j >= b.n) continue;
        a.w[j] = (const unsigned char*)b.w[j];
        a.scales[j] = (const unsigned char*)b.scales[j];
        a.biases[j] = (const unsigned char*)b.biases[j];
        a.out[j] = (uint16_t*)b.out[j];
        a.N[j] = b.N[j];
        a.block0[j] = a.blocks;
        a.blocks += (b.N[j] + 15u) / 16u;
    }
    a.x = (const unsigned char*)p.x;
    a.M = p.M;
    a.K = p.K;
    a.slices = 1;
    const uint32_t cus = runs_cus(), wgs = a.blocks < cus ? a.blocks : cus, xs = runs_steps(p.bits, p.K);
    const void* fn = runs_pick(p.dtype, p.bits, p.group_size, false, xs);
    void* args[] = {&a};
    hipError_t e = launch_kernel(fn, dim3(wgs), dim3(p.bits == 4 && (xs <= 1 || xs == 4) ? 512 : 1024), args, 0, lc);
    if (e != hipSuccess) return hip_fail(e, "K-run qmv kernel launch");
    return ERR_OK;
}

// Rows too long for the registers of one workgroup, in slices of up to 5120 codes: each workgroup works on one slice, f32 sums
// of the slices go to scratch and a second launch adds them in slice order.
static uint32_t slices_of(uint32_t K) { return (K + 5119u) / 5120u; }

bool qmv_slices_takes(const QmmParams& p) {
    const uint32_t G = p.group_size, M = p.M, N = p.N, K = p.K;
    if ((p.dtype != DT_F16 && p.dtype != DT_BF16) || (p.bits != 4 && p.bits != 8) || (G != 32 && G != 64 && G != 128)) return false;
    if (M == 0 || M > 16 || N == 0 || K % 128 || K % G || K <= 5120 || slices_of(K) > 16u) return false;
    if (!runs_aligned(p.w, p.scales, p.biases, p.x) || (uint64_t)slices_of(K) * M * N >= (1ull << 31)) return false;
    return (uint64_t)N * K * p.bits / 8 < (1ull << 31) && (uint64_t)M * K * 2 < (1ull << 31) && (uint64_t)N * (K / G) * 2 < (1ull << 31);
}

size_t qmv_slices_scratch_bytes(const QmmParams& p) { return (size_t)slices_of(p.K) * p.M * p.N * sizeof(float); }

int launch_qmv_slices(const QmmParams& p, const LaunchCtx& lc, void* scratch) {
    if (!qmv_slices_takes(p) || !scratch) return fail(ERR_UNSUPPORTED, "K-sliced qmv: shape not taken");
    QmvRunsArgs a{};
    for (int j = 1; j < 4; j++) a.block0[j] = 0x7FFFFFFFu;
    a.w[0] = (const unsigned char*)p.w;
    a.scales[0] = (const unsigned char*)p.scales;
    a.biases[0] = (const unsigned char*)p.biases;
    a.out[0] = (uint16_t*)p.out;
    a.part[0] = (float*)scratch;
    a.N[0] = p.N;
    a.blocks = (p.N + 15u) / 16u;
    a.x = (const unsigned char*)p.x;
    a.M = p.M;
    a.K = p.K;
    a.slices = slices_of(p.K);
    const uint32_t per = runs_cus() / a.slices > 0 ? runs_cus() / a.slices : 1u, wgs = (a.blocks < per ? a.blocks : per) * a.slices;
    void* args[] = {&a};
    LaunchCtx l1 = lc, l2 = lc;
    l1.stop = nullptr;
    l2.start = nullptr;
    hipError_t e = launch_kernel(runs_pick(p.dtype, p.bits, p.group_size, true, 0), dim3(wgs), dim3(512), args, 0, l1);
    if (e != hipSuccess) return hip_fail(e, "K-sliced qmv kernel launch");
    return add_slices(p.dtype, (const float*)scratch, p.out, p.M * p.N, a.slices, l2);
}

}  // namespace mtq
