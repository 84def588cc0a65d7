// Host side of the K-run matrix-core GEMV (kernel in qmv_runs_impl.h): which shapes it takes and its geometry.
#include "qmv_runs_impl.h"

namespace mtq {

// Steps of a sixteenth of a row, rounded up: K / 16 codes in steps of 128 (64 of 8-bit codes). (Where eight waves share a row, a run is two sixteenths.)
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
RunsInstance qmv_runs_pick_f16(bool paired, int bits, uint32_t G, bool sliced, uint32_t xs, bool few);
RunsInstance qmv_runs_pick_bf16(bool paired, int bits, uint32_t G, bool sliced, uint32_t xs, bool few);
// Whether the steps of a row are dealt to the waves in pairs: of rows of whole 128-byte lines, 8-bit and sliced ones always (2 x 3072 x 1024,
// 8 bits, 4 rows 5.6 -> 5.4, 2 x 12288 x 4096 29.1 -> 21.1), 4-bit ones where that is the faster at every batch. bf16, groups of 64, us, runs -> pairs, three square
// matrices and two of twice or three times as many rows, 5 | 16 rows:
//   K = 512   5.0 5.0 -> 5.1 5.1 | 5.0 5.0 -> 5.1 5.2     1536  6.1 7.2 -> 6.1 7.0 | 6.1 7.2 -> 6.1 7.1      1792  6.3 7.3 -> 6.2 7.2 | 6.3 7.4 -> 6.2 7.3
//       2304  7.8 11.2 -> 7.9 11.2 | 8.3 11.6 -> 8.4 11.6   2560  8.0 11.8 -> 7.9 11.4 | 8.4 12.0 -> 8.5 11.9   3584  10.4 15.1 -> 9.4 13.9 | 10.9 15.3 -> 10.2 14.7
//       4096  11.3 -> 10.4, 2 x 14336 18.4 -> 16.6 | 11.7 -> 10.7, 18.7 -> 17.2      8192 (one)  14.7 -> 12.5 | 16.2 -> 16.1
// A wave of rows of 4097 to 6144 codes has a pair and some have a step of their own beside it, half of a line whose other half is another wave's. Which
// form is the faster there depends on the device and on how much of the weights its last-level cache still holds: three layers of 5120, 13824 wide, in groups
// of 128 at 16 rows, runs -> pairs on eight devices 185 -> 178, 185.5 -> 178, 187 -> 186, 188 -> 188, 187 -> 188, 188 -> 194, 189 -> 195, 195 -> 205. So
// runs there. (qmv.runs = 2 and 3: pairs wherever rows are whole lines.)
static bool runs_paired(int bits, uint32_t K, bool sliced) {
    if ((uint64_t)K * bits / 8 % 128) return false;
    if (bits == 8 || sliced || options().qmv_runs >= 2) return true;
    return K > 4096 ? K > 6144 : K > 2048 ? K >= 2560 : K >= 1792;
}
static RunsInstance runs_pick(int dtype, int bits, uint32_t G, uint32_t K, bool sliced, uint32_t xs, uint32_t M) {
    const bool paired = runs_paired(bits, K, sliced);
    return dtype == DT_BF16 ? qmv_runs_pick_bf16(paired, bits, G, sliced, xs, M <= 8) : qmv_runs_pick_f16(paired, bits, G, sliced, xs, M <= 8);
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
//   2048 x 2048     5.5  7.7  7.7 ->  4.9  5.0  5.2 | 11.0  8.2  8.2 ->  5.2  5.2  5.6     8 bits 14.8 10.4 10.6 ->  6.0  6.0  6.4
//   4096 x 4096     7.8 10.1 10.0 ->  6.8  7.2  7.4 | 15.6 19.7 20.8 ->  9.0  9.5  9.4     8 bits 17.2 22.3 23.6 -> 13.2 13.2 13.4
//   5120 x 5120    11.4 11.2 11.8 ->  9.8  9.7  9.7 | 22.9 22.3 23.6 -> 13.2 13.1 13.2     8 bits 33.3 28.6 30.2 -> 19.3 19.5 19.4
//   16384 x 2048    8.9  9.7  9.9 ->  8.7  8.6  8.8 | 18.6 19.4 19.7 -> 13.0 13.0 13.4     8 bits 24.2 23.5 24.2 -> 17.8 17.9 18.3
//   14336 x 4096   12.9 14.0 14.2 -> 13.6 13.6 14.1 | 25.1 27.8 28.0 -> 19.5 19.5 20.2     8 bits 39.1 37.7 38.5 -> 34.1 33.9 31.9
//   13824 x 5120   16.5 16.5 17.0 -> 15.1 15.7 15.3 | 33.0 32.7 33.9 -> 23.5 24.1 24.1     (70.8 M codes)
//   7168 x 7168    14.2 15.1 15.4 -> 13.7 13.5 14.1 | 28.0 30.3 30.8 -> 21.5 21.6 22.1
//   8192 x 8192    15.0 16.8 17.1 -> 16.3 16.3 16.3 | 30.0 33.1 35.2 -> 25.4 25.3 25.6
//   1024 x 8192     9.8  9.7 10.3 -> 10.3 10.3 10.3 | 11.1 11.0 11.8 -> 10.7 10.7 10.8
//   2048 x 8192     9.4  9.4  9.5 -> 10.4 10.4 10.5 | 18.5 18.6 18.8 -> 12.3 12.3 12.4
//   8192 x 1024     5.6  6.6  6.7 ->  6.0  6.0  6.0 | 11.3  7.3  7.4 ->  7.7  7.7  7.8     8 bits 12.6  8.5  8.8 ->  7.9  7.9  7.9
//   16384 x 512     7.8  6.0  6.0 ->  7.4  7.5  7.5 | 15.7 11.9 12.0 -> 11.7 11.7 11.7     8 bits 15.6 12.5 12.7 -> 10.2 10.3 10.4
//   16384 x 5120   17.8 18.0 18.3 -> 15.9 15.5 15.6 | 34.4 35.3 36.7 -> 26.4 26.1 26.8     8 bits 76.9 48.2 50.5 -> 42.1 42.5 43.0     (83.9 M)
//   28672 x 4096   19.3 19.6 21.0 -> 19.7 20.4 20.7 | 37.3 38.4 41.9 -> 32.2 33.5 34.0     8 bits 63.2 66.5 69.7 -> 58.8 59.0 59.7     (117 M)
// and 3 and 4 rows (2 rows in the last lines):
//   512 x 1024       4.1  4.1 ->  4.7  4.8 |  8.3  8.1 ->  5.0  5.0     8 bits  4.3  4.7 ->  4.3  4.3 |  8.6  9.5 ->  4.5  4.6
//   2048 x 2048      4.3  4.3 ->  4.9  4.9 |  8.5  8.7 ->  5.1  5.2     8 bits  5.9  6.4 ->  5.5  5.5 | 11.7 12.7 ->  5.9  5.9
//   4096 x 2048      4.2  4.3 ->  5.3  5.3 |  8.4  8.6 ->  6.5  6.6     8 bits  5.8  5.9 ->  5.9  5.9 | 11.6 11.8 ->  7.7  7.6
//   1536 x 1536      4.3  4.3 ->  4.8  4.8 |  8.6  8.6 ->  5.1  5.1     8 bits  5.7  5.8 ->  5.4  5.4 | 11.4 11.5 ->  5.7  5.7
//   512 x 3584       7.0  7.5 ->  6.2  6.2 | 14.1 15.0 ->  6.4  6.5     8 bits  7.1  7.7 ->  6.5  6.5 | 14.2 15.3 ->  6.8  6.7
//   4096 x 4096      5.9  6.0 ->  6.8  6.8 | 11.8 12.0 ->  9.0  9.0     8 bits  7.5  7.8 ->  8.9  8.9 | 14.9 15.4 -> 13.2 13.3
//   5120 x 5120      8.5  8.9 ->  9.8  9.8 | 17.1 18.0 -> 13.2 13.1     8 bits 11.1 11.7 -> 13.5 13.4 | 22.0 23.2 -> 19.5 19.5
//   1024 x 5120      5.3  6.0 ->  7.3  7.3 | 10.7 11.8 ->  7.6  7.7     8 bits  6.5  7.1 ->  8.6  8.7 | 13.1 14.1 ->  9.2  9.2
//   6144 x 6144      9.3  9.5 -> 10.7 10.7 | 18.7 19.2 -> 15.4 14.7
//   4096 x 7168      7.4  7.8 -> 10.9 11.0 | 14.9 15.6 -> 13.8 13.8     (four steps a run, on eight waves)
//   6144 x 4096      6.8  7.0 ->  8.7  8.7 | 13.7 13.9 -> 11.4 11.4     8 bits  9.7 10.1 -> 11.6 11.7 | 19.4 20.2 -> 18.0 18.0
//   8192 x 4096      7.3  7.4 ->  8.9  8.9 | 14.6 14.8 -> 14.3 14.3     8 bits 10.3 10.8 -> 14.0 14.0 | 20.5 21.7 -> 21.8 22.0
//   10240 x 4096     9.6  9.7 -> 11.0 11.1 | 19.4 19.3 -> 15.3 15.4     8 bits 15.5 16.0 -> 16.3 16.2 | 30.9 31.8 -> 26.2 26.6
//   13824 x 4096    10.0 10.0 -> 13.6 13.7 | 20.2 20.2 -> 19.3 19.2     8 bits 16.3 16.6 -> 19.3 19.4 | 32.7 33.8 -> 32.0 32.3
//   8192 x 5120     10.0  9.6 -> 10.5 10.5 | 18.9 19.2 -> 15.7 15.7     8 bits 13.7 14.2 -> 14.7 14.7 | 27.8 28.6 -> 23.9 23.9
//   13824 x 5120    13.0 13.4 -> 15.2 15.2 | 25.9 26.7 -> 23.7 24.0     8 bits 20.1 20.6 -> 23.0 22.9 | 40.6 41.1 -> 38.5 38.3
//   18944 x 3584    14.2 14.1 -> 14.3 14.4 | 28.4 28.5 -> 22.8 23.0     8 bits 38.5 39.9 -> 34.0 34.1
//   28672 x 2560    14.7 14.4 -> 16.3 16.2 | 28.6 29.7 -> 26.4 26.7     (seven blocks of 4096 rows each on a workgroup)
//   in groups of 32: 4096 x 2048 4.2 4.3 -> 5.9 5.9 | 8.5 8.6 -> 7.7 7.8, 4608 x 1536 5.0 4.9 -> 6.8 6.9 | 9.9 10.0 -> 8.4 8.4,
//     13824 x 5120 13.9 14.2 -> 16.8 16.9 | 27.7 28.3 -> 26.9 26.8
//   2 rows: 512 x 2048 3.9 -> 4.7 | 7.9 -> 4.9; 1024 x 4096 5.9 -> 6.2 | 11.7 -> 6.5; 18944 x 3584 13.8 -> 14.2 | 27.7 -> 22.7;
//     4096 x 4096 5.2 -> 6.8 | 10.3 -> 9.0, 5120 x 5120 8.2 -> 9.7 | 16.4 -> 13.1 (pairs gain less, a lone output projection loses more)
// The others' time steps up behind 4096, 8192 and 16384 weight rows (the GEMV's 256 workgroups of sixteen waves hold 16384 rows, four
// a wave), this kernel's with each 4096, 256 blocks of 16: so at 3 and 4 rows up to 6144 weight rows (2048 of 4-bit rows of up to 2048
// codes), from 8193 to 12288 and from 16385 to 24576 (of 2048 to 4096 codes), and up to 16384 where rows of more than 2048 bytes make the
// others slower, except rows of 4096 bytes, which are slower here (8192 x 4096 of 8 bits 14.0, 8192 x 3584 11.0); up to 75 M codes and
// three steps a run (8 bits: five). The four products of a dense layer, 22 families of sizes in groups of 32, 64 and 128, 4 and 8 bits:
// 1.16 and 1.18 times as fast at 3 and 4 rows, none slower (5120, 17408 wide, 8 bits in groups of 32 124 -> 118, 129 -> 121; 1536, 4608
// wide, whose down projection alone loses 2 us, 8 bits 42 -> 27, 4 bits 33 -> 27).
// 2 rows, 4 bits: the short matrices of grouped-query attention and 16385 to 24576 weight rows.
// From 5 rows up to 75 M codes (60 M of 8 bits), and from 9 rows, where the others take tiles, no more than 8192 weight rows of fewer than
// 2048 codes, and no more than 1024 of more than 6144. The last two lines and the 75 M are those of an earlier form of the kernel, with
// sixteen waves on every row length: past them this one has become the faster (7168 x 7168, 16384 x 5120, 8 bits 16384 x 512), but
// those calls would no longer have the tiles' bits.
bool qmv_runs_preferred(int bits, uint32_t G, uint32_t M, uint32_t N, uint32_t K) {
    if (M < 2 || M > 16) return false;
    const uint64_t codes = (uint64_t)N * K;
    if (M < 5 && codes > 75000000ull) return false;
    const bool tall = N > 16384 && N <= 24576 && K >= 2048 && K <= 4096 && G >= 64;
    if (M == 2) return bits == 4 && (tall || ((uint64_t)N * 2 <= K && codes <= 4500000ull && K >= 2048 && K <= 4096));
    if (M < 5) {
        if (K < 1024 || K > (bits == 4 ? 6144u : 5120u)) return false;
        const uint32_t row = K * (uint32_t)bits / 8u;   // bytes from weight row to weight row
        if (N <= 6144) return bits == 8 || K > 2048 || N <= 2048;
        if (N <= 16384 && row > 2048 && row != 4096 && (G >= 64 || N <= 8192)) return true;
        return tall || (N > 8192 && N <= 12288 && (G >= 64 || K <= 4096));
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
//     230 M codes where the tiles are register-staged (their scales do not fit LDS): 8192 x 28672, 5 / 16 rows 97.1 / 99.0 -> 66.4 /
//     69.6, groups of 32 6144 x 40960 138 / 140 -> 73 / 75; load-to-LDS tiles: groups of 128 8192 x 28672, 16 rows 56.5 -> 68.0, 16384 x
//     14336 54.9 -> 66.9, 14336 x 16384 59.6 -> 65.3 (but 10240 x 24576 84.6 -> 70.4: not there either). 16384 x 12288, 201 M: 51.9 -> 55.0
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
    const RunsInstance k = runs_pick(p.dtype, p.bits, p.group_size, p.K, false, xs, p.M);
    void* args[] = {&a};
    hipError_t e = launch_kernel(k.fn, dim3(wgs), dim3(k.threads), args, 0, lc);
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
    const RunsInstance k = runs_pick(p.dtype, p.bits, p.group_size, p.K, true, 0, p.M);
    hipError_t e = launch_kernel(k.fn, dim3(wgs), dim3(k.threads), args, 0, l1);
    if (e != hipSuccess) return hip_fail(e, "K-sliced qmv kernel launch");
    return add_slices(p.dtype, (const float*)scratch, p.out, p.M * p.N, a.slices, l2);
}

}  // namespace mtq
