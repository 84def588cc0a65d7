// Host side of the matrix-core GEMV on codes (kernel in qmv_codes_impl.h): which calls it takes and its geometry.
#include "qmv_codes_pick.h"

namespace mtq {

// (instances: one translation unit per element type, kind of group and row count)
CodesInstance qmv_codes_pick_f16(int bits, uint32_t mt);
CodesInstance qmv_codes_pick_f16_g32(int bits, uint32_t mt);
CodesInstance qmv_codes_pick_bf16(int bits, uint32_t mt);
CodesInstance qmv_codes_pick_bf16_g32(int bits, uint32_t mt);

static CodesInstance codes_pick(int dtype, int bits, uint32_t G, uint32_t mt) {
    if (dtype == DT_BF16) return G == 32 ? qmv_codes_pick_bf16_g32(bits, mt) : qmv_codes_pick_bf16(bits, mt);
    return G == 32 ? qmv_codes_pick_f16_g32(bits, mt) : qmv_codes_pick_f16(bits, mt);
}

constexpr uint32_t QC_LDS = 160u * 1024u;   // of a compute unit
static uint32_t codes_cus() {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    return (uint32_t)cus;
}

// Tiles of up to 48 activation rows, all of one height but the last.
struct CodesRows {
    uint32_t tiles, rows, mt;   // mt: 16-row operand tiles of one
};
static CodesRows codes_rows(uint32_t M) {
    CodesRows r;
    r.tiles = (M + 47u) / 48u;
    r.rows = (M + r.tiles - 1u) / r.tiles;
    r.mt = (r.rows + 15u) / 16u;
    r.tiles = (M + r.rows - 1u) / r.rows;
    return r;
}

bool qmv_codes_takes(const QmmParams& p) {
    const uint32_t G = p.group_size, M = p.M, N = p.N, K = p.K;
    if ((p.dtype != DT_F16 && p.dtype != DT_BF16) || (p.bits != 2 && p.bits != 3 && p.bits != 4 && p.bits != 5 && p.bits != 6 && p.bits != 8)) return false;
    if ((G != 32 && G != 64 && G != 128) || M == 0 || M > 1024 || N == 0 || K == 0 || K % 128 || K % G) return false;
    if ((uintptr_t)p.w % 16 || (uintptr_t)p.x % 16 || (uintptr_t)p.scales % 4 || (uintptr_t)p.biases % 4) return false;
    // offsets of 32 bits: into 32 weight rows, into x; workgroups and partial results
    return (uint64_t)K * p.bits / 8 * 32 < (1ull << 31) && (uint64_t)M * K * 2 < (1ull << 31) && N < (1u << 24) && (uint64_t)M * N < (1ull << 31);
}

// How a matrix is split, by what its own launch would take (us, about): workgroups fill the chip in rounds, one to a compute unit; a
// step of 128 codes takes a workgroup 1.45 us, of eight waves as of five; slices of K cost a second launch. Tall matrices come in pairs, whose
// waves cannot share rows in another way than those of one alone (2 x 8704 x 3712, 5 bits, 20 rows 37.9 -> 34.6).
CodesSplit qmv_codes_split(const QmmParams& p) {
    const CodesRows r = codes_rows(p.M);
    const CodesInstance k = codes_pick(p.dtype, p.bits, p.group_size, r.mt);
    const uint32_t N = p.N, steps = p.K / 128u, pair = N >= 2 * (uint64_t)p.K ? 2u : 1u, cus = codes_cus();
    const Options& o = options();
    // Where all but the smallest matrices have four waves that share rows and no slices, so have those: with slices of their own they take two
    // more launches in a batch (2176, 272, 272 x 2176, 4 bits, 17 rows 25.1 -> 13.9, on the tiles 18.1; 272 alone 11.1 -> 15.6, tiles 17.5).
    const bool alike = r.mt == 2 && p.K <= 3072 && 4 * (uint64_t)N <= p.K && !o.qmv_codes_kw && !o.qmv_codes_nw && !o.qmv_codes_slices;
    CodesSplit best;
    float least = 1e30f;
    for (uint32_t kwl = alike ? 2 : 0; kwl <= 2; kwl++) {
        if (o.qmv_codes_kw && (1u << kwl) != (uint32_t)o.qmv_codes_kw) continue;
        for (uint32_t nw = qc_min_nw(r.mt); nw << kwl <= QC_WAVES; nw++) {   // (two waves along N at least: four share rows at most)
            if ((o.qmv_codes_nw && nw != (uint32_t)o.qmv_codes_nw) || k.lds(1u << kwl, 1, nw << kwl) > QC_LDS) continue;
            const uint32_t tiles = (N + 32u * nw - 1u) / (32u * nw);
            const float step_us = (r.mt == 1 ? 1.2f : r.mt == 2 ? 1.45f : 1.8f) * ((nw << kwl) <= 4 ? 0.8f : 1.0f);
            for (uint32_t s = 1; s <= (alike ? 1u : 16u) && s <= steps; s++) {
                if (o.qmv_codes_slices && s != (uint32_t)o.qmv_codes_slices) continue;
                if (s > 1 && !o.qmv_codes_slices && (steps >> kwl) < 3u * s) break;
                const uint32_t wgs = (tiles * s + 7u) / 8u * 8u * r.tiles * pair, per = (((steps + s - 1u) / s + 1u) / 2u + (1u << kwl) - 1u) >> kwl;
                float us = 4.f + (float)((wgs + cus - 1u) / cus) * ((float)(2u * per) * step_us + 6.5f);
                if (s > 1) us += 4.f + (float)(pair * s) * (float)p.M * (float)N * 8.0f / 4e6f;
                if (us < least) { least = us; best = CodesSplit{kwl, s}; }
            }
        }
    }
    return best;
}
size_t qmv_codes_scratch_bytes(const QmmParams& p, const CodesSplit& s) { return s.slices > 1 ? ((size_t)s.slices * p.M * p.N * sizeof(float) + 255) & ~(size_t)255 : 0; }

// Where the kernel stands against the tile kernels, which split K over workgroups only where it is a multiple of 256: short of
// that a workgroup walks the whole row. us, bf16, groups of 64, tiles -> this:
//                                   20 rows            32                40                48                60                96               128
//   4736 x 4736, 5 bits             55.1 -> 17.2       56.1 -> 17.8                        57.4 -> 20.6      58.5 -> 24.7      53.9 -> 27.6     54.4 -> 31.2
//                4 bits             32.4 -> 15.4       32.6 -> 15.9                        33.2 -> 18.9      33.3 -> 21.4      32.5 -> 24.6     33.1 -> 27.3
//   4736 x 20096, 5 bits            259 -> 39          263 -> 39                           270 -> 43         278 -> 65         95 -> 64         101 -> 84
//                4 bits             111 -> 33          112 -> 34                           115 -> 38         120 -> 56         112 -> 55        45 -> 71
//   2 x 20096 x 4736, 5 bits        120.9 -> 70.7      124.3 -> 72.5     124.6 -> 74.3     125.9 -> 76.1     128.0 -> 112.5    132 -> 130
//                4 bits             66.3 -> 58.8       67.4 -> 60.6      68.2 -> 64.6      68.6 -> 66.8      69.4 -> 96.3
// (one of them alone, 4 bits, 20 / 48 rows 34.9 -> 35.9, 36.9 -> 42.1: 4 bits up to 32 rows)
//                8 bits             107.3 -> 71.9      108.1 -> 73.6     108.3 -> 75.9     108.7 -> 77.8     109.9 -> 115.1
//   2 x 9472 x 2176, 5 bits         28.2 -> 19.6       28.7 -> 20.3      28.8 -> 23.4      29.1 -> 23.9      29.3 -> 27.7
//                4 bits             21.2 -> 17.3       21.1 -> 18.1      21.3 -> 21.0      21.4 -> 21.4      21.8 -> 24.0
//                8 bits             25.5 -> 21.2       26.0 -> 21.9      26.2 -> 24.7      26.3 -> 25.0      26.7 -> 29.2
//   2 x 8704 x 3968, 5 bits         49.8 -> 27.9       51.0 -> 28.6      51.3 -> 32.6      51.8 -> 33.0      52.8 -> 55.4
//   1664, 1664, 1664 x 1664, 5 bits 21.7 -> 12.5       22.3 -> 13.0      22.4 -> 15.2      22.5 -> 16.0      22.9 -> 13.3
//                4 bits             16.6 -> 11.2       16.6 -> 11.6      16.7 -> 13.9      16.7 -> 14.8      16.8 -> 12.0
//   3968, 992, 992 x 3968, 4 bits   28.6 -> 15.4       28.9 -> 16.8      29.1 -> 21.1      29.5 -> 29.8      29.6 -> 26.6
// (2 bits as 4, 3 and 6 bits as 5; up to 16 rows 4- and 8-bit codes have the K-run kernel, but for more than 75 M codes: 4736 x 4736, 5 bits, 54.6 -> 14.2.) A
// matrix's route cannot depend on whether it comes in a batch, and the tile kernels take the matrices of a batch in the time of one
// as long as they fill the chip together no more than once; so the lines of square matrices lie where one of them alone and one with the two of an
// eighth or a quarter of its rows (q8, q4) gain more together than three of them lose (us, tiles -> this):
//                         alone          q8             q4             three
//   4 bits,  20 rows, 5760   38.2 -> 18.5                                39.2 -> 45.2     48 rows  39.0 -> 22.1                                40.3 -> 51.0
//            64 rows, 4992   35.2 -> 21.3   35.2 -> 34.5   35.6 -> 37.5   36.0 -> 40.8     8064     54.0 -> 30.9   54.8 -> 48.0   55.2 -> 54.5   57.1 -> 85.9
//            72 rows, 4992   34.0 -> 23.8   34.2 -> 37.5   34.4 -> 40.8   35.6 -> 57.0     8064     52.0 -> 35.8   52.5 -> 54.1   52.7 -> 59.8   106 -> 94.8  (neither)
//   2 bits,  64 rows, 6784   63.2 -> 26.0   61.5 -> 40.9   63.8 -> 48.7   65.5 -> 71.5
//   3 bits, 128 rows, 4992   52.9 -> 27.3   54.2 -> 44.6   52.9 -> 54.7   56.8 -> 69.1     8064     88.1 -> 55.2   88.9 -> 70.6   88.2 -> 76.3   179 -> 159
//   5 bits,  96 rows, 6784   84.5 -> 39.2   85.9 -> 59.0   87.0 -> 64.9   173 -> 103
//   8 bits, 112 rows, 4992   56.8 -> 31.1   55.0 -> 49.0   54.9 -> 62.2   57.2 -> 81.7     8064     92.3 -> 67.6   93.1 -> 81.2   93.4 -> 91.4   187 -> 197
// Where the tiles split K (rows of a multiple of 256 codes; a matrix of at most half as many tiles of 128 columns as there are compute units) they
// are the faster: 4096 x 4096, 5 bits, 32 rows 13.1 -> 14.8; 2 x 8192 x 2048, 4 bits, 20 rows 9.7 -> 11.8. Past that pairs of matrices are faster here up to
// 48 rows, but one of them alone is not, on half the workgroups (us, 6 bits, tiles -> this, 20 and 48 rows):
//   2 x 14336 x 4096   37.7 -> 33.3   51.7 -> 39.4    one   18.8 -> 21.2   25.9 -> 31.8
//   2 x 18944 x 3584   43.6 -> 39.5   62.7 -> 46.9    one   29.0 -> 29.7   42.6 -> 34.9
//   28672 x 4096                                      one   34.1 -> 33.7   49.1 -> 41.2
//   2 x 28672 x 8192   124.7 -> 98.1  176.9 -> 121.0  57344 x 8192 120.2 -> 98.4  202.1 -> 120.0
//   128256 x 4096                                     one   130.5 -> 111.1 147.5 -> 135.0
// So from 16385 rows of weights on, where a pair's workgroups come to one round over the chip or to full ones. 8 bits: the last two only (57344 x 8192 124.1 -> 112.3,
// 151.1 -> 128.9; 128256 x 4096 131.2 -> 130.1, 167.8 -> 145.7; 28672 x 4096 33.1 -> 38.6); 3 bits from 33 rows on (28672 x 4096, 20 / 48 rows 25.5 -> 30.9, 38.6
// -> 37.7); 4 bits are not (2 x 28672 x 8192 67.8 -> 79.8). Past 48 rows neither are
// the others (128256 x 4096, 6 bits, 77 rows 194.6 -> 241.8). On long rows: bit-stream widths past 8192 codes (4096 x 14336, 5 bits, 16 / 32 / 48 rows 28.1 -> 20.5,
// 29.1 -> 25.4, 32.9 -> 29.3; 5120 x 20480, 6 bits, 77 rows 85.0 -> 67.4, but 3584 x 18944 45.0 -> 47.9), 8 bits past 16384 (5120 x 20480, 48 / 77 rows 60.5 -> 44.0,
// 138 -> 66.7; 20 rows 30.9 -> 38.3), 4 bits there at few rows of weights (3584 x 18944, 77 rows 51.1 -> 42.0, 8192 x 28672 88.2 -> 95.0).
// Groups of 32 cost the tiles nothing and a second scaling per group here: 2- and 4-bit codes are left there on rows of 1152 (1152 x 1152, 20 rows 10.8
// -> 12.3), bit-stream widths on the smaller long rows (2560 x 10496, 3 bits, 30 rows 17.1 -> 18.8).
// A matrix of half its row length and less goes by its own times. Past 64 rows, where the square 2- and 4-bit ones of its row length stay on the tiles, two of them are worked
// out beside the square one's tiles for nothing, and here cost what one alone gains: of a quarter of its row length and less they stay on the tiles, which larger
// ones leave where the tiles need twice the time (bits, rows, us, tiles -> this, alone | two next to the square one):
//   768 x 6528     4  60   40.4 -> 13.6                    8  96   67.5 -> 17.7      1184 x 4736    8  80   49.3 -> 17.4
//   592 x 4736     8  120  41.7 -> 16.0 | 52.5 -> 48.7 (the square one too)                1792 x 7040  4  60   48.0 -> 15.4    5  96   82.6 -> 20.2
// and not taken: 1632 x 6528, 4 bits, 80 rows 43.5 -> 17.6 | 44.5 -> 71.8 (a layer of 7296 with 896 for keys and values, 71 rows, 397 -> 417), 1056 x 4224 27.3 -> 15.1 | 30.1 -> 48.8,
// 544 x 2176 17.6 -> 12.8 | 18.8 -> 31.0, 736 x 2944 21.0 -> 13.5 | 23.6 -> 37.0, 1184 x 4736 29.9 -> 16.5; 512 x 1664, 8 bits 16.4 -> 13.1.
bool qmv_codes_preferred(int bits, uint32_t G, uint32_t M, uint32_t N, uint32_t K) {
    const bool stream = bits == 3 || bits == 5 || bits == 6, tall = N >= 2 * (uint64_t)K, wide = K >= 2 * (uint64_t)N, g32 = G == 32 && !stream && bits != 8;
    const uint64_t codes = (uint64_t)N * K;
    if (M < 5 || M > 128 || K < 1024 || (g32 && K < 1280 && M > 16)) return false;
    if (K % 256 == 0) {
        if (wide) {
            if (stream) return K > 8192 && (M <= 48 || (M <= 96 && N >= 5120 && K > 16384)) && (G != 32 || (uint64_t)N * K > 33000000ull);
            return K > 16384 && M <= 96 && (bits == 8 ? M > 32 : M > 48 && N <= 5120);
        }
        if (!tall || M < 9 || M > 48) return false;
        if (M <= 16) return stream && N > 8192 && (bits != 3 || N <= 16384);
        if (N <= 16384 || (!stream && bits != 8) || (M <= 32 && (bits == 3 || K < 2048))) return false;
        const uint32_t cus = codes_cus(), tiles = 2 * ((N + 255) / 256), rounds = (tiles + cus - 1) / cus;
        return tiles * 5 >= rounds * cus * 4 ? stream || K >= 8192 || N > 65536 : stream && rounds == 1;
    }
    if (M <= 16) return stream || (uint64_t)N * K > 75000000ull;
    if (wide) return M <= 64 || (stream || bits == 8 ? K >= 2048 : M <= 96 && K >= 4608 && (K > 8192 ? 5 : 4) * (uint64_t)N > K);
    if (tall) return M <= (stream ? (K < 2304 || codes > 90000000ull ? 64u : 48u) : bits == 8 ? 48u : 32u);
    if (M <= 48 || (M <= 64 && codes <= 68000000ull)) return true;
    return (stream || bits == 8) && (M <= 64 || (K >= 2048 && codes <= 68000000ull));
}

struct CodesReduceArgs {
    const float* part[4];
    uint16_t* out[4];
    uint32_t total[4];    // results
    uint32_t slices[4];
    uint32_t first[4];    // first workgroup, of 1024 results each; 0x7FFFFFFF past the last matrix
};

// Adds the slices' f32 sums in slice order. One thread has four results in a row.
template <int DT> __global__ __launch_bounds__(256) void qmv_codes_reduce_kernel(CodesReduceArgs a) {
    uint32_t i = 0;
#pragma unroll
    for (uint32_t k = 1; k < 4; k++) i += blockIdx.x >= a.first[k] ? 1u : 0u;
    const float* part = a.part[0];
    uint16_t* out = a.out[0];
    uint32_t total = a.total[0], slices = a.slices[0], first = a.first[0];
#pragma unroll
    for (uint32_t k = 1; k < 4; k++)
        if (i == k) { part = a.part[k]; out = a.out[k]; total = a.total[k]; slices = a.slices[k]; first = a.first[k]; }
    const uint32_t at = ((blockIdx.x - first) * 256u + threadIdx.x) * 4u;
    if (at >= total) return;
    if (total % 4u == 0 && (uintptr_t)out % 8u == 0) {
        kr_f32x4 s = *(const kr_f32x4*)(part + at);
        for (uint32_t k = 1; k < slices; k++) s += *(const kr_f32x4*)(part + (size_t)k * total + at);
        *(kr_u32x2*)(out + at) = kr_u32x2{f32_to_elem_bits<DT>(s[0]) | ((uint32_t)f32_to_elem_bits<DT>(s[1]) << 16),
                                          f32_to_elem_bits<DT>(s[2]) | ((uint32_t)f32_to_elem_bits<DT>(s[3]) << 16)};
        return;
    }
    for (uint32_t e = at; e < at + 4u && e < total; e++) {
        float s = part[e];
        for (uint32_t k = 1; k < slices; k++) s += part[(size_t)k * total + e];
        out[e] = f32_to_elem_bits<DT>(s);
    }
}

// The matrices of `b` whose waves share rows alike, in one launch (p: dtype, bits, group size, x, M, K); the sums of sliced ones go to
// `scratch` from `at` on.
static int launch_codes_alike(const QmmParams& p, const QmvBatch& b, const CodesSplit* split, const bool* in, void* scratch, size_t& at, CodesReduceArgs& r, uint32_t& n_sliced,
                              uint32_t& rblocks, const LaunchCtx& lc) {
    const CodesRows rows = codes_rows(p.M);
    const CodesInstance k = codes_pick(p.dtype, p.bits, p.group_size, rows.mt);
    QmvCodesArgs a{};
    uint32_t n = 0, kwl = 0, nw = QC_WAVES;
    uint32_t tile_slices[4] = {};
    for (int j = 0; j < b.n; j++) {
        if (!in[j]) continue;
        kwl = split[j].kwl;
        a.w[n] = (const unsigned char*)b.w[j];
        a.scales[n] = (const unsigned char*)b.scales[j];
        a.biases[n] = (const unsigned char*)b.biases[j];
        a.out[n] = (uint16_t*)b.out[j];
        a.N[n] = b.N[j];
        a.slices[n] = split[j].slices;
        if (a.slices[n] > 1) {
            if (!scratch) return fail(ERR_UNSUPPORTED, "GEMV on codes: no scratch");
            a.part[n] = (float*)((char*)scratch + at);
            at += ((size_t)a.slices[n] * p.M * b.N[j] * sizeof(float) + 255) & ~(size_t)255;
            r.part[n_sliced] = a.part[n];
            r.out[n_sliced] = a.out[n];
            r.total[n_sliced] = p.M * b.N[j];
            r.slices[n_sliced] = a.slices[n];
            r.first[n_sliced++] = rblocks;
            rblocks += (p.M * b.N[j] + 1023u) / 1024u;
        }
        n++;
    }
    // waves along N: the fewest rounds of workgroups over the chip, and of those the most waves
    const uint32_t cus = codes_cus();
    uint32_t least = ~0u;
    for (uint32_t t = qc_min_nw(rows.mt); t << kwl <= QC_WAVES; t++) {
        if (k.lds(1u << kwl, 1, t << kwl) > QC_LDS) break;
        uint32_t wgs = 0;
        for (uint32_t j = 0; j < n; j++) wgs += ((a.N[j] + 32u * t - 1u) / (32u * t) * a.slices[j] + 7u) / 8u * 8u * rows.tiles;
        if ((wgs + cus - 1u) / cus < least) { least = (wgs + cus - 1u) / cus; nw = t; }
    }
    if (options().qmv_codes_nw) nw = (uint32_t)options().qmv_codes_nw;
    uint32_t stage = k.stage;
    if (options().qmv_codes_stage && (uint32_t)options().qmv_codes_stage < stage) stage = (uint32_t)options().qmv_codes_stage;
    while (stage > 1 && k.lds(1u << kwl, stage, nw << kwl) > QC_LDS) stage /= 2;
    const uint32_t shmem = k.lds(1u << kwl, stage, nw << kwl);
    if (nw < qc_min_nw(rows.mt) || (nw << kwl) > QC_WAVES || shmem > QC_LDS) return fail(ERR_BAD_ARG, "GEMV on codes: geometry");
    uint32_t wgs = 0;
    for (uint32_t j = 0; j < 4; j++) {
        a.first[j] = 0x7FFFFFFFu;
        if (j >= n) { a.slices[j] = 1; continue; }
        a.first[j] = wgs;
        tile_slices[j] = (a.N[j] + 32u * nw - 1u) / (32u * nw) * a.slices[j];
        wgs += (tile_slices[j] + 7u) / 8u * 8u * rows.tiles;
    }
    a.x = (const unsigned char*)p.x;
    a.M = p.M;
    a.K = p.K;
    a.m_tiles = rows.tiles;
    a.m_rows = rows.rows;
    while ((1u << a.log2g) < p.group_size) a.log2g++;
    a.log2kw = kwl;
    a.waves = nw << kwl;
    a.log2stage = stage == 4 ? 2u : stage == 2 ? 1u : 0u;
    hipError_t e = set_max_dynamic_lds(k.fn, shmem);
    if (e != hipSuccess) return hip_fail(e, "GEMV on codes: LDS");
    void* args[] = {&a};
    e = launch_kernel(k.fn, dim3(wgs), dim3(a.waves * 64u), args, shmem, lc);
    return e == hipSuccess ? ERR_OK : hip_fail(e, "GEMV on codes: kernel launch");
}

int launch_qmv_codes(const QmmParams& p, const QmvBatch& b, const CodesSplit* split, void* scratch, const LaunchCtx& lc) {
    bool done[4] = {}, any_sliced = false;
    for (int j = 0; j < b.n; j++) {
        QmmParams q = p;
        q.w = b.w[j]; q.scales = b.scales[j]; q.biases = b.biases[j]; q.out = b.out[j]; q.N = b.N[j];
        if (!qmv_codes_takes(q)) return fail(ERR_UNSUPPORTED, "GEMV on codes: shape not taken");
        if (split[j].slices == 0) return fail(ERR_BAD_ARG, "GEMV on codes: geometry");
        any_sliced = any_sliced || split[j].slices > 1;
    }
    CodesReduceArgs r{};
    uint32_t n_sliced = 0, rblocks = 0;
    size_t at = 0;
    int left = b.n;
    bool started = false;
    while (left) {
        bool in[4] = {};
        int kwl = -1;
        for (int j = 0; j < b.n; j++) {
            if (done[j] || (kwl >= 0 && split[j].kwl != (uint32_t)kwl)) continue;
            kwl = (int)split[j].kwl;
            in[j] = done[j] = true;
            left--;
        }
        LaunchCtx l = lc;
        if (started) l.start = nullptr;
        if (left || any_sliced) l.stop = nullptr;
        started = true;
        int rc = launch_codes_alike(p, b, split, in, scratch, at, r, n_sliced, rblocks, l);
        if (rc) return rc;
    }
    if (!n_sliced) return ERR_OK;
    for (uint32_t j = n_sliced; j < 4; j++) r.first[j] = 0x7FFFFFFFu;
    LaunchCtx l2 = lc;
    l2.start = nullptr;
    void* rargs[] = {&r};
    const void* fn = p.dtype == DT_BF16 ? (const void*)qmv_codes_reduce_kernel<DT_BF16> : (const void*)qmv_codes_reduce_kernel<DT_F16>;
    hipError_t e = launch_kernel(fn, dim3(rblocks), dim3(256), rargs, 0, l2);
    return e == hipSuccess ? ERR_OK : hip_fail(e, "GEMV on codes: reduce kernel launch");
}

}  // namespace mtq
