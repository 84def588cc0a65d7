// Host side of the GEMV with its activations in LDS (kernel in qmv_held_impl.h): which calls it takes and its geometry.
#include "qmv_held_pick.h"

namespace mtq {

// (instances: one translation unit per element type and kind of group)
HeldInstance qmv_held_pick_f16(int bits, int mode, uint32_t rows);
HeldInstance qmv_held_pick_f16_g32(int bits, int mode, uint32_t rows);
HeldInstance qmv_held_pick_bf16(int bits, int mode, uint32_t rows);
HeldInstance qmv_held_pick_bf16_g32(int bits, int mode, uint32_t rows);

static HeldInstance held_pick(int dtype, int bits, uint32_t G, int mode, uint32_t rows) {
    if (dtype == DT_BF16) return G == 32 ? qmv_held_pick_bf16_g32(bits, mode, rows) : qmv_held_pick_bf16(bits, mode, rows);
    return G == 32 ? qmv_held_pick_f16_g32(bits, mode, rows) : qmv_held_pick_f16(bits, mode, rows);
}

static uint32_t held_log2rp(uint32_t rows) {
    uint32_t l = 0;
    while ((1u << l) < rows) l++;
    return l;
}
static uint32_t held_cus() {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    return (uint32_t)cus;
}

// The waves of a workgroup: KP share 16 weight rows, NB such rows side by side.
struct HeldGeometry {
    HeldInstance k;
    uint32_t kpl, nb, per_cu;   // per_cu: workgroups on a compute unit
    uint32_t cus;               // of the device
    uint32_t lds;
};
static bool held_geometry(int dtype, int bits, uint32_t G, int mode, uint32_t rows, uint32_t K, uint32_t blocks, HeldGeometry& g) {
    const Options& o = options();
    const uint32_t cus = held_cus(), rpl = held_log2rp(rows), pairs = (K / 128u + 1u) / 2u;
    g.k = held_pick(dtype, bits, G, mode, rows);
    g.cus = cus;
    if (!g.k.fn) return false;
    // KP: what brings more than a thousand waves to the matrix, each with two and a half steps of 128 codes or more; at least four on long
    // rows. bf16, groups of 64, RMS norm included, KP 1 / 2 / 4 / 8, us: 1536 x 1280 7.0 5.8 5.6 5.5, 2816 x 2304 9.4 7.6 6.6 7.0, 14080 x 2304 11.7
    // 9.4 10.5 11.8, 88612 x 2816 27.7 29.0 29.7 39.3, 5 bits 20480 x 2560 14.3 14.9 15.1 15.1, 57344 x 7808 77.2 80.5 70.7 72.0, 6 bits 86686 x 1408
    // 24.6 26.5 26.0; without a norm 3 bits 5120 x 5120 15.3 11.8 9.0 9.9, 5 bits 2560 x 10240 29.3 17.8 11.4 10.1. A thousand and 24 waves, four to a compute unit,
    // are too few where two waves or one share rows, or a wave has more than 12 steps: 16384 x 4096, 2 bits 15.4 -> 10.8; 8192 x 2304 9.1 -> 7.8, x 3584, gated norm,
    // 14.3 -> 9.8; 4096 x 9216, 3 bits 13.4 -> 10.9, but x 4736 8.2 -> 9.0. For several rows by the row length alone, so that a matrix gives the
    // same bits alone and in a batch (5 rows, 5 bits, 3 x 3456 x 3456 13.0 12.0 14.6, 2 x 14720 x 3456 22.5 22.8 24.1).
    uint32_t kpl = K > 4608 ? 2 : 0;
    const bool fixed = mode == HELD_PLAIN && rows > 1;
    auto few = [&]() { return (blocks << kpl) < 1024u || ((blocks << kpl) == 1024u && (kpl < 2 || (K / 128u) >> kpl > 12u)); };
    while (kpl < (fixed ? 2u : 4u) && (fixed || few()) && (K / 128u) * 2u >= 5u << (kpl + 1)) kpl++;
    if (o.qmv_held_kp) for (kpl = 0; (2u << kpl) <= (uint32_t)o.qmv_held_kp; kpl++) {}
    while (kpl && (1u << kpl) > pairs) kpl--;
    // a normalised row: at most two pieces of 16 elements a thread
    const uint32_t least = mode == HELD_PLAIN ? 1u : (K / 16u + 127u) / 128u;
    for (uint32_t most = 8; most <= 16; most += 8) {   // waves
        if ((1u << kpl) > most) continue;
        uint32_t nb = most >> kpl;
        while (nb > 1 && g.k.lds(K, rpl, nb << kpl) > 160u * 1024u) nb--;
        g.lds = g.k.lds(K, rpl, nb << kpl);
        if (g.lds > 160u * 1024u) return false;
        g.per_cu = most == 8 && g.lds <= 80u * 1024u ? 2u : 1u;
        const uint32_t want = (blocks + cus * g.per_cu - 1u) / (cus * g.per_cu);
        if (nb > want) nb = want ? want : 1u;
        if (o.qmv_held_nb && (uint32_t)o.qmv_held_nb <= most >> kpl) nb = (uint32_t)o.qmv_held_nb;
        while ((nb << kpl) < least && ((nb + 1u) << kpl) <= most) nb++;
        g.kpl = kpl;
        g.nb = nb;
        g.lds = g.k.lds(K, rpl, nb << kpl);
        if ((nb << kpl) >= least && g.lds <= 160u * 1024u && (most == 16 || g.per_cu == 2)) return true;
    }
    return false;
}

// p: dtype, bits, group size, x, M, K; g: the geometry of a call that is taken
static bool held_plan(const QmvParams& p, const QmvBatch& b, const HeldNorm& n, HeldGeometry& g) {
    const uint32_t G = p.group_size, K = p.K, rows = n.mode == HELD_PLAIN ? p.M : 2u;
    if ((p.dtype != DT_F16 && p.dtype != DT_BF16) || (p.bits != 2 && p.bits != 3 && p.bits != 4 && p.bits != 5 && p.bits != 6 && p.bits != 8)) return false;
    if ((G != 32 && G != 64 && G != 128) || K == 0 || K % 128 || K % G || rows == 0 || rows > 16 || b.n < 1 || b.n > 4 || K > (1u << 17)) return false;
    if ((uintptr_t)p.x % 16) return false;
    if (n.mode != HELD_PLAIN && ((uintptr_t)n.weight % 16 || (uintptr_t)n.eps % 4)) return false;
    if (n.mode == HELD_GATED && ((uintptr_t)n.gate % 16 || n.dv < 16 || n.dv > 1024 || (n.dv & (n.dv - 1)))) return false;   // a head's pieces in neighbouring lanes of a wave
    uint64_t blocks = 0;
    for (int j = 0; j < b.n; j++) {
        if (b.N[j] == 0 || (uintptr_t)b.w[j] % 16 || (uintptr_t)b.scales[j] % 4 || (uintptr_t)b.biases[j] % 4) return false;
        blocks += (b.N[j] + 15u) / 16u;
    }
    return blocks < (1u << 26) && held_geometry(p.dtype, p.bits, G, n.mode, rows, K, (uint32_t)blocks, g);
}
bool qmv_held_takes(const QmvParams& p, const QmvBatch& b, const HeldNorm& n) {
    HeldGeometry g;
    return held_plan(p, b, n, g);
}

// Where the kernel stands against the others: they have a launch per matrix, or three where a row is normalised first and their
// row lengths are not the ones it is fused for. us, bf16, groups of 64, others -> this.
// RMS norm, 4 bits: 1280 x 1024 9.5 -> 5.0, 2816 x 2304 11.1 -> 6.8, 512 x 9216 11.8 -> 10.8 (norm, GEMV, sum); against the norm inside the
// matrix-core GEMV, from 24 M codes: 14080 x 2304 10.4 -> 9.4, 19200 x 3200 15.9 -> 14.7, 67882 x 2304 26.0 -> 21.3, 25600 x 3328 / 3968 / 4224 / 4608 / 4736 / 4864 / 4992 / 5248 / 5632
// 14.8 17.1 24.4 22.8 22.0 18.7 22.5 22.2 19.1 -> 15.1 17.7 19.4 19.2 22.4 20.8 23.0 24.1 22.7, 46080 x 4224 / 4736 / 4864 / 4992 34.3 32.6 28.0 33.5 -> 29.9 30.7 28.2 32.0. Rows of whole 2048 codes are
// the streaming kernel's, which takes them in one launch too: 512 x 2048 4.4 -> 5.2, 1000 x 4096 4.7 -> 6.5, 8192 5.1 -> 10.2, 1500 x 12288 11.3 -> 12.2. 4 bits in groups
// of 32, where each group is scaled for itself: 14080 x 2304 11.2 -> 10.1, 11936 / 25728 x 2176 10.6 / 15.0 -> 10.1 / 13.7, 86686 x 1280 20.2 -> 18.5, but from 24 M codes 15616 / 33648 x 1664
// 8.2 / 12.8 -> 9.0 / 14.7, 13536 / 29152 x 1920 8.2 / 11.4 -> 9.1 / 12.6, 20832 x 2688 13.2 -> 15.2, 8112 / 17488 x 3200 8.4 / 13.3 -> 9.3 / 17.4, 6144 / 9456 x 4224 9.9 / 11.6 -> 11.0 / 14.4, 86686 x 1664 21.5 -> 24.7.
// 2 bits 4096 x 1024 9.6 -> 5.4, 8192 x 8192 14.2 -> 11.7; 3 bits 14720 x 3456 16.3 -> 11.4, 5 bits 20480 x 2560 23.8 -> 14.4, 57344 x 8192 78.8 -> 73.5, 6 bits
// 131838 x 1408 54.6 -> 37; 8 bits 14336 x 1664 14.2 -> 9.3, 32768 x 4608 38.9 -> 27.8, but 20480 x 5120 23.1 -> 24.3.
// Heads of more than 65536 rows, of which the GEMV of the others reads 2- to 5-bit codes faster: 70000 / 100000 / 150000 x 3968, 2 bits 31.5 / 39.8 / 53.1 -> 36.7 / 50.7 / 64.3, 3 bits
// 43 / 56 / 75 -> 46 / 63 / 81, 100000 x 4096, 5 bits 73 -> 79; 100000 x 3328, 2 bits 35.0 -> 38.5, 3584, 3 bits 50.2 -> 52.5; 6656 and 7936, 2 bits 60 and 64 -> 62 and 69, 7936, 3 bits
// 150000 130 -> 135. Rows of more than 16384 codes leave a compute unit one workgroup, whose second round costs the most there: 5120 x 18944, 5 bits 32.2 -> 36.5, 8192 38.8 -> 38.9;
// 8192 x 28672, 2 bits 36.0 -> 42.1, 16384 55.5 -> 47.5.
// A workgroup to a compute unit has eight blocks of 16 rows at a time: a head of a few rows more than full rounds of those (32768 rows on 256 units) takes a round more, while the
// others' time goes with its rows. Up to two fifths of a round into the third or a later one, us, 68000 | 100651 | (full rounds) 131072 rows: 4 bits x 1792 18.0 -> 19.0 | 22.9 -> 25.6 |
// 27.3 -> 27.0, 1920 21.7 -> 21.8 | 27.5 -> 30.0 | 31.7 -> 31.6, 2688 29.5 -> 30.0 | 38.9 -> 41.3 | 46.4 -> 43.5, 2944 30.5 -> 32.3 | 40.6 -> 44.5 | 47.7 -> 47.2 (but 2816 27.3 -> 26.4 |
// 35.9 -> 36.1, 3072 27.8 -> 28.2 | 37.7 -> 39.2 | 46.1 -> 40.7, 2432 29.7 -> 26.8 | 39.6 -> 37.3), in groups of 32 x 1152 17.1 -> 18.1 | 21.5 -> 23.8 | 24.8 -> 24.5; groups of 32 at 70000 |
// 100651 | 131072 rows: 2 bits x 1920 21.2 -> 22.1 | 25.8 -> 29.8 | 29.8 -> 30.9, 2688 29.4 -> 30.5 | 39.0 -> 41.5 | 46.8 -> 43.6, 3 bits x 3200 39.9 -> 43.1 | 52.7 -> 58.8 | 62.7 -> 62.3, 5 bits x
// 3712 53.1 -> 60.6 | 72.1 -> 81.6 | 90.7 -> 87.9, 6 bits 58.9 -> 62.3 | 79.4 -> 83.2 | 97.2 -> 89.6, 8 bits 54.3 -> 60.5 | 74.3 -> 82.9 | 93.3 -> 87.8. At any number of rows: x 3200, 4 bits 31.2 -> 36.0 | 40.6 -> 49.4 | 48.5 -> 51.5, 2 bits 38.1 -> 40.7 at 100651, 43.0 -> 43.2 at 131072; 4 bits in
// groups of 32 x 1408 50257 / 78000 / 115000 rows 14.8 19.1 24.8 -> 15.3 20.4 26.8.
static bool held_norm_short_round(int bits, uint32_t G, uint32_t N, uint32_t K) {
    const bool odd = K % 256 != 0;
    const bool row = bits == 4 && G == 32                  ? K > 1024
                     : bits == 4 || (bits == 2 && G == 32) ? (K >= 1792 && K < 2048 && (odd || (bits == 4 && G == 64))) || (K > 2560 && odd)
                                                           : G == 32 && ((bits == 8 && K > 3328) || (odd && ((bits == 3 && K > 2688) || (bits == 5 && K > 2944) || (bits == 6 && K > 3584))));
    if (!row || K > 4096) return false;   // (first: most calls need not ask the device)
    const uint32_t round = 128u * held_cus(), over = N % round;
    return N > 2 * round && over != 0 && over * 5 <= 2 * round;
}
bool qmv_held_norm_preferred(int bits, uint32_t G, uint32_t N, uint32_t K) {
    if (held_norm_short_round(bits, G, N, K)) return false;
    if (bits == 8) return K < 5120;
    if (K > 16384 && N > 4096 && N < (K > 20480 ? 16384u : 8192u)) return false;
    if (N > 65536) {
        if (bits == 2 && ((K > 3072 && K <= 4096) || (K >= 6656 && K < 8192))) return false;
        if (bits == 3 && ((K > 3456 && K <= 4096) || (K > 7680 && K <= 8192))) return false;
        if (bits == 5 && K > 3968 && K <= 4096) return false;
    }
    if (bits != 4) return true;
    if (K % 2048 == 0) return false;
    const uint64_t codes = (uint64_t)N * K;
    if (codes < 24000000ull) return true;
    if (G == 32) return K <= (N > 32768 && K % 256 ? 1280 : 1600) || (K > 2048 && K <= 2304 && codes < 60000000ull);
    return K <= (N > 65536 ? 3072 : 3200) || (K > 4096 && K < 5120 && (K <= 4608 || K % 256));
}
// Gated norm, 4 bits, row lengths that the streaming kernel does not take (norm, GEMV of two rows and sum -> this): 512 / 2560 / 5120 / 16384 rows x 2304 9.3 8.7 10.2 13.2 -> 6.6
// 6.9 9.2 10.4, x 4608 9.6 10.6 12.8 18.4 -> 9.4 9.8 12.0 14.9. Longer rows take a compute unit's LDS for two workgroups of few waves: 512 / 2048 / 2560 / 4096 / 5120 / 8192 / 12288 rows x
// 5376 8.7 9.6 10.3 10.5 12.5 13.0 14.9 -> 9.3 9.8 9.6 9.8 13.7 13.8 16.5, x 6016 8.9 9.3 10.6 10.8 13.7 14.4 17.3 -> 9.4 10.0 9.6 9.7 13.9 14.1 16.7, x 7680 10.8 10.4 10.9 11.3 13.2 14.2 18.5 ->
// 9.8 10.2 10.1 10.2 15.3 15.4 18.7, x 9216 9.2 10.8 12.6 13.2 14.6 16.5 20.1 -> 11.9 12.5 12.1 12.3 14.8 15.0 21.3; 5120 / 8192 x 5120 12.5 12.9 -> 12.0 12.2.
bool qmv_held_gated_preferred(uint32_t N, uint32_t K) {
    if (K <= 4608) return true;
    if (K > 6144 && K <= 8192) return N <= 4096 || N > 8192;
    if (N <= 2048) return false;
    if (K > 8192) return N <= 8192;
    return N <= 4096 || K <= 5120 || K > 5632;
}
// Batches of 2..16 rows, of the widths that the K-run kernel has not. As there, a matrix's route cannot depend on whether it comes in a batch, so the
// lines lie where two matrices of a size, or a square one with the two of a quarter of its rows that come with it, together gain more than one alone
// loses. us on the device (bf16, groups of 64, weights from memory), others -> this, alone | together (q: 1, 1/4, 1/4; 2: two):
//                  2 rows                     4 rows                     8 rows                      16 rows
//   2 bits  2048 x 2048   4.2 -> 4.6 | q 12.1 -> 4.8    4.7 -> 4.7 | 14.7 -> 4.8    6.4 -> 5.3 | 15.8 -> 5.6     9.1 -> 6.4 | 9.5 -> 6.7
//           4096 x 4096   5.3 -> 6.1 | q 15.4 -> 7.4    5.8 -> 6.7 | 19.6 -> 8.2    8.0 -> 7.9 | 17.6 -> 8.6    10.7 -> 10.1 | 21.2 -> 13.1
//           14336 x 4096  9.4 -> 9.5 | 2 18.6 -> 15.1  10.1 -> 9.9 | 19.9 -> 15.6  12.9 -> 11.0 | 25.4 -> 18.2  15.6 -> 19.1 | 31.0 -> 28.3 (not taken)
//           8192 x 8192   7.9 -> 11.5 | q 18.7 -> 14.9 (not taken)  9.8 -> 11.7 | 22.9 -> 14.2  20.6 -> 13.4 | 38.0 -> 19.4
//           28672 x 8192 24.4 -> 25.4 | 2 49.0 -> 41.7 29.4 -> 26.6 | 58.8 -> 48.1 41.3 -> 31.4 | 81.9 -> 50.8
//   3 bits  1024 x 1024   3.7 -> 4.4 | q 10.5 -> 4.4    4.4 -> 4.4 | 12.5 -> 4.5    6.0 -> 4.9 | 12.0 -> 5.0     6.4 -> 6.1 | 6.8 -> 6.0
//           4096 x 4096   5.5 -> 6.8 | q 18.1 -> 8.2    6.3 -> 7.3 | 23.0 -> 9.4    8.2 -> 8.5 | 17.9 -> 9.7    11.0 -> 10.7 | 21.6 -> 13.9
//           14336 x 4096 11.2 -> 12.0 | 2 22.3 -> 19.1 11.4 -> 12.3 | 22.5 -> 19.5 14.6 -> 12.9 | 28.8 -> 21.4
//           28672 x 8192 29.9 -> 33.1 | 2 59.3 -> 54.4 31.5 -> 34.3 | 62.9 -> 62.6 (not taken)  44.0 -> 45.5 | 88.9 -> 83.6
//           8192 x 1024                                                                         7.0 -> 7.8 | 7.8 -> 7.9 (not taken)
//   5 bits  3072 x 3072   5.3 -> 7.0 | q 16.8 -> 8.6    6.5 -> 7.4 | 21.1 -> 9.4    8.0 -> 8.2 | 20.5 -> 9.5    14.0 -> 9.9 | 14.1 -> 10.9
//           4096 x 4096   5.8 -> 7.6 | q 18.4 -> 9.4    7.0 -> 8.2 | 23.9 -> 10.4   8.7 -> 9.3 | 18.8 -> 10.8   12.2 -> 11.4 | 23.7 -> 15.3
//           8192 x 4096   7.9 -> 9.7 | 2 15.6 -> 14.7   8.6 -> 10.7 | 16.8 -> 15.2 (neither taken)  10.8 -> 11.3 | 21.7 -> 17.0  14.8 -> 15.2 | 29.4 -> 22.7
//           14336 x 4096 12.8 -> 14.2 | 2 25.1 -> 23.9 13.0 -> 14.6 | 25.8 -> 24.5 (neither)        16.2 -> 15.4 | 32.1 -> 26.7
//           10240 x 5120 14.5 -> 16.2 | 2 28.7 -> 22.3 15.4 -> 17.0 | 30.5 -> 23.0 18.8 -> 15.4 | 37.5 -> 29.1
//           21504 x 6144 25.2 -> 25.4 | 2 50.2 -> 46.0 26.5 -> 31.5 | 52.4 -> 47.6 (not taken)      34.6 -> 28.5 | 68.1 -> 50.5
//   6 bits  2048 x 2048   3.9 -> 5.4 | q 12.5 -> 5.8    4.9 -> 5.4 | 15.5 -> 5.7    6.5 -> 6.2 | 16.5 -> 6.4     9.6 -> 7.2 | 10.9 -> 7.6
//           7168 x 2048   6.0 -> 7.1 | 2 11.8 -> 9.5    6.2 -> 7.1 | 12.2 -> 9.7    7.5 -> 8.6 | 14.8 -> 10.3   11.0 -> 8.8 | 11.6 -> 13.4
//           14336 x 4096 13.3 -> 13.6 | 2 26.4 -> 23.8 13.8 -> 14.1 | 27.1 -> 24.1 17.7 -> 15.2 | 34.6 -> 25.9
//           8192 x 8192  14.2 -> 15.4 | q 27.6 -> 21.9 15.2 -> 15.8 | 31.5 -> 21.0 23.8 -> 20.6 | 43.2 -> 26.9
// (3 rows as 4, 12 as 16. At 5 bits up to 4 rows the others lose little on rows of whole 2048 codes, whose steps of 512 the waves of the GEMV of up to 8 rows
// share evenly: tall matrices of those are left there.)
// From 9 rows past 8192 weight rows the tiles are ahead (14336 x 4096, 16 rows, 5 bits 18.6 -> 21.3), but at 2 bits; rows of more than 8192 codes leave a
// compute unit one workgroup: 3 bits, 4 rows 4096 x 11008 11.1 -> 13.4.
// In groups of 32 a group is scaled for itself, which costs a wave of up to four rows most on long rows of tall matrices (alone | two):
//   2 rows  2 bits 12032 x 6016 10.4 -> 15.2 | 20.5 -> 20.0, 20480 x 5120 14.4 -> 17.0 | 28.1 -> 26.5    3 bits 16384 x 8192 19.8 -> 21.9 | 39.5 -> 39.9    6 bits 28672 x 8192 41.6 -> 47.1 | 83.3 -> 79.5
//   4 rows  5 bits 18432 x 5120 23.1 -> 30.7 | 45.7 -> 44.6, x 6016 24.0 -> 35.6 | 47.7 -> 52.8    6 bits 18432 x 5120 24.4 -> 30.2 | 48.4 -> 44.2, 16384 x 8192 28.0 -> 35.8 | 55.7 -> 54.1 (none taken)
//           5 bits 24576 x 5120 27.3 -> 31.6 | 54.1 -> 47.8    6 bits 28672 x 5120 32.3 -> 32.5 | 64.4 -> 58.8    2 bits 16384 x 8192 19.4 -> 20.0 | 39.2 -> 34.2, square and nearly square ones: 5 bits
//           6016 x 6016 12.7 -> 13.6 | q 26.4 -> 16.8 (taken). Groups of 64, 5 bits: 18432 x 6016 26.2 -> 31.7 | 52.2 -> 47.3 (not)
// A head has no other beside it and goes by its own times (68000 | 100651 | 131072 rows):
//   2 rows  2 bits x 3328 23.9 30.5 36.0 -> 26.1 36.2 45.3, x 4096 24.6 32.3 39.7 -> 27.3 38.4 48.6, x 7168 40.1 54.7 70.5 -> 46.7 65.8 83.5, but x 2944 25.6 33.1 -> 23.8 32.6, x 5120 37.1 52.2 66.0 ->
//           34.6 49.9 61.1    3 bits x 4096 35.0 48.0 55.6 -> 35.0 48.8 60.5, x 6144 47.2 68.7 89.7 -> 50.8 73.6 90.8, x 8192 61.6 87.7 112.1 -> 67.9 97.4 120.2, but x 5120 47.0 67.0 86.6 -> 45.0 63.1 78.7
//           groups of 32, at 100651: 2 bits x 1536 / 2944 / 4096 / 5120 21.2 34.5 40.8 51.7 -> 26.8 39.2 46.1 59.2, 3 bits x 1536 / 2048 / 4096 27.4 29.2 50.3 -> 29.8 31.8 55.5, but x 2944 47.0 -> 46.0
//   8 rows  3 bits x 8192 90.3 140.9 173.9 -> 100.7 146.4 185.1    5 bits x 4096 51.1 70.9 89.5 -> 55.0 77.2 89.3, 34000 rows 30.6 -> 34.2, but x 3584 49.8 69.9 88.5 -> 49.4 68.0 78.9
//           groups of 32 x 2048, 34000 / 68000 rows: 5 bits 19.2 31.1 -> 22.1 34.7, 6 bits 19.9 31.9 -> 21.8 33.6, but x 1664 18.7 29.3 -> 17.6 27.4
static bool held_head_slower(int bits, uint32_t G, uint32_t M, uint32_t N, uint32_t K) {
    if (N <= 32768) return false;
    const bool most = N > 65536, mid = K > 3072 && K <= 4096;
    if (M > 4) return G == 32 ? bits >= 5 && K == 2048 : (bits == 5 && K > 3840 && K <= 4096) || (bits == 3 && most && K > 7168);
    if (bits == 2) return G == 32 ? most || K > 2048 : most && (mid || (K > 6144 && K < 8192));
    if (bits != 3 || !most) return false;
    return G == 32 ? K <= 2048 || mid : (M == 2 && K > 5120) || (N > 98304 && K > 3584 && K <= 4096);
}
bool qmv_held_preferred(int bits, uint32_t G, uint32_t M, uint32_t N, uint32_t K) {
    if (M < 2 || M > 16 || bits == 4 || bits == 8) return false;
    const bool tall = N >= 2 * (uint64_t)K;
    if (held_head_slower(bits, G, M, N, K)) return false;
    if (G == 32 && M <= 4) {
        const bool fewer = bits == 2 ? M == 2 && N > 16384 : bits == 3 ? M == 2 : M > 2 || N > 16384;
        if (K > 5120 && 2 * (uint64_t)N > 3 * (uint64_t)K && (K % 2048 || fewer)) return false;
        if (K > 4608 && K <= 5120 && N > 16384 && N <= 20480 && (bits >= 5 ? M > 2 : bits == 2 && M == 2)) return false;
    } else if (bits == 5 && (M == 3 || M == 4) && K > 5632 && N > 16384 && N <= 20480) {
        return false;
    }
    if (M > 8) return K <= 4096 && (N <= 8192 || (bits == 2 && (M <= 12 || K <= 3328))) && !(bits != 6 && K <= 1024 && N > 4096);
    if (K > 8192) return false;
    if (bits == 5 && M <= 4 && tall && K % 2048 == 0) return false;
    if (bits == 3 && M >= 3 && M <= 4 && K > 6144 && N >= 3 * (uint64_t)K) return false;
    return !(bits == 2 && M == 2 && K > 6144 && N <= 2 * (uint64_t)K);
}

int launch_qmv_held(const QmvParams& p, const QmvBatch& b, const HeldNorm& n, const LaunchCtx& lc) {
    HeldGeometry g;
    if (!held_plan(p, b, n, g)) return fail(ERR_UNSUPPORTED, "GEMV with its activations in LDS: shape not taken");
    const uint32_t rows = n.mode == HELD_PLAIN ? p.M : 2u;
    QmvHeldArgs a{};
    for (int j = 0; j < 4; j++) {
        a.first[j] = 0x7FFFFFFFu;
        if (j >= b.n) continue;
        a.w[j] = (const unsigned char*)b.w[j];
        a.scales[j] = (const unsigned char*)b.scales[j];
        a.biases[j] = (const unsigned char*)b.biases[j];
        a.out[j] = (uint16_t*)b.out[j];
        a.N[j] = b.N[j];
        a.first[j] = a.blocks;
        a.blocks += (b.N[j] + 15u) / 16u;
    }
    a.x = (const unsigned char*)p.x;
    a.norm_w = (const unsigned char*)n.weight;
    a.gate = (const unsigned char*)n.gate;
    a.eps = n.eps;
    a.dv = n.dv;
    a.M = n.mode == HELD_PLAIN ? p.M : 1u;
    a.K = p.K;
    while ((1u << a.log2g) < p.group_size) a.log2g++;
    a.log2kp = g.kpl;
    a.log2rp = held_log2rp(rows);
    a.waves = g.nb << g.kpl;
    const uint32_t tasks = (a.blocks + g.nb - 1u) / g.nb, most = g.cus * g.per_cu, wgs = tasks < most ? tasks : most;
    hipError_t e = g.lds > 64u * 1024u ? set_max_dynamic_lds(g.k.fn, g.lds) : hipSuccess;   // (what a launch may have unasked: no static LDS here)
    if (e != hipSuccess) return hip_fail(e, "GEMV with its activations in LDS: LDS");
    void* args[] = {&a};
    e = launch_kernel(g.k.fn, dim3(wgs), dim3(a.waves * 64u), args, g.lds, lc);
    return e == hipSuccess ? ERR_OK : hip_fail(e, "GEMV with its activations in LDS: kernel launch");
}

}  // namespace mtq
