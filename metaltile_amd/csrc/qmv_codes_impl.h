// The matrix-core GEMV on codes (see qmv_codes.hip for the routing and the geometry): kernel and argument block.
#pragma once
// Batches of activation rows (5 to 128 where it is chosen) against one or several weight matrices of the same row length, f16 / bf16, codes of
// 2, 3, 4, 5, 6 and 8 bits, rows of any whole number of 128 codes, with exact-dequant arithmetic:
// out[m][n] = sum_g (s[n][g] * sum_k q[n][k] x[m][k] + b[n][g] * sum_k x[m][k]), the rows of mt_qmm
// (crates/metaltile-std/src/mlx/quantized.rs:1330-1500).
//
// What bounds such a batch is the stream of weights, as long as nothing else in the compute unit takes longer. So the
// codes themselves are the operands of the 16x16x32 MFMA, as MAGIC + code in the element type (exact; one masked OR for
// two codes where they lie 16 bits apart), and the scale is applied to the sum of a group: 4 FMAs for 16 x 16 results
// and a group, against a conversion of every weight. The bias term, sum_g (b - MAGIC s)[n][g] * xsum[g][m], is a product
// of its own with K / group_size terms in place of K: it runs on the f32 matrix instruction, four groups at a time,
// with xsum worked out once per workgroup where the activations are staged.
//
// A workgroup has NW x KW waves. Each works on 32 weight rows (two blocks of 16: an activation operand out of LDS serves
// both) and one of KW runs of steps of 128 codes; the KW sums of a result meet in LDS at the end. Long rows of few weight rows
// are also dealt to several workgroups (slices), whose f32 sums a second launch adds in order. Which wave and workgroup
// works on which step depends on the row length, the row count and the matrix's own N: a matrix gives the same bits
// alone and in a batch.
//
// Activations go through LDS a step at a time, turned into operand order, two buffers. Weights are loaded with
// neighbouring lanes on neighbouring 16 bytes of a row (in operand order, 16 rows next to each other, a load occupies the
// compute unit's address path four times as long), two steps ahead, and turned in an LDS area of the wave's own; rows
// there are 16 bytes apart from a multiple of 32 (128 at 4 and 8 bits) so that the operand reads spread over the banks.
// A step of eight waves (256 x 128 codes) takes 1.2 / 1.45 / 1.8 us at 16 / 32 / 48 activation rows: 5.2 TB/s of 6-bit codes at 16 rows, less than half of that of
// 4-bit codes at 48, where the LDS traffic of operands (98 KB of activations and 48 KB of codes in and out) and the conversion stand beside the MFMAs. us, tiles -> this:
// 4736 x 20096, 5 bits, 32 rows 263 -> 39; 2 x 8704 x 3968, 8 bits, 40 rows 45.1 -> 34.7 (the table is at qmv_codes_preferred).
// Every load is a buffer load whose out-of-range offsets read zeros without a memory access: rows past the matrix or the
// batch and steps past the slice are given such offsets.
#include "codes16.h"
#include "mtq_internal.h"

namespace mtq {

struct QmvCodesArgs {
    const unsigned char* w[4];
    const unsigned char* scales[4];
    const unsigned char* biases[4];
    uint16_t* out[4];
    float* part[4];          // f32 sums [slice][M][N] of a sliced matrix
    uint32_t N[4];
    uint32_t slices[4];      // of K
    uint32_t first[4];       // first workgroup of each matrix; 0x7FFFFFFF past the last one
    const unsigned char* x;
    uint32_t M, K;
    uint32_t m_tiles, m_rows;   // tiles of activation rows, and the rows of each (the last one has what is left)
    uint32_t log2g;          // of the group size
    uint32_t log2kw, waves;  // waves of a workgroup: NW * KW
    uint32_t log2stage;      // steps of activations between barriers: 1, 2 or 4
};

// What the number of 16-row activation tiles fixes: the 16-element pieces of a step's activations that a thread stages, the least waves along N for that.
template <int MT> struct QcShape {
    static constexpr int XU = MT == 1 ? 1 : 2;
    static constexpr uint32_t STAGE = MT <= 2 ? 4 : 2;   // steps of activations between barriers, at most
};
constexpr uint32_t qc_min_nw(uint32_t mt) { return mt == 1 ? 2u : mt; }
constexpr uint32_t QC_WAVES = 8;   // of a workgroup at most

template <int BITS, bool G32, int MT> struct QcLds {
    static constexpr uint32_t ROWS = MT * 16;
    static constexpr uint32_t QS = ROWS * 16 + 16;             // one quarter of an operand of every row
    static constexpr uint32_t XB = 16 * QS;                    // a K-wave's step of activations: [64-code half][operand][quarter][row]
    static constexpr uint32_t GPS = G32 ? 4 : 2;               // sums per step and row
    static constexpr uint32_t XSB = ROWS * 4 * GPS;            // and of their sums: [group][row]
    static constexpr uint32_t TS = 32 * BITS + 16;             // a weight row's two steps
    static constexpr uint32_t TB = 32 * TS;
    static constexpr uint32_t SG = G32 ? 16 : 8;               // scales (and biases less MAGIC scales), f32, of four steps: [group or 64 codes][weight row]
    static constexpr uint32_t SB = 2 * SG * 128;
    static constexpr uint32_t bytes(uint32_t kw, uint32_t stage, uint32_t waves) {
        const uint32_t loop = kw * (2 * stage * XB + 8 * XSB) + waves * (TB + SB), red = waves * 2 * MT * 1024u;
        return loop > red ? loop : red;
    }
};

template <int DT, int BITS, bool G32, int MT> __global__ __launch_bounds__(QC_WAVES * 64) void qmv_codes_kernel(QmvCodesArgs a) {
    using L = QcLds<BITS, G32, MT>;
    constexpr int R = 2, NL = BITS, XU = QcShape<MT>::XU;
    constexpr int U = G32 ? 1 : 2;                      // steps per f32 MFMA of the bias term (four sums)
    constexpr uint32_t ROWS = L::ROWS, QS = L::QS, XB = L::XB, XSB = L::XSB;
    using C = QcCodes<DT, BITS, false>;
    constexpr float MAGIC = C::MAGIC;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t j = lane & 15u, q = lane >> 4;
    const uint32_t kwl = a.log2kw, KW = 1u << kwl, kw = wave & (KW - 1u), nw = wave >> kwl, threads = a.waves * 64u;
    const uint32_t K = a.K, wrow = K / 8u * BITS, gpr = K >> a.log2g;

    // this workgroup's matrix: its arguments are read from the argument segment by its number
    const __attribute__((address_space(4))) QmvCodesArgs* const ka = (const __attribute__((address_space(4))) QmvCodesArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    const uint32_t mat = (blockIdx.x >= a.first[1] ? 1u : 0u) + (blockIdx.x >= a.first[2] ? 1u : 0u) + (blockIdx.x >= a.first[3] ? 1u : 0u);
    const uint32_t N = ka->N[mat], slices = ka->slices[mat], id = blockIdx.x - ka->first[mat];
    // The row tiles of one tile of weights and slice stand 8 workgroups apart: on one XCD, whose L2 then gives the weights to all.
    const uint32_t octet = id / (8u * a.m_tiles), in = id - octet * (8u * a.m_tiles), part_id = octet * 8u + (in & 7u), m0 = (in >> 3) * a.m_rows;
    const uint32_t tile = part_id / slices, slice = part_id - tile * slices, M = min(a.M - m0, a.m_rows);
    const uint32_t steps = K / 128u, first = steps * slice / slices, all = steps * (slice + 1u) / slices - first, iters = (((all + 1u) / 2u + KW - 1u) >> kwl) * 2u;
    // K-wave i has steps [i * iters, (i + 1) * iters) of the slice, the last one what is left
    const uint32_t my = kw * iters, cnt = all > my ? min(all - my, iters) : 0u, mine = first + my;
    const uint32_t tile_rows = 32u * (a.waves >> kwl), tile0 = tile * tile_rows;
    if (tile0 >= N) return;   // (what fills up the last eight)
    const uint32_t row0 = min(tile0 + 32u * nw, N), rows = min(N - row0, 32u);

    const __amdgpu_buffer_rsrc_t wr = kr_rsrc((uint64_t)ka->w[mat] + (uint64_t)row0 * wrow, rows * wrow);
    const __amdgpu_buffer_rsrc_t sr = kr_rsrc((uint64_t)ka->scales[mat] + (uint64_t)row0 * gpr * 2u, (rows * gpr * 2u + 3u) & ~3u);   // (a dword whose second half lies past the end is read whole)
    const __amdgpu_buffer_rsrc_t br = kr_rsrc((uint64_t)ka->biases[mat] + (uint64_t)row0 * gpr * 2u, (rows * gpr * 2u + 3u) & ~3u);
    const __amdgpu_buffer_rsrc_t xr = kr_rsrc((uint64_t)a.x + (uint64_t)m0 * K * 2u, M * K * 2u);

    const uint32_t sgl = a.log2stage, SGM = (1u << sgl) - 1u;
    unsigned char* const xs0 = lds + ((2u * KW * XB) << sgl);
    unsigned char* const turn = xs0 + 8u * KW * XSB + wave * (L::TB + L::SB);
    float* const sbl = (float*)(turn + L::TB);

    // weights of two steps: 16-byte piece id % (2 BITS) of row id / (2 BITS)
    uint32_t woff[NL], wput[NL], wpast[NL];
#pragma unroll
    for (int l = 0; l < NL; l++) {
        const uint32_t id16 = l * 64u + lane, r = id16 / (2u * BITS), p = id16 - r * (2u * BITS);
        woff[l] = r * wrow + p * 16u + mine * (16u * BITS);
        wput[l] = r * L::TS + p * 16u;
        wpast[l] = p >= (uint32_t)BITS ? 1u : 0u;
    }
    kr_u32x4 ring[NL];
    auto load_w = [&](uint32_t it) {
#pragma unroll
        for (int l = 0; l < NL; l++) ring[l] = __builtin_amdgcn_raw_buffer_load_b128(wr, (int)((woff[l] + it * (16u * BITS)) | ((cnt - 1u - it - wpast[l]) & KR_OOB)), 0, KR_NT);
    };
    // scales and biases of four steps: 16 bytes of each of the 32 rows (groups of 32: in two halves, lanes 32 .. 63 the second),
    // from the even element at or before the first one needed (which is odd for groups of 128 codes or more only; those
    // need four of the eight). One load has 32 or 64 lines to find, so few and wide ones: as 2-byte loads of a step's own
    // values they kept the address path busier than the weights.
    const uint32_t lrow = lane & 31u;
    const bool wide_g = !G32 && a.log2g == 7u;   // groups of 128: each stands for two runs of 64 codes
    kr_u32x4 sraw, braw;
    const uint32_t s_at = lrow * gpr + (G32 ? mine * 4u : wide_g ? mine : mine * 2u);
    auto load_s = [&](uint32_t it) {
        const uint32_t dead = ((cnt - 1u - it) & KR_OOB) | (G32 ? 0u : (31u - lane) & KR_OOB);
        const int o = (int)((((s_at + (G32 ? it * 4u : wide_g ? it : it * 2u)) & ~1u) * 2u + (G32 ? (lane >> 5) * 16u : 0u)) | dead);
        sraw = __builtin_amdgcn_raw_buffer_load_b128(sr, o, 0, 0);
        braw = __builtin_amdgcn_raw_buffer_load_b128(br, o, 0, 0);
    };
    auto store_s = [&](uint32_t it) {   // (it: the first of the four steps)
        if (wide_g) {
            const uint32_t by = (s_at & 1u) * 2u;
            uint32_t s4[2], b4[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                s4[i] = __builtin_amdgcn_alignbyte(sraw[i + 1], sraw[i], by);
                b4[i] = __builtin_amdgcn_alignbyte(braw[i + 1], braw[i], by);
            }
            sraw = kr_u32x4{__builtin_amdgcn_perm(0u, s4[0], 0x01000100u), __builtin_amdgcn_perm(0u, s4[0], 0x03020302u), __builtin_amdgcn_perm(0u, s4[1], 0x01000100u), __builtin_amdgcn_perm(0u, s4[1], 0x03020302u)};
            braw = kr_u32x4{__builtin_amdgcn_perm(0u, b4[0], 0x01000100u), __builtin_amdgcn_perm(0u, b4[0], 0x03020302u), __builtin_amdgcn_perm(0u, b4[1], 0x01000100u), __builtin_amdgcn_perm(0u, b4[1], 0x03020302u)};
        }
        if (G32 || lane < 32u) {
            float* const to = sbl + (G32 ? (lane >> 5) * 256u : 0u) + lrow;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                // (a run's last block of four steps may end before it: what follows belongs to other weights)
                const uint32_t step = it + (G32 ? 2u * (lane >> 5) + (uint32_t)i / 4u : (uint32_t)i / 2u);
                const uint32_t live = (uint32_t)((int32_t)(step - cnt) >> 31);
                const float sv = kr_elem<DT>(sraw[i / 2] & live, i % 2), bv = kr_elem<DT>(braw[i / 2] & live, i % 2);
                to[i * 32] = sv;
                to[i * 32 + L::SG * 32] = fmaf(-MAGIC, sv, bv);
            }
        }
    };
    // activations: 16 elements of a row, in pairs (i, i + 8)
    constexpr int XP = 2;   // steps ahead of those in LDS
    kr_u32x4 xring[XP][XU][2];
    uint32_t xoff[XU], xrow[XU];
    const uint32_t pl = kwl + 3u;   // log2 of the pieces of a row
#pragma unroll
    for (int u = 0; u < XU; u++) {
        const uint32_t v = tid + u * threads;
        xrow[u] = v >> pl;
        const uint32_t c = v & ((8u << kwl) - 1u);   // pieces 8 i .. 8 i + 7 are K-wave i's step
        xoff[u] = xrow[u] < M ? (xrow[u] * K + (first + (c >> 3) * iters) * 128u + (c & 7u) * 16u) * 2u : KR_OOB;
    }
    const uint32_t xc = tid & ((8u << kwl) - 1u);   // (a thread's pieces are the same one of every row: the threads are a multiple of 8 KW)
    auto load_x = [&](kr_u32x4 (&xv)[XU][2], uint32_t it) {
        const uint32_t dead = ((all - 1u - (xc >> 3) * iters - it) | (iters - 1u - it)) & KR_OOB;
#pragma unroll
        for (int u = 0; u < XU; u++) {
            const uint32_t o = (xoff[u] + it * 256u) | dead;
            xv[u][0] = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)o, 0, 0);
            xv[u][1] = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)(o + 16u), 0, 0);
        }
    };
    auto store_x = [&](const kr_u32x4 (&xv)[XU][2], uint32_t it) {
        constexpr uint32_t ONE = DT == DT_BF16 ? 0x3F803F80u : 0x3C003C00u;
        const uint32_t ckw = xc >> 3, hb = (xc >> 2) & 1u, c = xc & 3u;
        unsigned char* const to = lds + ((((((it >> sgl) & 1u) << kwl) + ckw) << sgl) + (it & SGM)) * XB + hb * (8u * QS);
        float* const sums = (float*)(xs0 + (((it & 7u) << kwl) + ckw) * XSB);
#pragma unroll
        for (int u = 0; u < XU; u++) {
            const kr_u32x4 t = xv[u][0], v = xv[u][1];
            const kr_u32x4 o0 = {__builtin_amdgcn_perm(v.x, t.x, 0x05040100u), __builtin_amdgcn_perm(v.x, t.x, 0x07060302u),
                                 __builtin_amdgcn_perm(v.y, t.y, 0x05040100u), __builtin_amdgcn_perm(v.y, t.y, 0x07060302u)};
            const kr_u32x4 o1 = {__builtin_amdgcn_perm(v.z, t.z, 0x05040100u), __builtin_amdgcn_perm(v.z, t.z, 0x07060302u),
                                 __builtin_amdgcn_perm(v.w, t.w, 0x05040100u), __builtin_amdgcn_perm(v.w, t.w, 0x07060302u)};
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) s = dot2_acc<DT>(v[i], ONE, dot2_acc<DT>(t[i], ONE, s));
            s = seg_allreduce(s, G32 ? 2 : 4);
            if (xrow[u] < ROWS) {
                // groups of 32: an operand holds one group, the pairs of its two pieces in lanes (0, 2) and (1, 3)
                *(kr_u32x4*)(to + (G32 ? ((c >> 1) * 4u + (c & 1u)) : c) * QS + xrow[u] * 16u) = o0;
                *(kr_u32x4*)(to + (G32 ? ((c >> 1) * 4u + (c & 1u) + 2u) : 4u + c) * QS + xrow[u] * 16u) = o1;
                if ((c & (G32 ? 1u : 3u)) == 0u) sums[(G32 ? (hb * 2u + (c >> 1)) : hb) * ROWS + xrow[u]] = s;
            }
        }
    };
    auto barrier = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    kr_f32x4 tot[R][MT];
    const kr_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int t = 0; t < MT; t++) tot[r][t] = zero;

    uint32_t kor = C::KOR;
    asm volatile("" : "+v"(kor));

    load_s(0);
    // the first stage of activations, ahead of the weights (vector loads complete in order)
    kr_u32x4 xfirst[QcShape<MT>::STAGE][XU][2];
#pragma unroll
    for (uint32_t i = 0; i < QcShape<MT>::STAGE; i++) load_x(xfirst[i], i <= SGM ? i : iters);
    load_w(0);
#pragma unroll
    for (int i = 0; i < XP; i++) load_x(xring[i], SGM + 1u + (uint32_t)i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t i = 0; i < QcShape<MT>::STAGE; i++)
        if (i <= SGM) store_x(xfirst[i], i);
    barrier();

    const uint32_t odd = (BITS == 3 || BITS == 5) ? (q & 1u) * 2u : 0u;
    const uint32_t tread = j * L::TS + ((q * (2u * BITS)) & ~3u);
    const uint32_t xread = q * QS + j * 16u;

    auto step = [&](uint32_t it, auto p_c) {
        constexpr int p = decltype(p_c)::value;
        // what was loaded two steps ago goes to LDS, and its registers take the next
        if constexpr (p == 0) store_s(it);
        if constexpr (p % 2 == 0) {
            if (it < iters) {   // (the same in every wave of the workgroup)
#pragma unroll
                for (int l = 0; l < NL; l++) *(kr_u32x4*)(turn + wput[l]) = ring[l];
            }
            if constexpr (p == 0) load_s(it + 4u);
            load_w(it + 2u);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (it >= iters) return;
        kr_turned();
        const unsigned char* const xb = lds + ((((((it >> sgl) & 1u) << kwl) + kw) << sgl) + (it & SGM)) * XB + xread;
        uint32_t d[2][R][4];
        float sv[2][R][G32 ? 2 : 1];
#pragma unroll
        for (int hb = 0; hb < 2; hb++)
#pragma unroll
            for (int r = 0; r < R; r++) {
                qc_read<BITS>(turn + tread + r * 16u * L::TS + (p % 2 * 2 + hb) * 8 * BITS, odd, d[hb][r]);
#pragma unroll
                for (int g = 0; g < (G32 ? 2 : 1); g++) sv[hb][r][g] = sbl[(G32 ? p * 4 + hb * 2 + g : p * 2 + hb) * 32 + 16 * r + j];
            }
#pragma unroll
        for (int hb = 0; hb < 2; hb++) {
            kr_u32x4 wo[R][2];
#pragma unroll
            for (int r = 0; r < R; r++) {
                qc_convert<DT, BITS, false>(d[hb][r], kor, wo[r]);
                if constexpr (G32) {
                    // operand u of lanes 0..3: the pairs of pieces 2 u, 2 u + 1 (first halves), then their second halves
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const auto t = __builtin_amdgcn_permlane32_swap(wo[r][0][i], wo[r][1][i], false, false);
                        wo[r][0][i] = t[0];
                        wo[r][1][i] = t[1];
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const kr_u32x4 x0 = *(const kr_u32x4*)(xb + (hb * 2) * 4 * QS + t * 256), x1 = *(const kr_u32x4*)(xb + (hb * 2 + 1) * 4 * QS + t * 256);
#pragma unroll
                for (int r = 0; r < R; r++) {
                    if constexpr (G32) {
                        const kr_f32x4 p0 = kr_mfma<DT>(x0, wo[r][0], zero), p1 = kr_mfma<DT>(x1, wo[r][1], zero);
#pragma unroll
                        for (int i = 0; i < 4; i++) tot[r][t][i] = fmaf(sv[hb][r][1], p1[i], fmaf(sv[hb][r][0], p0[i], tot[r][t][i]));
                    } else {
                        const kr_f32x4 s = kr_mfma<DT>(x1, wo[r][1], kr_mfma<DT>(x0, wo[r][0], zero));
#pragma unroll
                        for (int i = 0; i < 4; i++) tot[r][t][i] = fmaf(sv[hb][r][0], s[i], tot[r][t][i]);
                    }
                }
            }
        }
        if constexpr (p % U == U - 1) {   // (iters is even)
            constexpr uint32_t back = U - 1;   // the four sums of groups of 64 codes and more begin with the step before
            const unsigned char* const sums = xs0 + (((((it - back) & 7u) + (G32 ? 0u : (q >> 1))) << kwl) + kw) * XSB + (G32 ? q : (q & 1u)) * (ROWS * 4u) + j * 4u;
            float bp[R];
#pragma unroll
            for (int r = 0; r < R; r++) bp[r] = sbl[(L::SG + (G32 ? p * 4 : (p - (int)back) * 2) + q) * 32u + 16 * r + j];
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const float xa = *(const float*)(sums + t * 64);
#pragma unroll
                for (int r = 0; r < R; r++) tot[r][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa, bp[r], tot[r][t], 0, 0, 0);
            }
        }
        store_x(xring[p % XP], it + SGM + 1u);
        __builtin_amdgcn_sched_barrier(0);
        load_x(xring[p % XP], it + SGM + 1u + (uint32_t)XP);
        if ((it & SGM) == SGM) barrier();
    };
    for (uint32_t it0 = 0; it0 < iters; it0 += 4u) kr_for<0, 4>([&](auto p) { step(it0 + (uint32_t)decltype(p)::value, p); });
    barrier();

    // With an infinite activation, or one that the offset or the codes carry past the f32 range, the two halves of the
    // formula are infinities of either sign and their sum no number. Such sums are worked out again with the weights
    // themselves as operands, rounded to the element type as in the tile kernels.
#pragma unroll
    for (int r = 0; r < R; r++) {
        bool bad = false;
#pragma unroll
        for (int t = 0; t < MT; t++) bad = bad || !(__builtin_isfinite(tot[r][t][0]) && __builtin_isfinite(tot[r][t][1]) && __builtin_isfinite(tot[r][t][2]) && __builtin_isfinite(tot[r][t][3]));
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(bad) == 0, 1)) continue;
        kr_f32x4 plain[MT];
#pragma unroll
        for (int t = 0; t < MT; t++) plain[t] = zero;
#pragma unroll 1
        for (uint32_t c = 0; c < iters * 4u; c++) {
            if ((c >> 2) >= cnt) break;
            const uint32_t k = (mine + (c >> 2)) * 128u + (c & 3u) * 32u + 8u * q, bit = k * BITS, n = 16u * r + j;
            const uint32_t wo = n * wrow + (bit >> 5) * 4u, so = (n * gpr + (k >> a.log2g)) * 2u;   // rows past the last: zeros
            uint64_t v = __builtin_amdgcn_raw_buffer_load_b32(wr, (int)wo, 0, 0) | ((uint64_t)__builtin_amdgcn_raw_buffer_load_b32(wr, (int)wo + 4, 0, 0) << 32);
            const uint32_t sh = bit & 31u;
            if (sh) v = (v >> sh) | ((uint64_t)__builtin_amdgcn_raw_buffer_load_b32(wr, (int)wo + 8, 0, 0) << (64u - sh));
            const float sv = kr_elem<DT>((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(sr, (int)so, 0, 0), 0), bv = kr_elem<DT>((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(br, (int)so, 0, 0), 0);
            kr_u32x4 o;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t c0 = (uint32_t)(v >> (2 * i * BITS)) & ((1u << BITS) - 1u), c1 = (uint32_t)(v >> ((2 * i + 1) * BITS)) & ((1u << BITS) - 1u);
                o[i] = f32_to_elem_bits<DT>(fmaf(sv, (float)c0, bv)) | ((uint32_t)f32_to_elem_bits<DT>(fmaf(sv, (float)c1, bv)) << 16);
            }
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const uint32_t m = 16u * t + j;
                plain[t] = kr_mfma<DT>(__builtin_amdgcn_raw_buffer_load_b128(xr, (int)(((m * K + k) * 2u) | ((M - 1u - m) & KR_OOB)), 0, 0), o, plain[t]);
            }
        }
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) tot[r][t][i] = __builtin_isfinite(tot[r][t][i]) ? tot[r][t][i] : plain[t][i];
    }

    // Result i of lane (j, q) is activation row 16 t + 4 q + i, weight row 16 r + j. The sums of the waves that share weight rows
    // meet in LDS, over what the steps are done with.
    uint16_t* const out = ka->out[mat] + (size_t)m0 * N;
    float* const part = ka->part[mat] + ((size_t)slice * a.M + m0) * N;
    float* const red = (float*)lds;   // [wave][r][t][i][lane]
    constexpr uint32_t WS = R * MT * 256;
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) red[wave * WS + ((r * MT + t) * 4 + i) * 64 + lane] = tot[r][t][i];
    barrier();
    // neighbouring threads on neighbouring columns
    const uint32_t live = min(N - tile0, tile_rows), row_l = tid / tile_rows, row_n = threads / tile_rows, col = tid - row_l * tile_rows;
    if (row_l >= row_n || col >= live) return;
    const uint32_t at = ((col >> 5) << kwl) * WS + ((col >> 4) & 1u) * (MT * 256u) + (col & 15u);
    for (uint32_t m = row_l; m < M; m += row_n) {
        const float* const from = red + at + (m >> 4) * 256u + (m & 3u) * 64u + ((m >> 2) & 3u) * 16u;
        float s = from[0];
        for (uint32_t o = 1; o < KW; o++) s += from[o * WS];
        if (slices > 1u) part[(size_t)m * N + tile0 + col] = s;
        else out[(size_t)m * N + tile0 + col] = f32_to_elem_bits<DT>(s);
    }
}

}  // namespace mtq
