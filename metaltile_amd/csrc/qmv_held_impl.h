// The matrix-core GEMV with its activations held in LDS (see qmv_held.hip for the routing and the geometry).
#pragma once
// A few activation rows (as many as fit the LDS: a normalised one of up to 18944 codes, 28672 at 2 bits; 16 of up to 4096) against one or several
// weight matrices of the same row length: f16 / bf16, codes of 2, 3, 4, 5, 6 and 8 bits, rows of any whole number of 128
// codes, groups of 32, 64 and 128, the row optionally RMS-normalised or gated and normalised per head first. Exact-dequant
// arithmetic: out[m][n] = sum_g (s[n][g] * sum_k q[n][k] x[m][k] + b[n][g] * sum_k x[m][k]), the rows of mt_qmv and mt_qmm
// (crates/metaltile-std/src/mlx/quantized.rs:1330-1500) and of the norm-fused projections
// (crates/metaltile-std/src/ffai/gated_rms_norm_qgemv.rs:88-291).
//
// The codes themselves are the operands of the 16x16x32 MFMA, as MAGIC + code in the element type (exact), and the scale is
// applied to the sum of a group: an FMA per result row and group in place of a conversion of every weight. The bias
// term, sum_g (b - MAGIC s)[n][g] * xsum[g][m], is a product of its own with a 64th of the terms: it runs on the f32 matrix
// instruction, four groups at a time.
//
// What bounds such a call on the small and middle matrices of a layer is what lies around the stream of weights: launches,
// the preparation of the row, round trips that wait for each other. So one launch takes all matrices and the norm;
// the first weights are asked for before the row is prepared; every wave then streams on its own, with no barrier but the
// one at which the KP waves that share 16 weight rows add their sums. The stream goes on across a wave's blocks.
// A normalised row is carried as its rounded value and rounded remainder, two operand rows of the same MFMA. Weights are loaded two
// steps of 128 codes at a time, neighbouring lanes on neighbouring 16 bytes of a row (in pieces of 64 bytes of a row a read of 58 MB
// takes 13.4 us, in pieces of 128 bytes 10.0; this kernel at 28672 x 4096, 4 bits, norm included, 26.0 -> 20.3), and turned in an LDS area
// of the wave's own whose rows are 16 bytes apart from a multiple of 32 so that the operand reads spread over the banks.
// Scales are read 16 bytes of a row at a time and kept as f32 (as 2-byte loads of the values of each step they kept the
// address path busier than the weights).
#include "codes16.h"
#include "mtq_internal.h"

namespace mtq {

struct QmvHeldArgs {
    const unsigned char* w[4];
    const unsigned char* scales[4];
    const unsigned char* biases[4];
    uint16_t* out[4];
    uint32_t N[4];
    uint32_t first[4];       // first block of 16 weight rows of each matrix; 0x7FFFFFFF past the last one
    uint32_t blocks;         // of all matrices
    uint32_t M, K;
    const unsigned char* x;  // f32 [K] for the gated norm
    const unsigned char* norm_w;
    const unsigned char* gate;
    const float* eps;
    uint32_t dv;             // gated norm: elements per head
    uint32_t log2g, log2kp, log2rp, waves;   // rp: rows in LDS, a power of two
};

enum HeldMode : int { HELD_PLAIN = 0, HELD_NORM = 1, HELD_GATED = 2 };

template <int BITS, bool G32> struct QhLds {
    static constexpr uint32_t TS = 32 * BITS + 16;    // a weight row's two steps of 128 codes
    static constexpr uint32_t TB = 16 * TS;
    static constexpr uint32_t SG = G32 ? 16 : 8;      // scales of four steps: [group or 64 codes][weight row], then biases less MAGIC scales
    static constexpr uint32_t WB = TB + 2 * SG * 64;  // a wave's own part
    static_assert(WB % 16 == 0, "16-byte LDS accesses");
    // rows and their sums; the waves' parts behind them begin on 16 bytes (one row in groups of 64: 264 bytes per 128 codes)
    static constexpr uint32_t xbytes(uint32_t K, uint32_t rpl) { return (((K * 2u + K / (G32 ? 32u : 64u) * 4u) << rpl) + 15u) & ~15u; }
    static constexpr uint32_t bytes(uint32_t K, uint32_t rpl, uint32_t waves) { return xbytes(K, rpl) + waves * WB + ((2u * waves * 64u) << rpl) + 64u; }
};

// DT, BITS, groups of 32 (else 64 or 128), NR: result registers that hold rows (1: one row, 2: value and remainder, 4), MODE
template <int DT, int BITS, bool G32, int NR, int MODE> __global__ __launch_bounds__(1024) void qmv_held_kernel(QmvHeldArgs a) {
    using L = QhLds<BITS, G32>;
    constexpr int NL = (BITS + 1) / 2;                  // 16-byte loads of two steps: 32 * BITS pieces
    // (one row of f16 4- and 8-bit codes came from the streaming and one-shot kernels)
    constexpr bool LEAST = NR == 1 && DT == DT_F16 && (BITS == 4 || BITS == 8);
    using C = QcCodes<DT, BITS, LEAST>;
    constexpr float MAGIC = C::MAGIC;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t j = lane & 15u, q = lane >> 4;
    const uint32_t kpl = a.log2kp, KP = 1u << kpl, kp = wave & (KP - 1u), NB = a.waves >> kpl, threads = a.waves * 64u;
    const uint32_t K = a.K, wrow = K / 8u * BITS, gpr = K >> a.log2g, rpl = a.log2rp, RPM = (1u << rpl) - 1u;
    const uint32_t steps = K / 128u, iters = (((steps + 1u) / 2u + KP - 1u) >> kpl) * 2u, my = kp * iters, cnt = steps > my ? min(steps - my, iters) : 0u;

    unsigned char* const xl = lds;
    float* const sums = (float*)(lds + ((K * 2u) << rpl));
    unsigned char* const own = lds + L::xbytes(K, rpl) + wave * L::WB;
    float* const sbl = (float*)(own + L::TB);
    float* const red = (float*)(lds + L::xbytes(K, rpl) + a.waves * L::WB);
    auto barrier = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    // ---- the stream: turns of four steps, a block's last ones possibly empty
    const uint32_t n_blocks = a.blocks, stride = gridDim.x * NB;
    // (the arguments of a block's matrix are read from the argument segment by its number)
    const __attribute__((address_space(4))) QmvHeldArgs* const ka = (const __attribute__((address_space(4))) QmvHeldArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    auto matrix_of = [&](uint32_t blk) { return (blk >= a.first[1] ? 1u : 0u) + (blk >= a.first[2] ? 1u : 0u) + (blk >= a.first[3] ? 1u : 0u); };
    uint32_t woff[NL], wput[NL], wpast[NL];
#pragma unroll
    for (int l = 0; l < NL; l++) {
        const uint32_t id16 = l * 64u + lane, r = id16 / (2u * BITS), p = id16 - r * (2u * BITS);
        woff[l] = (r * wrow + p * 16u + my * (16u * BITS)) | ((15u - r) & KR_OOB);
        wput[l] = r < 16u ? r * L::TS + p * 16u : 0u;
        wpast[l] = p >= (uint32_t)BITS ? 1u : 0u;   // of the second step
    }
    const bool wide_g = !G32 && a.log2g == 7u;
    const uint32_t s_row = j * gpr + (G32 ? my * 4u : wide_g ? my : my * 2u);   // (lanes 0 .. 15; groups of 32: 16 .. 31 the second half)
    const uint32_t s_dead = ((G32 ? 31u : 15u) - lane) & KR_OOB;
    struct Source { __amdgpu_buffer_rsrc_t w, s, b; };
    auto source = [&](uint32_t blk) {
        const uint32_t at = min(blk, n_blocks - 1u), mat = __builtin_amdgcn_readfirstlane(matrix_of(at)), N = ka->N[mat], row0 = (at - ka->first[mat]) * 16u;
        const uint32_t rows = blk < n_blocks ? min(N - row0, 16u) : 0u;
        // (a dword of scales whose second half lies past the end is read whole)
        return Source{kr_rsrc((uint64_t)ka->w[mat] + (uint64_t)row0 * wrow, rows * wrow), kr_rsrc((uint64_t)ka->scales[mat] + (uint64_t)row0 * gpr * 2u, (rows * gpr * 2u + 3u) & ~3u),
                      kr_rsrc((uint64_t)ka->biases[mat] + (uint64_t)row0 * gpr * 2u, (rows * gpr * 2u + 3u) & ~3u)};
    };
    kr_u32x4 ring[2][NL], sraw, braw;
    auto load_w = [&](const Source& s, uint32_t it, int p) {   // two steps
#pragma unroll
        for (int l = 0; l < NL; l++) ring[p][l] = __builtin_amdgcn_raw_buffer_load_b128(s.w, (int)((woff[l] + it * (16u * BITS)) | ((cnt - 1u - it - wpast[l]) & KR_OOB)), 0, KR_NT);
    };
    // scales and biases of four steps, from the even element at or before the first one (odd for groups of 128 only)
    auto load_s = [&](const Source& s, uint32_t it) {
        const uint32_t dead = ((cnt - 1u - it) & KR_OOB) | s_dead;
        const int o = (int)((((s_row + (G32 ? it * 4u : wide_g ? it : it * 2u)) & ~1u) * 2u + (G32 ? (lane >> 4) * 16u : 0u)) | dead);
        sraw = __builtin_amdgcn_raw_buffer_load_b128(s.s, o, 0, 0);
        braw = __builtin_amdgcn_raw_buffer_load_b128(s.b, o, 0, 0);
    };
    auto store_s = [&](uint32_t it) {
        if (wide_g) {
            const uint32_t by = (s_row & 1u) * 2u;
            uint32_t s4[2], b4[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                s4[i] = __builtin_amdgcn_alignbyte(sraw[i + 1], sraw[i], by);
                b4[i] = __builtin_amdgcn_alignbyte(braw[i + 1], braw[i], by);
            }
            sraw = kr_u32x4{__builtin_amdgcn_perm(0u, s4[0], 0x01000100u), __builtin_amdgcn_perm(0u, s4[0], 0x03020302u), __builtin_amdgcn_perm(0u, s4[1], 0x01000100u), __builtin_amdgcn_perm(0u, s4[1], 0x03020302u)};
            braw = kr_u32x4{__builtin_amdgcn_perm(0u, b4[0], 0x01000100u), __builtin_amdgcn_perm(0u, b4[0], 0x03020302u), __builtin_amdgcn_perm(0u, b4[1], 0x01000100u), __builtin_amdgcn_perm(0u, b4[1], 0x03020302u)};
        }
        if (lane < (G32 ? 32u : 16u)) {
            float* const to = sbl + (G32 ? (lane >> 4) * 128u : 0u) + j;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                // (a run's last four steps may reach past it: what follows belongs to other weights)
                const uint32_t step = it + (G32 ? 2u * (lane >> 4) + (uint32_t)i / 4u : (uint32_t)i / 2u);
                const uint32_t live = (uint32_t)((int32_t)(step - cnt) >> 31);
                const float sv = kr_elem<DT>(sraw[i / 2] & live, i % 2), bv = kr_elem<DT>(braw[i / 2] & live, i % 2);
                to[i * 16] = sv;
                to[i * 16 + L::SG * 16] = fmaf(-MAGIC, sv, bv);
            }
        }
    };

    // ---- the rows, in operand order: 16 elements as pairs (i, i + 8), and the sums over the codes of a scale
    auto put_row = [&](uint32_t m, uint32_t c, const kr_u32x4& t, const kr_u32x4& v) {
        constexpr uint32_t ONE = DT == DT_BF16 ? 0x3F803F80u : 0x3C003C00u;
        const kr_u32x4 o0 = {__builtin_amdgcn_perm(v.x, t.x, 0x05040100u), __builtin_amdgcn_perm(v.x, t.x, 0x07060302u),
                             __builtin_amdgcn_perm(v.y, t.y, 0x05040100u), __builtin_amdgcn_perm(v.y, t.y, 0x07060302u)};
        const kr_u32x4 o1 = {__builtin_amdgcn_perm(v.z, t.z, 0x05040100u), __builtin_amdgcn_perm(v.z, t.z, 0x07060302u),
                             __builtin_amdgcn_perm(v.w, t.w, 0x05040100u), __builtin_amdgcn_perm(v.w, t.w, 0x07060302u)};
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) s = dot2_acc<DT>(v[i], ONE, dot2_acc<DT>(t[i], ONE, s));
        s = seg_allreduce(s, G32 ? 2 : 4);
        const uint32_t kb = c >> 2, cq = c & 3u, p0 = kb * 8u + (G32 ? (cq >> 1) * 4u + (cq & 1u) : cq), p1 = p0 + (G32 ? 2u : 4u);
        *(kr_u32x4*)(xl + ((p0 << rpl) | m) * 16u) = o0;
        *(kr_u32x4*)(xl + ((p1 << rpl) | m) * 16u) = o1;
        if ((cq & (G32 ? 1u : 3u)) == 0u) sums[((G32 ? kb * 2u + (cq >> 1) : kb) << rpl) | m] = s;
    };
    const uint32_t upr = K / 16u;
    uint32_t blk = blockIdx.x * NB + (wave >> kpl);
    Source next = source(blk);
    auto first_weights = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        load_s(next, 0);
        kr_for<0, 2>([&](auto p) { load_w(next, 2u * (uint32_t)decltype(p)::value, decltype(p)::value); });
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (MODE == HELD_PLAIN) {
        const uint32_t units = a.M * upr;
        const __amdgpu_buffer_rsrc_t xr = kr_rsrc((uint64_t)a.x, units * 32u);
        kr_u32x4 xv[2][2];
        auto load = [&](uint32_t u0) {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int h = 0; h < 2; h++) xv[i][h] = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)((u0 + i * threads + tid) * 32u + h * 16u), 0, 0);
        };
        auto put = [&](uint32_t u0) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t u = u0 + i * threads + tid;
                if (u < units) {
                    const uint32_t m = NR == 1 ? 0u : u / upr;
                    put_row(m, u - m * upr, xv[i][0], xv[i][1]);
                }
            }
        };
        load(0);
        first_weights();
        put(0);
        for (uint32_t u0 = 2u * threads; u0 < units; u0 += 2u * threads) {
            load(u0);
            put(u0);
        }
    } else {
        // one row, at most two units a thread
        constexpr int XL = MODE == HELD_GATED ? 4 : 2;
        const __amdgpu_buffer_rsrc_t xr = kr_rsrc((uint64_t)a.x, K * (MODE == HELD_GATED ? 4u : 2u)), nr = kr_rsrc((uint64_t)a.norm_w, (MODE == HELD_GATED ? a.dv : K) * 2u);
        kr_u32x4 xv[2][XL], nv[2][2], zv[2][2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t u = i * threads + tid;
#pragma unroll
            for (int h = 0; h < XL; h++) xv[i][h] = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)(u * (16u * XL) + h * 16u), 0, 0);
            if constexpr (MODE == HELD_GATED) {
                const __amdgpu_buffer_rsrc_t zr = kr_rsrc((uint64_t)a.gate, K * 2u);
#pragma unroll
                for (int h = 0; h < 2; h++) zv[i][h] = __builtin_amdgcn_raw_buffer_load_b128(zr, (int)(u * 32u + h * 16u), 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t u = i * threads + tid, at = MODE == HELD_GATED ? (u * 16u) & (a.dv - 1u) : u * 16u;   // (dv: a power of two)
#pragma unroll
            for (int h = 0; h < 2; h++) nv[i][h] = __builtin_amdgcn_raw_buffer_load_b128(nr, (int)(at * 2u + h * 16u), 0, 0);
        }
        const float eps = a.eps[0];
        first_weights();
        auto up = [](uint32_t d, int odd) { return kr_elem<DT>(d, odd); };
        if constexpr (MODE == HELD_NORM) {
            float ssq = 0.f;
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int h = 0; h < 2; h++) ssq += raw_sumsq<DT>(__builtin_bit_cast(uint4, xv[i][h]));   // (past the row: zeros)
            ssq = seg_allreduce(ssq, 64);
            if (lane == 0) red[wave] = ssq;
            barrier();
            float tot = 0.f;
            for (uint32_t i = 0; i < a.waves; i++) tot += red[i];
            const float inv = 1.0f / sqrtf(tot / (float)K + eps);
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t u = i * threads + tid;
                if (u < upr) {
                    uint4 hi[2], lo[2];
#pragma unroll
                    for (int h = 0; h < 2; h++) raw_normed<DT>(__builtin_bit_cast(uint4, xv[i][h]), __builtin_bit_cast(uint4, nv[i][h]), inv, hi[h], lo[h]);
                    put_row(0, u, __builtin_bit_cast(kr_u32x4, hi[0]), __builtin_bit_cast(kr_u32x4, hi[1]));
                    put_row(1, u, __builtin_bit_cast(kr_u32x4, lo[0]), __builtin_bit_cast(kr_u32x4, lo[1]));
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                float ssq = 0.f;
#pragma unroll
                for (int h = 0; h < 4; h++) ssq += raw_sumsq<DT_F32>(__builtin_bit_cast(uint4, xv[i][h]));
                ssq = seg_allreduce(ssq, (int)(a.dv / 16u));   // (a head's lanes are neighbours: host)
                const float inv = 1.0f / sqrtf(ssq / (float)a.dv + eps);
                const uint32_t u = i * threads + tid;
                if (u < upr) {
                    kr_u32x4 hi[2], lo[2];
#pragma unroll
                    for (int e = 0; e < 16; e += 2) {
                        uint32_t h2[2], l2[2];
#pragma unroll
                        for (int o = 0; o < 2; o++) {
                            const float z = up(zv[i][e / 8][e % 8 / 2], o), gate = z / (1.0f + expf(0.0f - z));
                            const float v = __uint_as_float(xv[i][e / 4][e % 4 + o]) * inv * up(nv[i][e / 8][e % 8 / 2], o) * gate;
                            RemSplit<DT>::split(v, h2[o], l2[o]);
                        }
                        hi[e / 8][e % 8 / 2] = h2[0] | (h2[1] << 16);
                        lo[e / 8][e % 8 / 2] = l2[0] | (l2[1] << 16);
                    }
                    put_row(0, u, hi[0], hi[1]);
                    put_row(1, u, lo[0], lo[1]);
                }
            }
        }
    }
    barrier();

    uint32_t kor = C::KOR;
    asm volatile("" : "+v"(kor));
    const uint32_t odd = (BITS == 3 || BITS == 5) ? (q & 1u) * 2u : 0u;
    const uint32_t tread = j * L::TS + ((q * (2u * BITS)) & ~3u);
    const unsigned char* const xread = xl + (((my * 16u + q) << rpl) | (j & RPM)) * 16u;
    const float* const sread = sums + (((my * (G32 ? 4u : 2u) + q) << rpl) | (j & RPM));
    const kr_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    kr_f32x4 tot = zero;
    uint32_t par = 0;

    auto operands = [&](int hb, kr_u32x4 (&wo)[2]) {   // hb: half of 64 codes of the two steps
        uint32_t d[4];
        qc_read<BITS>(own + tread + hb * 8 * BITS, odd, d);
        qc_convert<DT, BITS, LEAST>(d, kor, wo);
        if constexpr (G32) {
            // operand u of lanes 0..3: the pairs of pieces 2 u, 2 u + 1 (first halves), then their second halves
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const auto t = __builtin_amdgcn_permlane32_swap(wo[0][i], wo[1][i], false, false);
                wo[0][i] = t[0];
                wo[1][i] = t[1];
            }
        }
    };
    auto put_w = [&](int p) {
#pragma unroll
        for (int l = 0; l < NL; l++)
            if ((l + 1) * 64 <= 32 * BITS || lane < (uint32_t)(32 * BITS - l * 64)) *(kr_u32x4*)(own + wput[l]) = ring[p][l];
    };
    // Two steps' products with the weights themselves as operands, rounded to the element type as in the tile kernels.
    auto steps_plain = [&](const Source& s, uint32_t it, kr_f32x4& plain) {
        load_w(s, it, 0);
        put_w(0);
        kr_turned();
#pragma unroll 1
        for (int hb = 0; hb < 4; hb++) {
            if (it + (uint32_t)hb / 2u >= cnt) break;
            kr_u32x4 wo[2];
            operands(hb, wo);
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const uint32_t g = (((my + it) * 128u + hb * 64u + (G32 ? u * 32u : 0u)) >> a.log2g);
                const float sv = kr_elem<DT>((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(s.s, (int)((j * gpr + g) * 2u), 0, 0), 0);
                const float bv = kr_elem<DT>((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(s.b, (int)((j * gpr + g) * 2u), 0, 0), 0);
#pragma unroll
                for (int i = 0; i < 4; i++)
                    wo[u][i] = f32_to_elem_bits<DT>(fmaf(sv, kr_elem<DT>(wo[u][i], 0) - MAGIC, bv)) | ((uint32_t)f32_to_elem_bits<DT>(fmaf(sv, kr_elem<DT>(wo[u][i], 1) - MAGIC, bv)) << 16);
                plain = kr_mfma<DT>(*(const kr_u32x4*)(xread + (((it * 16u + hb * 8u + u * 4u) << rpl) * 16u)), wo[u], plain);
            }
        }
        kr_turned();
    };

    for (uint32_t base = blockIdx.x * NB; base < n_blocks; base += stride, blk += stride) {
        const bool alive = blk < n_blocks;
        Source now = next;
        next = source(blk + stride);
        for (uint32_t t = 0; t < iters; t += 4u) {   // (the same in every wave of the workgroup)
            const bool last = t + 4u >= iters;
            const uint32_t t_next = last ? 0u : t + 4u;
            Source from = now;
            if (last) from = next;
            kr_for<0, 2>([&](auto p_c) {
                constexpr int p = decltype(p_c)::value;
                const uint32_t it = t + 2u * (uint32_t)p;   // and it + 1
                if constexpr (p == 0) {
                    store_s(t);
                    load_s(from, t_next);
                }
                put_w(p);
                load_w(from, t_next + 2u * (uint32_t)p, p);
                __builtin_amdgcn_sched_barrier(0);
                kr_turned();
                if (!alive || it >= cnt) return;   // (the same in every lane)
                // (a second step past the run: its weights are zeros and so are its scales, the rows behind it finite or not;
                // its products are left out)
                const int halves = it + 1u < cnt ? 4 : 2;
                float sv[4][G32 ? 2 : 1];
                kr_u32x4 xo[4][2];
#pragma unroll
                for (int hb = 0; hb < 4; hb++) {
#pragma unroll
                    for (int g = 0; g < (G32 ? 2 : 1); g++) sv[hb][g] = sbl[(G32 ? p * 8 + hb * 2 + g : p * 4 + hb) * 16 + j];
                }
                auto half = [&](int hb) {
                    kr_u32x4 wo[2];
                    operands(hb, wo);
#pragma unroll
                    for (int u = 0; u < 2; u++) xo[hb][u] = *(const kr_u32x4*)(xread + (((it * 16u + hb * 8u + u * 4u) << rpl) * 16u));
                    if constexpr (G32) {
                        const kr_f32x4 p0 = kr_mfma<DT>(xo[hb][0], wo[0], zero), p1 = kr_mfma<DT>(xo[hb][1], wo[1], zero);
#pragma unroll
                        for (int i = 0; i < NR; i++) tot[i] = fmaf(sv[hb][1], p1[i], fmaf(sv[hb][0], p0[i], tot[i]));
                    } else {
                        const kr_f32x4 s = kr_mfma<DT>(xo[hb][1], wo[1], kr_mfma<DT>(xo[hb][0], wo[0], zero));
#pragma unroll
                        for (int i = 0; i < NR; i++) tot[i] = fmaf(sv[hb][0], s[i], tot[i]);
                    }
                };
                auto bias = [&](int of, bool lone) {   // of: the step's four sums, or both steps'
                    float xa = sread[((it + (uint32_t)of) * (G32 ? 4u : 2u)) << rpl];
                    if (lone) xa = q < 2u ? xa : 0.f;
                    tot = __builtin_amdgcn_mfma_f32_16x16x4f32(xa, sbl[(L::SG + (G32 ? p * 8 + of * 4 : p * 4) + q) * 16u + j], tot, 0, 0, 0);
                };
                if (halves == 4) {
#pragma unroll
                    for (int hb = 0; hb < 4; hb++) half(hb);
                    bias(0, false);
                    if constexpr (G32) bias(1, false);
                } else {
                    half(0);
                    half(1);
                    bias(0, !G32);
                }
            });
        }
        // With an infinite activation, or one that the offset or the codes carry past the f32 range, the two halves of the formula are
        // infinities of either sign and their sum no number: such sums are worked out again. The weights in flight for the next
        // block are asked for once more.
        bool bad = false;
#pragma unroll
        for (int i = 0; i < NR; i++) bad = bad || (4u * q + i < (MODE == HELD_PLAIN ? a.M : 2u) && !__builtin_isfinite(tot[i]));
        if (__builtin_expect(alive && __builtin_amdgcn_ballot_w64(bad) != 0, 0)) {
            kr_f32x4 plain = zero;
#pragma unroll 1
            for (uint32_t it = 0; it < cnt; it += 2u) steps_plain(now, it, plain);
#pragma unroll
            for (int i = 0; i < NR; i++) tot[i] = __builtin_isfinite(tot[i]) ? tot[i] : plain[i];
            load_w(next, 0, 0);
        }
        // result i of lane (j, q) is activation row 4 q + i, weight row j
        if (kpl == 0) {
            if (alive) {
                const uint32_t mat = __builtin_amdgcn_readfirstlane(matrix_of(blk)), N = ka->N[mat], n = (blk - ka->first[mat]) * 16u + j;
                uint16_t* const out = ka->out[mat];
                if constexpr (MODE != HELD_PLAIN) {
                    if (q == 0 && n < N) out[n] = f32_to_elem_bits<DT>(tot[0] + tot[1] * (1.0f / RemSplit<DT>::kRemScale));
                } else {
#pragma unroll
                    for (int i = 0; i < NR; i++)
                        if (4u * q + i < a.M && n < N) out[(size_t)(4u * q + i) * N + n] = f32_to_elem_bits<DT>(tot[i]);
                }
            }
        } else {
            // two buffers: one barrier a block
            float* const rd = red + (((par ? a.waves : 0u) * 16u) << rpl);
            par ^= 1u;
#pragma unroll
            for (int i = 0; i < NR; i++)
                if (4u * q + i <= RPM) rd[(((wave << rpl) + 4u * q + i) << 4) + j] = tot[i];
            barrier();
            const uint32_t rows = MODE == HELD_PLAIN ? a.M : 1u;
            for (uint32_t i = tid; i < (NB << (4u + rpl)); i += threads) {
                const uint32_t b = base + (i >> (4u + rpl)), m = (i >> 4) & RPM, at = min(b, n_blocks - 1u);
                if (m >= rows || b >= n_blocks) continue;
                const uint32_t mat = matrix_of(at);
                const float* const f = rd + ((((i >> (4u + rpl)) << kpl << rpl) + m) << 4) + (i & 15u);
                float s = f[0];
                for (uint32_t o = 1; o < KP; o++) s += f[(o << rpl) << 4];
                if constexpr (MODE != HELD_PLAIN) {
                    float l = f[16];
                    for (uint32_t o = 1; o < KP; o++) l += f[((o << rpl) + 1u) << 4];
                    s += l * (1.0f / RemSplit<DT>::kRemScale);
                }
                const uint32_t N = mat == 0 ? a.N[0] : mat == 1 ? a.N[1] : mat == 2 ? a.N[2] : a.N[3];
                const uint32_t n = (b - (mat == 0 ? a.first[0] : mat == 1 ? a.first[1] : mat == 2 ? a.first[2] : a.first[3])) * 16u + (i & 15u);
                uint16_t* const out = mat == 0 ? a.out[0] : mat == 1 ? a.out[1] : mat == 2 ? a.out[2] : a.out[3];
                if (n < N) out[(size_t)m * N + n] = f32_to_elem_bits<DT>(s);
            }
        }
        tot = zero;
    }
}

}  // namespace mtq
