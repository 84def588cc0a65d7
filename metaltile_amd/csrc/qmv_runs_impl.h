// The K-run matrix-core GEMV (see qmv_runs.hip for the routing and the geometry): kernel and argument block.
#pragma once
// Batches of a few activation rows (up to 16) against one or several weight matrices of the same row length, f16 / bf16,
// with exact-dequant arithmetic: out[m][n] = sum_g (s[n][g] * sum_k q[n][k] x[m][k] + b[n][g] * sum_k x[m][k]), the
// rows of mt_qmm (crates/metaltile-std/src/mlx/quantized.rs:1330-1500) and of the batched projections
// (crates/metaltile-std/src/ffai/batched_qkv_qmm.rs:49-68, batched_4_qmm.rs:61-85).
//
// What bounds such a batch is the stream of weights; what kept the other kernels from it on matrices of 5 - 60 MB were
// the parts around the stream: a launch per matrix, activations staged in LDS by every workgroup before its first
// product, or f32 partial tiles of a split K and a second launch that adds them. Here one launch takes all matrices, and
// its workgroups (one per compute unit) walk their blocks of 16 weight rows. The waves of a workgroup (KP: sixteen, or eight) share a
// block, each with a run of K / KP codes of every row, whose activations it reads once, turns into the operand layout of the
// 16x16x32 MFMA and keeps in registers: from then on the only loads are weights, scales and biases, PF blocks ahead.
// (Vector loads complete in order: activations read along the way, even from the L2, make a wave wait for all weights
// asked for before them. The same kernel with activations read per block streamed at half the rate.) The KP sums of
// a result meet in LDS. The split of K depends on K and the code width: a matrix gives the same bits in whatever batch of matrices.
//
// A step is 128 codes of a row (64 of 8-bit codes), 64 bytes, two neighbouring ones of which are loaded together where rows are dealt in pairs; of a step lane (j, q) = (lane % 16, lane / 16) multiplies the
// 16 bytes of row j at 16 q: 32 codes (16). What bounded the kernel was finding the lines: with neighbouring lanes in sixteen different rows
// a load of 1 KB occupies the compute unit's address path four times as long as with four neighbours in one row, about 64 clk
// against 16, and that was all of a block's 5000 clk at 16 rows (64 weight and scale loads of it). So four neighbours load a row's
// step, and the pieces are turned in LDS (one write and one read of 16 bytes, conflict-free). 16 rows, us, groups of 128, before ->
// after, with the activations first and turned alike: 3 x 5120 x 5120 17.2 -> 13.5, 5120 x 5120 12.4 -> 8.9, 2 x 13824 x 5120 24.2 -> 21.0. An MFMA has to stay inside one group of codes, so for groups shorter than a step the four lanes
// of a row exchange dwords (v_permlane32_swap, and v_permlane16_swap for groups of 32 4-bit codes), and the activations
// are put in the order that leaves, once. The sums of the activations over each group, which
// the bias and the offset of the code conversion are multiplied by, come from one more MFMA per activation operand,
// against ones: its result has the layout of the products and needs no cross-lane step.
// Every load is a buffer load whose out-of-range offsets read zeros without a memory access: rows past the matrix or
// the batch, steps past a wave's run and blocks past the last one are given such offsets, so that every wave issues the
// same loads in the same order.
#include "mfma16.h"
#include "mtq_internal.h"

namespace mtq {

struct QmvRunsArgs {
    const unsigned char* w[4];
    const unsigned char* scales[4];
    const unsigned char* biases[4];
    uint16_t* out[4];
    uint32_t N[4];
    uint32_t block0[4];      // first block of 16 weight rows of each matrix; 0x7FFFFFFF past the last one
    uint32_t blocks;         // of all matrices
    const unsigned char* x;
    uint32_t M, K;
    uint32_t slices;         // of K, for the sliced kernel: workgroup i works on slice i % slices
    float* part[4];          // and its f32 sums [slice][M][N]
};

// An instance and the threads of its workgroups (qmv_runs_pick.h).
struct RunsInstance {
    const void* fn;
    uint32_t threads;
};

// What a code width fixes: the codes a lane loads per step, the MFMAs of a step, the dwords an MFMA's 8 codes per lane
// come in, and the offset its conversion adds to every code.
template <int DT, int BITS> struct KrCodes {
    static constexpr int LANE = 128 / BITS;       // codes in a lane's 16 bytes
    static constexpr int STEP = 4 * LANE;
    static constexpr int UNITS = STEP / 32;
    static constexpr int DPU = BITS / 4;          // dwords per unit
    static constexpr float MAGIC = BITS == 4 ? (DT == DT_BF16 ? 128.0f : 1024.0f) : (DT == DT_BF16 ? 0.0f : 1024.0f);
};

// 8 codes -> an MFMA operand of (MAGIC + code). 4-bit pairs come out as codes (0, 4), (1, 5), (2, 6), (3, 7).
template <int DT, int BITS> __device__ __forceinline__ kr_u32x4 kr_convert(const uint32_t* d, uint32_t kor) {
    if constexpr (BITS == 4) {
        const uint32_t m = 0x000F000Fu, v = d[0];
        return kr_u32x4{(v & m) | kor, ((v >> 4) & m) | kor, ((v >> 8) & m) | kor, ((v >> 12) & m) | kor};
    } else if constexpr (DT == DT_F16) {
        // bytes (code, 0x64, code, 0x64)
        return kr_u32x4{__builtin_amdgcn_perm(kor, d[0], 0x04010400u), __builtin_amdgcn_perm(kor, d[0], 0x04030402u),
                        __builtin_amdgcn_perm(kor, d[1], 0x04010400u), __builtin_amdgcn_perm(kor, d[1], 0x04030402u)};
    } else {
        // integers up to 255 are exact in bf16: the upper halves of their f32 forms
        kr_u32x4 o;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t v = d[i / 2] >> (16 * (i % 2));
            const uint32_t f0 = __float_as_uint((float)(v & 0xFFu)), f1 = __float_as_uint((float)((v >> 8) & 0xFFu));
            o[i] = __builtin_amdgcn_perm(f1, f0, 0x07060302u);
        }
        return o;
    }
}

// 8 codes -> an MFMA operand of weights scale * code + bias, rounded to the element type, in kr_convert's order.
template <int DT, int BITS> __device__ __forceinline__ kr_u32x4 kr_weights(const uint32_t* d, float sv, float bv) {
    kr_u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t a = BITS == 4 ? (d[0] >> (4 * i)) & 15u : (d[BITS == 4 ? 0 : i / 2] >> (16 * (i % 2))) & 255u;
        const uint32_t b = BITS == 4 ? (d[0] >> (4 * i + 16)) & 15u : (d[BITS == 4 ? 0 : i / 2] >> (16 * (i % 2) + 8)) & 255u;
        o[i] = f32_to_elem_bits<DT>(fmaf(sv, (float)a, bv)) | ((uint32_t)f32_to_elem_bits<DT>(fmaf(sv, (float)b, bv)) << 16);
    }
    return o;
}

// PAIRED: a row is a whole number of 128 bytes. DT, BITS (4 or 8), G (32, 64, 128), XS: steps of a wave at most, PF: blocks whose
// weights are in flight ahead of the one that is worked on.
template <bool PAIRED, int KP, bool SLICED, bool ORDERED, int DT, int BITS, int G, int XS, int PF> __device__ __forceinline__ void qmv_runs_body(const QmvRunsArgs& a) {
    static_assert(PAIRED || BITS == 4, "rows of 8-bit codes are whole lines");
    using C = KrCodes<DT, BITS>;
    constexpr int EG = G < C::STEP ? G : C::STEP;   // codes per scale within a step
    constexpr int GPS = C::STEP / EG;               // scales per step: 1, 2 or 4
    constexpr int UPG = EG / 32;                    // MFMAs per scale
    constexpr bool SWAP32 = EG * 2 <= C::STEP, SWAP16 = EG * 4 <= C::STEP;
    constexpr int SDW = GPS == 4 ? 2 : 1;           // dwords of scales per step and row
    constexpr int SR = (XS + 3) / 4;                // scale registers: lanes (j, q) hold steps q, q + 4 of row j
    constexpr bool HOLD = XS * GPS <= (KP == 16 ? 4 : 5);   // the activations' sums stay in registers
    constexpr bool SUMS = !HOLD && KP != 16;                // or in LDS
    constexpr int PAIRS = PAIRED ? XS / 2 : 0;              // pairs of steps of a wave; of an odd number the last step stands alone
    constexpr int SLOTS = C::UNITS;                         // KB of LDS in which a wave turns two steps' weights, or a step's activations
    static_assert(SLOTS >= 2, "a pair of steps is 2 KB");
    __shared__ float red[2][KP * 256];
    __shared__ kr_u32x4 turned[KP * SLOTS * 64];
    __shared__ __attribute__((aligned(16))) float sums[SUMS ? KP * XS * GPS * 16 : 4];

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t kp = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t j = lane & 15u, q = lane >> 4;
    const uint32_t K = a.K, wrow_bytes = K / 8u * BITS, gpr = K / (uint32_t)G;

    // this wave's run of steps
    const uint32_t all_steps = K / (uint32_t)C::STEP;
    uint32_t first_step = 0, steps = all_steps, slice = 0, wg = blockIdx.x, wgs = gridDim.x;
    if constexpr (SLICED) {
        // (the grid is a whole number of workgroups per slice)
        wg = blockIdx.x / a.slices;
        slice = blockIdx.x - wg * a.slices;
        wgs = gridDim.x / a.slices;
        const uint32_t unit = PAIRED ? 2u : 1u;   // (of paired rows a whole number of pairs)
        first_step = all_steps / unit * slice / a.slices * unit;
        steps = all_steps / unit * (slice + 1u) / a.slices * unit - first_step;
    }
    // Of the slice's steps, wave kp has the pairs kp, kp + KP, ... and, of what lies behind PAIRS * KP pairs, the kp-th step: two
    // neighbouring steps are the 128 bytes of a line, and the same loads streamed 58 MB at 4.4 TB/s in pieces of 64 bytes of
    // a row, at 5.8 in pieces of 128 (figures and lines: runs_paired). Where rows are an odd number of steps a pair of every second row
    // lies in two lines, and a run of steps a wave is the faster (4736 x 4736 9.6 against 10.1). steps <= XS * KP (host).
    const uint32_t run0 = steps * kp / KP, run = steps * (kp + 1u) / KP - run0;
    auto step_of = [&](uint32_t n) { return !PAIRED ? run0 + n : n < 2u * PAIRS ? 2u * (kp + KP * (n >> 1)) + (n & 1u) : 2u * (uint32_t)(KP * PAIRS) + kp; };
    auto has_step = [&](uint32_t n) { return PAIRED ? n < (uint32_t)XS && step_of(n) < steps : n < run; };

    // What a lane loads: slot ls of row lr, of the four 16-byte pieces that a step has of a row; the pieces of a row are dealt to
    // its slots so that the sixteen rows' reads from LDS do not meet in a bank.
    const uint32_t lr = lane >> 2, ls = lane & 3u, lpiece = (ls ^ (lr >> 1)) & 3u;
    const uint32_t my_row = j * 4u, my_turn = (j >> 1) & 3u;   // (row j, piece p) lies in slot my_row + (p ^ my_turn)
    kr_u32x4* const swap_lds = turned + kp * (uint32_t)(SLOTS * 64);

    // Weights of a pair: load 0 has rows 0 .. 7, load 1 rows 8 .. 15, slot lane % 8 of row lane / 8 of the eight pieces; these too
    // are dealt to the slots so that the reads do not meet in a bank. Of a step alone: as the activations.
    const uint32_t pr = lane >> 3, ppiece = (lane ^ pr) & 7u;
    const uint32_t plane = pr * wrow_bytes + (first_step + 2u * kp) * 64u + ppiece * 16u, wlane = lr * wrow_bytes + (first_step + (PAIRED ? kp : run0)) * 64u + lpiece * 16u;
    uint32_t pair_dead[PAIRS ? PAIRS : 1];   // this lane's piece lies past the slice
#pragma unroll
    for (int n = 0; n < PAIRS; n++) pair_dead[n] = (steps - 1u - step_of(2 * n) - (ppiece >> 2)) & KR_OOB;
    const uint32_t pair_row = (j >> 3) * 64u + (j & 7u) * 8u, pair_turn = j & 7u;   // (row j, piece p) lies in slot pair_row + (p ^ pair_turn)
    uint32_t slane[SR];
#pragma unroll
    for (int i = 0; i < SR; i++) {
        const uint32_t n = ls + 4u * i, at = first_step + step_of(n);
        slane[i] = has_step(n) ? lr * gpr * 2u + (G > C::STEP ? at / (uint32_t)(G / EG) : at * GPS) * 2u : KR_OOB;
    }
    uint32_t step_dead[XS];   // steps past the slice
#pragma unroll
    for (int n = 0; n < XS; n++) step_dead[n] = (PAIRED ? steps - 1u - step_of(n) : run - 1u - (uint32_t)n) & KR_OOB;

    // The matrix of a block, by sums of masked differences on the scalar unit. (Selections among the arguments become an
    // indexed read of a copy of them in scratch memory, with a wait for every load in flight.)
    const uint32_t n_blocks = a.blocks;
    auto pick = [&](const auto* f, uint32_t blk) {
        uint64_t v = (uint64_t)f[0];
#pragma unroll
        for (int i = 1; i < 4; i++) {
            const int64_t in = (int32_t)(a.block0[i] - 1u - blk) >> 31;   // all ones from the matrix's first block on
            v += ((uint64_t)f[i] - (uint64_t)f[i - 1]) & (uint64_t)in;
        }
        return v;
    };

    struct Block {   // a block's weights, scales and biases in flight
        kr_u32x4 w[XS];
        uint32_t s[SR][SDW], b[SR][SDW];
    };
    auto load_block = [&](Block& d, uint32_t blk) {
        // (Everything but the lane's own part is worked out on the scalar unit. The offsets are put out of range with the sign of
        // a difference: from a selection the optimiser makes a branch around the loads, and waits there for all in flight.)
        const uint32_t at_blk = min(blk, n_blocks - 1u), N = (uint32_t)pick(a.N, at_blk), first = (uint32_t)pick(a.block0, at_blk);
        const uint32_t row0 = (at_blk - first) * 16u, rows = blk < n_blocks ? N - row0 : 0u;   // (16 or more: a whole block)
        const __amdgpu_buffer_rsrc_t wr = kr_rsrc(pick(a.w, at_blk), N * wrow_bytes), sr = kr_rsrc(pick(a.scales, at_blk), N * gpr * 2u),
                                     br = kr_rsrc(pick(a.biases, at_blk), N * gpr * 2u);
        const uint32_t dead = (rows - 1u - lr) & KR_OOB;
        const uint32_t w0 = row0 * wrow_bytes, s0 = row0 * gpr * 2u, wo = (wlane + w0) | dead;
#pragma unroll
        for (int i = 0; i < SR; i++) {
            const uint32_t o = (slane[i] + s0) | dead;
            if constexpr (GPS == 1) {
                d.s[i][0] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(sr, (int)o, 0, 0);
                d.b[i][0] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(br, (int)o, 0, 0);
            } else if constexpr (GPS == 2) {
                d.s[i][0] = __builtin_amdgcn_raw_buffer_load_b32(sr, (int)o, 0, 0);
                d.b[i][0] = __builtin_amdgcn_raw_buffer_load_b32(br, (int)o, 0, 0);
            } else {
                const kr_u32x2 sv = __builtin_amdgcn_raw_buffer_load_b64(sr, (int)o, 0, 0), bv = __builtin_amdgcn_raw_buffer_load_b64(br, (int)o, 0, 0);
                d.s[i][0] = sv.x; d.s[i][1] = sv.y; d.b[i][0] = bv.x; d.b[i][1] = bv.y;
            }
        }
#pragma unroll
        for (int n = 0; n < PAIRS; n++)
#pragma unroll
            for (uint32_t h = 0; h < 2; h++)
                d.w[2 * n + h] = __builtin_amdgcn_raw_buffer_load_b128(wr, (int)((plane + w0 + 8u * h * wrow_bytes + 128u * KP * n) | pair_dead[n] | ((rows - 1u - pr - 8u * h) & KR_OOB)), 0, KR_NT);
#pragma unroll
        for (int n = 2 * PAIRS; n < XS; n++) d.w[n] = __builtin_amdgcn_raw_buffer_load_b128(wr, (int)((wo + 64u * (PAIRED ? 2 * KP * PAIRS : n)) | step_dead[n]), 0, KR_NT);
    };

    Block ring[PF + 1];

    // ---- the activations of the run, ahead of the first weights (loads complete in order, over the whole compute unit: behind
    // weights from memory they came late, 5120 x 5120 in groups of 128, 16 rows 11.6 us, so 10.1). They are turned in LDS: four neighbouring lanes read 64
    // contiguous bytes (read straight into the operand layout, 16 rows next to each other, a load of 1 KB took four times as long
    // to find its lines: 12.4 us, so 10.9), and unit u of lane (j, q) takes the piece of 8 codes that its weights will be.
    kr_u32x4 xop[XS][C::UNITS];
    {
        const __amdgpu_buffer_rsrc_t xr = kr_rsrc((uint64_t)a.x, a.M * K * 2u);
        const uint32_t xo = ((lr * K + (first_step + (PAIRED ? 0u : run0)) * (uint32_t)C::STEP + lpiece * 8u) * 2u) | ((a.M - 1u - lr) & KR_OOB);
#pragma unroll
        for (int n = 0; n < XS; n++)
#pragma unroll
            for (int k = 0; k < C::UNITS; k++) xop[n][k] = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)((xo + (PAIRED ? step_of(n) : (uint32_t)n) * (uint32_t)(C::STEP * 2) + (uint32_t)(k * 64)) | step_dead[n]), 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        // No wave's weights ahead of another's activations. Not where a run is short, as the wait for the last of the waves to start
        // costs more there (us, with -> without): 8 bits, 5 rows 4096 x 2048 6.5 -> 5.9; 4 bits 11008 x 2048 7.8 -> 7.4, groups of 32
        // 1024 x 2048 5.9 -> 5.4; two steps, 3584 x 3584, 5 rows 7.1 -> 6.8, but 11008 x 4096, 16 rows 11.4 -> 11.9.
        if constexpr (ORDERED) __builtin_amdgcn_s_barrier();
        kr_for<0, PF>([&](auto p) { load_block(ring[decltype(p)::value], wg + wgs * (uint32_t)decltype(p)::value); });
        __builtin_amdgcn_sched_barrier(0);
        uint32_t from[C::UNITS];
#pragma unroll
        for (uint32_t u = 0; u < C::UNITS; u++) {
            const uint32_t p = BITS == 4 ? (SWAP16 ? 4u * u + q : SWAP32 ? (u >> 1) * 8u + (u & 1u) + (q & 1u) * 4u + (q >> 1) * 2u : 4u * q + u)
                                         : (SWAP32 ? 4u * u + (q & 1u) * 2u + (q >> 1) : 2u * q + u);
            from[u] = p / 4u * 64u + my_row + ((p ^ my_turn) & 3u);
        }
#pragma unroll
        for (int n = 0; n < XS; n++) {
#pragma unroll
            for (int k = 0; k < C::UNITS; k++) swap_lds[k * 64 + lane] = xop[n][k];
            kr_turned();
#pragma unroll
            for (int u = 0; u < C::UNITS; u++) {
                const kr_u32x4 t = swap_lds[from[u]];
                if constexpr (BITS == 4)   // in the order the nibble masks deliver the codes
                    xop[n][u] = kr_u32x4{__builtin_amdgcn_perm(t.z, t.x, 0x05040100u), __builtin_amdgcn_perm(t.z, t.x, 0x07060302u),
                                         __builtin_amdgcn_perm(t.w, t.y, 0x05040100u), __builtin_amdgcn_perm(t.w, t.y, 0x07060302u)};
                else xop[n][u] = t;
            }
            kr_turned();
        }
    }
    const uint32_t kor = BITS == 8 ? 0x64646464u : magic_or_vgpr<DT>();
    constexpr uint32_t ONE = DT == DT_BF16 ? 0x3F803F80u : 0x3C003C00u;
    const kr_u32x4 ones = {ONE, ONE, ONE, ONE};
    const kr_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    auto x_sum = [&](int n, int g) {
        kr_f32x4 s = zero;
#pragma unroll
        for (int u = 0; u < UPG; u++) s = kr_mfma<DT>(xop[n][g * UPG + u], ones, s);
        return s;
    };
    kr_f32x4 held[HOLD ? XS : 1][HOLD ? GPS : 1];
    if constexpr (HOLD) {
#pragma unroll
        for (int n = 0; n < XS; n++)
#pragma unroll
            for (int g = 0; g < GPS; g++) held[n][g] = x_sum(n, g);
    }
    if constexpr (SUMS) {
        // [step][group][activation row], a wave's own: every column of the product is the same
#pragma unroll
        for (int n = 0; n < XS; n++)
#pragma unroll
            for (int g = 0; g < GPS; g++) {
                const kr_f32x4 s = x_sum(n, g);
                if (j == 0) *(kr_f32x4*)&sums[((kp * XS + n) * GPS + g) * 16 + 4 * q] = s;
            }
        kr_turned();
    }
    __builtin_amdgcn_sched_barrier(0);

    // a step's dwords with every MFMA inside one group of codes
    auto codes_of = [&](const kr_u32x4& w, uint32_t (&v)[4]) {
        v[0] = w.x; v[1] = w.y; v[2] = w.z; v[3] = w.w;
        if constexpr (SWAP32) {
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const auto t = __builtin_amdgcn_permlane32_swap(v[k], v[k + 2], false, false);
                v[k] = t[0];
                v[k + 2] = t[1];
            }
        }
        if constexpr (SWAP16) {
#pragma unroll
            for (int k = 0; k < 4; k += 2) {
                const auto t = __builtin_amdgcn_permlane16_swap(v[k], v[k + 1], false, false);
                v[k] = t[0];
                v[k + 1] = t[1];
            }
        }
    };
    uint32_t par = 0;
    uint32_t blk = wg;
    auto turn = [&](auto p_c) {
        constexpr int p = decltype(p_c)::value;
        load_block(ring[(p + PF) % (PF + 1)], blk + wgs * (uint32_t)PF);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t now = blk;
        blk += wgs;
        if (now >= n_blocks) return;   // (the same in every wave of the workgroup)
        Block& d = ring[p];
        kr_f32x4 tot = zero;
        kr_for<0, XS>([&](auto n_c) {
            constexpr int n = decltype(n_c)::value;
            uint32_t v[4];
            if constexpr (n < 2 * PAIRS) {
                constexpr int at = n / 2 * 2 % SLOTS * 64;
                if constexpr (n % 2 == 0) {
                    swap_lds[at + lane] = d.w[n];
                    swap_lds[at + 64 + lane] = d.w[n + 1];
                    kr_turned();
                }
                codes_of(swap_lds[at + pair_row + ((q + 4u * (n % 2)) ^ pair_turn)], v);
            } else {
                swap_lds[n % SLOTS * 64 + lane] = d.w[n];
                kr_turned();
                codes_of(swap_lds[n % SLOTS * 64 + my_row + (q ^ my_turn)], v);
            }
            const int src = (int)((my_row + (n % 4)) * 4u);   // the lane that holds this step's scales of row j
            kr_for<0, GPS>([&](auto g_c) {
                constexpr int g = decltype(g_c)::value;
                kr_f32x4 acc = zero;
#pragma unroll
                for (int u = g * UPG; u < (g + 1) * UPG; u++) acc = kr_mfma<DT>(xop[n][u], kr_convert<DT, BITS>(&v[u * C::DPU], kor), acc);
                const uint32_t sp = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)d.s[n / 4][g / 2]);
                const uint32_t bp = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)d.b[n / 4][g / 2]);
                const float sv = kr_elem<DT>(sp, g % 2), bv = kr_elem<DT>(bp, g % 2);
                const float bm = C::MAGIC == 0.f ? bv : fmaf(-C::MAGIC, sv, bv);
                kr_f32x4 xs;
                if constexpr (HOLD) xs = held[n][g];
                else if constexpr (SUMS) xs = *(const kr_f32x4*)&sums[((kp * XS + n) * GPS + g) * 16 + 4 * q];
                else xs = x_sum(n, g);
#pragma unroll
                for (int r = 0; r < 4; r++) tot[r] = fmaf(bm, xs[r], fmaf(sv, acc[r], tot[r]));
            });
        });
        // With an infinite activation, or one that the offset or the codes carry past the f32 range, the two halves of the
        // formula are infinities of either sign and their sum no number. Such sums are worked out again
        // with the weights themselves as operands, rounded to the element type as in the tile kernels.
        // (What the look at the sums costs: 13824 x 5120, 16 rows 19.0 -> 19.3 us, 4096 x 4096 8.9 -> 9.0.)
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(__builtin_isfinite(tot[0]) && __builtin_isfinite(tot[1]) && __builtin_isfinite(tot[2]) && __builtin_isfinite(tot[3]))) != 0, 0)) {
            // (From memory and in a rolled loop: the copies of the turn stay short. In the registers' order and unrolled the
            // code was three times as long.)
            kr_f32x4 plain = zero;
            const uint32_t at_blk = now, N = (uint32_t)pick(a.N, at_blk), row0 = (at_blk - (uint32_t)pick(a.block0, at_blk)) * 16u;
            const __amdgpu_buffer_rsrc_t wr = kr_rsrc(pick(a.w, at_blk), N * wrow_bytes), sr = kr_rsrc(pick(a.scales, at_blk), N * gpr * 2u),
                                         br = kr_rsrc(pick(a.biases, at_blk), N * gpr * 2u), xr = kr_rsrc((uint64_t)a.x, a.M * K * 2u);
#pragma unroll 1
            for (uint32_t i = 0; i < (uint32_t)(XS * C::UNITS); i++) {
                const uint32_t n = i / C::UNITS;
                if (!has_step(n)) continue;   // (the same in every lane)
                const uint32_t k = (first_step + step_of(n)) * (uint32_t)C::STEP + i % C::UNITS * 32u + 8u * q, wo = (row0 + j) * wrow_bytes + k / 8u * BITS, so = ((row0 + j) * gpr + k / (uint32_t)G) * 2u;   // rows past the last: zeros
                uint32_t d[2] = {};
                d[0] = __builtin_amdgcn_raw_buffer_load_b32(wr, (int)wo, 0, 0);
                if constexpr (BITS == 8) d[1] = __builtin_amdgcn_raw_buffer_load_b32(wr, (int)wo + 4, 0, 0);
                const uint32_t sp = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(sr, (int)so, 0, 0), bp = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(br, (int)so, 0, 0);
                kr_u32x4 xv = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)(((j * K + k) * 2u) | ((a.M - 1u - j) & KR_OOB)), 0, 0);
                if constexpr (BITS == 4)   // in the order of kr_weights
                    xv = kr_u32x4{__builtin_amdgcn_perm(xv.z, xv.x, 0x05040100u), __builtin_amdgcn_perm(xv.z, xv.x, 0x07060302u),
                                  __builtin_amdgcn_perm(xv.w, xv.y, 0x05040100u), __builtin_amdgcn_perm(xv.w, xv.y, 0x07060302u)};
                plain = kr_mfma<DT>(xv, kr_weights<DT, BITS>(d, kr_elem<DT>(sp, 0), kr_elem<DT>(bp, 0)), plain);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) tot[r] = __builtin_isfinite(tot[r]) ? tot[r] : plain[r];
        }
        // The runs meet in LDS: result r of lane (j, q) is activation row 4 q + r, weight row j. The
        // other half of the buffer takes the next block, so one barrier per block is enough.
        float* rd = red[par];
        par ^= 1u;
#pragma unroll
        for (int r = 0; r < 4; r++) rd[(kp * 4u + r) * 64u + lane] = tot[r];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        if (tid < 256u) {
            float s = rd[tid];
#pragma unroll
            for (uint32_t o = 1; o < KP; o++) s += rd[o * 256u + tid];
            __attribute__((address_space(1))) uint16_t* out = (__attribute__((address_space(1))) uint16_t*)pick(a.out, now);
            const uint32_t N = (uint32_t)pick(a.N, now), first = (uint32_t)pick(a.block0, now);
            const uint32_t arow = 4u * q + (tid >> 6), wrow = (now - first) * 16u + j;
            if (arow < a.M && wrow < N) {
                if constexpr (SLICED) {
                    __attribute__((address_space(1))) float* part = (__attribute__((address_space(1))) float*)pick(a.part, now);
                    part[((size_t)slice * a.M + arow) * N + wrow] = s;
                } else {
                    out[(size_t)arow * N + wrow] = f32_to_elem_bits<DT>(s);
                }
            }
        }
    };
    // (The way out lies behind the last turn only. From breaks between the turns the compiler makes one edge back to the loop's
    // head, on which it takes the loads of any turn to be still in flight, and waits at the head for all of them: with one block
    // ahead, none was in flight at every second turn.)
    do kr_for<0, PF + 1>(turn);
    while (blk < n_blocks);
}

// XS: steps of a sixteenth of K at most.
template <bool PAIRED, bool ORDERED, int KP, int DT, int BITS, int G, int XS, int PF> __global__ __launch_bounds__(KP * 64) void qmv_runs_kernel(QmvRunsArgs a) {
    qmv_runs_body<PAIRED, KP, false, ORDERED, DT, BITS, G, XS * 16 / KP, PF>(a);
}
// On one of a.slices slices of K, whose sums a second launch adds; XS: steps of an eighth of a slice at most.
template <bool PAIRED, int DT, int BITS, int G, int XS, int PF> __global__ __launch_bounds__(512) void qmv_slices_kernel(QmvRunsArgs a) {
    qmv_runs_body<PAIRED, 8, true, true, DT, BITS, G, XS, PF>(a);
}

}  // namespace mtq
