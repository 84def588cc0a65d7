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

// Blocks in flight: as many as the registers of sixteen waves hold beside the activations.
template <int DT, int BITS, int G> static const void* runs_pick_steps(uint32_t xs) {
    if constexpr (BITS == 4)
        return xs <= 1 ? (const void*)qmv_runs_kernel<DT, 4, G, 1, 3> : xs == 2 ? (const void*)qmv_runs_kernel<DT, 4, G, 2, 2> :
               xs == 3 ? (const void*)qmv_runs_kernel<DT, 4, G, 3, 1> : (const void*)qmv_runs_kernel<DT, 4, G, 4, 1>;
    else
        return xs <= 2 ? (const void*)qmv_runs_kernel<DT, 8, G, 2, 2> : xs <= 4 ? (const void*)qmv_runs_kernel<DT, 8, G, 4, 1> : (const void*)qmv_runs_kernel<DT, 8, G, 5, 1>;
}
template <int DT, int BITS> static const void* runs_pick_g(uint32_t G, uint32_t xs) {
    return G == 32 ? runs_pick_steps<DT, BITS, 32>(xs) : G == 64 ? runs_pick_steps<DT, BITS, 64>(xs) : runs_pick_steps<DT, BITS, 128>(xs);
}
static const void* runs_pick(int dtype, int bits, uint32_t G, uint32_t xs) {
    if (dtype == DT_BF16) return bits == 4 ? runs_pick_g<DT_BF16, 4>(G, xs) : runs_pick_g<DT_BF16, 8>(G, xs);
    return bits == 4 ? runs_pick_g<DT_F16, 4>(G, xs) : runs_pick_g<DT_F16, 8>(G, xs);
}

bool qmv_runs_takes(const QmvParams& p, const QmvBatch& b) {
    if (b.n < 1 || b.n > 4) return false;
    for (int j = 0; j < b.n; j++)
        if (!runs_shape(p.dtype, p.bits, p.group_size, p.M, b.N[j], p.K) || !runs_aligned(b.w[j], b.scales[j], b.biases[j], p.x)) return false;
    return true;
}

// Where the kernel stands against the others, us, bf16 / f16, weights from memory (others -> this; a single matrix, and the
// projections that a layer has in one call):
//                              4 rows         8 rows         16 rows               8-bit codes: 4 rows, 8 rows, 16 rows
//   1024 x 4096               8.4 ->  6.8    9.1 ->  7.7    9.3 ->  8.7          8.3 ->  8.1   9.7 ->  8.9  10.0 -> 10.2
//   4096 x 4096               6.5 ->  7.2    8.6 ->  7.8   10.5 ->  9.0          7.9 ->  9.2   9.3 ->  9.4  11.5 -> 10.6
//   5120 x 5120               9.6 -> 11.1   12.3 -> 11.9   11.7 -> 13.8         10.6 -> 14.5  17.0 -> 15.5  14.7 -> 17.6
//   14336 x 4096             10.2 -> 13.7   13.3 -> 14.3   13.8 -> 15.7         15.2 -> 18.7  18.6 -> 19.4  18.4 -> 20.8
//   128256 x 4096              55 -> 65       55 -> 66       57 -> 68             91 -> 116    105 -> 121    128 -> 126
//   4096 + 2 x 1024 x 4096   23.6 -> 10.0   26.2 -> 10.7   28.5 -> 11.7         24.4 -> 12.2  28.7 -> 12.7  32.4 -> 14.1
//   3 x 5120 x 5120          27.2 -> 16.7   36.4 -> 17.6   34.4 -> 19.2         31.5 -> 24.4  50.5 -> 25.5  43.4 -> 27.7
//   2 x 14336 x 4096         19.8 -> 18.9   25.7 -> 19.6   27.2 -> 21.0         30.0 -> 30.4  36.8 -> 31.5  36.2 -> 33.1
// A matrix's route cannot depend on whether it comes in a batch (it would not have the same bits), so the line lies where
// a layer gains: from 5 rows up to 75 M codes (60 M of 8 bits), where a long matrix alone loses 1 - 2 us to the 16-row
// kernel and the tiles and a batch of them gains 6 and more; below 5 rows, where those kernels keep up on all but the
// shortest matrices (the K and V projections of grouped-query attention), up to 4.5 M.
bool qmv_runs_preferred(int bits, uint32_t M, uint32_t N, uint32_t K) {
    if (M < 2 || M > 16) return false;
    const uint64_t codes = (uint64_t)N * K;
    return codes <= (M < 5 ? 4500000ull : bits == 4 ? 75000000ull : 60000000ull);
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
    const uint32_t cus = runs_cus(), wgs = a.blocks < cus ? a.blocks : cus;
    const void* fn = runs_pick(p.dtype, p.bits, p.group_size, runs_steps(p.bits, p.K));
    void* args[] = {&a};
    hipError_t e = launch_kernel(fn, dim3(wgs), dim3(1024), args, 0, lc);
    if (e != hipSuccess) return hip_fail(e, "K-run qmv kernel launch");
    return ERR_OK;
}

}  // namespace mtq
