// What a launch of the tile kernels (qmm_direct.hip) is: their argument block, and one matrix's kernel and geometry.
#pragma once
#include "mtq_internal.h"
#include "routed_deal.h"

namespace mtq {

constexpr uint32_t QD_ROUTED_ROWS = 160;   // the tall row tiles of expert-routed rows
constexpr uint32_t QD_RUN = 4;   // row tiles of an expert that go through its column tiles together

struct QmmDBase {
    const unsigned char* w;
    const unsigned char* scales;
    const unsigned char* biases;
    const unsigned char* x;
    void* out;
    uint32_t M, N, K;
    uint32_t log2g, gpr;
    uint32_t m_tiles, n_tiles, iters;
    uint32_t m_tile_rows;  // 32 (4 K-groups only), 64, 128 or 256; 160 for expert-routed rows (at most)
    uint32_t by_m;         // consecutive workgroup ids walk the N-tiles of one M-tile (else the M-tiles of one N-tile)
    // grouped mode (expert-routed rows): tiles[0 .. 3] = number of row tiles of each height class, then a table of m_tiles slots for
    // each class (one class and table but for the tall tiles) with one uint4 per tile
    // (expert, first row of the tile in the row order, rows in the tile, its place in its run of at most QD_RUN row tiles of the
    // expert | the run's length << 16); rowlist maps the row order to rows of x / out (null: identity). w / scales / biases
    // are the stacked experts'.
    const uint32_t* tiles;
    const uint32_t* rowlist;
    uint64_t w_expert_bytes, sb_expert_elems;
    // split K (few tiles, long rows): workgroup (x, y) works iterations [y * iters_per_split, +iters_per_split)
    // of tile x and writes its f32 partial tile to part[y][M][N]; a second kernel adds the splits in order.
    uint32_t ksplit, iters_per_split;
    float* part;
};

// Further matrices of the same launch (the projections of a layer against the same rows): their workgroups (blockIdx.x)
// follow the first matrix's, on the same tiling, rows, K and K split.
struct QmmDMore {
    uint32_t n = 0;                                       // 0..3
    uint32_t first[3] = {~0u, ~0u, ~0u};                  // first workgroup of each
    uint32_t N[3] = {}, n_tiles[3] = {}, by_m[3] = {};
    const unsigned char *w[3] = {}, *scales[3] = {}, *biases[3] = {};
    void* out[3] = {};
    float* part[3] = {};
};
struct QmmDArgs : QmmDBase {
    QmmDMore more;
};

// One matrix's call, planned: the kernel that the tiling picks, its geometry, and whether partial tiles follow.
struct QmmDLaunch {
    const void* fn = nullptr;
    int dtype = 0;
    uint32_t grid = 0, block = 0;   // workgroups per K split
    uint32_t cus = 256;             // compute units of the device
    size_t shmem = 0;
    bool split = false;
    bool dma = false;               // activations by load-to-LDS instructions
    size_t scratch = 0;             // bytes of f32 partial tiles (0 when K is not split), a multiple of 256
    QmmDArgs a;
};
// f16 / bf16 activations, any row count, any code width. ERR_UNSUPPORTED where the kernels do not take the shape.
int plan_qmm_direct(const QmmParams& p, QmmDLaunch& l);
// Launches up to four planned matrices against the same rows: those whose tilings come to the same kernel share a launch.
// scratch: the sum of their scratch bytes (null when that is 0). The order of `l` may change.
int launch_qmm_direct(QmmDLaunch* l, int n, void* scratch, const LaunchCtx& lc);

}  // namespace mtq
