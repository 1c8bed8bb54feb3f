// What the tiled GEMM kernels (q4_gemm.hip, q4_gemm_wide.hip) share: their arguments, the order of the tiles, the shares of
// the reduction.
#pragma once
#include "q4_common.hpp"
#include "q4_gemm_plan.hpp"
#include <type_traits>

namespace q4 {

struct GemmArgs {
    const half_t* a;          // fwd: x [M,K]      bwd: dy [M,N]
    const uint32_t* qweight;  // [K/8, N]
    const uint32_t* qzeros;   // [G, N/8]
    const half_t* scales;     // [G, N]
    const int32_t* g_idx;     // [K] or null
    int groupsize;
    uint32_t gs_inv31;        // ceil(2^31 / (groupsize / 64)): reduction offset -> group without a division
    const half_t* bias;       // fwd only, [N] or null
    const half_t* la;         // fwd: xa [M,R]     bwd: dyb [M,R]   (or null)
    const void* lb;           // adapter matrix (fp16 or fp32), element (r, c) at lb[r*lb_sr + c*lb_sc]; fwd: c = n, bwd: c = k
    int lb_sr, lb_sc, lb_is_f32;
    float lb_scale;           // multiplied into the adapter matrix when it is staged in LDS
    int R;
    half_t* out;              // fwd: y [M,N]      bwd: dx [M,K]
    int M, K, N, G;
    int phase_step;           // bits 0-7: rotation of the reduction loop per row tile, in steps of 64; bits 8+: row tiles per group of the tile order
    float* part;              // split-K: fp32 partial outputs [gridDim.z][M][part_cols] (gridDim.z > 1 only)
    int col_tile0;            // first column tile of this launch (a launch may cover a range of column tiles)
    int part_cols;            // columns held by `part`: those of this launch's column tiles
    DropArgs drop;            // thr15 != 0: the adapter term of out[m, c] is kept only where dropout keeps (m, c)
};

// Which output tile a workgroup computes.  Workgroups are handed to the 8 XCDs round-robin in dispatch order.  The ids are
// permuted so that one XCD owns a contiguous range of tiles, ordered in groups of `rg` row tiles: all column tiles of a
// group, then the next group.  The 32 workgroups an XCD runs at a time then share 2 slabs of activations and 16 column
// tiles of W (about 4 MB each at K = 4096, what its L2 holds) instead of every row tile of a few columns: with many row
// tiles the activations would otherwise stream from HBM once per column tile (8192 x 4096 x 4096: 306 -> 260 us; no shape
// slower).
struct TileMap {
    int tile_c, tile_r;
};
__device__ __forceinline__ TileMap map_tile(int phase_step, int col_tile0) {
    const int nc = gridDim.x, nr = gridDim.y, total = nc * nr;
    int id = blockIdx.y * nc + blockIdx.x;
    if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
    TileMap m;
    const int rg = phase_step >> 8;                   // row tiles per group (0: column-major over all row tiles)
    const int grouped = rg > 0 ? (nr / rg) * rg * nc : 0;
    if (id < grouped) {
        // groups of rg row tiles: all column tiles of a group, then the next group
        const int gi = id / (rg * nc), rem = id - gi * rg * nc;
        m.tile_c = rem / rg;
        m.tile_r = gi * rg + (rem - m.tile_c * rg);
    } else {
        const int left = rg > 0 ? nr % rg : nr, base = nr - left, rem = id - grouped;
        m.tile_c = rem / left;
        m.tile_r = base + (rem - m.tile_c * left);
    }
    m.tile_c += col_tile0;
    return m;
}
// Split-K: gridDim.z workgroups share an output tile; workgroup z owns `cnt` consecutive steps from `begin`.
struct StepRange {
    int begin, cnt;
};
__device__ __forceinline__ StepRange split_steps(int nsteps, int z, int S) {
    const int base = nsteps / S, rem = nsteps - base * S;
    StepRange r;
    r.cnt = base + (z < rem ? 1 : 0);
    r.begin = z * base + min(z, rem);
    return r;
}
// reduction offset of pipeline stage `stage` (stages past the end repeat the last one: harmless reloads)
__device__ __forceinline__ int red_of(int stage, StepRange sr, int phase) {
    int v = min(stage, sr.cnt - 1) + phase;
    if (v >= sr.cnt) v -= sr.cnt;
    return (sr.begin + v) * BK;
}

// Group of reduction row k (a multiple of 64; sequential groups of a multiple of 64 rows):
// floor((k/64) / (groupsize/64)) as a multiply-high, exact while k * groupsize < 2^40.
__device__ __forceinline__ int group_of(const GemmArgs& a, int k) {
    return (int)__umulhi((uint32_t)k >> 5, a.gs_inv31);
}

__device__ __forceinline__ float adapter_at(const GemmArgs& a, size_t idx) {
    return a.lb_is_f32 ? reinterpret_cast<const float*>(a.lb)[idx] : (float)reinterpret_cast<const half_t*>(a.lb)[idx];
}

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// Up to kGemmGroup layers that share M, K, the group size and (forward) the activations -- q|k|v, gate|up -- in ONE
// grid, each on its own tensors.
//   forward:    blockIdx.x walks the column tiles of layer 0, then of layer 1, ...; every workgroup computes one tile of
//               one layer's own output, over the whole reduction (no split).
//   grad-input: dx = sum_i dy_i @ W_i^T is ONE reduction over the layers' columns one after the other: a workgroup
//               walks the layers (all of them, or its share of the concatenated steps where the tiles are few) with
//               the sum in its accumulators, adapter term and dropout mask of each layer included.
struct GemmGroupArgs {
    GemmArgs layer[kGemmGroup];
    int tile_end[kGemmGroup];          // forward: running total of column tiles (tile width of the launch)
    int n;
};

// q4_gemm_wide.hip: grids of 256 x 256 tiles, or of 128 x 256 ones (`low`, forward only)
void launch_wide_tiles(bool fwd, bool low, const GemmArgs& a, dim3 grid, hipStream_t stream);
void launch_wide_group_tiles(bool fwd, bool low, const GemmGroupArgs& g, dim3 grid, hipStream_t stream);

}  // namespace q4
