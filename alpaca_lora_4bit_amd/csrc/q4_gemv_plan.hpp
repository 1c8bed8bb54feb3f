// Split of the weight-streaming product of 1..16 rows (gemv_stream_kernel).  Host arithmetic on the sizes alone, without HIP, so
// that it also compiles by itself for the CPU tests.
#pragma once
#include <stddef.h>

namespace q4 {

// LDS bytes of the block sums that `nb` blocks of a share leave behind: four wavefronts, M rows of 64 columns in fp32.
inline size_t stream_slab_bytes(int M, int nb) { return (size_t)nb * 4 * M * 64 * 4; }

// Blocks of 8 chunks of 128 reduction rows per workgroup of gemv_stream_kernel.  One block each (as many workgroups as it takes, 4
// wavefronts of two chunks), or about one workgroup per compute unit with a longer share, which pays its finish once and sends one
// atomic per output instead of one per block, but starts slower: it wins from some rows on, and only where the workgroups
// fill the chip.  us, one block / longer share: 216 strips, K = 5120 (84 % filled) 11.0 / 10.9 at 4 rows, 11.8 / 11.2 at 6,
// 15.2 / 12.7 at 16; 64 strips, K = 11008 (all) 8.0 / 8.2 at 4 rows, 9.0 / 8.6 at 8, 10.4 / 9.7 at 16; 192 strips, K = 4096 (75 %)
// 8.9 / 9.2 at 8 rows, 10.7 / 10.0 at 16; 144 strips, K = 3072 (56 %) 8.7 / 8.7 at 16.  Shares of two blocks and groups of 64
// or 32 rows do not gain.
inline int plan_stream_blocks(int M, int blocks, int strips, int groupsize) {
    const int least = blocks > 255 ? (blocks + 254) / 255 : 1;    // the 8-bit arrival counter
    if (strips > 256 || groupsize % 128 != 0 || M < 5) return least;
    const int S = 256 / strips < blocks ? 256 / strips : blocks;
    const int share = (blocks + S - 1) / S;
    const int fill = 100 * strips * ((blocks + share - 1) / share) / 256;
    if (share < 3 || share < least || stream_slab_bytes(M, share) > 128 * 1024) return least;
    return fill >= 80 || (fill >= 66 && M >= 11) ? share : least;
}

}  // namespace q4
