// Split of the weight-streaming product of 1..16 rows (gemv_stream_kernel).  Host arithmetic on the sizes alone, without HIP, so
// that it also compiles by itself for the CPU tests.
#pragma once
#include <stddef.h>

namespace q4 {

// LDS bytes of the block sums that `nb` blocks of a share leave behind: four wavefronts, M rows of 64 columns in fp32.
inline size_t stream_slab_bytes(int M, int nb) { return (size_t)nb * 4 * M * 64 * 4; }

// Which kernel takes a product of 1..16 rows over chunks of 128 rows with groups of 32, 64 or a multiple of 128: gemv_stream_kernel,
// or the burst of one chunk per wavefront and eight wavefronts (gemv_seq_kernel), with the same bits.  For one row the stream
// gains little (the activations cost the burst little) and its second chunk waits behind the first: the burst wins from two
// workgroups per compute unit on, and up to two rows with more than one group per chunk, whose sums the stream scales for four rows.
// us at one row, burst / stream: 64 strips, K = 4096 (256 workgroups) 4.67 / 4.57; 80, 5120 (400) 5.80 / 5.73; 96, 4096 (384) 6.31 / 6.04;
// 216, 2048 (432) 5.88 / 5.79; 64, 8192 (512) 6.13 / 6.24; 128, 4096 (512) 6.06 / 6.24; 64, 11008 (704) 7.24 / 7.43;
// 80, 13824 (1120) 9.65 / 10.02; 216, 5120 (1080) 9.81 / 10.06; against the rule 128, 2048 (256) 4.72 / 4.79.  Groups of 64 and 32 rows:
// 64 strips, K = 4096 4.82 / 4.96 and 5.17 / 5.83 at one row, 5.01 / 5.04 and 5.47 / 5.90 at two, 5.20 / 5.13 and 5.78 / 5.96 at three;
// 64, 11008 7.50 / 8.10 and 8.72 / 9.73, 7.88 / 8.30 and 9.19 / 9.78, 8.16 / 8.42 and 9.83 / 9.86; 216, 5120 at two 11.24 / 11.23 and 13.5 / 14.3,
// at three 11.60 / 11.43 and 14.4 / 14.4, at four 12.1 / 11.5 and 15.2 / 14.5.
inline bool plan_stream_takes(int M, int blocks, int strips, int groupsize) {
    if (blocks > 255 || M > 2) return true;                       // 255: the burst's 8-bit arrival counter
    return groupsize % 128 == 0 && (M == 2 || (long)strips * blocks < 512);
}

// Blocks of 8 chunks of 128 reduction rows per workgroup of gemv_stream_kernel.  One block each (as many workgroups as it takes, 4
// wavefronts of two chunks), or about one workgroup per compute unit with a longer share, which pays its finish once and sends one
// atomic per output instead of one per block, but starts slower: it wins from some rows on, and only where the workgroups
// fill the chip.  us, one block / longer share, where one workgroup takes the whole reduction: 216 strips, K = 5120 (84 % filled)
// 11.1 / 11.4 at 5 rows, 11.3 / 11.3 at 6, 11.5 / 11.3 at 7, 14.3 / 12.3 at 16; 240 strips 11.7 / 11.8, 12.0 / 11.8, 12.2 / 11.9, 15.3 / 13.1;
// 192 strips, K = 4096 (75 %) 9.0 / 9.0 at 8 rows, 10.1 / 10.4 at 11, 10.3 / 10.4 at 12, 10.9 / 10.5 at 16.  Where several share it:
// 64 strips, K = 11008 8.5 / 8.6 at 8 rows, 9.4 / 9.2 at 10, 9.6 / 9.2 at 11, 10.5 / 9.7 at 16; 80 strips, K = 13824 11.7 / 12.0 at 8, 12.5 / 12.7
// at 10, 12.7 / 12.6 at 11, 14.3 / 12.8 at 16; 128 strips, K = 8192 10.6 / 10.5 at 8, 11.7 / 11.3 at 11, 12.7 / 11.8 at 16.  Shares of two blocks and
// groups of 64 or 32 rows do not gain.  (The longer share's figures are of one team of wavefronts; with two, plan_stream_teams, it is
// 0.2 to 0.5 us shorter.)
inline int plan_stream_blocks(int M, int blocks, int strips, int groupsize) {
    const int least = blocks > 255 ? (blocks + 254) / 255 : 1;    // the 8-bit arrival counter
    if (strips > 256 || groupsize % 128 != 0 || M < 7) return least;
    const int S = 256 / strips < blocks ? 256 / strips : blocks;
    const int share = (blocks + S - 1) / S;
    const int fill = 100 * strips * ((blocks + share - 1) / share) / 256;
    if (share < 3 || share < least || stream_slab_bytes(M, share) > 128 * 1024) return least;
    return (fill >= 80 && (share == blocks || M >= 11)) || (fill >= 66 && M >= 13) ? share : least;
}

// Teams of four wavefronts in a workgroup of gemv_stream_kernel whose share is `nb` blocks, the blocks in turn to the teams: two
// where the sums of the blocks fit the LDS beside the second team's tiles.  Four wavefronts of one chunk ahead keep 16 KB per compute
// unit on the way, too little for the latency of HBM; eight twice that.  us, one team / two: q|k|v of 4096 features 10.21 / 9.97 at
// 16 rows, 11008 -> 4096 9.03 / 8.51 at 12, 9.45 / 8.99 at 16.  (Gate, up and activation in one launch move twice the words per chunk and
// are level with two teams at 16 rows, 0.9 us slower at 4.)
inline int plan_stream_teams(int M, int nb) { return nb >= 2 && stream_slab_bytes(M, nb) <= 96 * 1024 ? 2 : 1; }

}  // namespace q4
