// Tiled GEMMs whose weight operands are built in registers (sequential groups of a multiple of 64 rows):
//   forward   y [M,N] = x  [M,K] @ W      (+ bias) (+ xa  [M,R] @ lora_bt [R,N])
//   backward  dx[M,K] = dy [M,N] @ W^T             (+ dyb [M,R] @ lora_a  [R,K])
// the products of q4_gemm.hip for outputs that have enough large tiles (plan_gemm).
//
// What bounds them.  A full round of 256 x 256 tiles runs into the chip's power limit: products of normally distributed operands
// from registers alone reach 1.64 PFLOP/s at 1.6-1.7 GHz (2.4 PFLOP/s at 2.4 GHz on zeros), with a 128-bit LDS fragment per two
// MFMAs and two packed vector operations per MFMA beside them 1.50.  Speed is then energy per MFMA, not cycles: with parts of the
// loop taken out, the activations' way from L2 into LDS is 11 % of it, the operand build 13 %, the fragment reads 6 %, the
// packed words less than 1 %.
//
// Layout.  A workgroup computes 32*TM x 256 outputs with four wavefronts, one per SIMD, side by side: each has all rows of 64
// columns as TM x 2 accumulators of v_mfma_f32_32x32x16_f16 (256 registers at TM = 8).  No two wavefronts share a column, so
// every weight is decoded once per workgroup and its operand never goes through LDS: forward, a packed word IS the 8-deep
// reduction slice of one column that a lane feeds to the MFMA.  Grad-input, a word holds eight output columns of one reduction
// index; the workgroup turns each 8 x 8 block of codes around in registers (32 byte permutes and masks per thread and step) and
// passes the turned words, still packed, through 8 KB of LDS.  LDS otherwise holds activations only: four tiles of 64 reduction
// entries, written by the loads themselves (buffer_load ... lds) three steps ahead, units of 16 bytes swizzled by the row so
// that the 128-bit fragment reads meet no bank twice.  Per 256 x 256 x 64 step 32 KB are written and 128 KB read, where staging
// both operands (8 wavefronts of 128 x 64) writes 64 KB and reads 192.
//
// Operand build.  17 (forward) or 15 vector operations per word: masks, permutes, one conversion per pair (codes_of_bytes), product
// and difference rounded apart: the weights are the dense kernel's, bit for bit.  A pair's difference comes with the next pair's
// product: directly behind its own it waits for an issue slot (512 x (5120 -> 13824) 73 us instead of 67).  With the codes as
// (1024 + q, 64 + q) and the offset taken off by the product (16 operations) 70.
//
// Order of the sums.  That of q4_gemm.hip: the reduction rotated per 256 rows, adapter terms behind a layer's loop, masked ones in
// front of it, so that a product has the same bits on either file's tiles.
//
// us, 8 wavefronts of 128 x 64 with both operands in LDS -> now, one lease: forward 4096 x (4096 -> 4096) 113.5 -> 105.9,
// 4096 x (5120 -> 13824) 482 -> 454, 4096 x (13824 -> 5120) 482 -> 446; grad-input 113.7 -> 109.3, 487 -> 472, 485 -> 470.
//
// TM = 4, forward: tiles of 128 x 256 for outputs with too few of the large ones (one unsplit round of 256 x 128 tiles of
// q4_gemm.hip before: the same area, half the activations per weight decoded, but 64 KB of fragment reads per round of 1024 MFMA
// cycles instead of 128).  us, 256 x 128 with both operands in LDS -> 128 x 256: 2048 x (4096 -> 4096) 65.2 -> 61.0, 512 x (5120 -> 13824)
// 72.2 -> 67.4, 600 x (5120 -> 5120) 47.4 -> 41.7, 1024 x (11008 -> 4096) 95.0 -> 88.6, 2048 x (4096 -> 11008) 166.5 -> 158.6 (its last
// 88 tiles).  Grad-input the form is level to 2 % slower: the words turned around serve half the rows.
#include "q4_gemm_args.hpp"

namespace q4 {

// 16 bytes per lane from memory to LDS, lane l's at lds + 16 l
__device__ __forceinline__ void load_lds128(rsrc_t r, half_t* lds, int voff, int soff) {
    typedef __attribute__((address_space(3))) void lds_void;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds, 16, voff, soff, 0, 0);
}

constexpr int kStages = 4;               // activation tiles in LDS: one being multiplied, three on their way
constexpr int kWideCols = 256;
constexpr int kFar = 0x70000000;         // beyond every buffer: reads as zero, without traffic

// Of `n` pieces of work spread over `span` places the first that goes to place i or a later one: piece l goes to place
// l * span / n.
constexpr int first_piece(int i, int n, int span) { return i <= 0 ? 0 : i >= span ? n : (i * n + span - 1) / span; }
template <int I, int N, int SPAN, typename F>
__device__ __forceinline__ void pieces_of(F&& f) {
    static_for<first_piece(I, N, SPAN), first_piece(I + 1, N, SPAN)>(f);
}

__device__ __forceinline__ uint32_t bfi(uint32_t mask, uint32_t a, uint32_t b) { return (a & mask) | (b & ~mask); }

// Keeps a block of accumulators in the accumulation registers: what vector operations make of it goes back there at once, instead
// of 256 of them drifting into the registers that the loop needs.
__device__ __forceinline__ void keep_acc(float16_t& a) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+a"(a));
#endif
}

template <int TM, bool FWD, bool MULTI>
__device__ __forceinline__ void wide_body(const GemmArgs* layers, const int nlay, const TileMap tm, const StepRange share,
                                          const int zsplit, const int nsplit) {
    constexpr int BM = 32 * TM, KS = BK / 16, NMK = 2 * TM;       // NMK: MFMAs of a sub-step of 16
    constexpr int kTile = BM * BK;                                // halves of an activation tile
    constexpr int kOther = FWD ? KS + 2 : 4;                      // loads of a step beside its activations
    constexpr int kLoads = TM + kOther;
    __shared__ __attribute__((aligned(16))) half_t sA0[kTile];
    __shared__ __attribute__((aligned(16))) half_t sA1[kTile];
    __shared__ __attribute__((aligned(16))) half_t sA2[kTile];
    __shared__ __attribute__((aligned(16))) half_t sA3[kTile];
    // grad-input: codes of a step, nibbles along the reduction: [octet][column], and (scales, zero terms) of a wavefront's step
    constexpr int kTw = kWideCols + 8;
    __shared__ __attribute__((aligned(16))) uint32_t sT0[FWD ? 4 : 8 * kTw];
    __shared__ __attribute__((aligned(16))) uint32_t sT1[FWD ? 4 : 8 * kTw];
    __shared__ __attribute__((aligned(16))) half_t sZ[FWD ? 1 : 4][2][2][FWD ? 4 : BK];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int lane = threadIdx.x & 63, lc = lane & 31, lg = lane >> 5;
    const GemmArgs& a0 = layers[0];
    const int NOUT = FWD ? a0.N : a0.K;
    const int m0 = tm.tile_r * BM, c0 = tm.tile_c * kWideCols, cw = c0 + 64 * wave;
    const int rows_valid = min(BM, a0.M - m0);

    float bias_v[2] = {0.f, 0.f};
    if (FWD && a0.bias) {
#pragma unroll
        for (int j = 0; j < 2; ++j) bias_v[j] = (float)a0.bias[cw + 2 * lc + j];
    }
    float16_t acc[TM][2];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    auto keep_all = [&] {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) keep_acc(acc[i][j]);
    };
    if constexpr (TM == 8) keep_all();

    // Adapter terms: operands straight from memory, added where q4_gemm.hip adds them.
    auto adapter_row = [&](const GemmArgs& a, int i, int ks) {    // columns past R and rows past M read as zero
        const rsrc_t rl = make_rsrc(a.la + (size_t)m0 * a.R, (unsigned)rows_valid * (unsigned)a.R * 2u);
        return __builtin_bit_cast(half8_t, buf_load128(rl, 16 * ks + 8 * lg < a.R ? ((32 * i + lc) * a.R + 16 * ks + 8 * lg) * 2 : kFar, 0));
    };
    // columns cw + 2 lc, + 1, rows 16 ks + 8 lg .. + 7 of the adapter matrix (rows past R: of row 0), as they lie in memory
    auto adapter_load = [&](const GemmArgs& a, int ks, uint32_t (&raw)[2][8]) {
        const int r0 = 16 * ks + 8 * lg < a.R ? 16 * ks + 8 * lg : 0;
        auto load = [&](auto tag) {
            using T = decltype(tag);
            constexpr int per = 16 / sizeof(T);
            if (FWD && a.lb_sr == 1 && a.lb_sc % per == 0 && reinterpret_cast<uintptr_t>(a.lb) % 16 == 0) {
                // lora_B as it is kept, [N, R]: a lane's rows of a column lie together (one by one its loads touch 64 lines each,
                // 1024 x (4096 -> 4096) at rank 64 takes 51.9 us instead of 47.3)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int h = 0; h < 8 / per; ++h) {
                        const uint4_t u = *reinterpret_cast<const uint4_t*>(reinterpret_cast<const T*>(a.lb) + r0 + per * h + (size_t)(cw + 2 * lc + j) * a.lb_sc);
                        const uint32_t d[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                        for (int e = 0; e < per; ++e) raw[j][per * h + e] = sizeof(T) == 4 ? d[e & 3] : d[(e / 2) & 3] >> (16 * (e & 1));
                    }
                return;
            }
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 8; ++e) raw[j][e] = reinterpret_cast<const T*>(a.lb)[(size_t)(r0 + e) * a.lb_sr + (size_t)(cw + 2 * lc + j) * a.lb_sc];
        };
        if (a.lb_is_f32) load(uint32_t{});
        else load((unsigned short)0);
    };
    // the operand they make (zero past R)
    auto adapter_cols = [&](const GemmArgs& a, int ks, const uint32_t (&raw)[2][8], half8_t (&b)[2]) {
        uint32_t in = 16 * ks + 8 * lg < a.R ? 0xFFFFFFFFu : 0u;
        asm volatile("" : "+v"(in));                              // opaque: one mask instead of a branch around every value
        // fp32 values scaled and rounded to fp16 at once, as q4_gemm.hip's staging of the matrix compiles (left to itself the
        // compiler makes a product and a conversion of pairs: a rounding more)
        auto pair = [&](uint32_t u0, uint32_t u1) -> uint32_t {
            if (a.lb_is_f32) {                                    // uniform
                uint32_t h = 0;
#if defined(__HIP_DEVICE_COMPILE__)
                asm("v_fma_mixlo_f16 %0, %1, %3, 0\n\tv_fma_mixhi_f16 %0, %2, %3, 0" : "=&v"(h) : "v"(u0), "v"(u1), "s"(a.lb_scale));
#endif
                return h;
            }
            return as_u32(half2_t{(half_t)(a.lb_scale * (float)__builtin_bit_cast(half_t, (unsigned short)u0)),
                                  (half_t)(a.lb_scale * (float)__builtin_bit_cast(half_t, (unsigned short)u1))});
        };
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32_t o[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) o[p] = pair(raw[j][2 * p], raw[j][2 * p + 1]) & in;
            b[j] = __builtin_bit_cast(half8_t, uint4_t{o[0], o[1], o[2], o[3]});
        }
    };
    // behind the layer's loop; the next sub-step of the rank is on its way while one is multiplied
    auto add_adapter = [&](const GemmArgs& a) {
        uint32_t raw[2][8];
        half8_t v[TM], b[2];
        auto request = [&](int ks) {
            adapter_load(a, ks, raw);
#pragma unroll
            for (int i = 0; i < TM; ++i) v[i] = adapter_row(a, i, ks);
        };
        request(0);
#pragma unroll 1
        for (int ks = 0; 16 * ks < a.R; ++ks) {
            half8_t row[TM];
            adapter_cols(a, ks, raw, b);
#pragma unroll
            for (int i = 0; i < TM; ++i) row[i] = v[i];
            if (16 * (ks + 1) < a.R) request(ks + 1);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(row[i], b[j], acc[i][j], 0, 0, 0);
            if constexpr (TM == 8) keep_all();
        }
    };
    // Dropout on the adapter input: its share of out[m, c] exists only where the mask keeps (m, c); the kept values carry
    // 1 / (1 - p) through lb_scale.  Summed by itself and added block by block, in front of the layer's loop, before anything
    // of it is live.
    auto add_masked_adapter = [&](const GemmArgs& a) {
        if constexpr (!FWD && TM == 8) {
            static_assert(kTile >= 4 * 2 * 256 * 8, "a layer's operands fill one tile");
            auto operand = [&](int ks, int j) {                   // the lane's own
                return reinterpret_cast<half8_t*>(sA0 + ((2 * ks + j) * 256 + threadIdx.x) * 8);
            };
            for (int ks = 0; 16 * ks < a.R; ++ks) {
                uint32_t raw[2][8];
                half8_t b[2];
                adapter_load(a, ks, raw);
                adapter_cols(a, ks, raw, b);
                *operand(ks, 0) = b[0];
                *operand(ks, 1) = b[1];
            }
            half8_t v[4], next[4];                                // a block's rows, and the following block's on their way
            auto request = [&](int i) {
#pragma unroll
                for (int ks = 0; ks < 4; ++ks)
                    if (ks == 0 || 16 * ks < a.R) next[ks] = adapter_row(a, i, ks);
            };
            request(0);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) v[ks] = next[ks];
                if (i + 1 < TM) request(i + 1);
                float16_t term[2];
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) term[j][r] = 0.f;
#pragma unroll
                for (int ks = 0; ks < 4; ++ks)
                    if (ks == 0 || 16 * ks < a.R) {
#pragma unroll
                        for (int j = 0; j < 2; ++j) term[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[ks], *operand(ks, j), term[j], 0, 0, 0);
                    }
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + 32 * i + 8 * (r >> 2) + 4 * lg + (r & 3);
                    const uint32_t dw = drop_word(a.drop, drop_row_key(a.drop, (uint32_t)m), (uint32_t)(cw + 2 * lc) >> 1);
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const float kept = ((dw >> (16 * j)) & 0x7FFFu) < a.drop.thr15 ? 0.f : term[j][r];
                        acc[i][j][r] = MULTI ? acc[i][j][r] + kept : 0.f + kept;
                    }
                }
#pragma unroll
                for (int j = 0; j < 2; ++j) keep_acc(acc[i][j]);
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads();                                      // before the loads write over the operands
        }
    };

    auto run_layer = [&](const GemmArgs& a, const StepRange sr) {
        const int RED = FWD ? a.K : a.N;
        const int phase = (tm.tile_r * TM / 8 * (a.phase_step & 0xff)) % sr.cnt;     // of the 256 rows that the tile belongs to
        const rsrc_t ra = make_rsrc(a.a + (size_t)m0 * RED, (unsigned)rows_valid * (unsigned)RED * 2u);
        const rsrc_t rw = make_rsrc(a.qweight, (unsigned)(a.K >> 3) * (unsigned)a.N * 4u);
        const rsrc_t rs = make_rsrc(a.scales, (unsigned)a.G * (unsigned)a.N * 2u);
        const rsrc_t rz = make_rsrc(a.qzeros, (unsigned)a.G * (unsigned)(a.N >> 3) * 4u);

        // activations: load q of a wavefront brings rows 8 (4q + wave) .. + 7, lane (row, slot); 16-byte unit u of row r sits
        // in slot u ^ (r / 2 % 8)
        int va[TM];
#pragma unroll
        for (int q = 0; q < TM; ++q)
            va[q] = ((8 * (4 * q + wave) + (lane >> 3)) * RED + 8 * ((lane & 7) ^ (4 * (wave & 1) + (lane >> 4)))) * 2;
        auto load_a = [&](half_t* dst, int q, int red) {
            load_lds128(ra, dst + (4 * q + wave) * 512, va[q], red * 2);
        };
        auto stage_ptr = [&](auto st) -> half_t* {
            constexpr int S = decltype(st)::value & 3;
            if constexpr (S == 0) return sA0;
            else if constexpr (S == 1) return sA1;
            else if constexpr (S == 2) return sA2;
            else return sA3;
        };
        int fo[KS];                                               // fragment of sub-step ks, halves from the tile's start
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) fo[ks] = lc * BK + 8 * ((2 * ks + lg) ^ ((lc >> 1) & 7));

        // packed words.  Forward: word-row 2 ks + lg of the step, columns cw + 2 lc, + 1: the lane's own B operands.
        // Grad-input: word-row t % 32 of the tile's 256 output columns, octet t / 32 of the step's 64 columns n.
        uint2_t w[FWD ? kStages : 2][KS];                         // grad-input: read back from sT, turned around
        uint4_t wr[FWD ? 1 : kStages][2];
        uint32_t sraw[kStages], zraw[kStages];
        const int twr = (threadIdx.x >> 3) & 31, toc = threadIdx.x & 7;
        const int g_out = FWD ? 0 : cw / a.groupsize;
        const int vw = FWD ? (lg * a.N + cw + 2 * lc) * 4 : (((c0 >> 3) + twr) * a.N + 8 * toc) * 4;
        const int vs = FWD ? (cw + 2 * lc) * 2 : (g_out * a.N + lane) * 2;
        const int vz = FWD ? ((cw + 2 * lc) >> 3) * 4 : (g_out * (a.N >> 3) + (lane >> 3)) * 4;
        // load number l of the step that multiplies reduction offset red; `slot` its registers
        auto load_other = [&](auto slot, auto lt, int red) {
            constexpr int S = decltype(slot)::value & 3, l = decltype(lt)::value;
            if constexpr (FWD) {
                if constexpr (l < KS) w[S][l] = buf_load64(rw, vw, ((red >> 3) + 2 * l) * a.N * 4);
                else if constexpr (l == KS) sraw[S] = buf_load32(rs, vs, group_of(a, red) * a.N * 2);
                else zraw[S] = buf_load32(rz, vz, group_of(a, red) * (a.N >> 3) * 4);
            } else {
                if constexpr (l < 2) wr[S][l] = buf_load128(rw, vw, (red + 4 * l) * 4);
                else if constexpr (l == 2) sraw[S] = buf_load16(rs, vs, red * 2);
                else zraw[S] = buf_load32(rz, vz, (red >> 3) * 4);
            }
        };

        // forward: (scale, zero term) of the lane's two columns
        half2_t s2[2], z2[2];
        auto prep = [&](uint32_t s, uint32_t z) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                s2[j] = as_half2(__builtin_amdgcn_perm(s, s, j ? 0x03020302u : 0x01000100u));
                const uint32_t zz = (z >> (4 * ((2 * lc + j) & 7))) & 0xFu;
                z2[j] = zero_term(s2[j], zz, zz);
            }
        };
        // grad-input: scales and zero terms of the octet the lane multiplies in a sub-step
        uint4_t so[2], zo[2];
        uint32_t bo[2][2][4];                                     // B operands [sub-step parity][j][pair]
        half8_t af[2][TM];
        auto read_sz = [&](auto st, auto kt) {
            constexpr int P = decltype(st)::value & 1, ks = decltype(kt)::value;
            so[ks & 1] = *reinterpret_cast<const uint4_t*>(&sZ[FWD ? 0 : wave][P][0][FWD ? 0 : 8 * (2 * ks + lg)]);
            zo[ks & 1] = *reinterpret_cast<const uint4_t*>(&sZ[FWD ? 0 : wave][P][1][FWD ? 0 : 8 * (2 * ks + lg)]);
        };
        // The operands of sub-step ks of a stage in 12 pieces for as many MFMAs' shadows: the codes of column j as bytes
        // (pieces 0..3: the two halves of j = 0, of j = 1), then one pair of weights each.
        uint32_t bt[2][2];
        half2_t bp[2];
        auto build = [&](auto st, auto kt, auto ut) {
            constexpr int ks = decltype(kt)::value, u = decltype(ut)::value, S = decltype(st)::value & (FWD ? 3 : 1);
            if constexpr (u % 6 < 2) {
                constexpr int j = u / 6, h = u % 6;
                const uint32_t c = j ? w[S][ks].y : w[S][ks].x;
                if constexpr (!FWD) bt[j][h] = (h ? c >> 4 : c) & 0x0F0F0F0Fu;
                else if constexpr (h == 0) { bt[j][0] = c & 0x0F0F0F0Fu; bt[j][1] = (c >> 4) & 0x0F0F0F0Fu; }
                else {                                            // rows 0..3 and 4..7 in order
                    const uint32_t lo = bt[j][0], hi = bt[j][1];
                    bt[j][0] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
                    bt[j][1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
                }
            } else {
                // the zero term comes off with the next pair: right behind its product the difference waits for a slot
                constexpr int j = u / 6, p = u % 6 - 2;
                bp[p & 1] = codes_of_bytes<p & 1>(bt[j][p >> 1]) * (FWD ? s2[j] : as_half2(so[ks & 1][p]));
                auto less_zero = [&](auto pt) {
                    constexpr int P = decltype(pt)::value;
                    bo[ks & 1][j][P] = as_u32(bp[P & 1] - (FWD ? z2[j] : as_half2(zo[ks & 1][P])));
                };
                if constexpr (p > 0) less_zero(std::integral_constant<int, p - 1>{});
                if constexpr (p == 3) less_zero(std::integral_constant<int, p>{});
            }
        };
        auto build_all = [&](auto st, auto kt) {
            static_for<0, 12>([&](auto ut) { build(st, kt, ut); });
        };
        // grad-input: the eight words of a thread turned around and stored, in pieces
        uint32_t tx[8];
        auto turn = [&](auto slot, auto par, auto it) {
            constexpr int S = decltype(slot)::value & 3, P = decltype(par)::value & 1, I = decltype(it)::value;
            if constexpr (!FWD) {
                if constexpr (I == 0 || I == 1) {                 // 16-bit halves: rows 0-3 against 4-7
                    const uint4_t lo = wr[S][0], hi = wr[S][1];
                    const uint32_t x[8] = {lo.x, hi.x, lo.y, hi.y, lo.z, hi.z, lo.w, hi.w};      // nibble 2 c of a turned word is column c, 2 c + 1 column c + 4
#pragma unroll
                    for (int i = 2 * I; i < 2 * I + 2; ++i) {
                        tx[i] = __builtin_amdgcn_perm(x[i + 4], x[i], 0x05040100u);
                        tx[i + 4] = __builtin_amdgcn_perm(x[i + 4], x[i], 0x07060302u);
                    }
                } else if constexpr (I == 2 || I == 3) {          // bytes
                    constexpr int b = 4 * (I - 2);
#pragma unroll
                    for (int i = b; i < b + 2; ++i) {
                        const uint32_t u = tx[i], v = tx[i + 2];
                        tx[i] = __builtin_amdgcn_perm(v, u, 0x06020400u);
                        tx[i + 2] = __builtin_amdgcn_perm(v, u, 0x07030501u);
                    }
                } else if constexpr (I < 8) {                     // nibbles
                    constexpr int i = 2 * (I - 4);
                    const uint32_t u = tx[i], v = tx[i + 1];
                    tx[i] = bfi(0x0F0F0F0Fu, u, v << 4);
                    tx[i + 1] = bfi(0x0F0F0F0Fu, u >> 4, v);
                } else if constexpr (I == 8) {
                    uint32_t* d = (P ? sT1 : sT0) + toc * kTw + 8 * twr;
                    *reinterpret_cast<uint4_t*>(d) = uint4_t{tx[0], tx[1], tx[2], tx[3]};
                    *reinterpret_cast<uint4_t*>(d + 4) = uint4_t{tx[4], tx[5], tx[6], tx[7]};
                } else {                                          // scale and zero term of column n = lane of the step
                    const half_t s = __builtin_bit_cast(half_t, (unsigned short)sraw[S]);
                    const half_t z = (half_t)(float)(((zraw[S] >> (4 * (lane & 7))) & 0xFu) + 1u);
                    sZ[wave][P][0][FWD ? 0 : lane] = s;
                    sZ[wave][P][1][FWD ? 0 : lane] = s * z;
                }
            }
        };
        constexpr int kTurns = 10;
        auto read_t = [&](auto st) {
            constexpr int P = decltype(st)::value & 1;
            if constexpr (!FWD) {
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    w[P][ks] = *reinterpret_cast<const uint2_t*>((P ? sT1 : sT0) + (2 * ks + lg) * kTw + 64 * wave + 2 * lc);
            }
        };
        constexpr int kAhead = FWD ? 3 : 4;                       // stage whose words, scales, zeros a step requests
        constexpr int BAR = TM / 2;                               // slot of the last sub-step behind which the barrier sits

        // multiplies stage s (ring position C = s % 4); on entry af[0] and bo[0] hold its sub-step 0.  LEFT: most steps that can
        // follow it.  The last three (LEFT < 3) request nothing, and their barriers await everything: a counted wait holds only
        // while every request of the last two steps exists, and the compiler deletes those to registers that no later step reads.
        auto step = [&](int s, auto ct, auto leftt) {
            constexpr int C = decltype(ct)::value, LEFT = decltype(leftt)::value;
            constexpr bool more = LEFT >= 3;
            const int red3 = red_of(s + 3, sr, phase), redx = red_of(s + kAhead, sr, phase);
            static_for<0, KS>([&](auto kt) {
                constexpr int ks = decltype(kt)::value, kn = (ks + 1) % KS;
                constexpr int sn = ks + 1 == KS ? C + 1 : C;      // stage of the operands built in this sub-step
                constexpr bool next = LEFT > 0 || ks + 1 < KS;    // whether there can be such a stage
                static_for<0, NMK>([&](auto it) {
                    constexpr int i = decltype(it)::value, g = ks * NMK + i;
                    acc[i / 2][i % 2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[ks & 1][i / 2],
                        __builtin_bit_cast(half8_t, uint4_t{bo[ks & 1][i % 2][0], bo[ks & 1][i % 2][1], bo[ks & 1][i % 2][2], bo[ks & 1][i % 2][3]}),
                        acc[i / 2][i % 2], 0, 0, 0);
                    // requests, one at a time over the first three sub-steps
                    constexpr int SL = 3 * NMK;
                    if constexpr (more) pieces_of<g, kLoads, SL>([&](auto lt) {
                        constexpr int l = decltype(lt)::value;
                        if constexpr (l < kOther) load_other(std::integral_constant<int, C + kAhead>{}, lt, redx);
                        else load_a(stage_ptr(std::integral_constant<int, C + 3>{}), l - kOther, red3);
                    });
                    // activation fragments of the next sub-step
                    constexpr int first = ks + 1 == KS ? BAR + 1 : 0, span = NMK - 1 - first;
                    if constexpr (next && ks + 1 == KS && i == BAR) {
                        constexpr int kYounger = more ? 2 * kLoads : 0;     // requested since the next stage's activations
                        __builtin_amdgcn_sched_barrier(0);
                        __builtin_amdgcn_s_waitcnt(0x0070 | (kYounger & 15) | ((kYounger >> 4) << 14));
                        asm volatile("" ::: "memory");
                        __builtin_amdgcn_s_barrier();
                        asm volatile("" ::: "memory");
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if constexpr (next) pieces_of<i - first, TM, span>([&](auto rt) {
                        constexpr int r = decltype(rt)::value;
                        af[kn & 1][r] = *reinterpret_cast<const half8_t*>(stage_ptr(std::integral_constant<int, sn>{}) + fo[kn] + r * 32 * BK);
                    });
                    // operands of the next sub-step
                    if constexpr (FWD) {
                        if constexpr (next && ks + 1 == KS && i == 0) prep(sraw[(C + 1) & 3], zraw[(C + 1) & 3]);
                    } else {
                        if constexpr (i == 0 && (LEFT > 0 || ks + 2 < KS)) read_sz(std::integral_constant<int, ks + 2 >= KS ? C + 1 : C>{}, std::integral_constant<int, (ks + 2) % KS>{});
                        if constexpr (LEFT > 0 && ks == KS - 2 && i == 1) read_t(std::integral_constant<int, C + 1>{});
                        if constexpr (LEFT > 1) pieces_of<g - NMK / 2, kTurns, 2 * NMK>([&](auto qt) {      // words of stage s + 2
                            turn(std::integral_constant<int, C + 2>{}, std::integral_constant<int, C>{}, qt);
                        });
                    }
                    if constexpr (next) pieces_of<i, 12, NMK - 1>([&](auto ut) {
                        build(std::integral_constant<int, sn>{}, std::integral_constant<int, kn>{}, ut);
                    });
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
        };

        // the first stages
        static_for<0, kAhead>([&](auto st) {
            constexpr int S = decltype(st)::value;
            const int red = red_of(S, sr, phase);
            static_for<0, kOther>([&](auto lt) { load_other(st, lt, red); });
            if constexpr (S < 3) {
#pragma unroll
                for (int q = 0; q < TM; ++q) load_a(stage_ptr(st), q, red);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (!FWD) {
            static_for<0, kTurns>([&](auto qt) { turn(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, qt); });
            static_for<0, kTurns>([&](auto qt) { turn(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{}, qt); });
        }
        constexpr int kBehind = FWD ? 2 * kLoads : 2 * kLoads + kOther;     // requested behind stage 0
        __builtin_amdgcn_s_waitcnt(0x0070 | (kBehind & 15) | ((kBehind >> 4) << 14));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if constexpr (FWD) prep(sraw[0], zraw[0]);
        else {
            read_t(std::integral_constant<int, 0>{});
            read_sz(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
            read_sz(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) af[0][i] = *reinterpret_cast<const half8_t*>(sA0 + fo[0] + i * 32 * BK);
        build_all(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);
        int s = 0;
        for (; s + 4 <= sr.cnt; s += 4) {
            step(s, std::integral_constant<int, 0>{}, std::integral_constant<int, 3>{});
            step(s + 1, std::integral_constant<int, 1>{}, std::integral_constant<int, 3>{});
            step(s + 2, std::integral_constant<int, 2>{}, std::integral_constant<int, 3>{});
            step(s + 3, std::integral_constant<int, 3>{}, std::integral_constant<int, 3>{});
        }
        if (s < sr.cnt) step(s, std::integral_constant<int, 0>{}, std::integral_constant<int, 2>{});
        if (s + 1 < sr.cnt) step(s + 1, std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
        if (s + 2 < sr.cnt) step(s + 2, std::integral_constant<int, 2>{}, std::integral_constant<int, 0>{});
        if constexpr (TM == 8) keep_all();
        // nothing on its way into the tiles any more, and every wavefront done with them
        __builtin_amdgcn_s_waitcnt(0x0070);
        __syncthreads();
    };

    auto layer = [&](const GemmArgs& a, const StepRange sr, const bool with_adapter) {
        if constexpr (MULTI) {                // opaque per layer, or everything derived from it is kept in registers over the layers (and spills)
            asm volatile("" : "+v"(lane));
            lc = lane & 31;
            lg = lane >> 5;
        }
        const bool adapter = with_adapter && a.R > 0, masked = adapter && !FWD && a.drop.thr15 != 0;     // uniform
        if (masked) add_masked_adapter(a);
        run_layer(a, sr);
        if (adapter && !masked) add_adapter(a);
    };
    if constexpr (MULTI) {
        int base = 0;
#pragma unroll 1
        for (int li = 0; li < nlay; ++li) {
            const int steps = (FWD ? layers[li].K : layers[li].N) / BK;
            const int lo = max(share.begin, base) - base, hi = min(share.begin + share.cnt, base + steps) - base;
            base += steps;
            if (lo >= hi) continue;                               // uniform
            layer(layers[li], StepRange{lo, hi - lo}, lo == 0);   // the share that holds a layer's first step carries its adapter term
        }
    } else {
        layer(a0, share, zsplit == 0);
    }

    // acc[i][j][r]: row 32 i + 8 (r / 4) + 4 (lane / 32) + r % 4, column cw + 2 (lane % 32) + j
    if (nsplit > 1) {
        float* const pz = a0.part + (size_t)zsplit * a0.M * a0.part_cols - (size_t)a0.col_tile0 * kWideCols;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + 32 * i + 8 * (r >> 2) + 4 * lg + (r & 3);
                typedef float float2_t __attribute__((ext_vector_type(2)));
                const float2_t v = {acc[i][0][r] + (zsplit == 0 ? bias_v[0] : 0.f), acc[i][1][r] + (zsplit == 0 ? bias_v[1] : 0.f)};
                if (m < a0.M) *reinterpret_cast<float2_t*>(pz + (size_t)m * a0.part_cols + cw + 2 * lc) = v;
            }
        return;
    }
    constexpr int kRow = 64 + 8;                                  // halves of a staged row of 64 outputs
    half_t* stage = (wave < 2 ? sA0 : sA1) + (wave & 1) * (32 * kRow);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const half2_t h = {(half_t)(acc[i][0][r] + bias_v[0]), (half_t)(acc[i][1][r] + bias_v[1])};
            *reinterpret_cast<half2_t*>(stage + (8 * (r >> 2) + 4 * lg + (r & 3)) * kRow + 2 * lc) = h;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int rr = (lane >> 3) + 8 * p, m = m0 + 32 * i + rr;
            const uint4_t v = *reinterpret_cast<const uint4_t*>(stage + rr * kRow + 8 * (lane & 7));
            if (m < a0.M) *reinterpret_cast<uint4_t*>(a0.out + (size_t)m * NOUT + cw + 8 * (lane & 7)) = v;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

template <int TM, bool FWD>
__global__ __launch_bounds__(256) void gemm_wide_kernel(GemmArgs a) {
    const StepRange sr = split_steps((FWD ? a.K : a.N) / BK, blockIdx.z, gridDim.z);
    wide_body<TM, FWD, false>(&a, 1, map_tile(a.phase_step, a.col_tile0), sr, blockIdx.z, gridDim.z);
}

// Several layers in one grid (see GemmGroupArgs).
template <int TM, bool FWD>
__global__ __launch_bounds__(256) void gemm_wide_group_kernel(GemmGroupArgs g) {
    TileMap tm = map_tile(g.layer[0].phase_step, g.layer[0].col_tile0);
    if constexpr (FWD) {
        const int li = (tm.tile_c >= g.tile_end[0]) + (tm.tile_c >= g.tile_end[1]) + (tm.tile_c >= g.tile_end[2]);   // uniform
        tm.tile_c -= li == 0 ? 0 : g.tile_end[li - 1];
        const GemmArgs a = g.layer[li];
        wide_body<TM, FWD, false>(&a, 1, tm, split_steps(a.K / BK, 0, 1), 0, 1);
    } else {
        int nsteps = 0;
        for (int i = 0; i < g.n; ++i) nsteps += g.layer[i].N / BK;
        wide_body<TM, FWD, true>(g.layer, g.n, tm, split_steps(nsteps, blockIdx.z, gridDim.z), (int)blockIdx.z, (int)gridDim.z);
    }
}

void launch_wide_tiles(bool fwd, bool low, const GemmArgs& a, dim3 grid, hipStream_t stream) {
    if (low) hipLaunchKernelGGL((gemm_wide_kernel<4, true>), grid, dim3(256), 0, stream, a);
    else if (fwd) hipLaunchKernelGGL((gemm_wide_kernel<8, true>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((gemm_wide_kernel<8, false>), grid, dim3(256), 0, stream, a);
}
void launch_wide_group_tiles(bool fwd, bool low, const GemmGroupArgs& g, dim3 grid, hipStream_t stream) {
    if (low) hipLaunchKernelGGL((gemm_wide_group_kernel<4, true>), grid, dim3(256), 0, stream, g);
    else if (fwd) hipLaunchKernelGGL((gemm_wide_group_kernel<8, true>), grid, dim3(256), 0, stream, g);
    else hipLaunchKernelGGL((gemm_wide_group_kernel<8, false>), grid, dim3(256), 0, stream, g);
}

}  // namespace q4
