// Rank-R helper products of the LoRA adapter around the fused 4-bit GEMMs (HBM-bound: each reads
// one [M, C] activation / gradient matrix exactly once).
//
//   down:  out fp16 [M, R]   = in fp16 [M, C] @ W^T          xa = x @ A^T,  dyb = dy @ B
//   grad:  out fp32 [R, C]^  = alpha * P^T fp16 [R, M] @ in   dA = s * dyb^T @ x,  dB^T = s * xa^T @ dy
//
// (^ written through strides, so dB lands directly in lora_B.weight's [N, R] layout.)
// Together with the adapter step inside the GEMMs they replace what torch autograd does over
// lora_B(lora_A(x)) * scaling in the reference (src/alpaca_lora_4bit/models.py:58-66).
// W is read in place with strides and in its own dtype (fp32 or fp16): no cast or transpose
// kernels around the adapter.
#include "q4_common.hpp"
#include "q4_gptq.h"
#include <algorithm>

namespace q4 {

constexpr int kFarOffset = 0x70000000;      // beyond any buffer accepted here: such loads return zero, no traffic

__device__ __forceinline__ half8_t to_half8(float4_t a, float4_t b) {
    half8_t r;
#pragma unroll
    for (int e = 0; e < 4; ++e) { r[e] = (half_t)a[e]; r[4 + e] = (half_t)b[e]; }
    return r;
}

// ---- down projection -------------------------------------------------------------------
// Workgroup = 16 wavefronts on 16 rows; wavefront w multiplies the C/16-wide slice w of those rows
// with v_mfma_f32_16x16x32_f16 (A operand = 16 rows x 32 columns of `in`, B operand = the same 32
// columns of up to 16 rows of W); the partial 16 x 16 results are added through LDS.  R <= 64 is
// handled as RB = ceil(R/16) column blocks.
// All loads are buffer loads whose out-of-range lanes (rows past M, adapter rows past R, steps past
// the wavefront's slice) return zero: no branch sits between the loads of a batch of UN steps, so they
// are all in flight together.  Three ways to fetch W[j][c] -> the B operand (8 consecutive c per lane):
//   kRowsT c contiguous in memory (lora_A.weight [R, C]), R <= 16: each adapter row's 256-column piece is
//          loaded as one fully coalesced instruction (4 values per lane), converted, and passed to the
//          operand layout through a wavefront-private LDS tile
//   kCols  j contiguous in memory (lora_B.weight [C, R] seen as W = B^T), R <= 16, R % 4 == 0: groups of 4
//          adapter rows are loaded coalesced and transposed through the same LDS tile
//   kRows  c contiguous, any R <= 64: one or two 16-byte loads per lane and step straight into the operand
//   kAny   arbitrary strides: eight scalar loads per lane and step
enum WLayout { kRows = 0, kCols = 1, kAny = 2, kRowsT = 3 };
constexpr int kDownWaves = 16;

// The adapters of layers that run together (q | v) go out side by side, blockIdx.y = the problem: a single one of a few hundred
// rows fills a fifth of the chip and its time is the latency of one burst of loads.  us for q and v of 4096 features at rank 8
// with dropout, one launch each -> one launch: 200 rows
// 12.1 -> 6.4, 1024 13.5 -> 7.1 (dy @ B without: 8.6 -> 4.6, 9.5 -> 5.8), 4096 of 5120 features 25.1 -> 23.4.  2048 rows at rank 64: 98 -> 50.
constexpr int kDownProbs = 4;
struct DownProb {
    const half_t* in;         // [M, C]
    const void* w;            // [R, C] through w_sr, w_sc
    half_t* out;              // [M, R]
    int w_sr, w_sc, C;
    DropArgs drop;
};
struct DownArgs { DownProb p[kDownProbs]; };

// LDS of a workgroup: the partial products, and the transposition tile of the staged layouts
template <int RB, int WL> struct DownLds {
    static constexpr bool kStaged = WL == kCols || WL == kRowsT;
    static constexpr int UN = WL == kAny ? (RB == 1 ? 4 : RB == 2 ? 2 : 1) : (RB == 1 ? 8 : 4);   // steps whose loads are issued together
    static constexpr int TRW = UN * 32 + 8;                     // padded row of the transposition tile (halves)
    float red[kDownWaves][RB][256];
    __attribute__((aligned(16))) half_t tr[kStaged ? kDownWaves : 1][16][kStaged ? TRW : 8];
};

// Leaves the wavefronts' partial 16 x 16 products of rows m0 .. m0 + rows - 1 in lds.red (no barrier after the last write).
template <int RB, int WL, bool F32, int RQ>   // RQ: ceil(R/4) for kCols / kRowsT, else unused
__device__ __forceinline__ void lora_down_rows(DownLds<RB, WL>& lds, const half_t* __restrict__ in, const void* __restrict__ w,
                                               int w_sr, int w_sc, int m0, int M, int C, int R, int rows, const DropArgs& drop) {
    constexpr int NW = kDownWaves, UN = DownLds<RB, WL>::UN;
    constexpr int ES = F32 ? 4 : 2;
    constexpr bool kStaged = DownLds<RB, WL>::kStaged;
    auto& tr = lds.tr;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kk = lane >> 4, c = lane & 15;
    const int steps = C / 32;                                   // C is a multiple of 32
    const int s_begin = (steps * wave) / NW, s_end = (steps * (wave + 1)) / NW;
    const rsrc_t rs_in = make_rsrc(in + (size_t)m0 * C, (unsigned)min(rows, M - m0) * (unsigned)C * 2u);
    const rsrc_t rs_w = make_rsrc(w, ((unsigned)(R - 1) * (unsigned)w_sr + (unsigned)(C - 1) * (unsigned)w_sc + 1u) * ES);
    const int voff_in = (c * C + 8 * kk) * 2;
    float4_t acc[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) acc[b] = float4_t{0.f, 0.f, 0.f, 0.f};
    // dropout of `in` (uniform branch): this lane's operand is row m0 + c, columns 32*s + 8*kk .. + 7 of step s
    const uint32_t drop_key = drop_row_key(drop, (uint32_t)(m0 + c));
    const uint32_t thr_pair = drop.thr15 | (drop.thr15 << 16);

    for (int s0 = s_begin; s0 < s_end; s0 += UN) {
        uint4_t av[UN];
        half8_t bv[UN][RB];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int s = s0 + u;
            av[u] = buf_load128(rs_in, voff_in, s < s_end ? s * 64 : kFarOffset);
        }
        if constexpr (WL == kRows) {
            uint4_t raw[UN][RB][F32 ? 2 : 1];
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int s = s0 + u;
                const int soff = s < s_end ? s * 32 * ES : kFarOffset;
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    const int j = 16 * b + c;
                    const int voff = j < R ? (j * w_sr + 8 * kk) * ES : kFarOffset;
                    raw[u][b][0] = buf_load128(rs_w, voff, soff);
                    if constexpr (F32) raw[u][b][1] = buf_load128(rs_w, voff + 16, soff);
                }
            }
#pragma unroll
            for (int u = 0; u < UN; ++u)
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    if constexpr (F32) bv[u][b] = to_half8(__builtin_bit_cast(float4_t, raw[u][b][0]), __builtin_bit_cast(float4_t, raw[u][b][1]));
                    else bv[u][b] = __builtin_bit_cast(half8_t, raw[u][b][0]);
                }
        } else if constexpr (kStaged) {
            // fill the tile tr[j][column within the batch] with fp16 values of W
            if constexpr (WL == kCols) {
                // UN*32 columns x RQ groups of 4 adapter rows, 64 items per load instruction
                constexpr int NT = UN * 32 * RQ / 64;
                uint4_t raw[NT];
                const int soff = s0 * 32 * w_sc * ES;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int i = lane + 64 * t, cl = i / RQ, q = i - cl * RQ;
                    const int voff = (s0 * 32 + cl) < s_end * 32 ? (cl * w_sc + 4 * q) * ES : kFarOffset;
                    if constexpr (F32) raw[t] = buf_load128(rs_w, voff, soff);
                    else { const uint2_t v = buf_load64(rs_w, voff, soff); raw[t] = uint4_t{v.x, v.y, 0u, 0u}; }
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int i = lane + 64 * t, cl = i / RQ, q = i - cl * RQ;
                    half_t h[4];
                    if constexpr (F32) {
                        const float4_t f = __builtin_bit_cast(float4_t, raw[t]);
#pragma unroll
                        for (int e = 0; e < 4; ++e) h[e] = (half_t)f[e];
                    } else {
                        const half2_t lo = as_half2(raw[t].x), hi = as_half2(raw[t].y);
                        h[0] = lo[0]; h[1] = lo[1]; h[2] = hi[0]; h[3] = hi[1];
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) tr[wave][4 * q + e][cl] = h[e];
                }
            } else {
                // 4*RQ adapter rows; per row the batch's UN*32 columns, 4 per lane
                constexpr int NL = UN * 32 / 256;                 // load instructions per row (1 for UN = 8)
                static_assert(NL >= 1, "a batch must cover at least 256 columns");
                uint4_t raw[4 * RQ][NL];
                const int soff = s0 * 32 * ES;
#pragma unroll
                for (int j = 0; j < 4 * RQ; ++j)
#pragma unroll
                    for (int t = 0; t < NL; ++t) {
                        const int cl = 4 * (lane + 64 * t);
                        const int voff = (j < R && (s0 * 32 + cl) < s_end * 32) ? (j * w_sr + cl) * ES : kFarOffset;
                        if constexpr (F32) raw[j][t] = buf_load128(rs_w, voff, soff);
                        else { const uint2_t v = buf_load64(rs_w, voff, soff); raw[j][t] = uint4_t{v.x, v.y, 0u, 0u}; }
                    }
#pragma unroll
                for (int j = 0; j < 4 * RQ; ++j)
#pragma unroll
                    for (int t = 0; t < NL; ++t) {
                        const int cl = 4 * (lane + 64 * t);
                        uint2_t packed;
                        if constexpr (F32) {
                            const float4_t f = __builtin_bit_cast(float4_t, raw[j][t]);
                            const half2_t lo = {(half_t)f[0], (half_t)f[1]}, hi = {(half_t)f[2], (half_t)f[3]};
                            packed = uint2_t{as_u32(lo), as_u32(hi)};
                        } else {
                            packed = uint2_t{raw[j][t].x, raw[j][t].y};
                        }
                        *reinterpret_cast<uint2_t*>(&tr[wave][j][cl]) = packed;
                    }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const half8_t v = *reinterpret_cast<const half8_t*>(&tr[wave][c][32 * u + 8 * kk]);
#pragma unroll
                for (int e = 0; e < 8; ++e) bv[u][0][e] = c < 4 * RQ ? v[e] : (half_t)0.f;   // rows past R were never written
            }
            __builtin_amdgcn_wave_barrier();
        } else {
            uint32_t raw[UN][RB][8];
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int s = s0 + u;
                const int soff = s < s_end ? s * 32 * w_sc * ES : kFarOffset;
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    const int j = 16 * b + c;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const int voff = j < R ? (j * w_sr + (8 * kk + e) * w_sc) * ES : kFarOffset;
                        raw[u][b][e] = F32 ? buf_load32(rs_w, voff, soff) : buf_load16(rs_w, voff, soff);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < UN; ++u)
#pragma unroll
                for (int b = 0; b < RB; ++b)
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        bv[u][b][e] = F32 ? (half_t)__builtin_bit_cast(float, raw[u][b][e])
                                          : __builtin_bit_cast(half_t, (uint16_t)raw[u][b][e]);
        }
        // dropout of `in`, after every load of the batch has been issued (steps past the slice hold zeros anyway)
        if (drop.thr15) {
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const uint32_t pair0 = (uint32_t)(s0 + u) * 16u + 4u * kk;
                av[u].x &= drop_keep_mask(drop_word(drop, drop_key, pair0), thr_pair);
                av[u].y &= drop_keep_mask(drop_word(drop, drop_key, pair0 + 1), thr_pair);
                av[u].z &= drop_keep_mask(drop_word(drop, drop_key, pair0 + 2), thr_pair);
                av[u].w &= drop_keep_mask(drop_word(drop, drop_key, pair0 + 3), thr_pair);
            }
        }
        // steps past the slice were loaded as zeros: they add nothing
#pragma unroll
        for (int u = 0; u < UN; ++u)
#pragma unroll
            for (int b = 0; b < RB; ++b)
                acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, av[u]), bv[u][b], acc[b], 0, 0, 0);
    }
    // acc[b][r]: row 4*kk + r, column 16*b + c
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) lds.red[wave][b][(4 * kk + r) * 16 + c] = acc[b][r];
}

template <int RB, int WL>
__device__ __forceinline__ float lora_down_sum(const DownLds<RB, WL>& lds, int b, int i) {     // element i of column block b
    float v = 0.f;
#pragma unroll
    for (int wv = 0; wv < kDownWaves; ++wv) v += lds.red[wv][b][i];
    return v;
}

template <int RB, int WL, bool F32, int RQ>
__global__ __launch_bounds__(64 * kDownWaves) void lora_down_kernel(DownArgs da, int M, int R, int rows) {
    __shared__ DownLds<RB, WL> lds;
    const DownProb& p = da.p[blockIdx.y];
    const int m0 = blockIdx.x * rows;                           // rows = 16, 8 or 4: operand rows past it read as zero
    const DropArgs drop = p.drop;
    lora_down_rows<RB, WL, F32, RQ>(lds, p.in, p.w, p.w_sr, p.w_sc, m0, M, p.C, R, rows, drop);
    __syncthreads();
    for (int e = threadIdx.x; e < RB * 256; e += 64 * kDownWaves) {
        const int b = e >> 8, i = e & 255;
        const float v = lora_down_sum(lds, b, i);
        const int m = m0 + (i >> 4), j = 16 * b + (i & 15);
        if ((i >> 4) < rows && m < M && j < R) p.out[(size_t)m * R + j] = (half_t)(v * drop.scale);
    }
}

// ---- rank-R update of a few rows -----------------------------------------------------------
// y[m, n] += alpha * sum_r xa[m, r] * B[n, r] in place, one rounding: the second half of the adapter at decode sizes.
// Launch-bound (a few hundred KB at most): one thread per column, kUpRows rows per workgroup, B read in place with its
// strides and in its own type, xa from LDS.  At 4 x 4096, R = 8 it stands for a library product of 6.9 us (whose 256-row
// tile is mostly padding) and for the fp16 copy of B that it needed: 8 blocks of the 7B step at 4 rows with adapters on q
// and v, called one by one, 1289 -> 937 us.
constexpr int kUpRows = 4, kUpCols = 64;

template <bool F32, bool VEC>           // VEC: B rows contiguous, R % 4 == 0, 16 (fp32) / 8 (fp16) byte aligned
__global__ __launch_bounds__(kUpCols) void lora_up_kernel(const half_t* __restrict__ xa, const void* __restrict__ w, int w_sn, int w_sr,
                                                          half_t* __restrict__ y, float alpha, int M, int N, int R) {
    __shared__ float sx[kUpRows][64];
    const int m0 = blockIdx.y * kUpRows, rows = min(kUpRows, M - m0);
    for (int i = threadIdx.x; i < kUpRows * R; i += kUpCols) {
        const int m = i / R, r = i - m * R;
        sx[m][r] = m < rows ? (float)xa[(size_t)(m0 + m) * R + r] : 0.f;
    }
    __syncthreads();
    const int n = blockIdx.x * kUpCols + threadIdx.x;
    if (n >= N) return;
    float old[kUpRows];
#pragma unroll
    for (int m = 0; m < kUpRows; ++m) old[m] = m < rows ? (float)y[(size_t)(m0 + m) * N + n] : 0.f;
    float acc[kUpRows] = {0.f, 0.f, 0.f, 0.f};
    const size_t base = (size_t)n * w_sn;
    auto add = [&](float b, int r) {
#pragma unroll
        for (int m = 0; m < kUpRows; ++m) acc[m] = fmaf(sx[m][r], b, acc[m]);
    };
    if constexpr (VEC) {
        for (int r = 0; r < R; r += 4) {
            if constexpr (F32) {
                const float4_t b = *reinterpret_cast<const float4_t*>(reinterpret_cast<const float*>(w) + base + r);
#pragma unroll
                for (int e = 0; e < 4; ++e) add(b[e], r + e);
            } else {
                const half4_t b = *reinterpret_cast<const half4_t*>(reinterpret_cast<const half_t*>(w) + base + r);
#pragma unroll
                for (int e = 0; e < 4; ++e) add((float)b[e], r + e);
            }
        }
    } else {
        for (int r = 0; r < R; ++r) {
            const size_t i = base + (size_t)r * w_sr;
            add(F32 ? reinterpret_cast<const float*>(w)[i] : (float)reinterpret_cast<const half_t*>(w)[i], r);
        }
    }
#pragma unroll
    for (int m = 0; m < kUpRows; ++m)
        if (m < rows) y[(size_t)(m0 + m) * N + n] = (half_t)fmaf(alpha, acc[m], old[m]);
}

// ---- the whole adapter of up to 16 rows in one launch ----------------------------------------
// y += alpha * fp16(x @ A^T) @ B^T for the adapters of layers that share x.  Every workgroup forms x @ A^T for itself, exactly as
// lora_down_kernel does (whose grid is one to four workgroups here: A comes from L2 either way, R * K * 4 bytes a workgroup),
// and then updates 256 columns with lora_up_kernel's products in its order: the results are the two kernels' to the bit.  B and y
// are on their way while x @ A^T is formed.  us for q and v of 4096 features at rank 8,
// four launches -> one: 11.8 -> 4.5 at 1 row, 13.6 -> 5.4 at 4, 14.0 -> 7.9 at 16; rank 16 15.3 -> 9.2 at 16 rows.
constexpr int kUpdCols = 256, kUpdRows = 16;
struct UpdProb {
    const void* a;            // [R, K], rows a_sr apart, contiguous and 16-byte aligned
    const void* b;            // [N, R], rows b_sn apart, contiguous and 4 values aligned
    half_t* y;                // [M, N]
    int a_sr, b_sn, N;
    float alpha;
};
struct UpdArgs { UpdProb p[kDownProbs]; };

template <bool F32, int RQ>             // R == 4 * RQ
__global__ __launch_bounds__(64 * kDownWaves) void lora_update_kernel(UpdArgs ua, const half_t* __restrict__ x, int M, int K) {
    constexpr int R = 4 * RQ, RG = 64 * kDownWaves / kUpdCols, MR = kUpdRows / RG;    // RG groups of up to MR rows
    __shared__ DownLds<1, kRowsT> lds;
    __shared__ float sx[kUpdRows][R];
    const UpdProb& p = ua.p[blockIdx.y];
    if ((int)blockIdx.x * kUpdCols >= p.N) return;              // uniform: past a narrower layer of the launch
    const int n = blockIdx.x * kUpdCols + (threadIdx.x & (kUpdCols - 1));
    const int per = (M + RG - 1) / RG, m0 = (threadIdx.x / kUpdCols) * per, rows = n < p.N ? min(per, M - m0) : 0;
    constexpr bool kLate = F32 && RQ > 3;                       // 16 more fp32 values would spill beside the loads of the products
    float bv[R], old[MR];
    auto load_b = [&] {
#pragma unroll
        for (int r = 0; r < R; r += 4) {
            if constexpr (F32) {
                float4_t b = {0.f, 0.f, 0.f, 0.f};
                if (rows > 0) b = *reinterpret_cast<const float4_t*>(reinterpret_cast<const float*>(p.b) + (size_t)n * p.b_sn + r);
#pragma unroll
                for (int e = 0; e < 4; ++e) bv[r + e] = b[e];
            } else {
                half4_t b = {(half_t)0.f, (half_t)0.f, (half_t)0.f, (half_t)0.f};
                if (rows > 0) b = *reinterpret_cast<const half4_t*>(reinterpret_cast<const half_t*>(p.b) + (size_t)n * p.b_sn + r);
#pragma unroll
                for (int e = 0; e < 4; ++e) bv[r + e] = (float)b[e];
            }
        }
    };
    if constexpr (!kLate) load_b();
#pragma unroll
    for (int m = 0; m < MR; ++m) old[m] = m < rows ? (float)p.y[(size_t)(m0 + m) * p.N + n] : 0.f;
    const DropArgs none{0u, 0u, 0u, 1.0f};
    lora_down_rows<1, kRowsT, F32, RQ>(lds, x, p.a, p.a_sr, 1, 0, M, K, R, kUpdRows, none);
    if constexpr (kLate) load_b();
    __syncthreads();
    if (threadIdx.x < 256 && (threadIdx.x & 15) < R)
        sx[threadIdx.x >> 4][threadIdx.x & 15] = (float)(half_t)lora_down_sum(lds, 0, threadIdx.x);
    __syncthreads();
    const float alpha = p.alpha;
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        if (m >= rows) break;
        float acc = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) acc = fmaf(sx[m0 + m][r], bv[r], acc);
        p.y[(size_t)(m0 + m) * p.N + n] = (half_t)fmaf(alpha, acc, old[m]);
    }
}

// ---- gradient of an adapter matrix --------------------------------------------------------
// out[j, c] = alpha * sum_m P[m, j] * in[m, c] as v_mfma_f32_16x16x32_f16 products whose reduction index is the ROW m:
//   A operand  P^T: lane (j = l % 16, kk = l / 16) holds P[mb + 8*kk .. + 7][j]   (rows j >= R are zero)
//   B operand  in:  lane (cg = l % 16, kk) holds in[mb + 8*kk .. + 7][col]         for ONE column per MFMA
// A lane loads eight 16-byte pieces, rows mb + 8*kk + e (e = 0..7) x columns c0 + 8*cg .. + 7 (256 contiguous bytes
// per 16 lanes and row), and turns the 8 x 8 block around in registers with 32 byte permutes; MFMA i of the eight
// then multiplies column c0 + 8*cg + i.  A wavefront so consumes a block of 32 rows x 128 columns (8 KB) with 8
// loads, 32 permutes and 8 MFMAs per 16 adapter rows; the kernel is bound by its loads.  P for the block (32 x R
// values) is fetched with 4-byte loads (R even, at most 32) or 16-byte ones (40, 48, 56, 64) and transposed through a
// wavefront-private LDS tile.
// Workgroup = 4 wavefronts on one 128-column strip and `rows_per_wg` rows (wavefront w takes the 32-row blocks
// w, w + 4, ...); the sum over wavefronts goes through LDS, the sum over the gridDim.y workgroups of a strip through
// fp32 partial tiles [split][strip][R][128] that lora_grad_reduce_kernel adds in a fixed order (bit-reproducible).
// Above 32 adapter rows `in` is still read once, at the price of one workgroup per CU for ranks 56 and 64 (32 accumulator
// tiles a wavefront).  As two problems of half the rank, each reading `in` and leaving partial tiles, both gradients of
// 2048 rows of 13824 and 13824 features took 72 us at rank 64 (77.5 with dropout) where library products take 44; now 31
// with dropout; 4096 x 4096 features 33.8 -> 20.5, 512 rows of 5120 and 13824 39 -> 17.  One block of 64 rows alone
// takes longer (7.8 -> 8.8 us).
constexpr int kG2Waves = 4, kG2Cols = 128, kG2PadRows = 40;

// Up to kGradProbs gradients per launch (blockIdx.z): the two adapter gradients of a layer, and those of the layers that run
// together, share M and R and are independent, so they go out side by side.  Workgroups beyond a problem's own grid leave at
// once.  us, gradients and reduction of q and v of 4096 features at rank 8 with dropout, two launches each -> two together:
// 200 rows 13.5 -> 7.4, 1024 15.2 -> 12.6, 4096 of 5120 features 36.2 -> 29.4.
constexpr int kGradProbs = 8;
struct GradProb {
    const half_t* P;          // [M, R]
    const half_t* in;         // [M, C]
    float* out;               // through o_sr, o_sc
    float* part;              // partial tiles [splits][col_blocks][R][128]
    int o_sr, o_sc, C, col_blocks, splits, rows_per_wg;
    float alpha;
    DropArgs drop;            // dropout mask applied to `in` (thr15 == 0: none); the result carries drop.scale
};
struct GradArgs {
    GradProb p[kGradProbs];
    int M;
};

// Above 32 adapter rows a result whose adapter rows lie side by side (lora_B.weight's layout) goes out along them, partial
// tiles included: 64-byte pieces instead of single words (64 rows of 4096 features at rank 64: 0.7 us).
__device__ __forceinline__ bool grad_jfast(const GradProb& q) { return q.o_sr < q.o_sc; }

template <int RB>
struct G2Regs { uint4_t d[8]; uint32_t p[4 * RB]; };

template <bool DROP, int RB>    // RB = ceil(R / 16) A operands; R is even, above 32 a multiple of 8
__global__ __launch_bounds__(64 * kG2Waves, RB == 3 ? 2 : 1) void lora_grad_kernel(GradArgs ga, int R) {
    const GradProb& q = ga.p[blockIdx.z];
    if ((int)blockIdx.x >= q.col_blocks || (int)blockIdx.y >= q.splits) return;       // uniform over the workgroup
    constexpr bool PV = RB > 2;                                                       // P in 16-byte pieces
    constexpr int NPL = PV ? RB : 4 * RB;                                             // loads of P per lane and block
    __shared__ __attribute__((aligned(16))) float red[kG2Waves][16][kG2Cols + (PV ? 4 : 0)];   // 32 KB; + 4: grad_jfast's reads
    __shared__ __attribute__((aligned(16))) half_t pt[kG2Waves][16 * RB][kG2PadRows]; // P^T of the current block
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cg = lane & 15, kk = lane >> 4;
    const int C = q.C, M = ga.M;
    const int row_bytes = C * 2;
    const int c0 = blockIdx.x * kG2Cols + 8 * cg;
    const int m_wg = blockIdx.y * q.rows_per_wg;
    const int m_end = min(m_wg + q.rows_per_wg, M);
    const rsrc_t rs_in = make_rsrc(q.in, (unsigned)m_end * (unsigned)row_bytes);       // rows past m_end read as zero
    const rsrc_t rs_p = make_rsrc(q.P, (unsigned)m_end * (unsigned)(R * 2));
    int voff[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) voff[e] = c0 < C ? (8 * kk + e) * row_bytes + c0 * 2 : kFarOffset;
    // this lane's share of a block of P: the pairs i = lane, lane + 64, ... of the 32 x R block
    // (row i / (R/2), columns 2 * (i % (R/2)) and the next); PV: row lane % 32, columns 16 * t + 8 * (lane / 32) and the
    // seven next (32 lanes then write 64 contiguous bytes of P^T)
    const int hr = R >> 1;
    int pvoff[NPL], pdst[NPL];
#pragma unroll
    for (int t = 0; t < NPL; ++t) {
        const int i = lane + 64 * t;
        const int m = PV ? lane & 31 : i / hr, j = PV ? 16 * t + 8 * (lane >> 5) : 2 * (i - m * hr);
        const bool mine = PV ? j < R : i < 32 * hr;
        pvoff[t] = mine ? (m * R + j) * 2 : kFarOffset;
        pdst[t] = mine || PV ? j * kG2PadRows + m : -1;             // PV: columns beyond R read as zero and fill their rows
    }
    half_t* const ptw = &pt[wave][0][0];
    if constexpr (!PV)
        for (int i = lane; i < 16 * RB * kG2PadRows; i += 64) ptw[i] = (half_t)0.f;   // rows j >= R stay zero
    const DropArgs drop = q.drop;
    const uint32_t thr_pair = drop.thr15 | (drop.thr15 << 16);

    float4_t acc[RB][8];
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[b][i] = float4_t{0.f, 0.f, 0.f, 0.f};

    auto load_block = [&](G2Regs<RB>& x, int mb) {
        const bool live = mb < m_end;
        const int soff = live ? mb * row_bytes : kFarOffset;
        const int soff_p = live ? mb * R * 2 : kFarOffset;
#pragma unroll
        for (int t = 0; t < NPL; ++t) {
            if constexpr (PV) *reinterpret_cast<uint4_t*>(&x.p[4 * t]) = buf_load128(rs_p, pvoff[t], soff_p);
            else x.p[t] = buf_load32(rs_p, pvoff[t], soff_p);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) x.d[e] = buf_load128(rs_in, voff[e], soff);
    };
    auto consume = [&](G2Regs<RB>& x, int mb) {
        if (DROP && drop.thr15) {                 // uniform: the mask belongs to one problem of a pair
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t key = drop_row_key(drop, (uint32_t)(mb + 8 * kk + e));
                const uint32_t pr = (uint32_t)(c0 >> 1);
                x.d[e].x &= drop_keep_mask(drop_word(drop, key, pr), thr_pair);
                x.d[e].y &= drop_keep_mask(drop_word(drop, key, pr + 1), thr_pair);
                x.d[e].z &= drop_keep_mask(drop_word(drop, key, pr + 2), thr_pair);
                x.d[e].w &= drop_keep_mask(drop_word(drop, key, pr + 3), thr_pair);
            }
        }
#pragma unroll
        for (int t = 0; t < NPL; ++t)
            if (PV || pdst[t] >= 0) {
                constexpr int W = PV ? 4 : 1;                                         // words of a load
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const uint32_t v = x.p[W * t + w];
                    ptw[pdst[t] + 2 * w * kG2PadRows] = __builtin_bit_cast(half_t, (uint16_t)(v & 0xFFFFu));
                    ptw[pdst[t] + (2 * w + 1) * kG2PadRows] = __builtin_bit_cast(half_t, (uint16_t)(v >> 16));
                }
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        half8_t aop[RB];
#pragma unroll
        for (int b = 0; b < RB; ++b) aop[b] = *reinterpret_cast<const half8_t*>(ptw + (16 * b + cg) * kG2PadRows + 8 * kk);
        __builtin_amdgcn_wave_barrier();
        // 8 x 8 turn: tr[c][q] = (row 2q, row 2q + 1) of column c of this lane's block
        uint32_t tr[8][4];
#pragma unroll
        for (int qq = 0; qq < 4; ++qq) {
            const uint4_t r0 = x.d[2 * qq], r1 = x.d[2 * qq + 1];
            const uint32_t a0[4] = {r0.x, r0.y, r0.z, r0.w}, a1[4] = {r1.x, r1.y, r1.z, r1.w};
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                tr[2 * p][qq] = __builtin_amdgcn_perm(a1[p], a0[p], 0x05040100u);
                tr[2 * p + 1][qq] = __builtin_amdgcn_perm(a1[p], a0[p], 0x07060302u);
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint4_t bq = {tr[i][0], tr[i][1], tr[i][2], tr[i][3]};
#pragma unroll
            for (int b = 0; b < RB; ++b)
                acc[b][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aop[b], __builtin_bit_cast(half8_t, bq), acc[b][i], 0, 0, 0);
        }
    };

    // blocks w, w + 4, ... of the workgroup's rows; the next block's loads are in flight while one is consumed
    const int step = 32 * kG2Waves;
    G2Regs<RB> xa, xb;
    int mb = m_wg + 32 * wave;
    load_block(xa, mb);
    if constexpr (RB == 4) {                  // one copy of the products: with two the accumulators are copied between register
                                              // files on the way (2048 rows, 4096 features: 22.1 against 20.5 us)
        for (; mb < m_end; mb += step) {
            load_block(xb, mb + step);
            consume(xa, mb);
            xa = xb;
        }
    } else {
        for (; mb < m_end; mb += 2 * step) {
            load_block(xb, mb + step);
            consume(xa, mb);
            load_block(xa, mb + 2 * step);
            if (mb + step < m_end) consume(xb, mb + step);
        }
    }
    const bool direct = q.splits == 1;
    const bool jfast = PV && grad_jfast(q);
    const float alpha = q.alpha * drop.scale;
    float* tile = q.part + ((size_t)blockIdx.y * q.col_blocks + blockIdx.x) * (size_t)(R * kG2Cols);
#pragma unroll
    for (int b = 0; b < RB; ++b) {
        if (b > 0) __syncthreads();
        // acc[b][i][r]: adapter row j = 16*b + 4*kk + r, column 8*cg + i of the strip
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float* dst = &red[wave][4 * kk + r][8 * cg];
            *reinterpret_cast<float4_t*>(dst) = float4_t{acc[b][0][r], acc[b][1][r], acc[b][2][r], acc[b][3][r]};
            *reinterpret_cast<float4_t*>(dst + 4) = float4_t{acc[b][4][r], acc[b][5][r], acc[b][6][r], acc[b][7][r]};
        }
        __syncthreads();
        const int nj = min(16, R - 16 * b);
        auto write = [&](int o) {
            int jl = o >> 7, cl = o & (kG2Cols - 1);
            if (jfast) {                                                              // nj is 8 or 16
                jl = o & (nj - 1);
                cl = nj == 16 ? o >> 4 : o >> 3;
            }
            const int j = 16 * b + jl;
            const float v = (red[0][jl][cl] + red[1][jl][cl]) + (red[2][jl][cl] + red[3][jl][cl]);
            if (direct) {
                const int cc = blockIdx.x * kG2Cols + cl;
                if (cc < C) q.out[(size_t)j * q.o_sr + (size_t)cc * q.o_sc] = alpha * v;
            } else {
                tile[jfast ? cl * R + j : j * kG2Cols + cl] = v;
            }
        };
        if constexpr (PV) {                    // nj is 8 or 16; four LDS sums under way at a time: 0.3-0.5 us of 7 to 16
            for (int o = threadIdx.x; o < nj * kG2Cols; o += 4 * 64 * kG2Waves) {
#pragma unroll
                for (int u = 0; u < 4; ++u) write(o + u * 64 * kG2Waves);
            }
        } else {
            for (int o = threadIdx.x; o < nj * kG2Cols; o += 64 * kG2Waves) write(o);
        }
    }
}

// Adds the `splits` partial tiles of every strip in order and writes the scaled result through the caller's strides.
template <bool WIDE>            // R > 32
__global__ __launch_bounds__(256) void lora_grad_reduce_kernel(GradArgs ga, int R) {
    const GradProb& q = ga.p[blockIdx.y];
    const int total = q.col_blocks * R * kG2Cols;              // one split's tiles: [strip][j][column] or [strip][column][j]
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (q.splits <= 1 || t >= total) return;                   // a single split was written directly
    const float* __restrict__ part = q.part;
    float v = 0.f;
    int s = 0;
    for (; s + 8 <= q.splits; s += 8) {
        float u[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) u[i] = part[(size_t)(s + i) * total + t];
#pragma unroll
        for (int i = 0; i < 8; ++i) v += u[i];
    }
    for (; s < q.splits; ++s) v += part[(size_t)s * total + t];
    const int bx = t / (R * kG2Cols), o = t - bx * (R * kG2Cols);
    int j = o >> 7, cl = o & (kG2Cols - 1);
    if (WIDE && grad_jfast(q)) {
        cl = o / R;
        j = o - cl * R;
    }
    const int cc = bx * kG2Cols + cl;
    if (cc < q.C) q.out[(size_t)j * q.o_sr + (size_t)cc * q.o_sc] = q.alpha * q.drop.scale * v;
}

// keep[m, c] = 1 where dropout keeps element (m, c), else 0: the mask the kernels above regenerate, written out
// for callers (and tests) that need to see it.
__global__ __launch_bounds__(256) void dropout_keep_kernel(uint8_t* __restrict__ keep, int M, int C, DropArgs drop) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;              // one column pair per thread
    const long pairs = (long)M * (C / 2);
    if (i >= pairs) return;
    const int m = (int)(i / (C / 2)), pr = (int)(i - (long)m * (C / 2));
    const uint32_t w = drop_word(drop, drop_row_key(drop, (uint32_t)m), (uint32_t)pr);
    keep[(size_t)m * C + 2 * pr] = (w & 0x7FFFu) >= drop.thr15;
    keep[(size_t)m * C + 2 * pr + 1] = ((w >> 16) & 0x7FFFu) >= drop.thr15;
}

// 128-column strips; enough row splits for about two workgroups per CU over both problems of a pair (their partial
// tiles cost 2 * splits * R * C * 4 bytes of traffic); rows per workgroup a multiple of 128 (4 wavefronts x 32 rows).
// Above 32 adapter rows at most one workgroup per CU over two problems of this size: a second round costs more than the
// parallel rows give (512 rows, two gradients of 5120 features at rank 64: 320 workgroups 27 us, 160 of them 16), and wide
// strips then need no partial tiles at all (13824 features, 2048 rows: 45 -> 35 us).
struct GradPlan { int col_blocks, splits, rows_per_wg; };
inline GradPlan plan_grad(int M, int C, int R) {
    GradPlan g;
    g.col_blocks = (C + kG2Cols - 1) / kG2Cols;
    int splits = R > 32 ? 128 / g.col_blocks : (384 + g.col_blocks - 1) / g.col_blocks;
    if (splits > 64) splits = 64;
    if (splits < 1) splits = 1;
    const int unit = 32 * kG2Waves;
    g.rows_per_wg = ((M + splits - 1) / splits + unit - 1) / unit * unit;
    g.splits = (M + g.rows_per_wg - 1) / g.rows_per_wg;
    return g;
}

}  // namespace q4

template <int RB, int WL, bool F32, int RQ>
static void launch_down_kernel(const q4::DownArgs& da, int n, int M, int R, hipStream_t stream) {
    // rows of `in` per workgroup: 16 fill the MFMA operand, but with few rows that leaves compute units idle and
    // the kernel is bound by the latency of its single burst of loads, so smaller blocks spread it out
    int rows = 16;
    while (rows > 4 && (M + rows - 1) / rows * n < 256) rows >>= 1;
    hipLaunchKernelGGL((q4::lora_down_kernel<RB, WL, F32, RQ>), dim3((M + rows - 1) / rows, n), dim3(64 * q4::kDownWaves), 0,
                       stream, da, M, R, rows);
}

template <int WL, bool F32>
static void launch_down_rb(const q4::DownArgs& da, int n, int M, int R, hipStream_t stream) {
    switch ((R + 15) / 16) {
        case 1: launch_down_kernel<1, WL, F32, 0>(da, n, M, R, stream); break;
        case 2: launch_down_kernel<2, WL, F32, 0>(da, n, M, R, stream); break;
        case 3: launch_down_kernel<3, WL, F32, 0>(da, n, M, R, stream); break;
        default: launch_down_kernel<4, WL, F32, 0>(da, n, M, R, stream); break;
    }
}

template <int WL, bool F32>
static void launch_down_staged(const q4::DownArgs& da, int n, int M, int R, hipStream_t stream) {
    switch ((R + 3) / 4) {
        case 1: launch_down_kernel<1, WL, F32, 1>(da, n, M, R, stream); break;
        case 2: launch_down_kernel<1, WL, F32, 2>(da, n, M, R, stream); break;
        case 3: launch_down_kernel<1, WL, F32, 3>(da, n, M, R, stream); break;
        default: launch_down_kernel<1, WL, F32, 4>(da, n, M, R, stream); break;
    }
}

static q4::WLayout down_layout(const void* w, int w_sr, int w_sc, int w_is_f32, int R) {
    using namespace q4;
    const bool base16 = (reinterpret_cast<uintptr_t>(w) & 15u) == 0;
    const int vec = w_is_f32 ? 4 : 8;                       // elements per 16 bytes
    if (w_sc == 1 && base16 && w_sr % 4 == 0 && R <= 16) return kRowsT;
    if (w_sc == 1 && base16 && w_sr % vec == 0) return kRows;
    if (w_sr == 1 && base16 && w_sc % 4 == 0 && R % 4 == 0 && R <= 16 && w_sc >= R) return kCols;
    return kAny;
}

template <bool F32>
static void launch_down(q4::WLayout layout, const q4::DownArgs& da, int n, int M, int R, hipStream_t stream) {
    using namespace q4;
    switch (layout) {
        case kRowsT: launch_down_staged<kRowsT, F32>(da, n, M, R, stream); break;
        case kRows: launch_down_rb<kRows, F32>(da, n, M, R, stream); break;
        case kCols: launch_down_staged<kCols, F32>(da, n, M, R, stream); break;
        default: launch_down_rb<kAny, F32>(da, n, M, R, stream); break;
    }
}

// `n` products of M rows; neighbours of the same rank, type and layout of w share a launch.  drops[i] null: no dropout.
extern "C" int q4_launch_lora_down(const q4_lora_down_t* probs, const q4::DropArgs* const* drops, int n, int M, hipStream_t stream) {
    using namespace q4;
    for (int i = 0; i < n;) {
        const q4_lora_down_t& f = probs[i];
        const WLayout layout = down_layout(f.w, f.w_sr, f.w_sc, f.w_is_f32, f.R);
        DownArgs da;
        int k = 0;
        for (; i + k < n && k < kDownProbs; ++k) {
            const q4_lora_down_t& g = probs[i + k];
            if (g.R != f.R || g.w_is_f32 != f.w_is_f32 || down_layout(g.w, g.w_sr, g.w_sc, g.w_is_f32, g.R) != layout) break;
            da.p[k] = {reinterpret_cast<const half_t*>(g.in), g.w, reinterpret_cast<half_t*>(g.out), g.w_sr, g.w_sc, g.C,
                       drops[i + k] ? *drops[i + k] : DropArgs{0u, 0u, 0u, 1.0f}};
        }
        if (f.w_is_f32) launch_down<true>(layout, da, k, M, f.R, stream);
        else launch_down<false>(layout, da, k, M, f.R, stream);
        i += k;
    }
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

// One launch takes up to 16 rows, ranks 4, 8, 12 and 16, and matrices of one type read in whole vectors.  A single adapter above
// eight rows stays with the two launches, whose first spreads the rows: us, 4096 features at rank 8, two launches -> one: 5.9 -> 4.4
// at 1 row, 6.9 -> 6.0 at 8, 7.1 -> 7.8 at 16; 13824 features 13.7 -> 12.7 at 4, 13.9 -> 20.6 at 16 (two adapters 27.5 -> 20.8).
extern "C" int q4_lora_update_fits(const q4_lora_update_t* probs, int n, int M) {
    if (n < 1 || n > q4::kDownProbs || M > (n == 1 ? q4::kUpdRows / 2 : q4::kUpdRows)) return 0;
    for (int i = 0; i < n; ++i) {
        const q4_lora_update_t& g = probs[i];
        if (g.R != probs[0].R || g.a_is_f32 != probs[0].a_is_f32 || g.b_is_f32 != g.a_is_f32 || g.R % 4 != 0 || g.R > 16) return 0;
        if (down_layout(g.a, g.a_sr, g.a_sc, g.a_is_f32, g.R) != q4::kRowsT) return 0;
        if (g.b_sr != 1 || g.b_sn % 4 != 0 || (reinterpret_cast<uintptr_t>(g.b) & (g.b_is_f32 ? 15u : 7u)) != 0) return 0;
    }
    return 1;
}

template <bool F32>
static void launch_update(const q4::UpdArgs& ua, int R, const q4::half_t* x, int M, int K, dim3 grid, hipStream_t stream) {
    const dim3 block(64 * q4::kDownWaves);
    switch (R / 4) {
        case 1: hipLaunchKernelGGL((q4::lora_update_kernel<F32, 1>), grid, block, 0, stream, ua, x, M, K); break;
        case 2: hipLaunchKernelGGL((q4::lora_update_kernel<F32, 2>), grid, block, 0, stream, ua, x, M, K); break;
        case 3: hipLaunchKernelGGL((q4::lora_update_kernel<F32, 3>), grid, block, 0, stream, ua, x, M, K); break;
        default: hipLaunchKernelGGL((q4::lora_update_kernel<F32, 4>), grid, block, 0, stream, ua, x, M, K); break;
    }
}

extern "C" int q4_launch_lora_update(const q4_lora_update_t* probs, int n, const void* x, int M, int K, hipStream_t stream) {
    using namespace q4;
    UpdArgs ua;
    int gx = 1;
    for (int i = 0; i < n; ++i) {
        const q4_lora_update_t& g = probs[i];
        ua.p[i] = {g.a, g.b, reinterpret_cast<half_t*>(g.y), g.a_sr, g.b_sn, g.N, g.alpha};
        gx = std::max(gx, (g.N + kUpdCols - 1) / kUpdCols);
    }
    const half_t* xp = reinterpret_cast<const half_t*>(x);
    if (probs[0].a_is_f32) launch_update<true>(ua, probs[0].R, xp, M, K, dim3(gx, n), stream);
    else launch_update<false>(ua, probs[0].R, xp, M, K, dim3(gx, n), stream);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

extern "C" int q4_launch_lora_up(const void* xa, const void* w, int w_sn, int w_sr, int w_is_f32, void* y, float alpha,
                                 int M, int N, int R, hipStream_t stream) {
    using namespace q4;
    const half_t* xp = reinterpret_cast<const half_t*>(xa);
    half_t* yp = reinterpret_cast<half_t*>(y);
    const dim3 grid((N + kUpCols - 1) / kUpCols, (M + kUpRows - 1) / kUpRows), block(kUpCols);
    const bool vec = w_sr == 1 && R % 4 == 0 && w_sn % 4 == 0 && (reinterpret_cast<uintptr_t>(w) & (w_is_f32 ? 15u : 7u)) == 0;
    if (w_is_f32 && vec) hipLaunchKernelGGL((lora_up_kernel<true, true>), grid, block, 0, stream, xp, w, w_sn, w_sr, yp, alpha, M, N, R);
    else if (w_is_f32) hipLaunchKernelGGL((lora_up_kernel<true, false>), grid, block, 0, stream, xp, w, w_sn, w_sr, yp, alpha, M, N, R);
    else if (vec) hipLaunchKernelGGL((lora_up_kernel<false, true>), grid, block, 0, stream, xp, w, w_sn, w_sr, yp, alpha, M, N, R);
    else hipLaunchKernelGGL((lora_up_kernel<false, false>), grid, block, 0, stream, xp, w, w_sn, w_sr, yp, alpha, M, N, R);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

extern "C" size_t q4_lora_grad_workspace(int M, int C, int R) {
    const q4::GradPlan g = q4::plan_grad(M, C, R);
    return g.splits == 1 ? 0 : (size_t)g.splits * g.col_blocks * R * q4::kG2Cols * sizeof(float);
}

template <int RB>
static void launch_grad_rb(const q4::GradArgs& ga, bool any_drop, dim3 grid, int R, hipStream_t stream) {
    const dim3 block(64 * q4::kG2Waves);
    if (any_drop) hipLaunchKernelGGL((q4::lora_grad_kernel<true, RB>), grid, block, 0, stream, ga, R);
    else hipLaunchKernelGGL((q4::lora_grad_kernel<false, RB>), grid, block, 0, stream, ga, R);
}

static int launch_grad(const q4::GradArgs& ga, int nprob, int R, hipStream_t stream) {
    using namespace q4;
    int gx = 0, gy = 0, rx = 0;
    bool any_split = false, any_drop = false;
    for (int i = 0; i < nprob; ++i) {
        gx = ga.p[i].col_blocks > gx ? ga.p[i].col_blocks : gx;
        gy = ga.p[i].splits > gy ? ga.p[i].splits : gy;
        const int rb = (ga.p[i].col_blocks * R * kG2Cols + 255) / 256;
        rx = rb > rx ? rb : rx;
        any_split = any_split || ga.p[i].splits > 1;
        any_drop = any_drop || ga.p[i].drop.thr15 != 0;
    }
    const dim3 grid(gx, gy, nprob);
    switch ((R + 15) / 16) {
        case 1: launch_grad_rb<1>(ga, any_drop, grid, R, stream); break;
        case 2: launch_grad_rb<2>(ga, any_drop, grid, R, stream); break;
        case 3: launch_grad_rb<3>(ga, any_drop, grid, R, stream); break;
        default: launch_grad_rb<4>(ga, any_drop, grid, R, stream); break;
    }
    if (any_split && R > 32) hipLaunchKernelGGL(lora_grad_reduce_kernel<true>, dim3(rx, nprob), dim3(256), 0, stream, ga, R);
    else if (any_split) hipLaunchKernelGGL(lora_grad_reduce_kernel<false>, dim3(rx, nprob), dim3(256), 0, stream, ga, R);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

extern "C" int q4_launch_dropout_keep(uint8_t* keep, int M, int C, const q4::DropArgs* drop, hipStream_t stream) {
    const long pairs = (long)M * (C / 2);
    hipLaunchKernelGGL(q4::dropout_keep_kernel, dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, stream, keep, M, C, *drop);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

// Up to kGradProbs gradients with the same M and R in one launch (plus one launch for their reductions); the workspace holds
// the partial tiles of one problem after the other.
extern "C" int q4_launch_lora_grad(const q4_lora_grad_t* probs, const q4::DropArgs* const* drops, int n, int M, int R,
                                   void* workspace, hipStream_t stream) {
    using namespace q4;
    GradArgs ga;
    float* ws = reinterpret_cast<float*>(workspace);
    for (int i = 0; i < n; ++i) {
        const q4_lora_grad_t& p = probs[i];
        const GradPlan g = plan_grad(M, p.C, R);
        ga.p[i] = {reinterpret_cast<const half_t*>(p.p), reinterpret_cast<const half_t*>(p.in), p.out, ws, p.o_sr, p.o_sc, p.C,
                   g.col_blocks, g.splits, g.rows_per_wg, p.alpha, drops[i] ? *drops[i] : DropArgs{0u, 0u, 0u, 1.0f}};
        if (ws) ws += q4_lora_grad_workspace(M, p.C, R) / sizeof(float);
    }
    ga.M = M;
    return launch_grad(ga, n, R, stream);
}
