// Weight streaming for 1..16 activation rows over chunks of 128 reduction rows: the loop of q4_gemv.hip's product and of
// q4_mlp.hip's gate / up / activation launch.  Four wavefronts a workgroup, about one workgroup per compute unit; wavefront
// w walks the chunks w, w + 4, ... of its workgroup's share of the reduction on one strip of 64 columns of NL layers.
//
// What bounds it and why it is laid out this way.  The packed words have to stream from HBM once; what a launch adds to
// that is fixed latencies, the finish of every workgroup (an LDS sum, one atomic per output and split) and, from a few rows
// on, the activations, which every strip reads again.  One burst of a single chunk per wavefront, eight wavefronts a workgroup
// with the activations straight into the operand registers, touched 16 cache lines per activation load and summed twice
// as many wavefronts per KB of weights.  Here the next chunk's words and activations are on their way while one is multiplied,
// and the activations come row-contiguous into the wavefront's own LDS tile by the loads themselves (buffer_load ... lds).
// us at 2 / 4 / 16 rows, launches replayed as a graph over cold weights, burst -> stream: 4096 -> 4096 4.8 / 5.1 / 6.3 ->
// 4.7 / 4.8 / 6.2, 11008 -> 4096 7.5 / 7.9 / 10.1 -> 7.6 / 7.8 / 9.5, q|k|v of 4096 features 8.2 / 8.5 / 10.3 -> 8.1 / 8.3 / 10.2, in groups
// of 64 rows at 4 / 16 rows 9.1 / 10.9 -> 9.1 / 11.3, of 32 rows 11.3 / 13.9 -> 10.4 / 12.6, q|k|v of 5120 features 11.1 / 12.1 / 15.7 ->
// 11.0 / 11.3 / 12.9, 5120 -> 13824 10.2 / 10.9 / 14.9 -> 10.3 / 10.7 / 12.2; one row and small groups: plan_stream_takes.  Eight wavefronts of half
// the length time the same, words two chunks ahead 0.3 us more, both chunks requested at once 0.2 us more, rows below four skipped by
// a uniform branch in the scaling 0.1 to 0.6 us more.
#pragma once
#include "q4_gemv_core.hpp"
#include <type_traits>

namespace q4 {

constexpr int kStreamTile = 16 * 128;                 // halves of one activation tile: 16 rows of one chunk
constexpr int kStreamLds = kStreamWaves * 2 * kStreamTile * 2;   // bytes: two tiles per wavefront

// Chunk i lies in group floor(i / (groupsize / 128)) = mulhi(2 i, inv), exact while i * (groupsize / 128) < 2^31.
inline uint32_t stream_group_inv(int groupsize) {
    const unsigned per = groupsize >= 128 ? (unsigned)groupsize / 128u : 1u;
    return (uint32_t)(((1ull << 31) + per - 1) / per);
}

// The reduction goes in blocks of 8 chunks, two neighbouring chunks per wavefront; `flush(b)` follows block b of the nb blocks
// from `block0` on with the sums of this wavefront's two chunks in yacc[layer][j][r]: row 4 * (lane / 16) + r, column
// n0 + 4 * (lane % 16) + j.  Chunks from `end` on are left out.  The layers share x, M, K, N and the group size.
// TEAMS: teams of four wavefronts that take the blocks in turn, team t the blocks t, t + TEAMS, ... of the nb.
// NG groups per chunk (1, 2, 4; 1: groupsize % 128 == 0).  `tile`: this wavefront's two activation tiles in LDS.  ONE: a single
// block, in straight line and with nothing requested past it.
// The operands are built as in gemv_core: codes as 1024 + q or 64 + q, and per group (sum x*(offset + q) - sum x*offset) -
// (z + 1) * sum x in the same order.
template <int NL, int NG, bool ONE, int TEAMS = 1, typename Flush>
__device__ __forceinline__ void stream_blocks(const GemvArgs* const (&l)[NL], uint32_t inv, int n0, int block0, int nb, int end,
                                              half_t* tile, float4_t (&yacc)[NL][4], Flush&& flush) {
    typedef __attribute__((address_space(3))) void lds_void;
    constexpr int kFar = 0x70000000;                  // beyond every buffer: zeros, without traffic
    constexpr int GS = 4 / NG;                        // steps of 32 rows per group
    constexpr int kBehind = NL * (4 + 2 * NG);        // loads requested behind a chunk's activations (words, scales, zeros)
    const int lane = threadIdx.x & 63;
    const int kk = lane >> 4, c = lane & 15;
    const GemvArgs& a = *l[0];
    const int M = a.M, K = a.K, N = a.N, ncol8 = N >> 3;
    rsrc_t rw[NL], rs[NL], rz[NL];
#pragma unroll
    for (int q = 0; q < NL; ++q) {
        rw[q] = make_rsrc(l[q]->qweight, (unsigned)((size_t)(K >> 3) * N * 4));
        rs[q] = make_rsrc(l[q]->scales, (unsigned)((size_t)a.G * N * 2));
        rz[q] = make_rsrc(l[q]->qzeros, (unsigned)((size_t)a.G * ncol8 * 4));
    }
    const rsrc_t rx = make_rsrc(a.x, (unsigned)M * (unsigned)K * 2u);          // rows past M read as zero
    const int vw = (kk * N + n0 + 4 * c) * 4, vs = (n0 + 4 * c) * 2, vz = ((n0 >> 3) + (c >> 1)) * 4;
    // lane (kk, c) of load t fetches unit c ^ row of row 4t + kk and lands at unit c: unit q of row r sits at q ^ r, so the
    // column-wise reads below are conflict-free
    int vx[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) vx[t] = ((4 * t + kk) * K + 8 * (c ^ (4 * t + kk))) * 2;

    uint4_t w[2][NL][4];
    uint2_t sv[2][NL][NG];
    uint32_t zv[2][NL][NG];
    auto load_x = [&](int i, int buf) {
        const int off = i < end ? i << 8 : kFar;
#pragma unroll
        for (int t = 0; t < 4; ++t)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void*)(tile + buf * kStreamTile + 512 * t), 16, vx[t], off, 0, 0);
    };
    auto load_w = [&](auto slot, int i) {
        constexpr int S = decltype(slot)::value;
        const int g = i < end ? (NG == 1 ? (int)__umulhi((uint32_t)i * 2u, inv) : i * NG) : 0, far = i < end ? 0 : kFar;
#pragma unroll
        for (int q = 0; q < NL; ++q)
#pragma unroll
            for (int e = 0; e < NG; ++e) {
                sv[S][q][e] = buf_load64(rs[q], vs, far + (g + e) * N * 2);
                zv[S][q][e] = buf_load32(rz[q], vz, far + (g + e) * ncol8 * 4);
            }
        // the order in which they are needed, which is the order in which they return: the scheduler would put a zero last
        __builtin_amdgcn_sched_barrier(0);
        const int row = i < end ? i << 4 : 0;         // packed rows; read exactly once per product: streaming loads
#pragma unroll
        for (int q = 0; q < NL; ++q)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                w[S][q][t] = buf_load128_stream(rw[q], vw, far + (row + 4 * t) * N * 4);
                __builtin_amdgcn_sched_barrier(0);
            }
    };
    const half8_t offs = make_half8(0x64006400u, 0x54005400u, 0x64006400u, 0x54005400u);
    const half8_t ones = make_half8(0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u);
    // masks in scalar, magic numbers in vector registers (opaque): one and-or instruction instead of an AND and an OR
    uint32_t m_lo = 0x000F000Fu, m_hi = 0x00F000F0u, g_lo = 0x64006400u, g_hi = 0x54005400u;
    asm volatile("" : "+s"(m_lo), "+s"(m_hi));
    asm volatile("" : "+v"(g_lo), "+v"(g_hi));

    // multiplies a chunk (words and activations in `slot`), chunk `next` requested on the way; without a branch
    // around the requests (past the end: no traffic), or every wait below would have to assume the shorter queue
    auto step = [&](auto slot, auto more, int next) {              // slot 0: the first chunk of a block
        constexpr int S = decltype(slot)::value;
        // the chunk's activations have landed: of everything requested, only what was asked for behind them may be missing
        __builtin_amdgcn_s_waitcnt(0x0F70 | (kBehind & 15) | ((kBehind >> 4) << 14));
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        half8_t av[4];                                // A operands in nibble order: (e0,e4)(e1,e5)(e2,e6)(e3,e7)
        const uint4_t* st = reinterpret_cast<const uint4_t*>(tile + S * kStreamTile);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint4_t u = st[c * 16 + ((4 * t + kk) ^ c)];
            av[t] = make_half8(__builtin_amdgcn_perm(u.z, u.x, 0x05040100u), __builtin_amdgcn_perm(u.z, u.x, 0x07060302u),
                               __builtin_amdgcn_perm(u.w, u.y, 0x05040100u), __builtin_amdgcn_perm(u.w, u.y, 0x07060302u));
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(more)::value) {
            load_x(next, S ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            load_w(std::integral_constant<int, S ^ 1>{}, next);
            __builtin_amdgcn_sched_barrier(0);
        }
        float4_t acco[NG], accx[NG];
#pragma unroll
        for (int e = 0; e < NG; ++e) {
            acco[e] = float4_t{0.f, 0.f, 0.f, 0.f};
            accx[e] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = e * GS; t < (e + 1) * GS; ++t) {
                acco[e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[t], offs, acco[e], 0, 0, 0);
                accx[e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[t], ones, accx[e], 0, 0, 0);
            }
        }
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            float4_t p[4];                            // the chunk's share of the output
#pragma unroll
            for (int e = 0; e < NG; ++e) {
                float4_t acc[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int t = e * GS; t < (e + 1) * GS; ++t) {
                    const uint32_t ww[4] = {w[S][q][t].x, w[S][q][t].y, w[S][q][t].z, w[S][q][t].w};
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t hi = ww[j] >> 8;
                        const half8_t bv = make_half8((ww[j] & m_lo) | g_lo, (ww[j] & m_hi) | g_hi, (hi & m_lo) | g_lo, (hi & m_hi) | g_hi);
                        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[t], bv, acc[j], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);     // consume the words in the order they return
                }
                const half2_t s01 = as_half2(sv[S][q][e].x), s23 = as_half2(sv[S][q][e].y);
                const float sf[4] = {(float)s01[0], (float)s01[1], (float)s23[0], (float)s23[1]};
                const uint32_t zw = zv[S][q][e] >> ((c & 1) * 16);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float zf = (float)(((zw >> (4 * j)) & 0xFu) + 1u);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float v = sf[j] * ((acc[j][r] - acco[e][r]) - zf * accx[e][r]);
                        p[j][r] = e == 0 ? v : p[j][r] + v;
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                yacc[q][j] = S == 0 ? p[j] : yacc[q][j] + p[j];
                asm volatile("" : "+v"(yacc[q][j]));       // added here: left to itself the compiler keeps every chunk's sums to the end
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), team = TEAMS > 1 ? wave / kStreamWaves : 0;
    int i = ((block0 + team) * kStreamWaves + wave % kStreamWaves) * 2;
    load_x(i, 0);
    __builtin_amdgcn_sched_barrier(0);
    load_w(S0{}, i);
    if constexpr (ONE) {
        step(S0{}, std::true_type{}, i + 1);
        step(S1{}, std::false_type{}, 0);
        flush(0);
        return;
    }
    // one copy of the two steps: with copies of their own for the last ones a launch took 0.2 to 1.2 us longer
    for (int b = team; b < nb; b += TEAMS) {
        step(S0{}, std::true_type{}, i + 1);
        i += 2 * kStreamWaves * TEAMS;
        step(S1{}, std::true_type{}, i);
        flush(b);
    }
    // what was requested past the end wrote zeros into the tiles: landed before their LDS is used again
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace q4
