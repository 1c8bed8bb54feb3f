// Launch plans of the tiled GEMMs: which tiles, how many shares of the reduction, which columns go to a second launch.
// Host arithmetic on the sizes alone, without HIP, so that it also compiles by itself for the CPU tests.
//
// The thresholds and the estimate below were fitted to kernels with both operands in LDS, which the tiles of
// q4_gemm_wide.hip have replaced since on sequential groups (all launches of 256 x 256, forward ones of 256 x 128 as 128 x 256); their
// figures are of that time where they do not say otherwise.  Since then forward takes 5 to 10 % less from 250 rows on, grad-input 1 to
// 5 %, no shape measured more; 256-row tiles are still counted where forward launches run ceil(M / 128) rows of 128 x 256 ones.
#pragma once
#include <stddef.h>

namespace q4 {

constexpr int BN = 128, BK = 64;         // columns of the narrow tiles, depth of a reduction step
constexpr int kGemmGroup = 4;            // most layers of one grouped launch

struct GemmPlan {
    int cfg, splits;
    int tail_cols, tail_splits;      // cfg 2, 3: 128-column tiles of the second launch (0: none), its reduction split
};

// More 256 x 256 tiles than whole rounds of the CUs: the wide tiles of the whole rounds run as they are, and the columns
// left over go to a second launch of 256 x 128 tiles that is one round at most, its reduction split when even that
// leaves CUs idle.  A full round of wide tiles takes 1.75-1.85 us per reduction step (1.65-1.7 in q4_gemm_wide.hip), one of
// narrow tiles 0.9-1.05 (0.95 forward, 1.03 grad-input now), so the
// remainder costs at most 0.6 of the round of wide tiles, or half of the two narrow ones, that it would cost otherwise:
// 2048 x (4096 -> 11008), 344 tiles: three rounds of narrow tiles 186 us, 118 + 57 us; grad-input of 4096 x
// (5120 -> 13824), 864 tiles: four rounds of wide tiles 561 us, 447 + 79 us.
// Taken for remainders of 1/8 to 1/2 of a round: below that the narrow tiles with their own remainder launch lose
// little, above it the remainder does not fit a round of narrow tiles.  Up to 128 rows the 128-row tiles stay: 100 rows
// of (2048 -> 81920), 320 wide tiles half empty, 54 us against 74.
struct WideTail { int tail_cols, tail_splits; };     // 128-column tiles; 0: does not apply
inline WideTail wide_tail(int M, int nsteps, int nout, bool may_split, size_t workspace_bytes) {
    WideTail w{0, 1};
    const int nr = (M + 255) / 256, nc = nout / 256;
    const long t = (long)nc * nr;
    if (nout % 256 != 0 || t <= 256 || M <= 128) return w;
    const int main_cols = (int)((t / 256) * 256 / nr);
    const long left = (long)(nc - main_cols) * nr;
    if (main_cols < 1 || left < 32 || left > 128) return w;
    int s = (int)(256 / (2 * left));
    while (s > 1 && (!may_split || nsteps < 8 * s ||
                     (size_t)s * (size_t)M * (size_t)(nc - main_cols) * 256 * sizeof(float) > workspace_bytes)) --s;
    w.tail_cols = 2 * (nc - main_cols);
    w.tail_splits = s;
    return w;
}

// Launch plan shared by q4_launch_gemm and q4_gemm_plan_workspace.  Few output tiles (small M) leave most CUs
// idle while each tile walks the whole reduction: the reduction is then split over gridDim.z workgroups that
// write fp32 partial tiles, about 1.5 workgroups per CU in total.
// `indexed`: the kernels that look every row's group up (groups of 32, g_idx).  On them wide tiles of whole rounds with a
// remainder launch are slower than the narrow tiles on every shape measured (30 shapes of groups of 32): forward by 37..53 %
// (1969 x (4352 -> 9472): 420 against 290 us), grad-input by 11..16 % (2605 x (8704 -> 4352): 318 against 279 us, where the
// wide kernel also spills 80 bytes a lane).
// `paired`: the launches of 256 x 128 tiles run as 128 x 256 ones where their columns come in whole pairs (forward, sequential groups).
inline GemmPlan plan_gemm(int M, int red, int nout, size_t workspace_bytes, bool indexed, bool paired = false) {
    GemmPlan p;
    p.tail_cols = 0; p.tail_splits = 1;
    const int nsteps = red / BK;
    // Tiles of 256 rows (8 wavefronts, one dequantized slab of W for 256 activation rows) do about twice the work per
    // CU and unit of time that 128-row tiles do, so they are used from 129 rows on: as they are when there are more
    // than 128 of them (even 130 of them on 256 CUs beat 260 tiles of 128 rows), otherwise with the reduction split
    // floor(256 / tiles) ways so that every CU gets one workgroup (never more than 256 workgroups: a second, nearly
    // empty round costs more than the split gains).
    const long t256 = (long)(nout / BN) * ((M + 255) / 256);
    int splits = 1;
    // 256 x 256 tiles from 144 of them on (a workgroup does the work of two 256 x 128 ones in about 1.7 times their
    // time), unless their last round would leave more than a fifth of the CUs' slots empty where the narrower tiles
    // fill theirs better: 3072 x (4096 -> 11008) has 516 wide tiles = 3 rounds for 2.02 rounds of work and stays
    // with the narrow ones (270 against 294 us), 4096 rows have 688 (313 against 356 us).
    const long twide = (nout % 256 == 0) ? (long)(nout / 256) * ((M + 255) / 256) : 0;
    const WideTail wt = indexed ? WideTail{0, 1} : wide_tail(M, nsteps, nout, true, workspace_bytes);
    if (wt.tail_cols > 0) {
        p.cfg = 3; p.splits = 1;
        p.tail_cols = wt.tail_cols;
        p.tail_splits = wt.tail_splits;
        return p;
    }
    if (twide >= 144 &&
        (twide <= 256 || 5 * twide >= 4 * 256 * ((twide + 255) / 256))) {
        p.cfg = 3; p.splits = 1;
        return p;
    }
    if (t256 > 128 && M > 128) {
        p.cfg = 2;
        // More tiles than CUs and a last round that fills at most half of them: the column tiles of that
        // remainder run as a second launch with the reduction split so that it takes a fraction of a round.
        const int nr = (M + 255) / 256;
        const long rem = t256 % 256;
        if (t256 > 256 && rem > 0) {
            const int tcols = (int)((rem + nr - 1) / nr);
            const long tt = (long)tcols * nr;
            int ts = tt <= 128 ? (int)(256 / tt) : 1;
            if (ts > 8) ts = 8;
            while (ts > 1 && nsteps < 8 * ts) --ts;
            if (ts > 1 && (size_t)ts * (size_t)M * (size_t)tcols * BN * sizeof(float) <= workspace_bytes) {
                p.tail_cols = tcols;
                p.tail_splits = ts;
                // An odd remainder of an even width takes one more column, in as many shares as the same scratch holds, so that
                // both launches are whole pairs; not where only one share would be left.  us, odd / even: 640 x (4096 -> 11008)
                // 76.4 / 71.9, 1536 rows 141.7 / 136.6, 3072 rows 270 / 258, 3328 x (13824 -> 5120) 460 / 434, 768 x (4096 -> 11008)
                // 79.0 / 79.1; one share: 520 x (1024 -> 11008) 31.1 / 32.1.
                const int fewer = ts * tcols / (tcols + 1);
                if (paired && (nout / BN) % 2 == 0 && tcols % 2 == 1 && fewer > 1) {
                    p.tail_cols = tcols + 1;
                    p.tail_splits = fewer;
                }
            }
        }
    } else if (t256 <= 128 && M > 128 && nsteps >= 8 * (int)(256 / t256) &&
               (size_t)(256 / t256 > 8 ? 8 : 256 / t256) * (size_t)M * (size_t)nout * sizeof(float) <= workspace_bytes) {
        p.cfg = 2;                                             // only with room for all its partial tiles
        splits = (int)(256 / t256);
        if (splits > 8) splits = 8;
    } else {
        p.cfg = 0;
        const long tiles = (long)(nout / BN) * ((M + 127) / 128);
        if (tiles < 192) {
            splits = (int)((384 + tiles - 1) / tiles);
            if (splits > 8) splits = 8;                        // measured: more splits only add prologues and partial tiles
            if (splits > nsteps / 4) splits = nsteps / 4;      // at least four steps per workgroup
        }
    }
    while (splits > 1 && (size_t)splits * (size_t)M * (size_t)nout * sizeof(float) > workspace_bytes) --splits;
    p.splits = splits < 1 ? 1 : splits;
    return p;
}

// fp32 partial sums of a plan
inline size_t plan_workspace(const GemmPlan& p, int M, int nout) {
    if (p.tail_cols > 0)
        return p.tail_splits > 1 ? (size_t)p.tail_splits * (size_t)M * (size_t)p.tail_cols * BN * sizeof(float) : 0;
    return p.splits > 1 ? (size_t)p.splits * (size_t)M * (size_t)nout * sizeof(float) : 0;
}

// cfg as in launch_gemm_cfg (2: 256 x 128 tiles, 3: 256 x 256 tiles; -1: not applicable), the split of the reduction, and
// the 128-column tiles of the second launch (0: none) with the split of its reduction.
struct GroupPlan { int cfg, splits, tail_cols, tail_splits; };

// Forward: one tile of one layer per workgroup, no split, so the launch needs enough tiles by itself: from 96 tiles of
// 256 x 128 on (q|k|v of 4096 features at 129..256 rows).  Forward + grad-input of 200 rows apart / grouped, us: 96 tiles
// 110 / 92 (with adapters on q and v 143 / 101), 120 tiles of 5120 features 165 / 115.  Below the line, 90 tiles of 3840
// features 124 / 88 and 48 of 2048 63 / 57: the line could lie lower for training.
// Grad-input: one reduction over all layers' columns.  Of the tilings, splits and remainder launches the one with the
// shortest estimate in us: the rounds of the CUs, each as long as a workgroup's steps (a round that leaves CUs idle runs up
// to a fifth faster) plus its prologue and epilogue, a second launch, and the sum of the partial tiles where a reduction is
// split.  Against every plan measured on 130 shapes (2..4 layers, 129..4096 rows, 2048..13824 features) the choice is
// 0.2 % slower than the best on average and 3 % at most; splits of one round alone and remainders of wide tiles alone were
// 4.9 % and up to 44 % slower (1006 rows, three layers 8832 -> 9600, 276 narrow tiles: 736 -> 553 us).
inline GroupPlan plan_gemm_group(int fwd, int n, int M, int K, const int* N) {
    GroupPlan p{-1, 1, 0, 1};
    if (n < 2 || n > kGemmGroup || M <= 128) return p;
    const int nr = (M + 255) / 256;
    if (fwd) {
        long tot = 0;
        bool all256 = true;
        for (int i = 0; i < n; ++i) { tot += N[i]; all256 = all256 && N[i] % 256 == 0; }
        const long twide = all256 ? (tot / 256) * nr : 0, t256 = (tot / BN) * nr;
        const WideTail wt = all256 && tot < (1l << 30) ? wide_tail(M, K / BK, (int)tot, false, 0) : WideTail{0, 1};
        if (wt.tail_cols > 0) { p.cfg = 3; p.tail_cols = wt.tail_cols; }
        else if (twide >= 144 && (twide <= 256 || 5 * twide >= 4 * 256 * ((twide + 255) / 256))) p.cfg = 3;
        else if (t256 >= 96) p.cfg = 2;
        return p;
    }
    constexpr double kWide = 1.6, kNarrow = 1.0, kEnds = 5.0, kIdle = 0.8, kLaunch = 3.0, kBytesPerUs = 4.5e6;
    long nsteps = 0;
    for (int i = 0; i < n; ++i) nsteps += N[i] / BK;
    auto tiles_us = [&](int cfg, long tiles, int s) {
        const double steps = (double)((nsteps + s - 1) / s) * (cfg == 3 ? kWide : kNarrow);
        const long last = tiles * s % 256;
        return (double)(tiles * s / 256) * (steps + kEnds) + (last ? steps * (kIdle + (1.0 - kIdle) * last / 256.0) + kEnds : 0.0);
    };
    auto sum_us = [&](int s, long cols) { return s > 1 ? kLaunch + 8.0 * s * M * cols / kBytesPerUs : 0.0; };
    auto worth = [&](long tiles, int s) { return s == 1 || (tiles * s <= 512 && nsteps >= 8 * s); };
    double best = 0.0;
    auto offer = [&](double us, GroupPlan q) { if (p.cfg < 0 || us < best) { best = us; p = q; } };
    for (int cfg = 3; cfg >= 2; --cfg) {
        const int tw = cfg == 3 ? 256 : BN;
        if (K % tw != 0) continue;
        const long t = (long)(K / tw) * nr;
        for (int s = 1; s <= 8 && worth(t, s); ++s) offer(tiles_us(cfg, t, s) + sum_us(s, K), GroupPlan{cfg, s, 0, 1});
        const int main_cols = (int)(t / 256 * 256 / nr), tail = (K / tw - main_cols) * (tw / BN);
        if (main_cols < 1 || tail < 1) continue;
        for (int s = 1; s <= 8 && worth((long)tail * nr, s); ++s)
            offer(tiles_us(cfg, (long)main_cols * nr, 1) + kLaunch + tiles_us(2, (long)tail * nr, s) + sum_us(s, (long)tail * BN),
                  GroupPlan{cfg, 1, tail, s});
    }
    return p;
}
inline size_t group_workspace(const GroupPlan& p, int M, int K) {
    const size_t main = p.splits > 1 ? (size_t)p.splits * (size_t)M * (size_t)K * sizeof(float) : 0;
    const size_t tail = p.tail_cols > 0 && p.tail_splits > 1
        ? (size_t)p.tail_splits * (size_t)M * (size_t)p.tail_cols * BN * sizeof(float) : 0;
    return main > tail ? main : tail;
}

}  // namespace q4
