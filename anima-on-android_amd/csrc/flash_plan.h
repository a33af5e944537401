// Launch plans of the D == 128 flash kernels: which query tiles run whole and
// whose keys are shared out over several workgroups, and how.  Host code without
// HIP, so that a CPU test can ask for the shape of a call.
#pragma once

#include "flash_deal.h"

#include <cstddef>
#include <cstdint>

namespace anima_hip {

constexpr int kFlashD = 128;      // head dim
constexpr int kFlashKeys = 64;    // keys per tile of the flash kernels
constexpr int kFlashRows8 = 256;  // query rows of an 8-wave workgroup
constexpr size_t kPairBytes = 2 * sizeof(float);  // (max, sum) of a partial row
constexpr size_t kFlashSlotBytes = size_t(kFlashRows8) * (kFlashD * sizeof(float) + kPairBytes);

inline int64_t flash_ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline size_t flash_round_up256(size_t n) { return (n + 255) / 256 * 256; }

// Launch shape of the D == 128 flash kernels: T = B*H*ceil(S_q/256) query
// tiles of 8-wave workgroups, or twice as many of 4 waves, over n key tiles of
// 64 keys, on 256 CUs that hold one workgroup each.  Five shapes:
//   whole     8-wave workgroups, one query tile each;
//   small     4-wave workgroups, one query tile each (T < 256);
//   split     4-wave workgroups, the key range of every query tile split over
//             `splits` of them ("split-KV"): split s takes key tiles
//             [s*tiles, (s+1)*tiles);
//   balanced  the largest multiple of 256 query tiles whole, and the key tiles
//             of the `ntail` others as one list dealt out evenly, `u` to each
//             of the last workgroups (T = 288 over 36 key tiles: 36 + 5 tiles
//             a CU, where a second round of whole query tiles takes 36 + 36);
//   keys      (bf16 MFMA) 8-wave workgroups of 64 query rows whose waves share
//             the keys among them (flash_keys.hip): at most 256 of them.
// A workgroup that sees part of a query tile's keys writes its output
// normalised by its own row sum, plus that row's (max, sum), to scratch, and
// flash_combine merges the parts into O.
struct FlashPlan {
    bool keys = false;    // the keys shape
    int waves = 8;
    int splits = 1;
    int tiles = 1 << 30;  // key tiles per split
    int full = 0;         // balanced: query tiles run whole
    int ntail = 0;        // balanced: query tiles dealt out
    int nk = 0;           // balanced: key tiles of a query tile
    int u = 0;            // balanced: key tiles per workgroup (0: another shape)
    size_t bytes = 0;     // scratch for the partials (0 when every tile runs whole)
};
// What a kernel takes per 64-key tile (us) in a 4-wave and in an 8-wave
// workgroup when every CU holds one, measured on MI355X (4-wave: 32 heads x
// 256 queries, unsplit grids over 4 and 8 key tiles; 8-wave: 32 heads x 4096
// queries and keys).  The bf16-MFMA kernels are bound by power: an 8-wave
// round of at most about 0.7 of the CUs clocks higher, down to `part` of w8
// (x3, T = 288 .. 800: 0.66 .. 0.76 of the full rounds' time per tile); the
// f32 MFMA runs at full clock either way.
// The keys shape: `round` for every 64 KiB of K that its four key groups take
// together (keys_round of them), and `merge` once, both against what a 4-wave
// workgroup spends beside its tiles (256 and 1024 queries and keys, 16 heads;
// 0: the mode has no such kernel).
// What split and balanced grids cost beside their tiles (every part loads its
// query tile and writes f32 partials, which the combine pass reads back): a
// fixed part, and a part for every MB of partials.  These four and the f32x3 w4
// are fitted to whole calls in every shape, 5, 16 and 32 heads, 1 to 2048 queries
// and 65 to 4096 keys.  With 13 a split and 27 a balanced grid in every mode, f32x3
// took the keys shape for 64 queries on 512 keys of 16 heads (31.4 us; split
// 27.6), and f32 4-wave workgroups for 257 on 257 of 32 (59.1; split 51.4).  Still
// off, at most: f32x3 keys for 128 to 256 queries on 512 keys of 32 heads (37.4
// against 33.2 for split, which loses 31.9 to 34.4 with the same grid of 16 heads).
struct FlashTimes {
    float w4, w8, part, merge, round;
    int keys_round;
    float split, split_mb, balance, balance_mb;
};
constexpr FlashTimes kTimesF32{9.1f, 15.7f, 1.0f, 0.0f, 0.0f, 0, 7.0f, 0.3f, 3.0f, 0.5f},
    kTimesBF16{1.3f, 1.9f, 0.7f, 1.5f, 2.8f, 256, 13.0f, 0.0f, 27.0f, 0.0f},
    kTimesX3{2.7f, 4.6f, 0.7f, 1.0f, 3.2f, 128, 10.0f, 0.1f, 27.0f, 0.0f};
// A balanced grid behind whole query tiles (25 to 31 us at T = 288, every mode).
constexpr float kBalanceTailUs = 27.0f;
// Scratch a flash launch may use, 16-byte aligned; either may be null.
struct FlashScratch {
    void *part = nullptr;
    size_t part_bytes = 0;
    void *balance = nullptr;
    size_t balance_bytes = 0;
    bool keys = false;  // the keys shape may run (the caller needs no other shape's bits)
    // What it saves (us) because it alone takes the query rows raw: a row pass
    // of its own before the kernel.
    float keys_saves = 0.0f;
};

// The split shape, which every mode's scratch must hold: 4-wave workgroups,
// the key range over ~256 of them.
inline FlashPlan split_plan(int64_t BH, int S_q, int S_kv, int D)
{
    FlashPlan pl;
    if (D != kFlashD || BH <= 0 || S_q <= 0 ||
        BH * flash_ceil_div(S_q, kFlashRows8) >= kFlashTargetBlocks)
        return pl;
    pl.waves = 4;
    const int64_t units = BH * flash_ceil_div(S_q, 128);
    const int64_t ntiles = flash_ceil_div(S_kv, kFlashKeys);
    const int64_t want = flash_ceil_div(kFlashTargetBlocks, units);
    if (want < 2 || ntiles < 2)
        return pl;
    const int64_t tiles = flash_ceil_div(ntiles, std::min(want, ntiles));
    const int64_t splits = flash_ceil_div(ntiles, tiles);
    if (splits < 2)
        return pl;
    pl.splits = int(splits);
    pl.tiles = int(tiles);
    const size_t rows = size_t(splits) * size_t(BH) * size_t(S_q);
    pl.bytes = flash_round_up256(rows * kFlashD * sizeof(float)) + rows * kPairBytes;
    return pl;
}

// The longest series of key tiles on a CU of a split grid: `tiles` a round of
// workgroups.  One more round is as short as the last split, where each engine's
// (8 CUs) extra workgroups are fewer than its workgroups of that split, which end
// first (T4 = 96 on 5 key tiles, three splits of 2, 2 and 1, f32: 3 tiles' time).
inline double split_tiles(const FlashPlan &sp, int64_t T4, int64_t n, bool causal)
{
    constexpr int64_t kEngines = 32;
    // Causal: a split beyond its queries ends at once, about (splits - 1) / 2 of them
    // (7 heads of 2500, f32, two splits: call 1359 us, 4-wave workgroups 1450).
    const int64_t blocks = causal ? T4 * (sp.splits + 1) / 2 : T4 * sp.splits;
    const int64_t extra = blocks - kFlashTargetBlocks;
    const int64_t whole = flash_ceil_div(blocks, kFlashTargetBlocks) * sp.tiles;
    if (extra <= 0 || flash_ceil_div(extra, kEngines) >= 8 / sp.splits)
        return double(whole);
    return double(std::min(whole, n - int64_t(sp.splits - 2) * sp.tiles));
}

// The balanced shape; u == 0 where the query tiles come out even, or where a
// share would be a whole tile anyway.
inline FlashPlan balanced_plan(int64_t BH, int S_q, int S_kv, int D)
{
    FlashPlan pl;
    if (D != kFlashD || BH <= 0 || S_q <= 0 || S_kv <= 0)
        return pl;
    const int64_t T = BH * flash_ceil_div(S_q, kFlashRows8), nk = flash_ceil_div(S_kv, kFlashKeys);
    const int64_t tail = T % kFlashTargetBlocks;
    if (tail == 0 || T > INT32_MAX / 2 || nk > INT32_MAX / kFlashTargetBlocks)
        return pl;
    const int64_t u = flash_ceil_div(tail * nk, kFlashTargetBlocks);
    if (u >= nk)
        return pl;
    pl.full = int(T - tail);
    pl.ntail = int(tail);
    pl.nk = int(nk);
    pl.u = int(u);
    pl.bytes = size_t(tail + flash_ceil_div(tail * nk, u) - 1) * kFlashSlotBytes;
    return pl;
}

// The shape with the least predicted time among those whose partials fit:
// s.part_bytes for `split`, s.balance_bytes for `balanced` (causal calls, whose
// tiles differ in length, are not balanced, and `keys` has no mask).
inline FlashPlan flash_plan(int64_t BH, int S_q, int S_kv, int D, const FlashTimes &t,
                            bool causal, const FlashScratch &s)
{
    FlashPlan best;
    if (D != kFlashD || BH <= 0 || S_q <= 0)
        return best;
    const int64_t T = BH * flash_ceil_div(S_q, kFlashRows8), T4 = BH * flash_ceil_div(S_q, 128);
    const double n = double(flash_ceil_div(S_kv, kFlashKeys));
    const auto rounds = [](int64_t blocks) {
        return double(flash_ceil_div(blocks, kFlashTargetBlocks));
    };
    // Whole rounds of 8-wave workgroups, and one that fills part of the CUs.
    const double tail = double(T % kFlashTargetBlocks) / kFlashTargetBlocks;
    double us = (double(T / kFlashTargetBlocks) +
                 (tail > 0 ? std::max(tail, double(t.part)) : 0)) *
                n * t.w8;
    const auto consider = [&](const FlashPlan &pl, double cost) {
        if (cost < us) {
            us = cost;
            best = pl;
        }
    };
    if (T < kFlashTargetBlocks) {
        FlashPlan small;
        small.waves = 4;
        consider(small, rounds(T4) * n * t.w4);
        const FlashPlan sp = split_plan(BH, S_q, S_kv, D);
        if (sp.splits > 1 && sp.bytes <= s.part_bytes)
            consider(sp, split_tiles(sp, T4, int64_t(n), causal) * t.w4 + t.split +
                             t.split_mb * 1e-6 * double(sp.bytes));
    }
    const FlashPlan bal = balanced_plan(BH, S_q, S_kv, D);
    if (bal.u > 0 && !causal && bal.bytes <= s.balance_bytes)
        consider(bal, (bal.full / kFlashTargetBlocks * n + bal.u) * t.w8 +
                          (bal.full ? kBalanceTailUs
                                    : t.balance + t.balance_mb * 1e-6 * double(bal.bytes)));
    // One key tile of 64 has nothing to share (64 queries and keys, 16 heads:
    // 14.1 us whole against 16.1), and a second round of workgroups loses to
    // the taller tiles (576 queries and keys, 32 heads, f32x3: 46 against 60).
    if (s.keys && t.keys_round > 0 && !causal && S_kv > kFlashKeys &&
        BH * flash_ceil_div(S_q, 64) <= kFlashTargetBlocks) {
        FlashPlan keys;
        keys.keys = true;
        consider(keys, t.merge + flash_ceil_div(S_kv, t.keys_round) * t.round - s.keys_saves);
    }
    return best;
}

// Scratch that holds the partials of a split grid in every mode, and that of
// a balanced grid (0 where none would run).
inline size_t flash_split_bytes(int64_t BH, int S_q, int S_kv, int D)
{
    return split_plan(BH, S_q, S_kv, D).bytes;
}

inline size_t flash_balance_bytes(int64_t BH, int S_q, int S_kv, int D, const FlashTimes &t)
{
    FlashScratch any;
    any.part_bytes = any.balance_bytes = SIZE_MAX;
    const FlashPlan pl = flash_plan(BH, S_q, S_kv, D, t, false, any);
    return pl.u > 0 ? pl.bytes : 0;
}

constexpr size_t kMaxFlashBalanceBytes = 511 * kFlashSlotBytes;  // 65 MiB

// A grid of 8-wave workgroups with at least one for each CU.
inline bool flash_fills_gpu(int64_t BH, int S_q, int D)
{
    return D != kFlashD || BH <= 0 || S_q <= 0 ||
           BH * flash_ceil_div(S_q, kFlashRows8) >= kFlashTargetBlocks;
}

}  // namespace anima_hip
