// Plans of the deep kernel (deep.hip), host side, plain C++.
#include "deep_plan.hpp"

#include <algorithm>

namespace nne {

// Problems with at most half as many workgroups as CUs (decode steps of
// small batches, few-query cross-attention) split each unit's keys into up to
// kDeepMaxSplit parts of at least 4 tiles, one round of workgroups over the
// CUs, as far as max_bytes of records allow.  (Measured at d = 512, decode
// over L ~ U[512, 4096]: B = 8 601 -> 190 us with 4 parts; at B = 32, where
// every CU already has a head, 4 parts per head cost 667 -> 775 us: each
// extra workgroup pays its cold start, its record and the merge.)
uint64_t deep_split_plan(DeepParams& p, int max_tiles, int cus, uint64_t max_bytes) {
    p.n_split = 1;
    p.split_tiles = 0;
    const int64_t rows = (int64_t)p.G * p.Tq;
    p.rpu = (int)(rows < 32 ? rows : 32);
    const int64_t wg = (int64_t)p.B * p.Hkv * ((rows + 31) / 32) * ((p.d + kDeepChunk - 1) / kDeepChunk);
    if (wg == 0 || 2 * wg > (int64_t)cus || max_tiles < 8) return 0;
    int64_t sp = (int64_t)cus / wg;
    if (sp > kDeepMaxSplit) sp = kDeepMaxSplit;
    if (sp > max_tiles / 4) sp = max_tiles / 4;
    const uint64_t per = (uint64_t)wg * (uint64_t)p.rpu * (kDeepChunk + 2) * 4u;
    while (sp > 1 && per * (uint64_t)sp > max_bytes) --sp;
    if (sp <= 1) return 0;
    p.n_split = (int)sp;
    p.split_tiles = (int)((max_tiles + sp - 1) / sp);
    return per * (uint64_t)sp;
}

// Decode over ragged lengths (one unit and one output chunk per (sequence,
// KV head) pair, at most kDeepMaxHeads pairs and no more than the CUs): each
// pair's keys are cut into parts of `target` tiles -- at least 4, at most
// kDeepMaxSplit parts per pair, all parts in one round of workgroups over the
// CUs -- so a long sequence no longer sets the step's time on one CU while
// the others idle.  Used when that shortens the longest workgroup by a
// quarter or more.  (Measured at d = 512, L ~ U[512, 4096], Hq = 32,
// Hkv = 8: B = 8 571 -> 148 us, against 190 us for equal parts per pair;
// allowing two rounds, so that B = 32 could split too, made B = 8 261 us and
// B = 32 916 against 628 us unsplit: a part dispatched in the second round
// starts only when a CU's first one ends.)
uint64_t deep_ragged_plan(DeepParams& p, const int32_t* seq_keys, int cus, uint64_t max_bytes) {
    p.ragged = 0;
    const int64_t rows = (int64_t)p.G * p.Tq;
    const int64_t heads = (int64_t)p.B * p.Hkv;
    // With more pairs than CUs no part fits in the one round.
    if (rows > 32 || p.d > kDeepChunk || heads == 0 || heads > kDeepMaxHeads || heads > cus || !seq_keys)
        return 0;
    int64_t total = 0, longest = 0;
    for (int b = 0; b < p.B; ++b) {
        const int64_t t = ((int64_t)(seq_keys[b] > 0 ? seq_keys[b] : 0) + 31) / 32;
        total += t * p.Hkv;
        longest = longest > t ? longest : t;
    }
    auto parts = [](int64_t t, int64_t target) { return t > target ? (t + target - 1) / target : 1; };
    auto parts_of = [&](int64_t target) {
        int64_t n = 0;
        for (int b = 0; b < p.B; ++b)
            n += parts(((int64_t)(seq_keys[b] > 0 ? seq_keys[b] : 0) + 31) / 32, target) * p.Hkv;
        return n;
    };
    int64_t target = (total + cus - 1) / cus;
    if (target < 4) target = 4;
    if (target < (longest + kDeepMaxSplit - 1) / kDeepMaxSplit) target = (longest + kDeepMaxSplit - 1) / kDeepMaxSplit;
    // The smallest target whose parts fit the CUs (parts_of falls as target
    // grows; at target >= longest every pair is one part, and heads <= cus).
    if (parts_of(target) > cus) {
        int64_t lo = target, hi = longest > target ? longest : target;   // parts_of(hi) <= cus
        while (hi - lo > 1) {
            const int64_t mid = lo + (hi - lo) / 2;
            if (parts_of(mid) > cus) lo = mid;
            else hi = mid;
        }
        target = hi;
    }
    if (4 * longest < 5 * target) return 0;   // no pair's time shrinks enough to pay the split
    const int64_t n = parts_of(target);
    p.rpu = (int)(rows < 32 ? rows : 32);
    const uint64_t bytes = (uint64_t)n * (uint64_t)p.rpu * (kDeepChunk + 2) * 4u;
    if (bytes > max_bytes || n > 65535) return 0;
    int64_t at = 0;
    for (int b = 0; b < p.B; ++b) {
        const int64_t np = parts(((int64_t)(seq_keys[b] > 0 ? seq_keys[b] : 0) + 31) / 32, target);
        for (int k = 0; k < p.Hkv; ++k) {
            p.part_prefix[b * p.Hkv + k] = (uint16_t)at;
            at += np;
        }
    }
    p.part_prefix[heads] = (uint16_t)at;
    p.ragged = 1;
    p.n_split = kDeepMaxSplit;   // marks a split launch; parts per pair come from part_prefix
    p.split_tiles = (int)target;
    return bytes;
}

// With at most as many 32-row units as CUs (causal above 256 dims: two per CU,
// whose lengths even out) the deep kernel spreads or key-splits them over every
// CU, where the 8-wave kernel would leave most idle (deep / 8-wave, us: d = 256, T =
// 1024, 8 heads 164 / 163; T = 64, 128 heads 18 / 20; d = 512 non-causal, T = 512, 16
// heads 88 / 120; causal, T = 1024, 16 heads 178 / 228).  With more, the 8-wave
// kernel is 1.25 to 1.8 times as fast per unit and tile while its workgroups of 4
// units of one KV head (2 above 256 dims), one per CU, are full; KV heads of few
// units leave waves without a unit, and a few workgroups past a round of the CUs
// cost another round.  So the time of each is estimated as rounds of its
// workgroups (deep: 4 units at once on a CU, 2 above 256 dims), each a start and
// its tiles; the constants are fitted to calls of 257 to 3000 units, all measured
// on both (deep / 8-wave): d = 192, 300 heads of 65 rows 33 / 42, of 65 over 333 keys 89
// / 102, 600 of 40 rows 42 / 47, 90 of 100 34 / 25; d = 256, 257 heads of 32 rows 16 / 33;
// d = 320, 300 heads of 65 58 / 77, causal 51 / 67, 9 of 1024 222 / 183; d = 512, 257 of
// 32 over 1000 keys 355 / 484, 100 of 96 over 1000 319 / 241.  Estimates within 10 %
// keep the 8-wave kernel (d = 508, 150 heads of 530 rows over 42 keys 219 / 194).
bool deep_prefill_faster(int64_t heads, int64_t G, int64_t Tq, int64_t Tk, int d, bool causal,
                         int64_t q_offset, int cus) {
    const int64_t units = G * ((Tq + 31) / 32);
    if (heads * units <= (int64_t)cus * (d > 256 && causal ? 2 : 1)) return true;
    struct Cost { double start, tile; };   // us
    static constexpr Cost kWide[4] = {{7.5, 4.1}, {12.0, 4.7}, {8.0, 5.6}, {11.5, 7.05}};
    static constexpr Cost kDeep[4] = {{6.6, 7.1}, {8.5, 8.0}, {6.5, 7.0}, {10.0, 9.0}};
    const int at = d <= 192 ? 0 : d <= 256 ? 1 : d <= 384 ? 2 : 3;
    const auto tiles_of = [&](int64_t unit) {
        const int64_t keys = causal ? std::min(Tk, std::min((unit / G + 1) * 32, Tq) + q_offset) : Tk;
        return (double)((std::max<int64_t>(keys, 0) + 31) / 32);
    };
    // (The deep kernel's units run across the query heads of a KV head.)
    const auto us = [&](const Cost& c, int64_t per_wg, int64_t slots) {
        const int64_t n = heads * (per_wg > 1 ? (units + per_wg - 1) / per_wg : (G * Tq + 31) / 32);
        const double first = tiles_of(std::min(per_wg, units) - 1), last = tiles_of(units - 1);
        const double rounds = (double)((n + slots - 1) / slots);
        return rounds * c.start + c.tile * std::max({last, rounds * first, n * (first + last) / 2 / slots});
    };
    return us(kDeep[at], 1, (int64_t)cus * (d <= 256 ? 4 : 2)) < 0.9 * us(kWide[at], d <= 256 ? 4 : 2, cus);
}

}  // namespace nne
