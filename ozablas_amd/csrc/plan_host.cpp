// plan_host.cpp — how a single call's GEMM is cut into work items (host only).
//
// The persistent GEMMs run one 256 x 256 tile per CU at a time.  Where the items do not fill whole
// rounds of the CUs (Scheme II), or the longest item outlasts the rest (Scheme I), items are split along
// K: their parts are exact integer sums (digits add modulo m_s, group products in INT32), so the result
// does not depend on the split.  The plans are fixed functions of the shape, for an MI355X's 256 CUs and
// the measured item time below, so that workspace sizes and calls agree on them.
#include <algorithm>

#include "oza_internal.hpp"

namespace oza {

namespace {

constexpr int64_t kPlanCus = 256;
// An item lasts about 3.5 us plus 1.52 us per 128-byte K step (4096^2, S = 8, K = 128, 512, 1024, 2048: 5.0,
// 9.8, 16.0, 28.0 us per round).
constexpr double kItemUs = 3.5, kStepUs = 1.52;
// A Scheme I item stores INT32, four times the bytes of digits.
constexpr double kS1ItemUs = 9.0;
// The reconstruction of split items: their extra bytes, and its longer chain of loads.
constexpr double kBytesPerUs = 4.0e6, kPartsUs = 2.0;

double item_us(int64_t steps) { return kItemUs + kStepUs * (double)steps; }
int64_t div_up(int64_t a, int64_t b) { return (a + b - 1) / b; }
// Calls with this many items or more are not split; a split call adds at most this many partial tiles.
// With K below kS2LongKp the parts fill one round at most (more rounds of shorter parts pay for long K only:
// 192 items in fours are 3 rounds of a quarter).
constexpr int64_t kS2Items = 16 * kPlanCus, kS2Extra = 2 * kPlanCus, kS2LongKp = 4096;
constexpr int64_t kS1Items = 8 * kPlanCus, kS1Extra = kPlanCus;
constexpr int64_t kS1MinStages = 4;  // per part
int64_t tiles_of(const Dims& d) { return div_up(d.M, kS2TileRows) * div_up(d.N, kS2TileRows); }

}  // namespace

// Tile edge.  Calls, us, with 256 x 256 tiles (in parts where that is the plan) / 128 x 128 / 64 x 64:
//   64: at most 512 items (two workgroups per CU), and their stages, one item after the other, not past what
//   parts along K would take: 256^3, S = 4 15.0 / 14.0 / 13.5; 256^2 x 2048, S = 12 36.2 / 30.3 / 26.3;
//   512^2 x 2048, S = 8 36.7 / 29.9 / 28.2; 256^2 x 12000, S = 16 105 / 97 / 78; 100^2 x 4000, S = 10 43 / 38 / 30;
//   beyond: 512^2 x 16384, S = 8 130 / 161 / 152; 64^2 x 20000, S = 15 59 / 98 / 68; 512^2 x 256, S = 20 (1280
//   items) 21.4 / 19.3 / 21.6.
//   128: at most 512 items; with K past 2048 not where some CUs have two of them and most one:
//   512^2 x 1024, S = 14 31.5 / 24.1 / 26.8; 1024^3, S = 8 35.5 / 30.5 / 37.8; 1000^2 x 1500, S = 8 40.5 / 36.6 / 45.6;
//   512^2 x 4096, S = 14 57 / 50.5 / 58; beyond: 1024^3, S = 16 (1024 items) 44.6 / 46.5 / 61; 768^2 x 4096, S = 8 (288)
//   58.9 / 62.0 / 69.5; 512^2 x 8192, S = 14 98.7 / 100.5 / 113.7.
static int small_edge(const Dims& d) {
    const auto items = [&](int64_t edge) { return div_up(d.M, edge) * div_up(d.N, edge) * d.S; };
    const int64_t n64 = items(64), n128 = items(128), most = 2 * kPlanCus;
    if (n64 <= most && d.Kp <= 16384 && n64 * d.Kp <= most * 8192) return 64;
    if (n128 <= most && (d.Kp <= 2048 || (d.Kp <= 4096 && (n128 <= kPlanCus || n128 >= most * 7 / 8)))) return 128;
    return kS2TileRows;
}

// Candidates: every item in p parts, or only those past the last full round of the CUs (2048^3, S = 6:
// 384 items are 1.5 rounds; the last 128 in halves take 1 + 0.5: 95.4 -> 92.7 us for the call; 1500 x 900 x
// 3000, S = 12, 288 items: 124 -> 112 us; 777 x 1501 x 1003, S = 14: 55.7 -> 54.2 us).  From 16 rounds on row
// bands may run instead and the last round matters little.
S2Plan scheme2_plan(const Dims& d) {
    S2Plan best;  // unsplit
    const int64_t KT = d.Kp / 128, items = tiles_of(d) * d.S;
    best.kts = (int)KT;
    best.whole = items;
    if (items == 0 || items >= kS2Items) return best;
    best.edge = small_edge(d);
    if (best.edge != kS2TileRows) return best;
    const int64_t full = items / kPlanCus * kPlanCus;
    double best_us = 0.97 * (double)div_up(items, kPlanCus) * item_us(KT);  // a split has to pay
    for (const int64_t whole : {full, (int64_t)0}) {
        const int64_t tail = items - whole;
        if (tail == 0) continue;
        for (int64_t p = 2; p <= kMaxParts && 2 * p <= KT; ++p) {
            const int64_t kts = div_up(KT, p);
            if (div_up(KT, kts) != p) continue;  // some part would be empty
            if (d.Kp < kS2LongKp ? p * tail > kPlanCus : (p - 1) * tail > kS2Extra) break;
            const double us = (double)(whole / kPlanCus) * item_us(KT) + (double)div_up(tail * p, kPlanCus) * item_us(kts) +
                              (double)((p - 1) * tail * kTileBytes) / kBytesPerUs + kPartsUs;
            if (us < best_us) {
                best_us = 0.98 * us;  // more parts only where they pay clearly
                best.parts = (int)p;
                best.kts = (int)kts;
                best.whole = whole;
            }
        }
        if (full == 0) break;
    }
    return best;
}

// Four slots of 64 K-bytes instead of two of 128: three stages (96 KiB per CU) on their way from memory while
// one is computed, instead of one of 64 KiB, for twice the barriers.  That pays where the operand planes come
// from memory (past some 90 MB, that is with K past a few thousand) and each of their bytes meets few products.
// Calls, us, two slots / four: 600^2 x 16384, S = 12 227 / 206; 512^2 x 32768, S = 14 327 / 317; 1024^2 x 16384,
// S = 12 390 / 366; 300 x 8000 x 2048, S = 12 189 / 178; 1500^2 x 8192, S = 12 355 / 344.  Beyond the lines:
// 2048^3, S = 6 93 / 96; 2100^3, S = 15 216 / 220; 8192^3, S = 17 8459 / 8619; 1800^2 x 8192, S = 12 463 / 467;
// 1200^2 x 3000, S = 12 (86 MB) 109 / 110; 500^2 x 3000, S = 14 (45 MB) 53.9 / 54.5.
// The bytes are counted with rows padded to 256, although only 32-row blocks that hold a row are read: few rows by
// a long K gain as well (64^2 x 20000, S = 15, 39 of 154 MB read, 61.3 / 59.5; 30 x 40 x 60000, S = 6, 35 of 184, 76.3 / 72.7;
// 96 x 13 x 30000, S = 10, 39 of 154, 65.1 / 62.9; 128^2 x 20000, S = 14, 72 of 144, 79.2 / 78.9).
// (p.parts * p.kts - KT: what the last part is short of kts K steps; it needs two of them for its four stages.)
bool s2_deep_ring(const Dims& d, const S2Plan& p) {
    constexpr int64_t kDeepBytes = 90000000, kDeepWidth = 800;
    const bool pays = d.S * (d.Mp + d.Np) * d.Kp >= kDeepBytes && d.M * d.N <= kDeepWidth * (d.M + d.N);
    return pays && p.edge == kS2TileRows && d.Kp >= 256 &&
           (p.parts == 1 || (int64_t)p.parts * p.kts - d.Kp / 128 <= p.kts - 2);
}

int64_t s2_plan_tiles(const Dims& d, const S2Plan& p) {
    const int64_t items = tiles_of(d) * d.S;
    return p.parts > 1 ? items + (p.parts - 1) * (items - p.whole) : items;
}

// At least every plan's tiles, and growing with each of M, N, K and S, so that buffers made for the
// largest of a program's shapes hold the smaller ones (whose plans may have more parts).
static int64_t most_tiles(int64_t items, int64_t most_parted, int64_t split_items, int64_t extra) {
    return std::max(items, std::min({most_parted, items + extra, split_items + extra}));
}
int64_t s2_most_tiles(const Dims& d) {
    const int64_t items = tiles_of(d) * d.S, parted = items * std::clamp<int64_t>(d.Kp / 256, 1, kMaxParts);
    if (d.Kp >= kS2LongKp) return most_tiles(items, parted, kS2Items, kS2Extra);
    return items >= kS2Items ? items : std::min(parted, div_up(items, kPlanCus) * kPlanCus);
}
int64_t s1_most_tiles(const Dims& d) {
    int64_t parts = 0;
    for (int g = 0; g < d.S; ++g) parts += div_up((g + 1) * (d.Kp / 128), kS1MinStages);
    return most_tiles(tiles_of(d) * d.S, tiles_of(d) * std::min<int64_t>(parts, kMaxS1Planes), kS1Items, kS1Extra);
}

// Tile edge, by the items and the 128-byte K steps of the longest.  Calls, us, 256 x 256 (in parts) / 128 x 128 /
// 64 x 64: 256^3, S = 4 (64 items of 64 x 64, longest 8) 24.8 / 18.4 / 15.0; 512^3, S = 8 (512, 32) 40.9 / 36.5 / 27.6;
// 300^2 x 2000, S = 6 (150, 96) 58 / 78 / 50; 100^2 x 4000, S = 7 (28, 224) 52 / 145 / 80; 768^3, S = 6 (864, 36) 49 / 42 / 39;
// 1000^2 x 300, S = 4 (1024, 12; 256 of 128 x 128) 38.6 / 28.5 / 30.8; 1024^2 x 256, S = 6 (1536, 12; 384) 41.7 / 31.8 /
// 36.9; 1000^2 x 500, S = 9 (2304, 36; 576) 66 / 56 / 73; 1200^3, S = 6 (2166, 60; 600) 85 / 81 / 102; 2000^2 x 1000, S = 6
// (1536 of 128 x 128) 137 / 153 / 203.
static int small_edge_s1(const Dims& d) {
    const auto items = [&](int64_t edge) { return div_up(d.M, edge) * div_up(d.N, edge) * d.S; };
    const int64_t n64 = items(64), n128 = items(128), most = 2 * kPlanCus, longest = d.S * d.Kp / 128;
    if (longest <= 100 && (n64 <= most || (n64 <= 2 * most && longest > 32))) return 64;
    if (longest <= 64 && n128 <= 600) return 128;  // the third workgroups of a few CUs are short ones
    return kS2TileRows;
}

// Groups of at most `limit` stages per item, the limit with the least modelled time: the longest load of
// a workgroup in the launch's order (one list, longest item first, back and forth over the CUs; sampled
// workgroups), plus the extra planes' bytes.  Calls, us, whole / with this plan: 184 x 499 x 10597, S = 6
// 622 / 122; 700^2 x 3000, S = 6 208 / 88; 1200^3, S = 6 102 / 86; 1499 x 1200 x 1801, S = 8 199 / 191;
// 1500^3, S = 8 stays whole (179, in two parts 187), as does 2000^2 x 1000, S = 6 (136, 174).
S1Plan scheme1_plan(const Dims& d) {
    S1Plan best;
    const int64_t KT = d.Kp / 128, tiles = tiles_of(d);
    auto plan_us = [&](int64_t limit, S1Plan& p) -> double {
        double len[kMaxS1Planes];  // entries of `tiles` items each
        p.planes = 0;
        for (int g = 0; g < d.S; ++g) {  // g + 1 pairs
            const int64_t stages = (g + 1) * KT;
            p.parts[g] = (int)div_up(stages, limit);
            if (p.planes + p.parts[g] > kMaxS1Planes) return 1e30;
            for (int j = 0; j < p.parts[g]; ++j) len[p.planes++] = kS1ItemUs + kStepUs * (double)div_up(stages, p.parts[g]);
        }
        std::sort(len, len + p.planes, [](double a, double b) { return a > b; });
        const int64_t items = tiles * p.planes;
        double longest = 0.0;
        for (int64_t b = 0; b < kPlanCus; b += 15) {
            double load = 0.0;
            for (int64_t r = 0; r * kPlanCus < items; ++r) {
                const int64_t k = r & 1 ? (r + 1) * kPlanCus - 1 - b : r * kPlanCus + b;
                if (k < items) load += len[k / tiles];
            }
            longest = std::max(longest, load);
        }
        const int extra = p.planes - d.S;
        return longest + (extra ? (double)(extra * tiles) * 8.0 * kTileBytes / kBytesPerUs + kPartsUs : 0.0);
    };
    const int64_t most = (int64_t)d.S * KT;
    best.edge = small_edge_s1(d);
    if (tiles == 0 || tiles * d.S >= kS1Items || best.edge != kS2TileRows) {  // enough items to balance, or small ones
        best.planes = d.S;
        std::fill(best.parts, best.parts + d.S, 1);
        return best;
    }
    double best_us = 0.95 * plan_us(most, best);
    int64_t last = most;
    for (const int p : {2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32}) {
        const int64_t limit = std::max(kS1MinStages, div_up(most, p));
        if (limit == last) continue;
        last = limit;
        S1Plan cand;
        const double us = plan_us(limit, cand);
        if (us < best_us && (cand.planes - d.S) * tiles <= kS1Extra) {
            best_us = 0.96 * us;
            best = cand;
        }
    }
    return best;
}

}  // namespace oza
