// Which tiles a product of many rows is made of, and how it is cut: plain C++, without a device.
#pragma once

#include <stdint.h>

namespace nvmai {

// Which tile, and how many parts of k: those whose rounds over the compute units take the least time.  A step of 64 k takes `full` where every unit
// has a tile and `lone` where few have one (in 10 ns; fitted to every tile and part at k 1024 .. 8192 over 20 .. 2900 rows and 128 .. 11,264 weight
// rows).  Large tiles read each operand less often, small
// ones leave fewer units idle.
//   Tiles that are fewer than the units are cut along k, in 2, 3, 4, 6, 8 or 12 parts of two steps at least, as long as every part has a unit of its
// own: a step's latency is then paid by all units at once.  The join costs a trip to memory and back, the parts' sums that the last block takes back and
// the sums of all.  Rows x n x k, cold weights, uncut and cut, us: 65 x 2048 x 8192 26.9 and 13.8, 128 x 2048 x 5632 28.8 and 13.9, 300 x 1024 x 4096
// 18.4 and 11.7, 700 x 2048 x 8192 48.6 and 40.5, 300 x 2048 x 4096 18.9 and 17.1, 128 x 256 x 2048 7.9 and 6.4; 32-bit rows 20 x 1024 x 4096 39 and 14, 128 x 1024 x 2816
// 27.6 and 15.1, 500 x 1024 x 4096 48 and 32, 300 x 1024 x 1024 14.5 and 13.3.  A cut has to save 0.3 us by these costs (700 x 2048 x 4096 saves 0.4 by them, 28.2 and 24.5;
// 32-bit 70 x 4112 x 1024 less, 14.4 and 15.5), and 1 us past 1024 rows, where little is left to gain and a prompt of any length keeps one sum per output: 1250 x 256 x 2048 10.2
// and 9.3 is cut, 1501 x 256 x 2048 10.0 and 9.0 and 2048 x 256 x 2048 10.9 and 9.7 are not (weights from memory; where the caches hold them whole is the faster, 7.9 and 8.3).
// Sums against 64 bits, whole and in parts: 5.7e-7 and 2.7e-7 (65 x 2048 x 8192), 4.0e-7 and 2.7e-7 (500 x 1024 x 4096), 32-bit 1.6e-7 and 1.0e-7 there.
struct DenseTile {
    uint32_t bn, bm, lone, full;
};
constexpr DenseTile DENSE_TILES[] = {{64, 64, 16, 23}, {128, 64, 25, 38}, {128, 128, 43, 58}, {256, 128, 76, 100}, {256, 256, 114, 162}};
constexpr uint32_t DENSE_PARTS[] = {2, 3, 4, 6, 8, 12};
constexpr int DENSE_CUT_TILES = 3;                           // of these the first may be cut along k
constexpr float DENSE_CUT_SAVES = 300.0f, DENSE_CUT_SAVES_TALL = 1000.0f;      // ns at least: parts end in other roundings than a sum in one piece
constexpr uint32_t DENSE_TALL = 1024;                        // rows past which the larger saving is asked for

struct DensePlan {
    int tile;
    uint32_t parts;
    float ns;
};

// planes: the stages of 64 k.  cut: whether there is a place for the sums of parts.  (Few divisions, and those of 32 bits: the choice is made in every
// call, and short prompts are bound by the host.)
inline DensePlan dense_plan_tile(uint32_t n, uint32_t rows, uint32_t k, uint32_t planes, uint32_t cus, int count, bool cut) {
    DensePlan whole{0, 1, 1e30f}, parted{0, 1, 1e30f};
    const uint32_t steps = k / 64u;
    const float units = 1.0f / (float)cus, stages = 10.0f * (float)planes;
    for (int c = 0; c < count; ++c) {
        const DenseTile& t = DENSE_TILES[c];
        const uint64_t all = (uint64_t)((n + t.bn - 1) / t.bn) * ((rows + t.bm - 1) / t.bm);
        const uint32_t tiles = all > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)all, rounds = tiles < cus ? 0u : tiles / cus, rest = tiles - rounds * cus;
        const float lone = (float)t.lone, rise = (float)(t.full - t.lone) * units;
        const float cost = (float)rounds * (float)t.full + (rest ? lone + rise * (float)rest : 0.0f);
        const float ns = cost * stages * (float)steps + 4750.0f;             // and a launch, the first requests, the stores
        if (ns < whole.ns) whole = {c, 1, ns};
        if (!cut || rounds != 0 || c >= DENSE_CUT_TILES) continue;
        const float area = (float)(t.bn * t.bm);
        for (uint32_t parts : DENSE_PARTS) {
            if (parts * 2u > steps || tiles * parts > cus) break;
            const float blocks = (float)(tiles * parts);
            const float join = 1000.0f + area * ((float)parts * (1.0f / 16.0f) + blocks * (1.0f / 3500.0f));
            const float ns = (lone + rise * blocks) * stages * (float)((steps + parts - 1) / parts) + 4750.0f + join;
            if (ns < parted.ns) parted = {c, parts, ns};
        }
    }
    return parted.ns + (rows > DENSE_TALL ? DENSE_CUT_SAVES_TALL : DENSE_CUT_SAVES) <= whole.ns ? parted : whole;
}

// The matrix's rows in one launch, or in two where that is shorter: a last round that few units take part in is left to
// smaller tiles (8208 weight rows, 2048 tokens: one round of 256 x 256 and a sixteenth of one, 105 -> 76 us in all).
// Past 1024 rows the second is not cut along k: all outputs of such a product are sums in one order (cut, those sixteen rows would save 3 us of the 76, and end in
// other roundings than the rows beside them).
struct DenseSplit {
    uint32_t first;                                          // rows of the first launch
    DensePlan head, tail;
    float ns;
};

inline DenseSplit dense_plan(uint32_t n, uint32_t rows, uint32_t k, uint32_t planes, uint32_t cus, int count, bool split) {
    DenseSplit best{n, dense_plan_tile(n, rows, k, planes, cus, count, split), DensePlan{}, 0.0f};
    best.ns = best.head.ns;
    for (int c = 0; c < count; ++c) {
        const uint32_t tm = (rows + DENSE_TILES[c].bm - 1) / DENSE_TILES[c].bm, tn = n / DENSE_TILES[c].bn;
        if ((uint64_t)tn * tm < cus) continue;
        const uint32_t rounds = (uint32_t)((uint64_t)tn * tm / cus);
        const uint32_t cut = (uint32_t)((uint64_t)rounds * cus / tm) * DENSE_TILES[c].bn;
        if (cut == 0 || cut >= n) continue;
        const DensePlan head = dense_plan_tile(cut, rows, k, planes, cus, count, false), tail = dense_plan_tile(n - cut, rows, k, planes, cus, count, split && rows <= DENSE_TALL);
        if (head.ns + tail.ns < best.ns) best = {cut, head, tail, head.ns + tail.ns};
    }
    return best;
}

}  // namespace nvmai
