// How ops_flash.hip cuts the keys of causal attention's query tiles into runs: host code that needs no device, and what the kernels share of it.
#pragma once

#include <algorithm>

namespace pgk {

constexpr int FL_BQ = 128, FL_BKV = 64;                          // query rows and keys of a tile

constexpr int fl_ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }
// KV tiles and runs of query tile qt where runs hold `run` tiles
constexpr int flash_tiles(int qt, int q_len, int kv_len) {
    const int last = qt * FL_BQ + FL_BQ < q_len ? qt * FL_BQ + FL_BQ : q_len, end = kv_len - q_len + last;
    return ((end < kv_len ? end : kv_len) + FL_BKV - 1) / FL_BKV;
}
constexpr int flash_runs(int qt, int q_len, int kv_len, int run) { return (flash_tiles(qt, q_len, kv_len) + run - 1) / run; }

// runs: of the heaviest query tile, and of every one where run is 0; sides: of a workgroup (1 or 2: half a run's tiles each); fp32: of partial rows; run > 0: KV tiles of a run, of which
// a query tile takes as many as it has tiles for
struct FlashPlan { int runs, sides; bool fp32; int run; };

// The same number of runs for every query tile, or two sides.
// Where the causal edge is most of the work (contexts under twice the rows) a launch lasts as long as its heaviest tile; two sides take three quarters to nine tenths of
// one workgroup's time, and merge in LDS.
//  * Few workgroups (short of 5/8 of the CUs, 1200 positions and more): as many runs as two to a CU hold, of at least 2.5 KV tiles - more where many rows make the merge's
//    traffic count -, at most 8, or 12 where 8 would leave part of a round.  Us with two runs / this rule: head dim 128, 1 head, 1531 rows 20.3 / 13.4, 5000 47.3 / 23.4; 4 heads, 2048
//    26.6 / 24.4.
//  * Up to a workgroup per CU (and no runs of flash_run_tiles): two runs, of which a heavy and a light one share a CU.  12 heads, 2400 rows 37.7 (two sides 40.8), but 16 heads, 1800 34.5 (33.8).
//  * Shorter contexts, at most a workgroup to four CUs: three or four runs whose rows stay fp32.  In 16 bits they were rounded twice: 2.27e-3 of float64 for 700 rows of 4 heads
//    where two sides leave 2.00e-3 and these 1.98e-3.  1 head, 1024 rows 20.4 (two sides) / 12.8, 8 heads, 900 19.8 / 19.9.
//  * Otherwise two sides beyond ten KV tiles, up to five workgroups to four CUs: 16 heads, 2300 rows 46.6 (one side) / 41.4; 24 heads, 1531 34.3 / 31.5; 32 heads, 1100 27.0 / 25.1.  Up to two to a CU only where
//    nearly all of the context is causal and long: 16 heads, 3000 rows 63.4 / 53.8; but 64 heads, 900 rows 27.8 / 35.2, 32 heads, 1300 of 1950 47.7 / 52.1, 2500 68.6 / 81.6.  Beyond, two workgroups
//    of their own time per CU do more (one barrier makes the sides wait for each other).  Since the loop takes two tiles a pass the line is late by 3 %: 32 heads, 1600 rows 38.7 / 39.9, 2000 51.4 / 52.8, 28
//    heads, 1800 43.6 / 45.0.
// Longer contexts: as many runs as one round of workgroups holds, at least four KV tiles each: of two per CU (the kernel's occupancy), or of one per CU where all runs are alike and
// that many still cut it well.  A second round costs more than the shorter runs save, and every run costs the merge: 16 heads, 1000 of 4000 50.4 (2) 46.1 (4); 384 of 3585 27.3 (5)
// 29.8 (8); 250 of 2250 20.4 (4) 19.5 (8); 32 heads, 600 of 3000 48.0 (2) 45.3 (3).  Two sides there: 384 of 3585 52.4, 600 of 3000 48.7.
// (Results that are rounded to e4m3 next, by whichever kernel, ask for one side: the codes magnify a sum's last bit to a sixteenth, and a prompt in one pass and in pieces would
// no longer agree - 4096 rows of 32 heads at once and as two of 2048, which alone had two sides, were 0.028 apart in the logits, with one side each under 0.01.)
inline FlashPlan flash_even_plan(int cus, long long wgs, int q_len, int kv_len, int most) {
    if (kv_len < 2LL * q_len) {
        const int nt = fl_ceil_div(kv_len, FL_BKV);
        const bool fp32 = kv_len < 1200;
        long long n = 1;
        if (!fp32) n = 8 * wgs <= 5 * cus ? std::min({8 * wgs > cus ? 12LL : 8LL, 2 * cus / wgs, nt * 40 / (100 + wgs * 256 / cus)}) : wgs <= cus ? 2 : 1;
        else if (4 * wgs <= cus) n = 8 * wgs <= cus ? std::min(nt / 3, 4) : std::min(nt / 4, 3);
        if (fp32 && n < 3) n = 1;
        n = std::min<long long>(n, most);
        if (n > 1) return {(int)n, 1, fp32, 0};
        return {1, nt > 10 && (4 * wgs <= 5 * cus || (wgs <= 2 * cus && !fp32 && 4LL * kv_len <= 5LL * q_len)) ? 2 : 1, false, 0};
    }
    long long n = cus / wgs;
    if (n < 4 || kv_len < 4LL * q_len) n = 2 * cus / wgs;
    if (n > most) n = most;
    if (n > fl_ceil_div(kv_len, FL_BKV) / 4) n = fl_ceil_div(kv_len, FL_BKV) / 4;
    return {n < 1 ? 1 : (int)n, 1, false, 0};
}
// with a sliding window: up to four runs over the `span` keys that the heaviest query tile walks, until two workgroups per CU are reached
inline int flash_window_runs(int cus, long long wgs, int span) {
    int n = 1;
    while (n < 4 && wgs * n < 2LL * cus && fl_ceil_div(span, FL_BKV) >= 4 * (n * 2)) n *= 2;
    return n;
}

// KV tiles of a run where every query tile is cut into as many as it takes, so that the heavy ones do not decide: the fewest, four or more, with which a workgroup has a CU to itself (a few of
// the lightest may share one: two to a CU take 1.8 times as long).  0: flash_even_plan, for shapes that would need runs of more than 16 tiles.  Us with the merge, one launch behind another,
// even runs / this: 16 heads, 1200 rows 26.1 / 22.2, 1400 29.0 / 24.7, 1600 31.6 / 28.4; 8 heads, 1600 24.5 / 21.4, 2000 28.2 / 25.2; 4 heads, 1600 20.9 / 17.2, 2049 24.4 / 20.1.  Up to 16 runs for the heaviest
// tile: 1 head, 3900 rows 20.0, with at most 8 20.3 (head dim 64 14.7 / 15.3).  Under 1200 keys partial rows are fp32.
// Deeper in a context nearly every row has partial rows, which lose a bit where they are rounded to 16 bits (1 % more error than the even runs leave) and time where they are not (800 at 700
// 30.1 / 32.1, 900 at 800 32.2 / 35.5, with the loop of one tile a pass).
inline int flash_run_tiles(int cus, int hq, int q_len, int kv_len, int most) {
    const int tiles = fl_ceil_div(q_len, FL_BQ);
    for (int run = 4; run <= 16; ++run) {
        long long wgs = 0;
        int runs = 1, over = 0;                                  // over: the largest run beyond the CUs
        for (int qt = tiles - 1; qt >= 0; --qt) {
            const int n = flash_runs(qt, q_len, kv_len, run);
            runs = std::max(runs, n);
            wgs += (long long)n * hq;
            if (wgs > cus) over = std::max(over, fl_ceil_div(flash_tiles(qt, q_len, kv_len), n));
        }
        if (runs <= most && (wgs <= cus || (2 * over <= run && 4 * wgs <= 5LL * cus))) return run;
    }
    return 0;
}
// `even`: flash_even_plan's.  It stays where it is one run: a call that needs no scratch memory, as under capture, goes on needing none.  And where it has few workgroups: its runs are shorter than four tiles
// there, or few of the CUs work.  Us, even / runs of as many tiles, up to 7/16 of the CUs in workgroups: head dim 128, 1 head, 1200 rows 12.6 / 13.6, 1400 13.0 / 13.7, 1600 13.5 / 13.9, 2 heads, 1000 of 1240
// 13.5 / 14.1; beyond, 1 head, 3300 18.7 / 17.9, 3 heads, 1400 16.7 / 15.2.  Head dim 64, whose partial rows cost half, up to 3/4: 1 head, 1200 9.6 / 10.6, 2700 12.1 / 12.9, 2 heads, 1400 10.6 / 11.0;
// beyond, 3 heads, 1400 11.7 / 11.5, 4 heads, 1400 12.5 / 11.8.  More than eight even runs stay for the one head of 5000 rows and more that has them (23.4 / 23.6, 8000 34.3 / 34.1); they cost where few rows
// have them: 2 heads, 2049 20.9 / 16.4, 3 heads, 2300 23.1 / 19.7, 1 head, 4200 22.8 / 20.6.
inline FlashPlan flash_plan(int cus, const FlashPlan& even, int hq, int q_len, int kv_len, int d, int most) {
    if (kv_len < 1200 || 4LL * kv_len > 5LL * q_len || even.runs == 1 || even.runs > 8) return even;
    if (16LL * even.runs * fl_ceil_div(q_len, FL_BQ) * hq <= (d == 64 ? 12 : 7) * cus) return even;
    const int run = flash_run_tiles(cus, hq, q_len, kv_len, most);
    return run ? FlashPlan{flash_runs(fl_ceil_div(q_len, FL_BQ) - 1, q_len, kv_len, run), 1, false, run} : even;
}

// The plan, or where grant(runs) refuses scratch memory for the heaviest tile's runs the even one, which takes less, or where that is refused too, one run
template <class Grant> FlashPlan flash_granted(const FlashPlan& plan, const FlashPlan& even, Grant grant) {
    if (plan.runs == 1 || grant(plan.runs)) return plan;
    if (even.runs > 1 && even.runs < plan.runs && grant(even.runs)) return even;
    return {1, plan.sides, plan.fp32, 0};
}

}  // namespace pgk
