// Which tile and how many shares of K a product of wide_tile.h takes.
#pragma once

#include <stddef.h>

namespace esp {

struct WideForm { int bm = 0, bn = 0, per = 0, splits = 0; float us = 0.0f; };   // rows and weight rows of a tile (0: none), steps of 64 k of a share of K, shares, expected time

struct WideProduct {
    int rows = 0, weight_rows = 0, steps = 0, compute_units = 0;
    float stored_mb = 0.0f;                 // what a launch without shares writes
    size_t plane_floats = 0;                // room for planes of sums (0: no shares of K)
    float after = 0.0f, after_share = 0.0f; // us that adding the planes takes besides reading them, and for each of them
    bool wide_weights = true;               // whether a tile may hold 256 weight rows
    int forced = 0;                         // rows of a tile * 10000 + weight rows * 10 + shares of K (0: by cost)
    int shares = 0;                         // as many shares of K and no others (0: by cost)
};

// us: a launch's start, a step of 64 k with one workgroup on a compute unit and with two (0: one is resident), filling and emptying a tile
struct WideFormCost { int bm, bn; float start, step, step_of_two, fill; };
constexpr WideFormCost kWideForms[] = {{64, 128, 3.6f, 0.394f, 0.763f, 0.0f}, {64, 256, 4.0f, 0.666f, 0.0f, 0.0f}, {128, 128, 4.1f, 0.479f, 1.039f, 0.0f}, {128, 256, 3.9f, 0.782f, 0.0f, 1.24f},
                                       {192, 128, 2.1f, 0.577f, 0.0f, 2.53f}, {192, 256, 3.7f, 0.927f, 0.0f, 2.87f}, {256, 128, 2.05f, 0.693f, 0.0f, 3.32f}, {256, 256, 2.07f, 1.11f, 0.0f, 6.17f}};
inline bool wide_form_known(int form) {
    for (const WideFormCost &f : kWideForms)
        if (form / 10000 == f.bm && form / 10 % 1000 == f.bn && form % 10 >= 1) return true;
    return false;
}

// The form by its expected time: rounds of one or two workgroups per compute unit, what they store, and for shares of K the planes that the next kernel reads once more.  Constants fitted to
// 3500 launches with fp16 weights that no cache holds (fourteen shapes of 576 to 28672 weight rows and 576 to 14336 columns, 3 to 2048 rows): off by 7 % at the median, and what the rule
// chooses takes 1 % longer than the best form on average, 17 % at worst (two launches of 576 and 1152 weight rows, 3 us of 6, apart).
inline WideForm choose_wide_form(const WideProduct &p) {
    WideForm best;
    const int cus = p.compute_units > 0 ? p.compute_units : 256;
    const int kShares[] = {1, 2, 3, 4, 6, 8};
    for (const WideFormCost &f : kWideForms) {
        if (p.forced > 0 && (p.forced / 10000 != f.bm || p.forced / 10 % 1000 != f.bn)) continue;
        if ((p.forced == 0 && f.bm > 64 && f.bm - 64 >= p.rows) || (f.bn > 128 && !p.wide_weights)) continue;   // rows that no activation fills
        const long tiles = (long)((p.weight_rows + f.bn - 1) / f.bn) * ((p.rows + f.bm - 1) / f.bm);
        for (int want : kShares) {
            if ((p.forced > 0 && p.forced % 10 != want) || (p.shares > 0 && p.shares != want)) continue;
            const int per = (p.steps + want - 1) / want, splits = (p.steps + per - 1) / per;
            if ((splits != want && p.forced == 0) || (splits > 1 && (size_t)splits * p.rows * p.weight_rows > p.plane_floats)) continue;
            const float two = f.step_of_two > 0.0f ? f.step_of_two : f.step;
            const long wgs = tiles * splits, at_once = f.step_of_two > 0.0f ? 2 * cus : cus, whole = wgs / at_once, rest = wgs % at_once;
            const float steps = (float)per * ((float)whole * two + (rest == 0 ? 0.0f : rest > cus ? two : f.step));
            const float mb = splits > 1 ? (float)splits * (float)p.rows * (float)p.weight_rows * 4e-6f : p.stored_mb;
            float us = f.start + steps + (float)(whole + (rest > 0)) * f.fill + 0.18f * mb;
            if (splits > 1) us += 0.22f * mb + p.after + p.after_share * (float)splits;
            if (!best.bm || us < best.us) best = WideForm{f.bm, f.bn, per, splits, us};
        }
    }
    return best;
}

}  // namespace esp
