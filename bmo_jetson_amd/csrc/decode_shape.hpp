// decode_shape.hpp -- which workgroup shape a decode call takes (decode.hip).
// Plain C++, so that a host test can walk the rule.
#pragma once

#include <stdint.h>
#include <stdio.h>

#include <initializer_list>

namespace bmo {

// Waves per unit, groups in flight per wave, query heads per workgroup.
struct Shape {
    int nw, pf, r;
};

// The shapes launch_shape instantiates ({1, 3, 1} and {16, 1, 1} only for
// BMO_ATTN_SHAPE).
constexpr Shape kShapes[] = {{1, 1, 1}, {1, 2, 1}, {1, 3, 1}, {2, 1, 1},  {2, 2, 1}, {4, 1, 1}, {4, 2, 1},
                             {8, 1, 1}, {8, 2, 1}, {16, 1, 1}, {1, 2, 2}, {2, 2, 2}, {4, 2, 2}, {1, 2, 4}};

constexpr bool shape_instantiated(Shape s) {
    for (const Shape &k : kShapes)
        if (k.nw == s.nw && k.pf == s.pf && k.r == s.r) return true;
    return false;
}

// Threads of a launch along its first dimension: 64 a wave, units / r
// workgroups of r * nw waves.
constexpr uint64_t launch_threads(int64_t units, Shape s) { return (uint64_t) units * 64 * (uint64_t) s.nw; }

// Workgroup shape per call, from the units (entry, head) and the window's
// groups.  With two groups in flight a wave takes about 142 VGPRs, three
// waves fit a SIMD and 3072 the chip; a unit gets as many waves (4, 2 or 1)
// as leave every unit resident, and its window keeps busy.  us per launch, 32
// heads x d128, 512 slots (32 groups) unless noted, 4 / 2 / 1 waves (RoPE +
// append; plain in brackets):
//   256 units   7.6 /  9.7 / 13.6 (6.6 / 8.7 / 12.3)
//   768 units  13.5 / 13.9 / 15.3 (12.2 / 12.6 / 13.3)
//   1024       18.3 / 15.8 / 16.7 (16.2 / 15.4 / 14.8)
//   1536       23.7 / 22.7 / 24.2
//   2048       29.8 / 31.3 / 28.6 (27.1 / 29.9 / 25.9)
//   8192        108 /  106 /  105 (92.8 / 94.1 / 95.6)
//   1024 units, 3000 slots  72.8 / 70.9 / 67.4 (71.1 / 68.9 / 64.5)
//   576 units,  2 groups  6.39 / 5.48 / 5.15 (4.78 / 4.21 / 4.10)
//               5 groups  6.62 / 6.26 / 6.00 (5.57 / 5.03 / 5.00)
//               6 groups  6.80 / 6.39 / 6.50 (5.67 / 5.36 / 5.50)
//               8 groups  7.20 / 6.95 / 6.91 (5.96 / 6.16 / 5.88)
//              10 groups  7.95 / 7.50 / 8.08 (6.67 / 6.45 / 7.02)
//              17 groups  8.81 / 9.54 / 9.52 (8.72 / 8.06 / 8.45)
//   512 units,  3 and 4 groups  5.54 / 5.55 / 5.39 and 5.58 / 6.09 / 6.05
// Up to 511 units every window is worth four waves, at 512 one of more than
// three groups (plain: two), and up to 768, where workgroups of four waves
// share a SIMD, one of 14 (plain: 32); below that two waves, or one on the
// shortest windows and where its loop of three groups a pass ends with two
// left, the fewest it can (5, 8 and, fused, 11 groups).
// Past 2048 units, where one-wave units come in rounds, plain calls take
// four waves again from 32 groups on (2560 units 32.6 against 34.3 us, 5120
// 59.5 / 62.9, 3072 38.6 / 38.0; 8 groups, 8192 units: 40.3 / 28.9).
// Between 768 and 1536 units two waves win by overlapping the prologues of
// fused calls on short windows (3 to 64 groups; two groups, 800 units, 5.82
// against 5.57 us), and lose where the window's bytes dominate.  Below 128
// units 8 waves: one workgroup a CU at most, and on long windows more waves
// still pay (3000 slots, 32 units 16.3 against 17.5 us with 4, on 64 or more
// groups up to 256 units: 128 units 17.6 / 19.0; 32 groups, 32 units, 7.4 /
// 7.1).  Fewer groups than waves: fewer waves, with one group in flight, as
// where plain waves have one group each (64 units, 4 groups 3.60 against 3.79
// us, 192 units 3.64 / 3.84), but fused up to 256 units one more than the
// groups, for the new token (depformer frame, one group: 200 / 207 us; 288
// units 5.0 / 4.5).
//
// units are those of one layer, also where a launch serves several: the
// split of a unit's window, and with it every rounding of its output, is
// then that of the layer's call by itself.  With as few waves as leave every
// unit of the launch resident a step's error against 64 bits grew, since
// eight short runs round less than four or two longer ones (relative, 8 / 4,
// 2 or 1 waves: 20 layers of 128 slots 3.4e-7 / 3.7e-7, 64 layers of 512
// 4.1e-7 / 5.5e-7, 8 kv heads 4.0e-7 / 4.5e-7); 32 layers of 512 slots took
// 25.5 us then, 28.5 with eight waves.  Eight waves of several layers keep
// one group in flight each, which changes no result: 32 layers of 512 slots
// 28.5 us against 34.0, of 3000 slots 80.2 against 84.6.
//
// Grouped queries, an even number a kv head, from 257 units on: 2 or 4 of
// them share a workgroup, 8 waves of it up to 512 units, 4 up to 1536 (1280
// units of 64 groups: 27.8 us with 2 heads x 2 waves, 33.8 with 4 x 1, 36.4
// one head a workgroup; 512: 14.5 with 2 x 4, 15.2 with 2 x 2, 17.1).  Past
// that 4 x 1 (4096: 63.7 against 73.1 with 2 x 2 and 98.0), or with 2 heads
// a kv head 2 x 2 from 32 groups on (4096 of 64: 71.4, 2 x 1 79.9) and 2 x 1
// below (4800 of 19: 30.3, 2 x 2 32.0).  8 x 1 gains nothing over 4 x 1.
// Windows of two groups gain from it up to 512 units and, with four heads,
// past 1536 (288 units 4.6 against 5.4 us ungrouped, 4096 10.1 / 11.5; between
// them 544 units 5.4 / 5.2), windows of one group nowhere.
//
// A launch holds fewer than 2^32 threads a dimension: calls of so many units
// take as few waves as that needs.
constexpr Shape default_shape(int64_t units, int n_layers, int n_groups, int q_per_kv, bool fused) {
    Shape s{1, 2, 1};
    if (q_per_kv % 2 == 0 && units > 256 &&
        (n_groups > 2 || (n_groups == 2 && (units <= 512 || (units > 1536 && q_per_kv % 4 == 0))))) {
        s = units <= 512 ? Shape{4, 2, 2}
            : units <= 1536 ? Shape{2, 2, 2}
            : q_per_kv % 4 == 0 ? Shape{1, 2, 4}
            : n_groups >= 32 ? Shape{2, 2, 2} : Shape{1, 2, 2};
    } else if (units < 128) s = Shape{8, fused && n_groups < 64 ? 1 : 2, 1};
    else if (units <= 256 && n_groups >= 64) s = Shape{8, 2, 1};
    else if (units < 512) s = Shape{4, 2, 1};
    else if (units <= 768) {
        const bool few = n_groups <= (fused ? 3 : 2);
        const bool even = n_groups % 3 == 2 && n_groups <= (fused ? 11 : 8);
        if (!few && (units == 512 || n_groups >= (fused ? 14 : 32))) s = Shape{4, 2, 1};
        else if (!few && !even) s = Shape{2, 2, 1};
    } else if (units <= 1536 && fused && n_groups > 2 && n_groups <= 64) s = Shape{2, 2, 1};
    else if (units > 2048 && !fused && n_groups >= 32) s = Shape{4, 2, 1};
    while (s.nw > 1 && s.nw > n_groups + (fused && n_groups == 1 && units <= 256 ? 1 : 0)) {
        s.nw /= 2;
        if (s.r == 1) s.pf = 1;
    }
    if (!fused && s.r == 1 && n_groups == s.nw) s.pf = 1;
    while (s.nw > 1 && launch_threads(units, s) > UINT32_MAX) s.nw /= 2;
    if (n_groups == 1 || (s.nw == 8 && n_layers > 1)) s.pf = 1;
    return s;
}

constexpr bool default_shapes_instantiated() {
    for (int64_t units : {1, 127, 128, 256, 257, 511, 512, 513, 768, 769, 1536, 1537, 2048, 2049, 1 << 24, 1 << 25, 1 << 26})
        for (int n_groups : {1, 2, 3, 4, 7, 8, 14, 32, 63, 64, 65})
            for (int q_per_kv : {1, 2, 3, 4, 6, 8, 16})
                for (bool fused : {false, true})
                    for (int n_layers : {1, 2})
                        if (!shape_instantiated(default_shape(units, n_layers, n_groups, q_per_kv, fused))) return false;
    return true;
}
static_assert(default_shapes_instantiated(), "every default decode shape has a kernel");

// forced = "nw,pf[,r]" (the environment's BMO_ATTN_SHAPE, for tuning; null:
// none) overrides the default; a shape without a kernel, or with an r that
// does not divide the query heads of a kv head, falls back to one wave with
// one group in flight.
inline Shape pick_shape(int64_t units, int n_layers, int n_groups, int q_per_kv, bool fused, const char *forced) {
    Shape s = default_shape(units, n_layers, n_groups, q_per_kv, fused);
    if (forced) {
        Shape o{0, 0, 1};
        if (sscanf(forced, "%d,%d,%d", &o.nw, &o.pf, &o.r) >= 2) s = o;
    }
    if (!shape_instantiated(s) || q_per_kv % s.r != 0) s = Shape{1, 1, 1};
    return s;
}

}  // namespace bmo
