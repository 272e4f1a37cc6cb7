// prefill_shape.hpp -- which workgroup shapes a staged prefill call takes
// (prefill.hip).  Plain C++, so that a host test can walk the rule.
#pragma once

#include <stdint.h>

namespace bmo {

constexpr int kQB = 1;  // blocks of 16 queries per wave

// Workgroup of the staged path: qw waves, ks of them on each block of 16
// queries.
struct StagedShape {
    int qw, ks;
    constexpr int queries() const { return 16 * kQB * qw / ks; }
};
constexpr StagedShape kStagedShapes[] = {{16, 1}, {16, 2}, {8, 1}, {8, 2}};

// The time of a staged call's workgroups in units of one round of 256
// workgroups of 16 waves x 16 queries, one a CU.  A 16-wave workgroup fills a
// CU; two 8-wave ones fit, and slow each other down.  Measured with 8 of 32
// heads' K/V, 1024 slots, 500 and 256 tokens (us; 16 x 1, 16 x 2, 8 x 1, 8 x
// 2): 1 session 61.7 / 50.2 / 54.9 / 43.8, 2 sessions 62.9 / 51.0 / 56.1 /
// 59.6, 3 sessions 64.7 / 92.8 / 76.7 / 87.1, 16 x 256 tokens 124 / 178 / 140
// / 196; 24 sessions x 64 tokens 120.9 / 118.5 / 87.7 / 85.8.  The constants
// stand for other rings and for head_dim 64 too: of 40 staged calls of 1 to
// 24 sessions, 16 to 600 tokens, 64 to 3000 slots and both head dims, 38 take
// no longer than in 16 x 1 (22.0 against 26.1 us for 16 tokens of one session
// on 512 slots, 21.2 / 23.3 for 64 tokens at d64, 49.3 / 68.1 for 2 x 300
// tokens, 2048 slots, d64, 165 / 237 for 3 x 600, 3000 slots), and two on
// nearly empty rings at d64 a little (10 x 130 tokens 30.2 / 29.4, 6 x 128
// 15.7 / 14.6), since the window does not enter.
constexpr double staged_cost(const StagedShape &s, int64_t workgroups) {
    const int per_cu = s.qw == 16 ? 1 : 2;
    const double alone = s.qw == 16 ? (s.ks == 1 ? 1.0 : 0.81) : (s.ks == 1 ? 0.88 : 0.71);
    const double shared = s.ks == 1 ? 1.155 : 0.95;
    const int64_t round = 256 * per_cu;
    const int64_t rest = workgroups % round;
    return (double) (workgroups / round) * (per_cu == 1 ? alone : shared) +
           (rest == 0 ? 0.0 : rest <= 256 ? alone : shared);
}

// The cheapest shape; a smaller one only if it saves a twentieth.
constexpr StagedShape staged_shape(int64_t units, int n_tok) {
    StagedShape best = kStagedShapes[0];
    double cost = 0.95 * staged_cost(best, units * ((n_tok + best.queries() - 1) / best.queries()));
    for (int i = 1; i < 4; ++i) {
        const StagedShape s = kStagedShapes[i];
        const double c = staged_cost(s, units * ((n_tok + s.queries() - 1) / s.queries()));
        if (c < cost) {
            best = s;
            cost = c;
        }
    }
    return best;
}

// The units that go ahead in full rounds of the first shape, when the rest in
// a shape of its own then takes a twentieth less in all than every unit in
// one (0: one launch).  A second launch costs as much as about 0.05 rounds.
// 160 units of 500 tokens (8 of 32 heads' K/V, 1000 slots), 320 workgroups of
// 256 queries: 128 units in one round and 32 in 256 workgroups of 64 queries,
// 93.4 us a call against 104.9 in one launch.
constexpr int64_t staged_full_units(int64_t units, int n_tok) {
    auto cost = [=](int64_t n) {
        const StagedShape s = staged_shape(n, n_tok);
        return staged_cost(s, n * ((n_tok + s.queries() - 1) / s.queries()));
    };
    const int64_t n_qt = (n_tok + kStagedShapes[0].queries() - 1) / kStagedShapes[0].queries();
    const int64_t rounds = units * n_qt / 256;
    const int64_t full = rounds * 256 / n_qt;
    if (full == 0 || full == units) return 0;
    return (double) rounds + 0.05 + cost(units - full) < 0.95 * cost(units) ? full : 0;
}
static_assert(staged_full_units(160, 500) == 128 && staged_full_units(512, 256) == 0,
              "a quarter of a round goes apart, full rounds do not");
static_assert(staged_shape(512, 256).qw == 16 && staged_shape(512, 256).ks == 1, "full rounds: 256 queries");
static_assert(staged_shape(32, 500).qw == 8 && staged_shape(32, 500).ks == 2, "256 workgroups of 64 queries");
static_assert(staged_shape(64, 500).qw == 16 && staged_shape(64, 500).ks == 2, "256 workgroups of 128 queries");

}  // namespace bmo
