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
// stand for other rings and for head_dim 64 too, though the window does not
// enter: of 576 calls of 1 to 24 sessions (8 of 32 heads' K/V), 16 to 400
// tokens, 512 slots empty and full and 2048 full, both head dims, none takes
// longer than in the build that had 16 x 1 alone but 12 sessions x 256 tokens
// on an empty ring at d64 (31.1 against 30.0 us; full 52 / 57).
constexpr double staged_cost(const StagedShape &s, int64_t workgroups) {
    const int per_cu = s.qw == 16 ? 1 : 2;
    const double alone = s.qw == 16 ? (s.ks == 1 ? 1.0 : 0.81) : (s.ks == 1 ? 0.88 : 0.71);
    const double shared = s.ks == 1 ? 1.155 : 0.95;
    const int64_t round = 256 * per_cu;
    const int64_t rest = workgroups % round;
    return (double) (workgroups / round) * (per_cu == 1 ? alone : shared) +
           (rest == 0 ? 0.0 : rest <= 256 ? alone : shared);
}

// The cheapest shape; a smaller one only if it saves a twentieth.  Up to 128
// tokens 16 x 2 has as many workgroups as 16 x 1 and twice the waves that load
// queries, which only a long window repays: on rings of up to 512 slots 8 x 1
// takes its place (6 sessions x 128 tokens, d128, us in 8 x 1, 16 x 2 and 16
// x 1: 512 slots empty 17.0 / 19.8 / 17.4, full 34.7 / 35.2 / 35.3; 2048 slots
// full 79.7 / 69.3 / 80.6).
constexpr StagedShape staged_shape(int64_t units, int n_tok, int n_ctx) {
    StagedShape best = kStagedShapes[0];
    double cost = 0.95 * staged_cost(best, units * ((n_tok + best.queries() - 1) / best.queries()));
    for (int i = 1; i < 4; ++i) {
        const StagedShape s = kStagedShapes[i];
        if (s.qw == 16 && n_tok <= s.queries() && n_ctx <= 512) continue;
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
constexpr int64_t staged_full_units(int64_t units, int n_tok, int n_ctx) {
    auto cost = [=](int64_t n) {
        const StagedShape s = staged_shape(n, n_tok, n_ctx);
        return staged_cost(s, n * ((n_tok + s.queries() - 1) / s.queries()));
    };
    const int64_t n_qt = (n_tok + kStagedShapes[0].queries() - 1) / kStagedShapes[0].queries();
    const int64_t rounds = units * n_qt / 256;
    const int64_t full = rounds * 256 / n_qt;
    if (full == 0 || full == units) return 0;
    return (double) rounds + 0.05 + cost(units - full) < 0.95 * cost(units) ? full : 0;
}
static_assert(staged_full_units(160, 500, 1000) == 128 && staged_full_units(512, 256, 512) == 0,
              "a quarter of a round goes apart, full rounds do not");
static_assert(staged_shape(512, 256, 1024).qw == 16 && staged_shape(512, 256, 1024).ks == 1, "full rounds: 256 queries");
static_assert(staged_shape(32, 500, 1024).qw == 8 && staged_shape(32, 500, 1024).ks == 2, "256 workgroups of 64 queries");
static_assert(staged_shape(64, 500, 1024).qw == 16 && staged_shape(64, 500, 1024).ks == 2, "256 workgroups of 128 queries");

}  // namespace bmo
