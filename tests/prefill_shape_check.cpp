// Prints the shapes of each staged prefill call read from standard input, a
// line each: units, tokens and slots in; the units that go ahead in full rounds, and
// the waves per workgroup and waves per block of 16 queries of the rest, out.
// Built by tests/Makefile; tests/_shapes.py runs it.
#include <cinttypes>
#include <cstdio>

#include "prefill_shape.hpp"

int main() {
    int64_t units;
    int n_tok, n_ctx;
    while (std::scanf("%" SCNd64 " %d %d", &units, &n_tok, &n_ctx) == 3) {
        const int64_t full = bmo::staged_full_units(units, n_tok, n_ctx);
        const bmo::StagedShape s = bmo::staged_shape(units - full, n_tok, n_ctx);
        std::printf("%" PRId64 " %d %d\n", full, s.qw, s.ks);
    }
    return 0;
}
