// Prints the workgroup shape of each decode call read from standard input, a
// line each: units, layers, groups, query heads per kv head and fused (0 or 1)
// in; waves per unit, groups in flight, heads per workgroup and the launch's
// threads out.  Built by tests/Makefile; tests/_shapes.py runs it.
#include <cinttypes>
#include <cstdio>

#include "decode_shape.hpp"

int main() {
    int64_t units;
    int n_layers, n_groups, q_per_kv, fused;
    while (std::scanf("%" SCNd64 " %d %d %d %d", &units, &n_layers, &n_groups, &q_per_kv, &fused) == 5) {
        const bmo::Shape s = bmo::default_shape(units, n_layers, n_groups, q_per_kv, fused != 0);
        std::printf("%d %d %d %" PRIu64 "\n", s.nw, s.pf, s.r, bmo::launch_threads(units, s));
    }
    return 0;
}
