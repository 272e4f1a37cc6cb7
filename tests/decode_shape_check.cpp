// Prints the workgroup shape of each decode call read from standard input, a
// line each: units, layers, groups, query heads per kv head, fused (0 or 1) and
// the forced shape (- for none) in; waves per unit, groups in flight, heads per workgroup and the launch's
// threads out.  Built by tests/Makefile; tests/_shapes.py runs it.
#include <cinttypes>
#include <cstdio>

#include "decode_shape.hpp"

int main() {
    int64_t units;
    int n_layers, n_groups, q_per_kv, fused;
    char forced[32];
    while (std::scanf("%" SCNd64 " %d %d %d %d %31s", &units, &n_layers, &n_groups, &q_per_kv, &fused, forced) == 6) {
        const bmo::Shape s = bmo::pick_shape(units, n_layers, n_groups, q_per_kv, fused != 0,
                                             forced[0] == '-' ? nullptr : forced);
        std::printf("%d %d %d %" PRIu64 "\n", s.nw, s.pf, s.r, bmo::launch_threads(units, s));
    }
    return 0;
}
