// Host build of the patch kernel's division of a rule over the waves that share a chunk (cqbem_kernels.hpp:
// part_has_points, each_part_point),
// for tests/test_far_rule_parts.py: for every "npts split" read from stdin prints the points that the parts take, in part
// order, "-" after each part.
#include "../surfaceonlydeformables_amd/csrc/cqbem_kernels.hpp"

#include <cstdio>

int main() {
    int npts, split;
    while (std::scanf("%d %d", &npts, &split) == 2) {
        for (int part = 0; part < split; part++) {
            if (cqbem::part_has_points(npts, part))
                cqbem::each_part_point(npts, split, part, [](int q, auto) { std::printf("%d ", q); });
            std::printf("- ");
        }
        std::printf("\n");
    }
    return 0;
}
