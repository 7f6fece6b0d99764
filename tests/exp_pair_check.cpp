// Host build of the regular kernels' exponentials (cqbem_device.hpp: exp_table_plan, fill_exp_node, exp_pair), for
// tests/test_exp_pair.py.  Reads "s/c1 (x y) s/c2 (x y) reach n", then n distances; prints whether the frequency is beyond the
// table's reach, and for each distance the pair by the table (0s beyond its reach) and by the direct functions, as hex doubles.
#include "../surfaceonlydeformables_amd/csrc/cqbem_device.hpp"

#include <cstdio>

using namespace cqbem;

int main() {
    static const double E[64][2] = CQBEM_EXP_TABLE;
    static const double T[64][4] = CQBEM_TRIG_TABLE;
    static MathTables M;
    for (int k = 0; k < 64; k++) {
        M.e[k] = make_double2(E[k][0], E[k][1]);
        M.t[k] = make_double4(T[k][0], T[k][1], T[k][2], T[k][3]);
    }
    static double2 tab[kExpWords];
    Freq f{};
    double reach;
    int n;
    while (std::scanf("%lf %lf %lf %lf %lf %d", &f.sc1.x, &f.sc1.y, &f.sc2.x, &f.sc2.y, &reach, &n) == 6) {
        exp_table_plan(f, exp_table_cell(reach));
        TableFreq t{};
        t.sc1 = f.sc1, t.sc2 = f.sc2, t.h = f.h, t.ih = f.ih;
        for (int c = 0; c < 2; c++)
            for (int k = 0; k < kExpDeg; k++) t.q[c][k] = f.q[c][k];
        for (int k = 0; k < kExpCoarse - 1 + kExpFine && !f.direct; k++) fill_exp_node(t, k, tab);
        std::printf("%d\n", f.direct);
        for (int k = 0; k < n; k++) {
            double r;
            if (std::scanf("%lf", &r) != 1) return 1;
            const PointFreq<cd> p = t;
            const cd z1 = f.sc1 * r, z2 = f.sc2 * r;
            cd a{0, 0}, b{0, 0}, c, d;
            if (!f.direct) exp_pair(r, z1, z2, t, tab, a, b);
            exp_pair(r, z1, z2, p, reinterpret_cast<const double2 *>(&M), c, d);
            std::printf("%a %a %a %a %a %a %a %a\n", a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y);
        }
    }
    return 0;
}
