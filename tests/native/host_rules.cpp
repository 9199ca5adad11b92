// Prints the library's host-side choices for a case, for tests/test_host_rules.py.
//   host_rules leg DIM N0 N1 N2 P0 P1 P2 NU F32 BOXES: waves of the block in
//     which a multigrid level of N cells with periodic axes P runs its legs
//     (0: sweep by sweep); BOXES: a level whose couplings differ.
//   host_rules coop DIM N0 N1 N2: workgroups of the cooperative solve (0: the
//     grid does not fit) and their LDS bytes.
//   host_rules spread DIM N0 N1 N2 BLOCKS: whether a device that holds so many
//     blocks runs the cooperative solve, the blocks launched and the launches
//     tried, and the same for the next launch.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include <type_traits>

#include "cf_mg.hpp"

using namespace cfmi;

// The launch takes the plan that its caller keeps, and makes none.
static_assert(std::is_same<decltype(&launch_pcg_solve_coop<double>),
                           bool (*)(const Geo&, CoopPlan&, double*, double*, double*,
                                    PcgState*, void*, unsigned&, int, hipStream_t)>::value,
              "a launch of the cooperative solve is given its plan");

static int leg(char** a)
{
    MgLev L{};
    L.dim = std::atoi(a[0]);
    for (int d = 0; d < 3; ++d) {
        L.n[d] = std::atoi(a[1 + d]);
        L.periodic[d] = std::atoi(a[4 + d]);
        L.coarsen[d] = d < L.dim && L.n[d] > 2;
    }
    MgFused f{};
    const bool fused = mg_fused_level(L, std::atoi(a[7]), std::atoi(a[8]) != 0,
                                      std::atoi(a[9]) ? 0.0 : -1.0, f);
    std::printf("%d\n", fused ? f.waves : 0);
    return 0;
}

static Geo grid(char** a)
{
    Geo g{};
    g.dim = std::atoi(a[0]);
    g.h = 1;
    for (int d = 0; d < 3; ++d)
        g.n[d] = std::atoi(a[1 + d]);
    g.px = g.n[0] + 3;
    g.py = g.n[1] + 3;
    return g;
}

static int spread(char** a)
{
    CoopPlan c = coop_plan(grid(a));
    const int blocks = std::atoi(a[4]);
    int& every = c.strips.G ? c.strips.every : c.pencils.every;
    for (int launches = 0; launches < 2; ++launches) {
        int tried = 0;
        const bool ran = coop_spread(every, [&](int e) {
            ++tried;
            return c.groups * e <= blocks;
        });
        std::printf("%d %d %d ", (int)ran, c.groups * every, tried);
    }
    std::printf("\n");
    return 0;
}

static int coop(char** a)
{
    const CoopPlan c = coop_plan(grid(a));
    std::printf("%d %zu\n", c.groups, c.lds);
    return 0;
}

int main(int argc, char** argv)
{
    if (argc == 12 && !std::strcmp(argv[1], "leg"))
        return leg(argv + 2);
    if (argc == 6 && !std::strcmp(argv[1], "coop"))
        return coop(argv + 2);
    if (argc == 7 && !std::strcmp(argv[1], "spread"))
        return spread(argv + 2);
    return 2;
}
