// Prints the library's plans without a GPU: one line of input, one of output.
//   default VARIANT N n CUS -> variant i_per_lane jslice nslices li
//   newton VARIANT N n CUS  -> the same with a Newton step
//   tile n ni ACC64 CUS     -> li i_per_lane
//   tasks N CUS             -> tasks per block pair of the symmetric plan's blocks of 512
//   lead TASKS CUS OCC      -> whether that launch's first halves go first
//   tuned VARIANT N CUS     -> how many plans autotune times, and how many of them are the default
#include "nbody_internal.h"

#include <cstdio>
#include <iostream>
#include <string>

using namespace nbody;

int main()
{
    std::string what;
    while (std::cin >> what) {
        if (what == "default" || what == "newton") {
            int variant, cus;
            size_t N, n;
            std::cin >> variant >> N >> n >> cus;
            const nbody_hip_options o{variant, 0, 0, -1, what == "newton" ? 1 : 0, 0, 0};
            const ForcePlan p = detail::default_plan(variant, N, n, cus, &o);
            std::printf("%d %d %d %d %d\n", p.variant, p.ipl, p.jslice, p.nslices, p.li);
        } else if (what == "tile") {
            size_t n, ni;
            int acc64, cus, li = 0, ipl = 0;
            std::cin >> n >> ni >> acc64 >> cus;
            tile_shape(n, ni, acc64 != 0, cus, &li, &ipl);
            std::printf("%d %d\n", li, ipl);
        } else if (what == "tasks") {
            size_t N;
            int cus;
            std::cin >> N >> cus;
            nbody_hip_options o{NBODY_HIP_SYMMETRIC, 8, 512, -1, 0, 0, 0};
            const ForcePlan p = detail::default_plan(VAR_SYMMETRIC, N, N, cus, &o);
            const size_t one = (size_t)12 * 512 * p.nslices * p.nslices;
            std::printf("%zu\n", plan_scratch_bytes(p, (int)N) / one);
        } else if (what == "tuned") {
            int variant, cus, same = 0;
            size_t N;
            std::cin >> variant >> N >> cus;
            const ForcePlan p = detail::default_plan(variant, N, N, cus, nullptr);
            const auto all = detail::tune_candidates(variant, N, cus);
            for (const ForcePlan& c : all)
                same += c.li == p.li && c.ipl == p.ipl && c.jslice == p.jslice && c.nslices == p.nslices &&
                        c.comp == p.comp;
            std::printf("%zu %d\n", all.size(), same);
        } else if (what == "lead") {
            ForcePlan p;
            int tasks;
            std::cin >> tasks >> p.cus >> p.occ;
            std::printf("%d\n", deal_leads(p, tasks) ? 1 : 0);
        }
    }
    return 0;
}
