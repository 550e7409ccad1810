// Prints the library's plans without a GPU: one line of input, one of output.
//   default VARIANT N n CUS      -> variant i_per_lane jslice nslices li
#include "nbody_internal.h"

#include <cstdio>
#include <iostream>
#include <string>

using namespace nbody;

int main()
{
    std::string what;
    while (std::cin >> what) {
        int variant, cus;
        size_t N, n;
        std::cin >> variant >> N >> n >> cus;
        const ForcePlan p = detail::default_plan(variant, N, n, cus, nullptr);
        std::printf("%d %d %d %d %d\n", p.variant, p.ipl, p.jslice, p.nslices, p.li);
    }
    return 0;
}
