// Host build of the batched tuner's cut (idi_amd/csrc/planner.hpp: tuning_offsets) for
// tests/test_tuning_cpu.py, with sanitizers.  Input (stdin): npix cap nshots offset_0 .. offset_nshots, case
// after case.  Output, a line per case: the offsets of what is timed.
#include "../../idi_amd/csrc/planner.hpp"

#include <cstdio>
#include <vector>

int main()
{
    double npix, cap;
    long nshots;
    while (std::scanf("%lf %lf %ld", &npix, &cap, &nshots) == 3) {
        std::vector<int64_t> off((size_t)nshots + 1);
        for (int64_t& o : off) {
            long v;
            if (std::scanf("%ld", &v) != 1) return 2;
            o = v;
        }
        const std::vector<int64_t> t = idisim::tuning_offsets(off.data(), nshots, npix, cap);
        for (size_t i = 0; i < t.size(); ++i) std::printf(i ? " %ld" : "%ld", (long)t[i]);
        std::printf("\n");
    }
    return 0;
}
