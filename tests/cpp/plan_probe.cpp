// Prints what the engine's host rules (tmc_amd/csrc/dmc_plan.h) answer.
//   plan_probe key nx ny nz [nx ny nz ...]   the pass key of volumes, everything else equal (hex)
//   plan_probe groups n rs [n rs ...]        group shift of n volumes of rs (row, segment)s each, and these padded
//   plan_probe blocks n per_block limit grid_cap
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../tmc_amd/csrc/dmc_plan.h"

int main(int argc, char** argv) {
    if (argc > 4 && !strcmp(argv[1], "key")) {
        tmc::PassShape s{};
        for (int i = 2; i < argc; i++) s.dims.push_back(atoi(argv[i]));
        for (unsigned char c : tmc::pass_key(s)) printf("%02x", c);
        printf("\n");
        return 0;
    }
    if (argc == 6 && !strcmp(argv[1], "blocks")) {
        printf("%lld\n", (long long)tmc::blocks_for(atoll(argv[2]), atoll(argv[3]), atoll(argv[4]), atoll(argv[5])));
        return 0;
    }
    if (argc > 3 && !strcmp(argv[1], "groups")) {
        std::vector<int64_t> rs;
        for (int i = 2; i + 1 < argc; i += 2) rs.insert(rs.end(), atoi(argv[i]), atoll(argv[i + 1]));
        const int shift = tmc::group_shift(rs);
        int64_t padded = 0;
        for (int64_t x : rs) padded += tmc::in_groups(x, shift);
        printf("%d %lld\n", shift, (long long)padded);
        return 0;
    }
    return 2;
}
