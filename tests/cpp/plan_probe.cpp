// Prints what the engine's host rules (tmc_amd/csrc/dmc_plan.h) answer.
//   plan_probe key nx ny nz [nx ny nz ...]   the pass key of volumes, everything else equal (hex)
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
    return 2;
}
