// Which way a batch's small trajectories run (qs_batch_rule.hpp), for batches
// whose both ways were timed on the device.  Prints "ok" or what differs.
#include <cstdio>
#include <string>
#include <vector>

#include "../../qpp_amd/csrc/qs_batch_rule.hpp"

using namespace qs_batch_rule;

int main() {
    // passes of the depth-30 ladder circuits
    auto circuit = [](uint32_t n, uint64_t count) {
        const int passes = n <= 12 ? 15 : n <= 14 ? 19 : n <= 16 ? 23 : n <= 20 ? 30 : 40;
        return Circuit{n, count, std::vector<uint64_t>(passes, uint64_t{1} << (n - 12))};
    };
    const Machine c64{false, 4 * 256, 3 * 256, false}, c128{true, 2 * 256, 2 * 256, false};
    Machine exact = c128;
    exact.force_exact = true;
    struct Case {
        const char* name;
        const Machine* m;
        std::vector<Circuit> batch;
        bool by_pass;
    };
    std::vector<Circuit> each;  // many circuits of one trajectory each
    for (int i = 0; i < 64; ++i) each.push_back(circuit(16, 1));
    const Case cases[] = {
        {"c128 192x16", &c128, {circuit(16, 192)}, true},
        {"c128 192x16 + 16x20", &c128, {circuit(16, 192), circuit(20, 16)}, true},
        {"c128 1024x16", &c128, {circuit(16, 1024)}, true},
        {"c128 3000x12", &c128, {circuit(12, 3000)}, true},
        {"c128 10000x14", &c128, {circuit(14, 10000)}, true},
        {"c128 16x12", &c128, {circuit(12, 16)}, true},
        {"c128 2000x12 + 8x22", &c128, {circuit(12, 2000), circuit(22, 8)}, false},
        {"c128 64 circuits of one", &c128, each, false},
        {"c128 192x16 + 16x22, replayed", &exact, {circuit(16, 192), circuit(22, 16)}, false},
        {"c64 16x12", &c64, {circuit(12, 16)}, false},
        {"c64 1024x16", &c64, {circuit(16, 1024)}, true},
        {"c64 1024x16 + 128x{12,20,22}", &c64,
         {circuit(16, 1024), circuit(12, 128), circuit(20, 128), circuit(22, 128)}, false},
        {"c64 1000x14 + 64x22", &c64, {circuit(14, 1000), circuit(22, 64)}, false},
        {"c64 4096x16 + 512x{12,20,22}", &c64,
         {circuit(16, 4096), circuit(12, 512), circuit(20, 512), circuit(22, 512)}, true},
    };
    int bad = 0;
    for (const Case& c : cases)
        if (small_pass_by_pass(c.batch, *c.m) != c.by_pass) {
            std::printf("%s: pass by pass is %d\n", c.name, int(!c.by_pass));
            ++bad;
        }
    if (!bad) std::printf("ok\n");
    return bad;
}
