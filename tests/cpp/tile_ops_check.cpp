// Kinds of the ops in a program as the tile kernel runs it (native_fuse), for
// gates read from stdin: nb, low_bits, max_ops, the number of gates, then per
// gate its number of bits, the bits, cmask, cval and the matrix (column-major
// re im pairs).  Prints the counts of the select ops by their condition.
#include <cstdio>
#include <vector>

#include "../../qpp_amd/csrc/qs_fused.hpp"

namespace qs {
FusedProgram native_fuse(const FusedProgram& P);
}

int main() {
    unsigned nb, low, ng;
    unsigned long long max_ops;
    if (std::scanf("%u %u %llu %u", &nb, &low, &max_ops, &ng) != 4) return 2;
    std::vector<BitGate> gates(ng);
    for (BitGate& g : gates) {
        unsigned k;
        unsigned long long cm, cv;
        if (std::scanf("%u", &k) != 1) return 2;
        g.bits.resize(k);
        for (uint32_t& b : g.bits)
            if (std::scanf("%u", &b) != 1) return 2;
        if (std::scanf("%llu %llu", &cm, &cv) != 2) return 2;
        g.cmask = cm;
        g.cval = cv;
        g.m.resize(size_t{1} << (2 * k));
        for (auto& v : g.m) {
            double re, im;
            if (std::scanf("%lf %lf", &re, &im) != 2) return 2;
            v = {re, im};
        }
    }
    FusedOptions o;
    o.low_bits = low;
    o.max_ops = max_ops;
    FusedProgram P;
    if (qs::fused_compile(gates, nb, o, P)) return 3;
    const FusedProgram Q = qs::native_fuse(P);
    int u1_lane = 0, u1_tile = 0, u2_tile = 0, both = 0;
    for (const FOp& op : Q.ops) {
        if (op.kind != OP_U1S && op.kind != OP_U2S) continue;
        both += op.tmask != 0 && op.omask != 0;
        (op.kind == OP_U2S ? u2_tile : op.tmask ? u1_lane : u1_tile) += 1;
        both += op.kind == OP_U2S && op.tmask != 0;  // the tile kernel has no such case
    }
    std::printf("%d %d %d %d\n", u1_lane, u1_tile, u2_tile, both);
    return 0;
}
