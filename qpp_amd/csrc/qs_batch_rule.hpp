// qs_batch_rule.hpp -- which way a batch's small trajectories run (host).
#ifndef QPP_AMD_QS_BATCH_RULE_HPP_
#define QPP_AMD_QS_BATCH_RULE_HPP_

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

namespace qs_batch_rule {

// Trajectories of at least this many qubits always run pass by pass: one
// workgroup that streams a state of 2^18 amplitudes and more tile after tile
// is bound by its own latency.
constexpr uint32_t kWideBits = 18;

struct Circuit {
    uint32_t qubits;
    uint64_t count;               // trajectories of it in the batch
    std::vector<uint64_t> tiles;  // workgroups of each of its passes
};

struct Machine {
    bool f64;              // complex128
    uint64_t pass_groups;  // resident workgroups of k_traj_pass on the device
    uint64_t traj_groups;  // and of k_traj
    bool force_exact;      // every outcome is replayed exactly
};

// Whether trajectories of fewer than kWideBits qubits are expected to end no
// later when they run pass by pass (k_traj_pass, a workgroup per tile, before
// k_traj measures them) than with a workgroup each in k_traj.  Both ways in
// rounds of k_traj_pass's resident workgroups, 40 us:
//  - pass by pass, the launches of every circuit follow each other, each as
//    many rounds as its tiles take;
//  - with a workgroup each, a tile and pass takes 44 us where a CU holds one
//    workgroup and 56 where it holds two (complex64 29, and 48 at three): the
//    longest trajectory at the first rate, or all of them at the second;
//  - meanwhile the wide trajectories are measured, 2.4 us a tile of 4096
//    amplitudes, and an outcome within rounding of an edge (of N amplitudes
//    about 8 N^2 2^-53 of the draws) is replayed by its workgroup, 12 us a
//    tile.  Small trajectories with a workgroup each run beside that, passes
//    of theirs come before it.
// complex128 and complex64, ms with a workgroup each and pass by pass: 192
// trajectories of 16 qubits 16.4 and 5.9, 10.8 and 3.2; 1024 of 16 41 and 29,
// 23.6 and 15.0; 3000 of 12 6.5 and 4.8, 3.0 and 2.6; 16 of 12 0.90 and 0.71,
// 0.61 and 0.68.  1024 of 16 and 128 each of 12, 20 and 22 qubits in
// complex64 (two 22-qubit outcomes replayed, 15 ms): 200 and 207.
inline bool small_pass_by_pass(const std::vector<Circuit>& circuits, const Machine& m) {
    double passes = 0, longest = 0, all = 0, tail = 0;
    for (const Circuit& c : circuits) {
        if (!c.count) continue;
        if (c.qubits >= kWideBits) {
            const double N = std::ldexp(1.0, int(c.qubits)), tiles = N / 4096;
            const double replays = double(c.count) * std::min(1.0, std::ldexp(8 * N * N, -53));
            const double any = m.force_exact ? 1.0 : 1 - std::exp(-replays);
            tail = std::max(tail, tiles * (0.06 + 0.3 * any));
            continue;
        }
        double tiles = 0;
        for (uint64_t t : c.tiles) {
            passes += double((c.count * t + m.pass_groups - 1) / m.pass_groups);
            tiles += double(t);
        }
        longest = std::max(longest, tiles);
        all += tiles * double(c.count);
    }
    const double alone = m.f64 ? 1.1 : 0.72, full = m.f64 ? 1.4 : 1.2;
    const double each = std::max(alone * longest, full * all / double(m.traj_groups));
    return passes + tail <= std::max(each, tail);
}

}  // namespace qs_batch_rule

#endif  // QPP_AMD_QS_BATCH_RULE_HPP_
