// kk_lstm.h -- how many blocks the BiLSTM recurrences split a sequence over (host only).
//
// The blocks of a sequence wait for each other every step, so a launch must never hold slots with
// blocks whose partners cannot get one.  The rule and why it holds:
// * Block B of a launch is part (B / 8) mod P of group 8 (B / 8P) + B mod 8: 8 P consecutive blocks
//   hold 8 complete groups, the parts of one 8 apart, hence on one XCD (blocks go to the 8, 4, 2 or 1
//   XCDs of the device or partition in turn).  A launch's blocks start in order (on each XCD), and a
//   complete group ends without waiting on anything else.  So once the complete groups have ended, a
//   launch holds at most 8 (P - 1) slots: P - 1 parts of each of the 8 groups that it is in the middle of.
// * A hardware queue starts one launch's blocks before the next one's, so at most one launch per queue
//   is in the middle, and a process has four queues (HIP's default).  A context runs two recurrences at
//   once, the text encoder's beside the duration encoder's; several contexts share the queues.
// * While 4 * 8 (P - 1) is less than the device's slots, some launch can always start its next block,
//   and every group completes.  256 CUs: 480 of 512 slots at P = 16, 224 of 512 at 8, 96 of 256 at 4,
//   32 of 256 for the pairs; per XCD 60 of 64, 28 of 64, 12 of 32, 4 of 32.
// * Recurrences of other processes come on top (each with queues of its own): from the fifth launch in
//   the middle the slots can run out at P = 16.  Then the kernels' bounded waits end the launch and the
//   run is repeated on the one-CU kernel: time (the 2 s wait), not a wrong result.
#pragma once
#include <cstdint>

namespace kk {

constexpr int kLstmGroups = 64;              // groups of a launch at most: 256 CUs in groups of 4
constexpr int64_t kLstmQuadMinSteps = 1024;  // past 64 sequences: groups when a span has this many steps, else pairs
constexpr int kLstmAtOnce = 4;               // launches whose blocks start at the same time

inline int lstm_groups(int nb) { return 2 * nb < kLstmGroups ? 2 * nb : kLstmGroups; }

// Blocks that one CU holds: the kernels of 8 and 16 parts are compiled for two (their launch bounds), the
// one of 4 takes 176 registers per thread and the pairs most of the LDS.
constexpr int lstm_blocks_per_cu(int parts) { return parts >= 8 ? 2 : 1; }

constexpr bool lstm_fits(int parts, int n_cu) {
    return kLstmAtOnce * 8 * (parts - 1) < lstm_blocks_per_cu(parts) * n_cu;
}

// The blocks per sequence for nb items, the longest span of `longest` steps, on n_cu CUs: the most that
// fit (lstm_fits) and put every sequence's blocks on CUs of their own -- the fewer sequences, the
// shorter a step; groups of 4 also run lists of sequences when a span is long; else pairs.
// sel: 0 pairs, 1 groups wherever they fit, -1 by the rule.
inline int lstm_parts(int nb, int64_t longest, int n_cu, int64_t sel = -1) {
    if (sel == 0) return 2;
    const int g = lstm_groups(nb);
    for (int parts = 16; parts >= 8; parts /= 2)
        if (lstm_fits(parts, n_cu) && parts * g <= n_cu) return parts;
    const bool at_once = 2 * nb == g && 4 * g <= n_cu;
    return lstm_fits(4, n_cu) && (sel > 0 || at_once || longest >= kLstmQuadMinSteps) ? 4 : 2;
}

}  // namespace kk
