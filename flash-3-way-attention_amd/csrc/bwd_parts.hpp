// Workgroups per query tile ("parts") of the 16-bit triple-dot backward at D = 64 under a causal mask, by the time that a launch
// takes with s of them.  Host code alone, of plain numbers.  Work is counted in 32-key steps of eight rows; one workgroup fills a CU;
// a part's own prologue, dQ's shares and tail are worth about twelve steps beside the other role's parts, nine in a launch alone.
#pragma once
#include <algorithm>

namespace tritt {

struct BwdPartsCall {
    int BH, T;
    int k1_window, k2_window, kk_left, kk_right;  // (no window: T)
    int roles;  // of the two, {dq, dk2, dv2} and {dk1, dv1}, those whose gradients the caller wants
};
constexpr int kBwdParts[] = {1, 2, 3, 4, 6, 8, 12, 16};

// Both roles in one grid (tdp_bwd_rows_kernel), heaviest tiles first, from tile 1 on (tile 0 takes the fp32 kernel).  It takes the
// longest of: 1.3 of a heaviest part; the even share of all parts over the CUs and 0.3 of a heaviest part of tail; and, where many
// tiles cost the same, whole rounds of those.  Training steps, bf16, the parts it chooses (the best): B=2 H=4 T=256 6 parts 144 us (1
// to 16: 298 190 150 145 144 147 155 156), B=4 H=8 T=128 2 parts 127, T=256 2 parts 376, B=1 H=2 T=1500 16 parts 2.84 ms, B=1 H=8 T=700
// 6 parts 1.22, B=2 H=4 T=2048 window 512 3 parts 5.23, B=4 H=8 T=1024 window 200 1 part 2.49, B=1 H=8 T=90 window 70 8 parts 71 us (6:
// 70), T=128 window 100 6 parts 97; B=1 H=2 T=512 12 parts 234 (16: 229), B=6 H=8 T=160 window 70 1 part 231 (2: 221), B=2 H=8 T=1000
// window 200 1 part 1.40 ms (2: 1.35), B=1 H=2 T=512 window 200 6 parts 163 us (8: 149).  Over 190 shapes it is 0.6 % from the best in the
// mean.  (A sum of squares in the place of the tiles' own work, and no tail, were 1.2 to 2.1 % from it and up to 16.)
inline int one_grid_parts(const BwdPartsCall& a) {
    constexpr float kPart = 12.f;
    constexpr int kCus = 256;
    auto work = [&](int q0) {
        const int q1 = std::min(q0 + 31, a.T - 1);
        const int rows = q1 - std::max(0, q0 - std::min(a.k2_window, a.T)) + 1;
        const int keys = std::min(q1 - std::max(0, q0 - std::min(a.k1_window, a.T)) + 1, a.kk_left + a.kk_right + 8);
        return (float)((rows + 7) / 8) * (float)((keys + 31) / 32);
    };
    const int nqt = (a.T + 31) / 32;
    float total = 0.f, most = 1.f;
    for (int t = 1; t < nqt; ++t) {
        const float w = work(32 * t);
        total += w;
        most = std::max(most, w);
    }
    long long full = 0;  // tiles that cost nearly the most
    for (int t = 1; t < nqt; ++t) full += work(32 * t) >= 0.9f * most;
    const float grid = (float)a.roles * (float)a.BH;
    int best = 1;
    float least = 3.0e38f;
    for (int s : kBwdParts) {
        const float part = kPart + most / (float)s;
        const long long rounds = (a.roles * a.BH * full * s + kCus - 1) / kCus;
        const float share = grid * (total + (float)((nqt - 1) * s) * kPart) / kCus + 0.3f * part;
        const float t = std::max(std::max(1.3f * part, share), (float)rounds * part);
        if (t < least) least = t, best = s;
    }
    return best;
}

// A launch per role (tdp_bwd_rows_general_kernel under a window): each fills and empties the chip.  All tiles but those at the start
// of the sequence cost the same, so it takes the larger of whole rounds of the full tiles' parts over the CUs and of the even share and
// half a part of tail.  The other model's parts cost up to 28 % here: training steps, bf16, the grid's -> a launch's, k-k bands of 50 and
// 25: B=1 H=2 T=512 window 200 206 -> 161 us, T=1999 window 100 258 -> 197, B=2 H=8 T=300 window 100 261 -> 199, B=1 H=8 T=700 window 200
// 500 -> 450.
inline int launch_parts(const BwdPartsCall& a) {
    constexpr float kPart = 9.f;
    constexpr int kCus = 256;
    const int nqt = (a.T + 31) / 32, rows = std::min(a.k2_window, a.T - 1) + 32;
    const int keys = std::min(std::min(a.k1_window, a.T - 1) + 32, a.kk_left + a.kk_right + 8);
    const float w = (float)((rows + 7) / 8) * (float)((keys + 31) / 32);  // of a tile past the start of the sequence
    const int full = a.BH * std::max(nqt - rows / 32, 0), light = a.BH * std::min(nqt, rows / 32);
    const float total = ((float)full + 0.36f * (float)light) * w;
    int best = 1;
    float least = 3.0e38f;
    for (int s : kBwdParts) {
        const float part = kPart + w / (float)s;
        const float t = std::max((float)((full * s + kCus - 1) / kCus) * part,
                                 ((float)(full + light) * (float)s * kPart + total) / kCus + 0.5f * part);
        if (t < least) least = t, best = s;
    }
    return best;
}

}  // namespace tritt
