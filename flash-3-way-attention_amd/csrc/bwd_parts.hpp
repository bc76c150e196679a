// Workgroups per query tile ("parts") of the 16-bit triple-dot backward at D = 64.  Host code alone, of plain numbers.
#pragma once
#include <algorithm>

namespace tritt {

struct BwdPartsCall {
    int BH, T;
    int k1_window, k2_window, kk_left, kk_right;
    int roles;      // of the two, {dq, dk2, dv2} and {dk1, dv1}, those whose gradients the caller wants
    bool one_grid;  // they run in one grid (tdp_bwd_rows_kernel); else in launches of their own (tdp_bwd_rows_general_kernel)
};

// Under a window, by the time that a launch takes with s parts: one workgroup fills a CU, and all tiles but those at the start
// of the sequence cost the same, so it takes the larger of whole rounds of the full tiles' parts over the CUs and of the even
// share plus some of a part of tail.  Work in 32-key steps of eight rows; a part's own prologue, dQ's shares and tail are worth
// about nine of them.  The kernel that has both roles in one grid is modelled with both roles' parts and a third of a part of
// tail; the other one, whose launches each fill and empty the chip, with one role's and half a part.  The model of the one for
// the other costs up to 28 %: training steps, bf16, one grid's model -> a launch's, k-k bands of 50 and 25: B=1 H=2 T=512
// window 200 206 -> 161 us, T=1999 window 100 258 -> 197, B=2 H=8 T=300 window 100 261 -> 199, B=1 H=8 T=700 window 200 500 -> 450.
// In one grid, the parts it chooses (the best otherwise): B=2 H=4 T=2048 window 512 3 parts 5.52 ms (1 to 12: 6.01 5.64 5.52 5.57
// 5.59 5.65 5.70), B=1 H=8 T=700 window 100 3 parts 259 us, B=2 H=8 T=2048 window 100 1 part 1.23 ms, B=1 H=4 T=1500 window 300
// 3 parts 934 us, B=4 H=8 T=1024 window 200 1 part 2.52 ms, B=1 H=2 T=1999 window 77 1 part 167 us, all the best; B=1 H=16 T=1024
// window 400 3 parts 3.10 ms (1 part 3.05).
inline int windowed_parts(const BwdPartsCall& a) {
    constexpr float kPart = 9.f;
    constexpr int kCus = 256;
    const int nqt = (a.T + 31) / 32, rows = std::min(a.k2_window, a.T - 1) + 32, roles = a.one_grid ? a.roles : 1;
    const int keys = std::min(std::min(a.k1_window, a.T - 1) + 32, a.kk_left + a.kk_right + 8);
    const float w = (float)((rows + 7) / 8) * (float)((keys + 31) / 32);  // of a tile past the start of the sequence
    const float tail = a.one_grid ? 0.3f : 0.5f;
    const int full = a.BH * std::max(nqt - rows / 32, 0), light = a.BH * std::min(nqt, rows / 32);
    const float total = ((float)full + 0.36f * (float)light) * w;
    int best = 1;
    float least = 3.0e38f;
    for (int s : {1, 2, 3, 4, 6, 8, 12, 16}) {
        const float part = kPart + w / (float)s;
        const float t = std::max((float)((roles * full * s + kCus - 1) / kCus) * part,
                                 (float)roles * ((float)(full + light) * (float)s * kPart + total) / kCus + tail * part);
        if (t < least) least = t, best = s;
    }
    return best;
}

// Under a full causal mask, for grids of less than 1024 tiles (both roles in one grid).  The work of a tile grows with the square
// of its position and the heaviest parts start first, so the grid of both roles takes the even share of all parts over the CUs
// and 0.3 of its longest part of tail, and no less than 1.5 of its longest part (which starts late by what the parts before it
// differ, and shares the chip with the other role's).  Work in 32-key steps of eight rows; a part's own prologue, dQ's shares and
// tail are worth about twelve of them.  Training steps, the parts it chooses and the best: B=2 H=4 T=256 6 parts 144 us (1 to 16: 298
// 190 150 145 144 147 155 156), B=4 H=8 T=128 2 parts 127, T=256 2 parts 376, B=1 H=2 T=1500 16 parts 2.84 ms, B=1 H=8 T=700 6
// parts 1.22, all the best; B=1 H=2 T=512 12 parts 234 us (16: 229), B=4 H=8 T=64 3 parts 74 (4: 71), T=700 3 parts 4.94 ms (1: 4.86).
// Without the tail (the longer of the two alone) B=1 H=8 T=700 took 3 parts and 1.26 ms, B=1 H=2 T=1500 6 parts and 2.98, B=2 H=8
// T=1500 1 part and 21.4 (with it 6: 20.8; 2: 20.6).
// D = 32 and 128 measure within 1 % of their best at 1024 workgroups.
inline int causal_parts(const BwdPartsCall& a) {
    constexpr float kPart = 12.f;
    constexpr int kCus = 256;
    const int nqt = (a.T + 31) / 32;
    const float w = (float)((a.T + 7) / 8) * (float)nqt;  // the last tile's
    const float total = (float)a.BH * w * (float)((nqt + 1) * (2 * nqt + 1)) / (float)(6 * nqt);  // a sum of squares
    int best = 1;
    float least = 3.0e38f;
    for (int s : {1, 2, 3, 4, 6, 8, 12, 16}) {
        const float part = kPart + w / (float)s;
        const float t = std::max(1.5f * part, (float)a.roles * (total + (float)(a.BH * nqt * s) * kPart) / kCus + 0.3f * part);
        if (t < least) least = t, best = s;
    }
    return best;
}

}  // namespace tritt
