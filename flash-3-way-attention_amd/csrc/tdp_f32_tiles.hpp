// The deal of query and key tiles to workgroups, shared by the fp32 triple-dot kernels (tdp_f32_mfma.hip has the description),
// and the fp32 query tiles of a 16-bit backward on v_mfma_f32_32x32x2_f32: their statistics pass and their backward, as a
// header because the 16-bit backward appends the workgroups of query tile 0 to its own grid (tdp_bwd_mfma.hip).
#pragma once
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "mfma.hpp"

namespace tritt {
namespace {

constexpr int kF32Waves = 8;
constexpr float kNegBig = -1.0e30f;  // finite stand-in for "no maximum yet"

__device__ __forceinline__ f32x16 mma_f32(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Ranges of streamed rows / owner rows a tile of queries [q0, q1] can touch.
struct Range {
    int lo, hi;
};
__host__ __device__ __forceinline__ Range row_range(const TdpMask& m, int q0, int q1, int T) {
    if (!m.causal) return {0, T - 1};
    return {q0 - m.wb > 0 ? q0 - m.wb : 0, q1};
}
__device__ __forceinline__ Range streamed_range(const TdpMask& m, int q0, int q1, int b, int T) {
    if (!m.causal) return {0, T - 1};
    // a <= q, q - a <= wa, b - a <= lab, a - b <= rab
    return {max(0, max(q0 - m.wa, b - m.lab)), min(q1, b + m.rab)};
}

// The same with the roles of a backward's workgroups: they own queries (KEYS false: as above) or keys, [o0, o1], whose streamed
// rows are then queries.
template <bool KEYS>
__device__ __forceinline__ Range own_row_range(const TdpMask& m, int o0, int o1, int T) {
    if (!KEYS) return row_range(m, o0, o1, T);
    if (!m.causal) return {0, T - 1};
    // some q: max(a, b) <= q <= min(a + wa, b + wb)
    return {max(0, o0 - min(m.rab, m.wb)), min(T - 1, o1 + min(m.lab, m.wa))};
}
template <bool KEYS>
__device__ __forceinline__ Range own_streamed_range(const TdpMask& m, int o0, int o1, int b, int T) {
    if (!KEYS) return streamed_range(m, o0, o1, b, T);
    if (!m.causal) return {0, T - 1};
    return {max(o0, b), min(T - 1, min(o1 + m.wa, b + m.wb))};
}

// Workgroups per query tile.  The work of a tile is its (round of nw rows, 32-row stage) steps, which under a causal mask
// grows with the square of its position: a workgroup takes about 1 / inv_target of them, and a tile as many workgroups (its
// parts) as that asks for.  The grid is the list of all parts, heaviest tiles first, without gaps: workgroups that find
// nothing to do would land on the same shader engines again and again (the dispatcher takes those in turn), B=4 H=8 T=512
// 13.8 -> 15-16 ms per backward.
struct F32Deal {
    float inv_target;
    int max_parts, items;  // parts of the heaviest tile, and of all tiles of a slice
    int keys = 0;          // the tiles own keys (f32_key_tile_steps): the first one is the heaviest
};
__host__ __device__ __forceinline__ int f32_tile_steps(const TdpMask& m, int q0, int q1, int T, int nw, int* rounds_out) {
    const Range r = row_range(m, q0, q1, T);
    const int rounds = r.hi / nw - r.lo / nw + 1;
    *rounds_out = rounds;
    if (!m.causal) return rounds * ((T + 31) / 32);
    const int span = q1 - (q0 - m.wa > 0 ? q0 - m.wa : 0), band = m.lab + m.rab + nw;
    return rounds * ((span < band ? span : band) / 32 + 1);
}
__host__ __device__ __forceinline__ int f32_key_tile_steps(const TdpMask& m, int o0, int o1, int T, int nw, int* rounds_out) {
    auto least = [](int x, int y) { return x < y ? x : y; };
    const int stages = (T + 31) / 32;
    if (!m.causal) {
        *rounds_out = (T - 1) / nw + 1;
        return *rounds_out * stages;
    }
    const int lo = o0 - least(m.rab, m.wb) > 0 ? o0 - least(m.rab, m.wb) : 0, hi = least(T - 1, o1 + least(m.lab, m.wa));
    const int below = o1 / nw - lo / nw + 1, above = hi / nw - o1 / nw;  // rounds up to the tile's own rows, and past them
    *rounds_out = below + above;
    // queries o .. min(o + wa, b + wb) below, b .. the same above
    const int end = least(T - 1, o1 + least(m.wa, m.wb)), longest = (end - o0) / 32 + 1, shortest = end > hi ? (end - hi) / 32 + 1 : 1;
    return below * longest + above * (longest + shortest) / 2;
}
__host__ __device__ __forceinline__ int f32_tile_parts(const F32Deal& d, const TdpMask& m, int qt, int T, int nw) {
    if (d.max_parts <= 1) return 1;
    const int q0 = qt * 32, q1 = q0 + 31 < T - 1 ? q0 + 31 : T - 1;
    int rounds;
    const int steps = d.keys ? f32_key_tile_steps(m, q0, q1, T, nw, &rounds) : f32_tile_steps(m, q0, q1, T, nw, &rounds);
    const int want = 1 + (int)((float)steps * d.inv_target);
    const int most = rounds < d.max_parts ? rounds : d.max_parts;
    return want < most ? want : most;
}
// part `item` of a slice's list: its tile, its place among the tile's parts and their number (part >= parts: past the list)
struct F32Item {
    int qt, part, parts;
};
__device__ __forceinline__ F32Item f32_item(const F32Deal& d, const TdpMask& m, int item, int nqt, int T, int nw) {
    const int first = d.keys ? 0 : nqt - 1, step = d.keys ? 1 : -1, last = nqt - 1 - first;  // heaviest tiles first
    if (d.max_parts <= 1) return {first + step * item, 0, 1};
    F32Item it{first, item, f32_tile_parts(d, m, first, T, nw)};
    while (it.part >= it.parts && it.qt != last) {
        it.part -= it.parts;
        it.qt += step;
        it.parts = f32_tile_parts(d, m, it.qt, T, nw);
    }
    return it;
}

// statistics of the 16-bit backward's fp32 tiles: lse receives the fp32 log-sum-exp of the covered rows and delta their
// rowsum(dO * O) with O in fp32
template <typename E>
struct F32StatsParams {
    const E *q, *ka, *kb, *va, *vb;  // streamed = (ka, va), rows = (kb, vb)
    // where these five and d_o lie: H heads per batch entry and each tensor's strides (dense tensors: H = 1 and
    // sb = T D, st = D)
    int H;
    TensorAt at_q, at_ka, at_kb, at_va, at_vb, at_do;
    float* lse;
    const E* d_o;
    float* delta;
    // Query tile 0 alone, with its rounds dealt out to `split_rounds` workgroups (f32_stats_block's `round`): each writes its
    // partial (maximum, sum, sum_d dO * unnormalised O) to delta[((bh * 32 + q) * split_rounds + round) * 3 ..] and
    // the first one clears `zero_words` 4-byte words at zero_ptr + bh * zero_words
    int split_rounds;
    unsigned* zero_ptr;
    int zero_words;
    int T, BH, nqt;  // nqt: query tiles this launch covers (tiles 0 .. nqt - 1)
    float scale_log2;
    TdpMask mask;  // in terms of the streamed index a and the row index b
};

// Staging of 32 x D tiles of E through registers (16-byte pieces), converted to fp32 on the way into LDS.
// NW waves move the two tiles of a stage.
template <typename E, int D, int NW>
struct StageE {
    static constexpr int VE = 16 / (int)sizeof(E);           // elements per piece
    static constexpr int kPieces = 32 * D / VE;               // per tensor
    static constexpr int kThreads = NW * 32;                  // per tensor: half of the workgroup for each
    static constexpr int kPer = (kPieces + kThreads - 1) / kThreads;  // per thread
    uint4 x[kPer];
};
template <typename E, int D, int NW>
__device__ __forceinline__ void stage_fetch_e(StageE<E, D, NW>& r, const E* __restrict__ ka, const E* __restrict__ va, int a0,
                                              int T, unsigned pitch_ka, unsigned pitch_va) {
    using S = StageE<E, D, NW>;
    constexpr int kVec = D / S::VE;
    const int t = threadIdx.x & (S::kThreads - 1);
    const bool first = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < NW / 2;  // whole waves serve one tensor
    const E* src = first ? ka : va;
    const unsigned pitch = first ? pitch_ka : pitch_va;
    // a whole stage lies at per-lane offsets that never change from its (scalar) first row; 31 pitch < T pitch < 2^31
    const bool whole = a0 + 31 < T;
    const E* row0 = src + (size_t)a0 * pitch;
#pragma unroll
    for (int i = 0; i < S::kPer; ++i) {
        const int idx = t + i * S::kThreads;
        if (S::kPieces % S::kThreads == 0 || idx < S::kPieces) {
            const int row = idx / kVec, c = idx % kVec;
            if (whole) r.x[i] = *reinterpret_cast<const uint4*>(row0 + (unsigned)(row * pitch + c * S::VE));
            else r.x[i] = *reinterpret_cast<const uint4*>(src + (size_t)min(a0 + row, T - 1) * pitch + c * S::VE);
        }
    }
}
// SILU: the second tensor is V1; its SiLU, rounded to E, is stored
template <typename E, int D, int NW, bool SILU = false>
__device__ __forceinline__ void stage_store_e(const StageE<E, D, NW>& r, float* sk, float* sv) {
    using S = StageE<E, D, NW>;
    constexpr int kVec = D / S::VE, LD = D + 4;  // f32_pitch<D>()
    const int t = threadIdx.x & (S::kThreads - 1);
    const bool first = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < NW / 2;
    float* dst = first ? sk : sv;
#pragma unroll
    for (int i = 0; i < S::kPer; ++i) {
        const int idx = t + i * S::kThreads;
        if (S::kPieces % S::kThreads == 0 || idx < S::kPieces) {
            const int row = idx / kVec, c = idx % kVec;
            float* p = dst + row * LD + c * S::VE;
            const E* e = reinterpret_cast<const E*>(&r.x[i]);
#pragma unroll
            for (int k = 0; k < S::VE; k += 4) {
                typedef __attribute__((ext_vector_type(4))) float f4;
                f4 v = {(float)e[k], (float)e[k + 1], (float)e[k + 2], (float)e[k + 3]};
                if constexpr (SILU) {
                    if (!first) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) v[j] = (float)(E)silu_f(v[j]);
                    }
                }
                *reinterpret_cast<f4*>(p + k) = v;
            }
        }
    }
}

// Row pitch (floats) of the [rows][D] tiles in LDS: rows start on 16-byte boundaries and the pitch is an odd number of
// 16-byte units, so that the 16-byte operand reads of a wave (32 rows, one piece each) fall on distinct bank groups.
template <int D>
constexpr int f32_pitch() {
    return D + 4;
}
template <int N>
struct VecF {
    typedef __attribute__((ext_vector_type(N))) float type;
};
template <>
struct VecF<1> {
    typedef float type;
};
template <int N>
__device__ __forceinline__ float vec_at(const typename VecF<N>::type& v, int i) {
    if constexpr (N == 1) return v;
    else return v[i];
}
typedef VecF<4>::type f32x4v;

// The valid streamed rows of one (query, row b): a - lo <= span as unsigned numbers; nothing is valid for span 0, lo 2^30
struct Interval {
    int lo;
    unsigned span;
};
__device__ __forceinline__ Interval valid_interval(const TdpMask& m, int q, int b, int T) {
    if (!m.causal) return {0, (unsigned)(T - 1)};
    const int lo = max(0, max(q - m.wa, b - m.lab)), hi = min(min(q, b + m.rab), T - 1);
    const bool any = (b <= q) & (q <= b + m.wb) & (lo <= hi);
    return any ? Interval{lo, (unsigned)(hi - lo)} : Interval{1 << 30, 0u};
}

// whether all of tile (queries q0 .. q0 + 31, streamed rows a0 .. a0 + 31) of row b is valid
__device__ __forceinline__ bool all_valid(const TdpMask& m, int q0, int a0, int b, int T) {
    if (!m.causal) return a0 + 31 < T;
    return (b <= q0) & (q0 + 31 <= b + m.wb) & (a0 + 31 <= min(q0, b + m.rab)) & (a0 >= max(q0 + 31 - m.wa, b - m.lab));
}

// the same for a workgroup that owns queries (above) or keys o
template <bool KEYS>
__device__ __forceinline__ Interval own_interval(const TdpMask& m, int o, int b, int T) {
    if (!KEYS) return valid_interval(m, o, b, T);
    if (!m.causal) return o < T ? Interval{0, (unsigned)(T - 1)} : Interval{1 << 30, 0u};
    const int lo = max(o, b), hi = min(min(o + m.wa, b + m.wb), T - 1);
    const bool any = (b <= o + m.lab) & (o <= b + m.rab) & (lo <= hi);
    return any ? Interval{lo, (unsigned)(hi - lo)} : Interval{1 << 30, 0u};
}
template <bool KEYS>
__device__ __forceinline__ bool own_all_valid(const TdpMask& m, int o0, int a0, int b, int T) {
    if (!KEYS) return all_valid(m, o0, a0, b, T);
    if (!m.causal) return (a0 + 31 < T) & (o0 + 31 < T);
    return (a0 >= max(o0 + 31, b)) & (a0 + 31 <= min(min(o0 + m.wa, b + m.wb), T - 1)) & (b <= o0 + m.lab) & (o0 + 31 <= b + m.rab);
}

// The (round of rows, stage of streamed rows) sequence a workgroup walks, one stage per step; rounds whose rows see no
// streamed row at all are passed over.
struct Walk {
    int m, st, st_hi;
};
template <int NW, bool KEYS = false>
__device__ __forceinline__ bool open_round(Walk& w, const TdpMask& mask, int m, int m_hi, int step, int q0, int q1, int T) {
    for (; m <= m_hi; m += step) {
        // the union over the round's rows
        const Range ra = own_streamed_range<KEYS>(mask, q0, q1, min(m * NW, T - 1), T);
        const Range rb = own_streamed_range<KEYS>(mask, q0, q1, min(m * NW + NW - 1, T - 1), T);
        const int lo = min(ra.lo, rb.lo) / 32, hi = max(ra.hi, rb.hi) / 32;
        if (lo <= hi) {
            w = {m, lo, hi};
            return true;
        }
    }
    return false;
}

// ------------------------------------------------------------------------------------------ statistics
// The forward over the fp32 query tiles of a 16-bit backward, for their log-sum-exp and Delta (F32StatsParams).  Operand reads
// are as wide as the layout allows: the k-slots of four consecutive MFMAs are four consecutive d (16 bytes of a row), and
// output row r of value tile dt is column d = DT r + dt, so that the operands of the DT value tiles are DT consecutive columns.
// Stages and row operands are fetched one step ahead across the rounds' ends, one barrier per step.
// SILU: p.va is V1 (a launch that does not wait for U)
template <typename E, int D, int NW, bool SILU>
__device__ __forceinline__ void f32_stats_block(const F32StatsParams<E>& p, int block, int round) {
    constexpr int DT = D / 32, LD = f32_pitch<D>(), NT = 64 * NW;
    constexpr bool HOLD = D <= 64;
    using vDT = typename VecF<DT>::type;
    extern __shared__ __align__(16) float smem_f[];
    float* sM = smem_f;                 // [NW][32]    end of kernel: per-wave maxima and sums
    float* sL = sM + NW * 32;           // [NW][32]
    float* sQ = sL + NW * 32;           // [32][LD]    the tile's queries * scale
    float* sK = sQ + 32 * LD;           // [2][32][LD] streamed key rows
    float* sV = sK + 2 * 32 * LD;       // [2][32][LD] streamed value rows
    float* sKb = sV + 2 * 32 * LD;      // [2][NW][D]  row operands of a round
    float* sVb = sKb + 2 * NW * D;      // [2][NW][D]
    float* sO = sK;                     // [NW][D][33] end of kernel: the waves' outputs (alias everything from the stages on)

    int bh, order;
    if (!xcd_tile(p.BH, p.nqt, block >> 3, block & 7, bh, order)) return;
    const int qt = p.nqt - 1 - order;

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int T = p.T;
    const int b_ = bh / p.H, h_ = bh % p.H;
    auto slice = [&](const E* t, const TensorAt& at) { return t + (size_t)b_ * at.sb + (size_t)h_ * at.sh; };
    const E* __restrict__ KA = slice(p.ka, p.at_ka);
    const E* __restrict__ VA = slice(p.va, p.at_va);
    const E* __restrict__ KB = slice(p.kb, p.at_kb);
    const E* __restrict__ VB = slice(p.vb, p.at_vb);
    const E* __restrict__ Qs = slice(p.q, p.at_q);
    const TdpMask mask = p.mask;

    const int q0 = qt * 32, q1 = min(T - 1, q0 + 31);
    const int q = q0 + n;  // this lane's query (column of every tile)
    const Range rows = row_range(mask, q0, q1, T);
    int m_lo = rows.lo / NW, m_hi = rows.hi / NW;  // rounds of NW rows
    if (p.split_rounds) {
        m_lo = max(m_lo, round);  // this workgroup's round only (none at all if it is out of range)
        m_hi = min(m_hi, round);
        if (round == 0)
            for (int idx = tid; idx < p.zero_words; idx += NT) p.zero_ptr[(size_t)bh * p.zero_words + idx] = 0u;
    }

    f32x16 accO[DT], accT[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            accO[dt][i] = 0.f;
            accT[dt][i] = 0.f;
        }
    float m_run = kNegBig, l_run = 0.f;  // per query, over every (a, b) this wave has seen (l: this lane's half)

    StageE<E, D, NW> regs;
    constexpr int kRowPer = (NW * D + NT - 1) / NT;
    float row_k[kRowPer], row_v[kRowPer];
    auto fetch_rows = [&](int m) {
#pragma unroll
        for (int i = 0; i < kRowPer; ++i) {
            const int idx = min(tid + i * NT, NW * D - 1);
            const size_t row = (size_t)min(m * NW + idx / D, T - 1);
            row_k[i] = (float)KB[row * p.at_kb.st + idx % D];
            row_v[i] = (float)VB[row * p.at_vb.st + idx % D];
        }
    };
    auto store_rows = [&](int par) {
#pragma unroll
        for (int i = 0; i < kRowPer; ++i)
            if (tid + i * NT < NW * D) {
                sKb[par * NW * D + tid + i * NT] = row_k[i];
                sVb[par * NW * D + tid + i * NT] = row_v[i];
            }
    };

    Walk w{};
    bool have = open_round<NW>(w, mask, m_lo, m_hi, 1, q0, q1, T);
    if (have) {
        fetch_rows(w.m);
        stage_fetch_e<E, D, NW>(regs, KA, VA, w.st * 32, T, p.at_ka.st, p.at_va.st);
    }
    for (int idx = tid; idx < 32 * D; idx += NT) {
        const int r = idx / D, d = idx % D;
        sQ[r * LD + d] = (float)Qs[(size_t)min(q0 + r, T - 1) * p.at_q.st + d] * p.scale_log2;
    }
    if (have) {
        store_rows(0);
        stage_store_e<E, D, NW, SILU>(regs, sK, sV);
    }
    __syncthreads();

    int buf = 0, par = 0;
    float bq[HOLD ? D / 2 : 1];
    bool fresh = true;  // the first step of a round
    while (have) {
        const float* cK = sK + buf * 32 * LD;
        const float* cV = sV + buf * 32 * LD;
        const bool last = w.st == w.st_hi;  // of this round
        Walk nw{w.m, w.st + 1, w.st_hi};
        const bool more = last ? open_round<NW>(nw, mask, w.m + 1, m_hi, 1, q0, q1, T) : true;
        if (more) {
            stage_fetch_e<E, D, NW>(regs, KA, VA, nw.st * 32, T, p.at_ka.st, p.at_va.st);
            if (last) fetch_rows(nw.m);
        }
        const int b = w.m * NW + wave, a0 = w.st * 32;
        const bool row_ok = b <= rows.hi && b >= rows.lo;
        const Range mine = streamed_range(mask, q0, q1, min(b, T - 1), T);
        const float* ob = sKb + par * NW * D + wave * D;
        if constexpr (HOLD) {
            if (fresh) {
#pragma unroll
                for (int c = 0; c < D / 8; ++c) {
                    const f32x4v qv = *reinterpret_cast<const f32x4v*>(sQ + n * LD + 4 * g + 8 * c);
                    const f32x4v kb = *reinterpret_cast<const f32x4v*>(ob + 4 * g + 8 * c);
#pragma unroll
                    for (int e = 0; e < 4; ++e) bq[c * 4 + e] = qv[e] * kb[e];
                }
            }
            fresh = last;
        }
        if (row_ok && a0 + 31 >= mine.lo && a0 <= mine.hi) {
            f32x16 s;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = 0.f;
            // per-lane parts of the LDS addresses, opaque: every read is one of them plus an immediate offset
            int row_base = n * LD + 4 * g, own_base = 4 * g, out_base = 4 * g * LD + DT * n;
            asm volatile("" : "+v"(row_base), "+v"(own_base), "+v"(out_base));
            // MFMA 4 c + e contracts d = 8 c + e (lanes of half 0) and 8 c + 4 + e (half 1)
#pragma unroll
            for (int c = 0; c < D / 8; ++c) {
                const f32x4v ka = *reinterpret_cast<const f32x4v*>(cK + row_base + 8 * c);
                if constexpr (HOLD) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) s = mma_f32(ka[e], bq[c * 4 + e], s);
                } else {
                    const f32x4v qv = *reinterpret_cast<const f32x4v*>(sQ + row_base + 8 * c);
                    const f32x4v kb = *reinterpret_cast<const f32x4v*>(ob + own_base + 8 * c);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s = mma_f32(ka[e], qv[e] * kb[e], s);
                }
            }
            if (!all_valid(mask, q0, a0, b, T)) {
                const Interval ok = valid_interval(mask, q, b, T);
                const int x = a0 + 4 * g - ok.lo;
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = (unsigned)(x + c_row(0, i)) <= ok.span ? s[i] : -INFINITY;
            }
            // exponentials relative to the query's reference, which is some earlier tile's maximum: a sum that outgrows it
            // by 2^16 (or the first one of all) moves it to this tile's maximum.  fp32 sums lose no digits by a loose
            // reference, and the maximum need not be formed for every tile; what they lose is room below the end of fp32's
            // range, which 2^40 took from values whose products reach 1e26.  2^40 -> 2^16, forward: N(0, 1) operands the same
            // time, three times that (scores 27 times) B=4 H=8 T=512 D=64 3.39 -> 3.43 ms
            f32x16 pv;
            float psum = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                pv[i] = fast_exp2(s[i] - m_run);
                psum += pv[i];
            }
            if (__any(!(psum <= 65536.f))) {
                float tmax = kNegBig;
#pragma unroll
                for (int i = 0; i < 16; ++i) tmax = fmaxf(tmax, s[i]);
                tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
                const float m_new = fmaxf(m_run, tmax), sc = fast_exp2(m_run - m_new);
                l_run *= sc;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        accT[dt][i] *= sc;
                        accO[dt][i] *= sc;
                    }
                m_run = m_new;
                psum = 0.f;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    pv[i] = fast_exp2(s[i] - m_run);
                    psum += pv[i];
                }
            }
            l_run += psum;
            // Tv^T[d, q] += VA^T[d, a] P^T[a, q]: step i contracts the two streamed rows c_row(0, i), c_row(1, i)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const vDT va = *reinterpret_cast<const vDT*>(cV + out_base + c_row(0, i) * LD);
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) accT[dt] = mma_f32(vec_at<DT>(va, dt), pv[i], accT[dt]);
            }
        }
        if (last) {
            // the finished row: O^T[d, q] += Tv^T[d, q] * VB[b, d]   (register i of half g: d = DT c_row(g, i) + dt)
            if (row_ok) {
                const float* vb = sVb + par * NW * D + wave * D;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const vDT v = *reinterpret_cast<const vDT*>(vb + DT * (c_row(0, i) + 4 * g));
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) accO[dt][i] += accT[dt][i] * vec_at<DT>(v, dt);
                }
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) accT[dt][i] = 0.f;
        }
        if (more) {
            buf ^= 1;
            if (last) {
                par ^= 1;
                store_rows(par);
            }
            stage_store_e<E, D, NW, SILU>(regs, sK + buf * 32 * LD, sV + buf * 32 * LD);
            __syncthreads();
        }
        w = nw;
        have = more;
    }

    // ---- merge the waves' partial results: each leaves its own, relative to the common maximum, in a [D][33] slice of LDS,
    // and the slices are added in a fixed order (one wave after another into a common slice put a barrier and a chain of
    // LDS round trips per wave at the end of every workgroup)
    l_run += __shfl_xor(l_run, 32, 64);
    if (g == 0) {
        sM[wave * 32 + n] = m_run;
        sL[wave * 32 + n] = l_run;
    }
    __syncthreads();
    float M = kNegBig;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, sM[w * 32 + n]);
    const float mine_scale = fast_exp2(m_run - M);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) sO[wave * D * 33 + (DT * c_row(g, i) + dt) * 33 + n] = accO[dt][i] * mine_scale;
    __syncthreads();
    auto merged = [&](int d, int r) {
        float v = sO[d * 33 + r];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += sO[(w * D + d) * 33 + r];
        return v;
    };
    float L = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) L += sL[w * 32 + n] * fast_exp2(sM[w * 32 + n] - M);
    // Delta[q] = sum_d dO[q, d] O[q, d] with O in fp32: two threads of every wave per query, joined through LDS
    float* red = sQ;  // [2 NW][32]
    const int k16 = wave * 2 + g;
    float dsum = 0.f;
    if (q < T) {
        const E* dor = slice(p.d_o, p.at_do) + (size_t)q * p.at_do.st;
        for (int d = k16; d < D; d += 2 * NW) dsum += (float)dor[d] * merged(d, n);
    }
    red[k16 * 32 + n] = dsum;
    __syncthreads();
    if (wave == 0 && g == 0 && q < T) {
        dsum = 0.f;
#pragma unroll
        for (int k = 0; k < 2 * NW; ++k) dsum += red[k * 32 + n];
        if (p.split_rounds) {
            float* part = p.delta + (((size_t)bh * 32 + n) * p.split_rounds + round) * 3;
            part[0] = M; part[1] = L; part[2] = dsum;
        } else {
            p.delta[(size_t)bh * T + q] = dsum / L;
        }
    }
    if (p.split_rounds) return;
    if (wave == 0 && g == 0 && q < T) p.lse[(size_t)bh * T + q] = (M + fast_log2(L)) * kLn2;
}
template <typename E, int D, int NW>
__global__ __launch_bounds__(64 * NW, 2) void tdp_f32_stats_kernel(F32StatsParams<E> p) {
    f32_stats_block<E, D, NW, false>(p, blockIdx.x, blockIdx.y);
}

// ------------------------------------------------------------------------------------------ backward
// The fp32 query tiles of a 16-bit backward, in two roles: rows = (K2, V2), streamed = (K1, U) gives dQ, dK2, dV2; with the
// roles exchanged, dK1 and dU.  Per (query tile, row b, 32 streamed rows):
//   S^T, dP^T (D / 2 MFMAs each),  P = exp2(S - LSE2[q]),  dS = P (dP - Delta[q])   (both lane-local)
//   Yq^T[d, q] += KA^T[d, a] dS^T[a, q]      Tv^T[d, q] += VA^T[d, a] P^T[a, q]      (DOUT / 2 MFMAs each)
// and when the row is finished
//   dQ^T[d, q] += Yq^T[d, q] KB[b, d]                                  (registers, all rounds)
//   dKB[b, d]  += alpha sum_q Yq^T[d, q] Q[q, d],   dVB[b, d] += sum_q Tv^T[d, q] dO[q, d]
// The sums over the tile's 32 queries are lane reductions; the sums over query tiles (workgroups) go to shared
// accumulators: 64-bit fixed point with integer atomics (the result does not depend on the order of arrival), or
// fp32 atomics when the accumulators are fp32.
//
// The tensors may be 16-bit (E = bf16 / f16): they are converted as they are staged, everything after that is
// fp32.  That is how the 16-bit backward runs its first query tile: for the first few causal queries the softmax
// is nearly one-hot and dS = P (dP - Delta) cancels two O(10) numbers, which the 16-bit operands of the MFMA
// kernels (dO * V2 rounded to 16 bit) cannot resolve.
// The operand reads and the walk over rounds and stages are the forward's; four waves per workgroup and two workgroups to a
// CU at D <= 64 (B=4 H=8 T=512 D=64: 18.5 -> 13.5 ms, B=2 H=4 T=500: 20.0 -> 3.5; eight waves, one workgroup: 15.1 / 4.0).
// DOUT < D: a workgroup produces DOUT of the gradient columns (blockIdx.y picks them).

template <typename E>
struct F32BwdParams {
    const E *q, *d_o, *ka, *kb, *va, *vb;
    int H;  // layouts of the six inputs, as in F32StatsParams
    TensorAt at_q, at_ka, at_kb, at_va, at_vb, at_do;
    const float *lse, *delta;
    E* dq;                 // WITH_DQ, when acc_q is null
    void *acc_k, *acc_v;   // [BH][T][D] gradients of the rows: fixed point (long long) or float
    void* acc_q;           // WITH_DQ: when non-null, dQ / alpha is added here instead of being written to dq
    int acc_q_rows;        // 0: acc_q is [BH][T][D]; else it holds the first acc_q_rows queries only, [BH][rows][D]
    // when non-null, LSE and Delta of query tile 0 come from the partials the split STATS launch left here
    const float* stats_part;
    int split_rounds;      // tile 0 only: rounds dealt out to workgroups (see tdp_f32_tile0_kernel), else 0
    // tdp_f32_bwd_kernel: the rounds of a tile dealt out to f32_tile_parts() workgroups.  max_parts above one needs
    // acc_q where dQ is produced (each workgroup holds a share of it)
    F32Deal deal;
    // fixed-point accumulators (common.hpp); scale_parts null: the accumulators are float
    const unsigned* scale_parts;
    unsigned* poison;
    int scale_bias;
    unsigned bit_k, bit_v;  // poison bits of acc_k / acc_v
    int T, BH, nqt;        // nqt: query tiles this launch covers (tiles 0 .. nqt - 1)
    float alpha;
    TdpMask mask;
};

// Sums over the 32 lanes of a wave half, of 16 registers of two tensors at once: lane n ends with the sum of register
// 8 (n>>4 & 1) + 4 (n>>3 & 1) + 2 (n>>2 & 1) + (n>>1 & 1), of x in even lanes and of y in odd ones.  Every exchange halves
// what is left to exchange, and none goes through LDS: rows of 16 lanes are swapped between two registers, lanes of a row meet
// by DPP (8 apart, mirrored in 8, 2 and 1 apart).  77 vector instructions; written with selects of vector elements and
// __shfl_xor it was 850 (the compiler makes the selects into chains of compares) and 31 LDS round trips.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ float half_sum_step(bool up, float low, float high) {  // keeps `high` in the lanes `up`, `low` elsewhere
    asm("" : "+v"(low), "+v"(high));  // (two values: not one element picked by `up`)
    const float keep = up ? high : low, send = up ? low : high;
    return keep + dpp<CTRL>(send);
}
__device__ __forceinline__ float half_sum_16(const f32x16& x, int n) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        // even rows of 16 lanes get their x[i] and their odd row's, odd rows both x[i + 8]
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[i]), __float_as_uint(x[i + 8]), false, false);
        v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = half_sum_step<0x128>(n & 8, v[i], v[i + 4]);  // row_ror:8
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] = half_sum_step<0x141>(n & 4, v[i], v[i + 2]);  // row_half_mirror
    return half_sum_step<0x4e>(n & 2, v[0], v[1]);                                    // quad_perm [2, 3, 0, 1]
}
__device__ __forceinline__ float half_sum_16x2(const f32x16& x, const f32x16& y) {
    const int n = threadIdx.x & 31;
    return half_sum_step<0xb1>(n & 1, half_sum_16(x, n), half_sum_16(y, n));           // quad_perm [1, 0, 3, 2]
}
__device__ __forceinline__ int half_sum_register() {  // the register whose sum this lane ends with
    return (threadIdx.x >> 1) & 15;
}

// `only_round` >= 0: this workgroup walks that round of rows only; else every `parts`-th round from the `part`-th on.
// `bx` >= 0: the workgroup's place in a grid of its own (a kernel that runs these workgroups beside others passes it);
// else blockIdx.x, and blockIdx.y picks the gradient columns
template <typename E, int D, int DOUT, bool WITH_DQ, int NW>
__device__ __forceinline__ void f32_bwd_body(const F32BwdParams<E>& p, int only_round, int bx = -1) {
    constexpr int DTO = DOUT / 32, LD = f32_pitch<D>(), NT = 64 * NW;
    using vDT = typename VecF<DTO>::type;
    // dQ of the tile, summed over the rounds: in registers up to 64 columns; beyond that the accumulators of a round
    // leave no room for it and it lives in LDS, where the waves add their round's share one after another
    constexpr bool DQ_LDS = WITH_DQ && DOUT > 64;
    // B operands of the score products held in registers over a round, where the accumulators leave room for them;
    // otherwise formed as they are used (two more LDS reads and four multiplies per four MFMAs)
    constexpr bool HOLD_Q = D < 64 || (D == 64 && !WITH_DQ), HOLD_G = HOLD_Q;
    extern __shared__ __align__(16) float smem_f[];
    float* sK = smem_f;                 // [2][32][LD]
    float* sV = sK + 2 * 32 * LD;       // [2][32][LD]
    float* sQ = sV + 2 * 32 * LD;       // [32][LD]  Q * alpha * log2(e)
    float* sDO = sQ + 32 * LD;          // [32][LD]
    float* sKb = sDO + 32 * LD;         // [2][NW][D]
    float* sVb = sKb + 2 * NW * D;      // [2][NW][D]
    float* sO = DQ_LDS ? sVb + 2 * NW * D : sK;  // dQ of the tile: [DOUT][33], or at the end [NW][DOUT][33], aliasing everything

    int bh, order;
    const int block_x = bx < 0 ? (int)blockIdx.x : bx;
    const bool tile0 = only_round >= 0;
    if (!xcd_tile(p.BH, tile0 ? p.nqt : p.deal.items, block_x >> 3, block_x & 7, bh, order)) return;
    const F32Item item = tile0 ? F32Item{p.nqt - 1 - order, 0, 1} : f32_item(p.deal, p.mask, order, p.nqt, p.T, NW);
    const int qt = item.qt, part = item.part, step = item.parts;
    if (part >= step) return;
    const int c0 = (bx < 0 ? (int)blockIdx.y : 0) * DOUT;  // first gradient column of this workgroup

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int T = p.T;
    const size_t base = (size_t)bh * T * D;
    const int b_ = bh / p.H, h_ = bh % p.H;
    auto slice = [&](const E* t, const TensorAt& at) { return t + (size_t)b_ * at.sb + (size_t)h_ * at.sh; };
    const E* __restrict__ KA = slice(p.ka, p.at_ka);
    const E* __restrict__ VA = slice(p.va, p.at_va);
    const E* __restrict__ KB = slice(p.kb, p.at_kb);
    const E* __restrict__ VB = slice(p.vb, p.at_vb);
    const E* __restrict__ Qs = slice(p.q, p.at_q);
    const TdpMask mask = p.mask;
    const float scale_log2 = p.alpha * kLog2e;
    const int q0 = qt * 32, q1 = min(T - 1, q0 + 31);
    const int q = q0 + n;
    const Range rows = row_range(mask, q0, q1, T);
    int m_lo = rows.lo / NW + part, m_hi = rows.hi / NW;
    if (only_round >= 0) {
        m_lo = max(m_lo, only_round);
        m_hi = min(m_hi, only_round);
    }

    StageE<E, D, NW> regs;
    constexpr int kRowPer = (NW * D + NT - 1) / NT;
    float row_k[kRowPer], row_v[kRowPer];
    auto fetch_rows = [&](int m) {
#pragma unroll
        for (int i = 0; i < kRowPer; ++i) {
            const int idx = min(tid + i * NT, NW * D - 1);
            const size_t row = (size_t)min(m * NW + idx / D, T - 1);
            row_k[i] = (float)KB[row * p.at_kb.st + idx % D];
            row_v[i] = (float)VB[row * p.at_vb.st + idx % D];
        }
    };
    auto store_rows = [&](int par) {
#pragma unroll
        for (int i = 0; i < kRowPer; ++i)
            if (tid + i * NT < NW * D) {
                sKb[par * NW * D + tid + i * NT] = row_k[i];
                sVb[par * NW * D + tid + i * NT] = row_v[i];
            }
    };
    Walk w{};
    bool have = open_round<NW>(w, mask, m_lo, m_hi, step, q0, q1, T);
    if (have) {
        fetch_rows(w.m);
        stage_fetch_e<E, D, NW>(regs, KA, VA, w.st * 32, T, p.at_ka.st, p.at_va.st);
    }
    for (int idx = tid; idx < 32 * D; idx += NT) {
        const int r = idx / D, d = idx % D;
        const size_t row = (size_t)min(q0 + r, T - 1);
        sQ[r * LD + d] = (float)Qs[row * p.at_q.st + d] * scale_log2;
        sDO[r * LD + d] = (float)slice(p.d_o, p.at_do)[row * p.at_do.st + d];
    }
    // (here, where the first stage's loads are on their way)
    const float fscale = p.scale_parts ? fixed_scale_value(fixed_scale_field(p.scale_parts, bh, p.scale_bias)) : 0.f;
    // a query past the end of the sequence gets a huge LSE: its P is exactly 0
    float lse2 = 1.0e30f, delta = 0.f;
    if (q < T) {
        if (p.stats_part) {  // tile 0: join the partials of the rounds
            const float* sp = p.stats_part + ((size_t)bh * 32 + n) * p.split_rounds * 3;
            float M = kNegBig, L = 0.f, num = 0.f;
            for (int z = 0; z < p.split_rounds; ++z) M = fmaxf(M, sp[z * 3]);
            for (int z = 0; z < p.split_rounds; ++z) {
                const float wt = fast_exp2(sp[z * 3] - M);
                L += sp[z * 3 + 1] * wt;
                num += sp[z * 3 + 2] * wt;
            }
            lse2 = M + fast_log2(L);
            delta = num / L;
        } else {
            lse2 = p.lse[(size_t)bh * T + q] * kLog2e;
            delta = p.delta[(size_t)bh * T + q];
        }
    }

    f32x16 accDQ[DQ_LDS || !WITH_DQ ? 1 : DTO];
#pragma unroll
    for (int dt = 0; dt < (DQ_LDS || !WITH_DQ ? 1 : DTO); ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) accDQ[dt][i] = 0.f;
    if constexpr (DQ_LDS)
        for (int idx = tid; idx < DOUT * 33; idx += NT) sO[idx] = 0.f;
    f32x16 accQ[DTO], accT[DTO];
#pragma unroll
    for (int dt = 0; dt < DTO; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            accQ[dt][i] = 0.f;
            accT[dt][i] = 0.f;
        }
    if (have) {
        store_rows(0);
        stage_store_e<E, D, NW>(regs, sK, sV);
    }
    __syncthreads();

    int buf = 0, par = 0;
    f32x4v bq[HOLD_Q ? D / 8 : 1], bg[HOLD_G ? D / 8 : 1];
    bool fresh = true;  // the first step of a round
    while (have) {
        const float* cK = sK + buf * 32 * LD;
        const float* cV = sV + buf * 32 * LD;
        const bool last = w.st == w.st_hi;  // of this round
        Walk nw{w.m, w.st + 1, w.st_hi};
        const bool more = last ? open_round<NW>(nw, mask, w.m + step, m_hi, step, q0, q1, T) : true;
        if (more) {
            stage_fetch_e<E, D, NW>(regs, KA, VA, nw.st * 32, T, p.at_ka.st, p.at_va.st);
            if (last) fetch_rows(nw.m);
        }
        if (HOLD_Q && fresh) {
            const float *kr = sKb + par * NW * D + wave * D + 4 * g, *vr = sVb + par * NW * D + wave * D + 4 * g;
#pragma unroll
            for (int c = 0; c < D / 8; ++c) {
                const f32x4v qv = *reinterpret_cast<const f32x4v*>(sQ + n * LD + 4 * g + 8 * c);
                const f32x4v kb = *reinterpret_cast<const f32x4v*>(kr + 8 * c);
#pragma unroll
                for (int e = 0; e < 4; ++e) bq[HOLD_Q ? c : 0][e] = qv[e] * kb[e];
                if constexpr (HOLD_G) {
                    const f32x4v gv = *reinterpret_cast<const f32x4v*>(sDO + n * LD + 4 * g + 8 * c);
                    const f32x4v vb = *reinterpret_cast<const f32x4v*>(vr + 8 * c);
#pragma unroll
                    for (int e = 0; e < 4; ++e) bg[c][e] = gv[e] * vb[e];
                }
            }
        }
        fresh = last;
        const int b = w.m * NW + wave, a0 = w.st * 32;
        const bool row_ok = b <= rows.hi && b >= rows.lo;
        const Range mine = streamed_range(mask, q0, q1, min(b, T - 1), T);
        const float *kb_row = sKb + par * NW * D + wave * D, *vb_row = sVb + par * NW * D + wave * D;
        if (row_ok && a0 + 31 >= mine.lo && a0 <= mine.hi) {
            f32x16 s, dp;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s[i] = 0.f;
                dp[i] = 0.f;
            }
            // The per-lane parts of the LDS addresses, opaque to the compiler from here on: every read below is
            // then this base plus a compile-time offset (the instruction's immediate field).  Left to itself the
            // compiler computes the hundreds of addresses of the unrolled loops ahead of the loops and keeps them
            // in registers (D = 128: 150 of them spilled to scratch memory).
            int row_base = n * LD + 4 * g, own_base = 4 * g, out_base = 4 * g * LD + c0 + DTO * n;
            asm volatile("" : "+v"(row_base), "+v"(out_base), "+v"(own_base));
#pragma unroll
            for (int c = 0; c < D / 8; ++c) {
                const f32x4v ka = *reinterpret_cast<const f32x4v*>(cK + row_base + 8 * c);
                const f32x4v va = *reinterpret_cast<const f32x4v*>(cV + row_base + 8 * c);
                f32x4v oq, og;
                if constexpr (HOLD_Q) {
                    oq = bq[c];
                } else {
                    const f32x4v qv = *reinterpret_cast<const f32x4v*>(sQ + row_base + 8 * c);
                    const f32x4v kb = *reinterpret_cast<const f32x4v*>(kb_row + own_base + 8 * c);
#pragma unroll
                    for (int e = 0; e < 4; ++e) oq[e] = qv[e] * kb[e];
                }
                if constexpr (HOLD_G) {
                    og = bg[c];
                } else {
                    const f32x4v gv = *reinterpret_cast<const f32x4v*>(sDO + row_base + 8 * c);
                    const f32x4v vb = *reinterpret_cast<const f32x4v*>(vb_row + own_base + 8 * c);
#pragma unroll
                    for (int e = 0; e < 4; ++e) og[e] = gv[e] * vb[e];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s = mma_f32(ka[e], oq[e], s);
                    dp = mma_f32(va[e], og[e], dp);
                }
                // operand reads stay within a chunk or two of their use (registers)
                if (D > 64 || (c & 1)) __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = fast_exp2(s[i] - lse2);
            if (!all_valid(mask, q0, a0, b, T)) {
                const Interval ok = valid_interval(mask, q, b, T);
                const int x = a0 + 4 * g - ok.lo;
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = (unsigned)(x + c_row(0, i)) <= ok.span ? s[i] : 0.f;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) dp[i] = s[i] * (dp[i] - delta);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                // row c_row(g, i) = c_row(0, i) + 4 g
                const vDT va = *reinterpret_cast<const vDT*>(cV + out_base + c_row(0, i) * LD);
                const vDT ka = *reinterpret_cast<const vDT*>(cK + out_base + c_row(0, i) * LD);
#pragma unroll
                for (int dt = 0; dt < DTO; ++dt) {
                    accT[dt] = mma_f32(vec_at<DTO>(va, dt), s[i], accT[dt]);
                    accQ[dt] = mma_f32(vec_at<DTO>(ka, dt), dp[i], accQ[dt]);
                }
                if ((i & (DTO > 2 ? 1 : 3)) == (DTO > 2 ? 1 : 3)) __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (last) {
            if (row_ok) {
                int q_base = n * LD + c0 + 4 * DTO * g, kb_base = c0 + 4 * DTO * g;  // opaque bases, as above
                asm volatile("" : "+v"(q_base), "+v"(kb_base));
                if constexpr (WITH_DQ && !DQ_LDS) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const vDT k = *reinterpret_cast<const vDT*>(kb_row + kb_base + DTO * c_row(0, i));
#pragma unroll
                        for (int dt = 0; dt < DTO; ++dt) accDQ[dt][i] += accQ[dt][i] * vec_at<DTO>(k, dt);
                    }
                }
#pragma unroll
                for (int dt = 0; dt < DTO; ++dt) {
                    // register i of half g is column d = c0 + DTO c_row(g, i) + dt.  sQ holds Q * alpha * log2(e):
                    // alpha is wanted, log2(e) is not
                    f32x16 xk, xv;
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const vDT qv = *reinterpret_cast<const vDT*>(sQ + q_base + DTO * c_row(0, i));
                        const vDT gv = *reinterpret_cast<const vDT*>(sDO + q_base + DTO * c_row(0, i));
                        xk[i] = accQ[dt][i] * vec_at<DTO>(qv, dt);
                        xv[i] = accT[dt][i] * vec_at<DTO>(gv, dt);
                    }
                    const float sum = half_sum_16x2(xk, xv);
                    const bool odd = n & 1;
                    const int i = half_sum_register(), d = c0 + DTO * c_row(g, i) + dt;
                    shared_add(odd ? p.acc_v : p.acc_k, base + (size_t)b * D + d, odd ? sum : sum * kLn2, fscale,
                               p.poison + (size_t)bh * T + b, odd ? p.bit_v : p.bit_k);
                    __builtin_amdgcn_sched_barrier(0);  // one tile's products and sums in registers at a time
                }
            }
            if constexpr (DQ_LDS) {
                // dQ[q] += Yq (.) K2[b], one wave after another: a fixed summation order (every wave takes part in the
                // barriers, whether or not it had a row this round)
                for (int v = 0; v < NW; ++v) {
                    if (wave == v && row_ok) {
                        int kb_base = c0 + 4 * DTO * g, o_base = 4 * DTO * g * 33 + n;
                        asm volatile("" : "+v"(kb_base), "+v"(o_base));
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            const vDT k = *reinterpret_cast<const vDT*>(kb_row + kb_base + DTO * c_row(0, i));
#pragma unroll
                            for (int dt = 0; dt < DTO; ++dt)
                                sO[o_base + (DTO * c_row(0, i) + dt) * 33] += accQ[dt][i] * vec_at<DTO>(k, dt);
                        }
                    }
                    __syncthreads();
                }
            }
#pragma unroll
            for (int dt = 0; dt < DTO; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    accQ[dt][i] = 0.f;
                    accT[dt][i] = 0.f;
                }
        }
        if (more) {
            buf ^= 1;
            if (last) {
                par ^= 1;
                store_rows(par);
            }
            stage_store_e<E, D, NW>(regs, sK + buf * 32 * LD, sV + buf * 32 * LD);
            __syncthreads();
        }
        w = nw;
        have = more;
    }

    if constexpr (WITH_DQ) {
        __syncthreads();
        if constexpr (!DQ_LDS) {  // the waves' shares side by side (sO), added in a fixed order below
#pragma unroll
            for (int dt = 0; dt < DTO; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) sO[wave * DOUT * 33 + (DTO * c_row(g, i) + dt) * 33 + n] = accDQ[dt][i];
            __syncthreads();
        }
        auto merged = [&](int d, int r) {
            float v = sO[d * 33 + r];
            if constexpr (!DQ_LDS) {
#pragma unroll
                for (int w = 1; w < NW; ++w) v += sO[(w * DOUT + d) * 33 + r];
            }
            return v;
        };
        for (int idx = tid; idx < 32 * DOUT; idx += NT) {
            const int r = idx / DOUT, d = idx % DOUT;
            if (q0 + r < T) {
                const size_t off = base + (size_t)(q0 + r) * D + c0 + d;
                if (p.acc_q)
                    shared_add(p.acc_q, p.acc_q_rows ? ((size_t)bh * p.acc_q_rows + q0 + r) * D + c0 + d : off,
                               merged(d, r), fscale, p.poison + (size_t)bh * T + q0 + r, kPoisonDQ);
                else
                    p.dq[off] = (E)(merged(d, r) * p.alpha);
            }
        }
    }
}

template <typename E, int D, int DOUT, bool WITH_DQ, int NW>
__global__ __launch_bounds__(64 * NW, 2) void tdp_f32_bwd_kernel(F32BwdParams<E> p) {
    f32_bwd_body<E, D, DOUT, WITH_DQ, NW>(p, -1);
}

// Query tile 0 of a 16-bit backward, both launches' roles and all rounds at once: blockIdx.z = role * rounds + round
// (role 0: rows = (K2, V2), with dQ; role 1: rows = (K1, U)).  A tile of 32 queries has at most four rounds of
// eight rows; one workgroup walking them one after another is 4 x ~25 us of pure latency.
template <typename E, int D, int DOUT>
__device__ __forceinline__ void f32_tile0_block(const F32BwdParams<E>& r0, const F32BwdParams<E>& r1, int roles_mask, int z,
                                                int bx = -1) {
    const int role = z / r0.split_rounds, round = z % r0.split_rounds;
    if (!((roles_mask >> role) & 1)) return;
    if (role == 0) {
        if (roles_mask & 4) f32_bwd_body<E, D, DOUT, true, kF32Waves>(r0, round, bx);
        else f32_bwd_body<E, D, DOUT, false, kF32Waves>(r0, round, bx);
    } else {
        f32_bwd_body<E, D, DOUT, false, kF32Waves>(r1, round, bx);
    }
}
template <typename E, int D, int DOUT>
__global__ __launch_bounds__(512) void tdp_f32_tile0_kernel(F32BwdParams<E> r0, F32BwdParams<E> r1, int roles_mask) {
    f32_tile0_block<E, D, DOUT>(r0, r1, roles_mask, blockIdx.z);
}

template <int D, int NW = kF32Waves>
constexpr size_t f32_bwd_smem() {
    // stages, Q and dO, the rows of two rounds; D = 128: dQ of the tile (f32_bwd_body's DQ_LDS); at the end the waves' dQ
    constexpr int loop = 6 * 32 * f32_pitch<D>() + 4 * NW * D + (D > 64 ? D * 33 : 0), merge = NW * (D > 64 ? 64 : D) * 33;
    return sizeof(float) * (size_t)(loop > merge ? loop : merge);
}

template <int D, int NW>
constexpr size_t f32_stats_smem() {
    constexpr int loop = 4 * 32 * f32_pitch<D>() + 4 * NW * D, merge = NW * D * 33;
    return sizeof(float) * (size_t)(2 * NW * 32 + 32 * f32_pitch<D>() + (loop > merge ? loop : merge));
}


// where the six inputs lie (F32StatsParams::H and at_*)
struct InputsAt {
    int H;
    TensorAt q, d_o, k1, u, k2, v2;
};
InputsAt dense_inputs(int T, int D) {
    const TensorAt d = dense_at(1, T, D);
    return InputsAt{1, d, d, d, d, d, d};
}
InputsAt inputs_of(const FirstTileArgs& a) {
    if (a.H <= 0) return dense_inputs(a.T, a.D);
    return InputsAt{a.H, a.at_q, a.at_do, a.at_k1, dense_at(a.H, a.T, a.D), a.at_k2, a.at_v2};
}
// streamed = (K1, U), rows = (K2, V2), or the two exchanged
template <typename P>
void place_inputs(P& p, const InputsAt& at, bool exchanged) {
    p.H = at.H; p.at_q = at.q; p.at_do = at.d_o;
    p.at_ka = exchanged ? at.k2 : at.k1; p.at_va = exchanged ? at.v2 : at.u;
    p.at_kb = exchanged ? at.k1 : at.k2; p.at_vb = exchanged ? at.u : at.v2;
}

// Query tile 0 alone, first half: the parameters of the STATS pass (its rounds dealt out to `rounds` workgroups; V1 is the
// streamed value tensor where it is given) ...
template <typename E, int D>
F32StatsParams<E> tile0_stats(const FirstTileArgs& a, int rounds, const void* v1, const TensorAt& at_v1) {
    const bool own_dq_acc = a.want_q && !a.acc_q;  // dQ of the tile is summed over its rounds in a.dq0_acc
    F32StatsParams<E> p{};
    p.q = (const E*)a.q; p.ka = (const E*)a.k1; p.kb = (const E*)a.k2; p.va = (const E*)(v1 ? v1 : a.u); p.vb = (const E*)a.v2;
    place_inputs(p, inputs_of(a), false);
    if (v1) p.at_va = at_v1;
    p.lse = nullptr; p.d_o = (const E*)a.d_o; p.delta = a.delta_f32;
    p.split_rounds = rounds;
    p.zero_ptr = own_dq_acc ? (unsigned*)a.dq0_acc : nullptr;
    p.zero_words = own_dq_acc ? 32 * D * (a.scale_parts ? 2 : 1) : 0;
    p.T = a.T; p.BH = a.BH; p.nqt = 1;
    p.scale_log2 = a.alpha * kLog2e;
    p.mask = TdpMask{a.causal, a.k1_window, a.k2_window, a.kk_left, a.kk_right};
    return p;
}
inline int tile0_rounds(const FirstTileArgs& a) { return (std::min(a.T, 32) + kF32Waves - 1) / kF32Waves; }

// ... and those of the backward pass over the tile for both roles, which is (8 xcd_slots(BH, 1)) x (2 rounds) calls of
// f32_tile0_block: tdp_f32_tile0_kernel, or the tail of another grid.
template <typename E, int D>
void tile0_backward(const FirstTileArgs& a, F32BwdParams<E>& r0, F32BwdParams<E>& r1, int& roles) {
    const int rounds = tile0_rounds(a);
    const TdpMask natural{a.causal, a.k1_window, a.k2_window, a.kk_left, a.kk_right};
    r0 = F32BwdParams<E>{};
    r0.q = (const E*)a.q; r0.d_o = (const E*)a.d_o; r0.lse = nullptr; r0.delta = nullptr;
    r0.stats_part = a.delta_f32; r0.split_rounds = rounds; r0.deal = F32Deal{0.f, 1, 1};
    r0.dq = (E*)a.dq; r0.acc_q = a.acc_q ? a.acc_q : a.dq0_acc; r0.acc_q_rows = a.acc_q ? 0 : 32;
    r0.scale_parts = a.scale_parts; r0.poison = a.poison; r0.scale_bias = a.scale_bias;
    r0.T = a.T; r0.BH = a.BH; r0.nqt = 1; r0.alpha = a.alpha;
    r1 = r0;
    r0.ka = (const E*)a.k1; r0.va = (const E*)a.u; r0.kb = (const E*)a.k2; r0.vb = (const E*)a.v2;
    place_inputs(r0, inputs_of(a), false);
    r0.acc_k = a.acc_k2; r0.acc_v = a.acc_v2; r0.bit_k = kPoisonDK2; r0.bit_v = kPoisonDV2; r0.mask = natural;
    r1.ka = (const E*)a.k2; r1.va = (const E*)a.v2; r1.kb = (const E*)a.k1; r1.vb = (const E*)a.u;
    place_inputs(r1, inputs_of(a), true);
    r1.acc_k = a.acc_k1; r1.acc_v = a.acc_u; r1.bit_k = kPoisonDK1; r1.bit_v = kPoisonDU;
    r1.mask = TdpMask{natural.causal, natural.wb, natural.wa, natural.rab, natural.lab};
    roles = ((a.want_q || a.want_k2) ? 1 : 0) | (a.want_k1 ? 2 : 0) | (a.want_q ? 4 : 0);
}

}  // namespace
}  // namespace tritt
