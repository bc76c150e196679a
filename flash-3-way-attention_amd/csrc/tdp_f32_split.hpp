// The fp32 triple-dot kernels over whole problems (tdp_f32_mfma.hip launches them): fp32 operands, products as six bf16 products
// (f32_split.hpp).  Tiles, rounds, parts and masks as in tdp_f32_tiles.hpp.
#pragma once
#include <type_traits>
#include <utility>

#include "direct_lds.hpp"
#include "f32_split.hpp"
#include "tdp_f32_tiles.hpp"

namespace tritt {
namespace {

// The streamed tensors of a problem as images: every 32 rows as the three planes that a stage holds in LDS, swizzle and all, rows
// past the end zero.  A stage is then 6 KB x D / 32 of consecutive bytes per tensor, fetched direct to LDS.
template <int D>
constexpr size_t split_image_elems(int BH, int T) {
    return (size_t)BH * ((T + 31) / 32) * 3 * split_plane<D>();
}
// One image tile: thread t of NT takes pieces t, t + NT, ... of eight columns; x(row, column) -> eight floats
template <int D, typename X>
__device__ __forceinline__ void split_store_piece(__bf16* tile, int row, int piece, const X& x) {
    const Split8 s = split8_any(x);
    __bf16* at = tile + row * D + ((piece ^ split_swizzle<D>(row)) * 8);
    *reinterpret_cast<bf16x8*>(at) = s.h;
    *reinterpret_cast<bf16x8*>(at + split_plane<D>()) = s.m;
    *reinterpret_cast<bf16x8*>(at + 2 * split_plane<D>()) = s.l;
}

// The two streamed tensors of a kernel; waves 0 .. NW / 2 - 1 move the first one's stages, the others the second's.  PACKED: from
// images, direct to LDS.  Otherwise from the floats themselves, through registers, split on the way (short problems, where an
// image costs more than it saves; a forward that has no room for images).
template <int D, int NW, bool PACKED>
struct SplitStream {
    static constexpr int kStage = 3 * split_plane<D>();  // elements of one tensor's stage
    static constexpr int kBlocks = kStage * 2 / 1024 / (NW / 2), kThreads = NW * 32, kPer = 32 * D / 8 / kThreads;
    static_assert(kStage * 2 % (1024 * (NW / 2)) == 0 && 32 * D / 8 % kThreads == 0, "whole blocks and pieces");
    const void* src;  // of this wave's tensor, this slice
    __bf16* lds;      // [2][kStage] of this wave's tensor
    int T, silu;
    int slot = 0, fetched = 0;
    f32x4v x[PACKED ? 1 : 2 * kPer];
    // start on stage `st` into buffer `buf`
    __device__ __forceinline__ void fetch(int st, int buf) {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if constexpr (PACKED) {
            const char* at = reinterpret_cast<const char*>(src) + (size_t)st * (kStage * 2) + (wave & (NW / 2 - 1)) * (kBlocks * 1024);
            char* dst = reinterpret_cast<char*>(lds + buf * kStage) + (wave & (NW / 2 - 1)) * (kBlocks * 1024);
            const unsigned lane16 = (threadIdx.x & 63) * 16;
#pragma unroll
            for (int i = 0; i < kBlocks; ++i) direct_load_16(uniform_ptr(at + i * 1024), lane16, dst + i * 1024);
        } else {
            const int t = threadIdx.x & (kThreads - 1);
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                const int idx = t + i * kThreads, row = idx / (D / 8), c = idx % (D / 8) * 8;
                const f32x4v* at = reinterpret_cast<const f32x4v*>(reinterpret_cast<const float*>(src) + (size_t)min(st * 32 + row, T - 1) * D + c);
                x[2 * i] = at[0];
                x[2 * i + 1] = at[1];
            }
            slot = buf;
            fetched = 1;
        }
    }
    // before the barrier after which the stage fetched last is read
    __device__ __forceinline__ void complete() {
        if constexpr (PACKED) {
            wait_vmcnt<0>();
        } else if (fetched) {
            const int t = threadIdx.x & (kThreads - 1);
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                const int idx = t + i * kThreads;
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = x[2 * i + e / 4][e % 4];
                if (silu) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = silu_f(v[e]);
                }
                split_store_piece<D>(lds + slot * kStage, idx / (D / 8), idx % (D / 8), v);
            }
            fetched = 0;
        }
    }
};

// One 32-row tile of an image, from row r0 on, through SiLU or not; 256 threads
template <int D>
__device__ __forceinline__ void split_image_tile(const float* __restrict__ src, __bf16* __restrict__ dst, int r0, int T, bool silu) {
    for (int idx = threadIdx.x; idx < 32 * D / 8; idx += 256) {
        const int r = idx / (D / 8), c = idx % (D / 8), row = r0 + r;
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (row < T) {
            const f32x4v* at = reinterpret_cast<const f32x4v*>(src + (size_t)row * D + c * 8);
            const f32x4v lo = at[0], hi = at[1];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = e < 4 ? lo[e & 3] : hi[e & 3];
            if (silu) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = silu_f(v[e]);
            }
        }
        split_store_piece<D>(dst, r, c, v);
    }
}
// Images of two tensors, the second through SiLU when `silu1`: one workgroup per 32-row tile (x), slice (y) and tensor (z)
template <int D>
__global__ __launch_bounds__(256) void f32_split_images_kernel(const float* __restrict__ x0, const float* __restrict__ x1,
                                                               __bf16* __restrict__ image0, __bf16* __restrict__ image1, int silu1, int T) {
    const float* src = (blockIdx.z ? x1 : x0) + (size_t)blockIdx.y * T * D;
    __bf16* dst = (blockIdx.z ? image1 : image0) + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * (3 * split_plane<D>());
    split_image_tile<D>(src, dst, blockIdx.x * 32, T, blockIdx.z && silu1);
}

// B operand of a score product, k-step ks: columns 16 ks + 8 g .. + 7 of (query or key row n) times the round's row
struct Product8 {
    float x[8];
    __device__ __forceinline__ float operator[](int e) const { return x[e]; }
};
__device__ __forceinline__ Product8 row_product(const float* own, const float* row, int ks) {
    Product8 r;
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
        const f32x4v a = *reinterpret_cast<const f32x4v*>(own + 16 * ks + e), b = *reinterpret_cast<const f32x4v*>(row + 16 * ks + e);
#pragma unroll
        for (int k = 0; k < 4; ++k) r.x[e + k] = a[k] * b[k];
    }
    return r;
}
// Those of all k-steps, with one test for infinite and very large products: a test for each keeps the reads of the next k-step
// behind it (training step of B=2 H=4 T=500 D=64: no test 2566 us, one for each 2591, one for all 2551).
template <int KS>
__device__ __forceinline__ void split_products(Split8 (&s)[KS], const float* own, const float* row) {
    float most = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const Product8 x = row_product(own, row, ks);
        s[ks] = split8(x);
        most = fmaxf(most, largest8(x));
    }
    if (__builtin_expect(__any(most > kSplitMax), 0)) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s[ks] = split8_any(row_product(own, row, ks));
    }
}

// A backward that does not hold its operands (D = 128) has no round to test them in: whether the workgroup has met an own or a row
// operand above 2^63 (below, no product of the two is too large for split8).  A word per wave; that wave's staging writes it ahead
// of the barrier after which the operands are read, and a later one only sets it.  Backward of B=2 H=4 T=500 against no test: 6 % more
// with every product tested as it is formed (4.87 -> 5.17 ms), 1 % with this (4.97 -> 5.00).  With the words instead of the test of
// split_products the forward and D = 32, 64 were up to 2 % slower.
constexpr float kSplitFactor = 0x1p63f;
template <int NW>
struct LargeOperands {
    static_assert(NW == 4, "one 16-byte read");
    int* words;  // [NW], 16-byte aligned
    __device__ __forceinline__ void start(float most) const { words[threadIdx.x >> 6] = __any(most > kSplitFactor); }
    __device__ __forceinline__ void more(float most) const {
        if (__builtin_expect(__any(most > kSplitFactor), 0)) words[threadIdx.x >> 6] = 1;
    }
    __device__ __forceinline__ bool any() const {
        const int4 w = *reinterpret_cast<const int4*>(words);
        return __builtin_amdgcn_readfirstlane(w.x | w.y | w.z | w.w) != 0;
    }
};

// Split of a pair of floats in two slots of vector work: s's elements e, e + 1
struct SplitPair {
    f32x2 r;
};
__device__ __forceinline__ void split_pair_high(float a, float b, Split8& s, int e, SplitPair& t) {
    const f32x2 v = {a, b};
    const bf16x2 h = __builtin_convertvector(v, bf16x2);
    t.r = f32x2{a - (float)h[0], b - (float)h[1]};
    s.h[e] = h[0]; s.h[e + 1] = h[1];
}
__device__ __forceinline__ void split_pair_low(Split8& s, int e, const SplitPair& t) {
    const bf16x2 m = __builtin_convertvector(t.r, bf16x2);
    const f32x2 q = {t.r[0] - (float)m[0], t.r[1] - (float)m[1]};
    const bf16x2 l = __builtin_convertvector(q, bf16x2);
    s.m[e] = m[0]; s.m[e + 1] = m[1];
    s.l[e] = l[0]; s.l[e + 1] = l[1];
}

// The MFMAs of a wave are issued in order with its vector work, and the pipe takes one every 32 cycles: `tick` after each of them
// does one slot of up to eight vector instructions and pins both (the compiler's own order is all the MFMAs, then all the rest).
template <int I, typename F>
__device__ __forceinline__ void pinned(const F& slot) {
    slot(std::integral_constant<int, I>{});
    __builtin_amdgcn_sched_barrier(0);
}

// Sum over a stage's 32 rows of (columns 32 dt ..) x P or dS: twelve MFMAs from zero, the small products of both halves first.  The
// caller adds the result to its running sum, so that one is rounded once per stage and not twelve times.
template <int TICK0, typename F>
__device__ __forceinline__ f32x16 stage_product(const Split8 (&a)[2], const Split8 (&b)[2], const F& slot) {
    using M = Mma<__bf16>;
    f32x16 t;
#pragma unroll
    for (int i = 0; i < 16; ++i) t[i] = 0.f;
    t = M::mma(a[0].l, b[0].h, t); pinned<TICK0 + 0>(slot);
    t = M::mma(a[1].l, b[1].h, t); pinned<TICK0 + 1>(slot);
    t = M::mma(a[0].h, b[0].l, t); pinned<TICK0 + 2>(slot);
    t = M::mma(a[1].h, b[1].l, t); pinned<TICK0 + 3>(slot);
    t = M::mma(a[0].m, b[0].m, t); pinned<TICK0 + 4>(slot);
    t = M::mma(a[1].m, b[1].m, t); pinned<TICK0 + 5>(slot);
    t = M::mma(a[0].m, b[0].h, t); pinned<TICK0 + 6>(slot);
    t = M::mma(a[1].m, b[1].h, t); pinned<TICK0 + 7>(slot);
    t = M::mma(a[0].h, b[0].m, t); pinned<TICK0 + 8>(slot);
    t = M::mma(a[1].h, b[1].m, t); pinned<TICK0 + 9>(slot);
    t = M::mma(a[0].h, b[0].h, t); pinned<TICK0 + 10>(slot);
    t = M::mma(a[1].h, b[1].h, t); pinned<TICK0 + 11>(slot);
    return t;
}

struct F32FwdParams {
    const float *q, *ka, *kb, *va, *vb;  // streamed = (ka, va), rows = (kb, vb), dense [BH][T][D]
    const __bf16 *image_ka, *image_va;   // PACKED: the streamed tensors' images (ka and va are not read then)
    float *o, *lse;
    int silu_va;  // not PACKED: va is V1 itself, SiLU is applied as its stages go to LDS
    // deal.max_parts > 1: the rounds of a tile are dealt out to f32_tile_parts() workgroups; each leaves its unnormalised
    // output, reference maximum and row sum in part[((bh T + q) max_parts + y) (D + 4)] (O[D], M, L)
    F32Deal deal;
    float* part;
    int T, BH, nqt;
    float scale_log2;
    TdpMask mask;  // in terms of the streamed index a and the row index b
};

// ------------------------------------------------------------------------------------------ forward
// What bounds it: the matrix pipe and the clock.  A step (32 streamed rows of a wave's row) is 24 MFMAs of scores and 24 of
// values at D = 64, 1536 cycles, beside some 190 vector instructions (exponentials, the split of P) and 24 KB of operand
// reads; the pipe is busy 65 % of the cycles at a clock that falls to 1.7 GHz under random operands (2.2 GHz with zeros):
// 1.15 PFLOP/s of bf16 products executed, what library products reach here.  Hence: the scores of the next step are formed
// beside the exponentials of this one (one instruction stream holds both kinds of work), the streamed tensors come as images
// (splitting them as they are staged took 100 of 350 vector instructions per step, and every tile streams every row again), a
// workgroup is four waves of at most 256 registers and two share a CU (D = 128: one, 512 registers).  The operand of the
// score product is formed and split once per round and held.  fp32 MFMAs -> this, forward kernels and launches around them:
// B=2 H=4 T=500 D=64 875 -> 552 us, B=4 H=8 T=512 D=64 3353 -> 2111, B=2 H=4 T=500 D=128 1774 -> 1258, B=2 H=8 T=1000 D=32
// 6600 -> 4430; the output is 1.5 times nearer to 64 bits (B=2 H=4 T=200 D=64: 1.63e-7 -> 1.02e-7).
template <int D, int NW, bool PACKED>
__global__ __launch_bounds__(64 * NW, D > 64 ? 1 : 2) void tdp_f32_split_fwd_kernel(F32FwdParams p) {
    constexpr int DT = D / 32, KS = D / 16, LD = f32_pitch<D>(), NT = 64 * NW, STAGE = 3 * split_plane<D>();
    extern __shared__ __align__(16) float smem_f[];
    float* sM = smem_f;                 // [NW][32]    end of kernel: per-wave maxima and sums
    float* sL = sM + NW * 32;           // [NW][32]
    float* sQ = sL + NW * 32;           // [32][LD]    the tile's queries * scale
    float* sKb = sQ + 32 * LD;          // [3][NW][D]  row operands of a round
    float* sVb = sKb + 3 * NW * D;      // [3][NW][D]
    __bf16* sK = reinterpret_cast<__bf16*>(sVb + 3 * NW * D);  // [2][3][32][D] streamed key rows
    __bf16* sV = sK + 2 * STAGE;                               // [2][3][32][D] streamed value rows
    float* sO = sKb;                    // [NW][D][33] end of kernel: the waves' outputs (alias everything from the rows on)

    int bh, order;
    if (!xcd_tile(p.BH, p.deal.items, blockIdx.x >> 3, blockIdx.x & 7, bh, order)) return;
    const F32Item item = f32_item(p.deal, p.mask, order, p.nqt, p.T, NW);
    const int qt = item.qt, part = item.part, step = item.parts;
    if (part >= step) return;

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int T = p.T;
    const size_t base = (size_t)bh * T * D;
    const float* __restrict__ KB = p.kb + base;
    const float* __restrict__ VB = p.vb + base;
    const float* __restrict__ Qs = p.q + base;
    const TdpMask mask = p.mask;

    const int q0 = qt * 32, q1 = min(T - 1, q0 + 31);
    const int q = q0 + n;  // this lane's query (column of every tile)
    const Range rows = row_range(mask, q0, q1, T);
    // rounds of NW rows: workgroup `part` of a tile takes every step-th one from the part-th on
    const int m_lo = rows.lo / NW + part, m_hi = rows.hi / NW;

    // the (round, stage) steps: w0 is worked on, the scores of w1 are formed meanwhile, w2 is fetched
    Walk w0{}, w1{}, w2{};
    auto next = [&](const Walk& w, Walk& to) {
        to = Walk{w.m, w.st + 1, w.st_hi};
        return w.st < w.st_hi || open_round<NW>(to, mask, w.m + step, m_hi, step, q0, q1, T);
    };
    bool have = open_round<NW>(w0, mask, m_lo, m_hi, step, q0, q1, T);
    bool have1 = have && next(w0, w1);

    SplitStream<D, NW, PACKED> stream;
    const bool first = wave < NW / 2;  // this wave moves key stages
    stream.T = T;
    stream.silu = !first && p.silu_va;
    stream.lds = first ? sK : sV;
    if constexpr (PACKED) stream.src = (first ? p.image_ka : p.image_va) + (size_t)bh * ((T + 31) / 32) * STAGE;
    else stream.src = (first ? p.ka : p.va) + base;
    constexpr int kRowPer = (NW * D + NT - 1) / NT;
    float row_k[kRowPer], row_v[kRowPer];
    auto fetch_rows = [&](int m) {
#pragma unroll
        for (int i = 0; i < kRowPer; ++i) {
            const int idx = min(tid + i * NT, NW * D - 1);
            const size_t at = (size_t)min(m * NW + idx / D, T - 1) * D + idx % D;
            row_k[i] = KB[at];
            row_v[i] = VB[at];
        }
    };
    auto store_rows = [&](int slot) {
#pragma unroll
        for (int i = 0; i < kRowPer; ++i)
            if (tid + i * NT < NW * D) {
                sKb[slot * NW * D + tid + i * NT] = row_k[i];
                sVb[slot * NW * D + tid + i * NT] = row_v[i];
            }
    };

    if (have) {
        fetch_rows(w0.m);
        stream.fetch(w0.st, 0);
    }
    for (int idx = tid; idx < 32 * D; idx += NT) {
        const int r = idx / D, d = idx % D;
        sQ[r * LD + d] = Qs[(size_t)min(q0 + r, T - 1) * D + d] * p.scale_log2;
    }
    if (have) store_rows(0);
    stream.complete();
    bool fresh1 = have1 && w1.m != w0.m;  // w1 is the first step of its round
    if (have1 && first) stream.fetch(w1.st, 1);
    if (fresh1) {
        fetch_rows(w1.m);
        store_rows(1);
    }
    stream.complete();
    __syncthreads();

    const int row_base = split_row_base<D>(lane), col_base = split_col_base<D>(lane);
    Split8 bq[KS];
    auto form_operand = [&](int slot) {
        const float* ob = sKb + (slot * NW + wave) * D;
        split_products(bq, sQ + n * LD + 8 * g, ob + 8 * g);
    };
    auto scores = [&](const __bf16* tile) {
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.f;
        bf16x8 kh[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const Split8 ka = split_rows<D>(tile, row_base, ks);
            s = small_products(ka, bq[ks], s);
            kh[ks] = ka.h;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s = large_product(kh[ks], bq[ks].h, s);
        return s;
    };
    f32x16 accO[DT], accT[DT], s;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            accO[dt][i] = 0.f;
            accT[dt][i] = 0.f;
        }
    float m_run = kNegBig, l_run = 0.f;  // per query, over every (a, b) this wave has seen (l: this lane's half)
    if (have) {
        form_operand(0);
        s = scores(sK);
        __syncthreads();  // the first step's fetch of w2 overwrites the keys of w0
    }
    int buf = 0, slot0 = 0, slot1 = fresh1 ? 1 : 0;  // buffer of V(w0) (and of K(w0), K(w2)); places of the rounds' rows
    while (have) {
        const bool have2 = have1 && next(w1, w2), fresh2 = have2 && w2.m != w1.m;
        const int slot2 = fresh2 ? (slot1 == 2 ? 0 : slot1 + 1) : slot1;
        if (first ? have2 : have1) stream.fetch(first ? w2.st : w1.st, first ? buf : buf ^ 1);
        if (fresh2) fetch_rows(w2.m);
        if (fresh1) form_operand(slot1);

        const int b = w0.m * NW + wave, a0 = w0.st * 32;
        const bool row_ok = b <= rows.hi && b >= rows.lo;
        if (!row_ok || !all_valid(mask, q0, a0, b, T)) {
            const Interval ok = valid_interval(mask, q, b, T);
            const int x = a0 + 8 * g - ok.lo;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = row_ok && (unsigned)(x + key_of(0, i)) <= ok.span ? s[i] : -INFINITY;
        }
        // exponentials relative to the query's reference, which is some earlier tile's maximum: a sum that outgrows it by 2^16
        // (or the first one of all) moves it to this tile's maximum.  fp32 sums lose no digits by a loose reference, and the
        // maximum need not be formed for every tile; what they lose is room below the end of fp32's range, which 2^40 took
        // from values whose products reach 1e26
        float psum = 0.f;
        Split8 bp[2];  // registers 8 half .. + 7 of a lane are its k-slots of streamed rows 16 half ..
        auto exponentials = [&] {
            psum = 0.f;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    x[e] = fast_exp2(s[8 * half + e] - m_run);
                    psum += x[e];
                }
                bp[half] = split8(x);
            }
        };
        const f32x16 s1 = scores(sK + (buf ^ 1) * STAGE);  // of w1 (of no use after the last step)
        exponentials();
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
            exponentials();
        }
        l_run += psum;
        // Tv^T[d, q] += VA^T[d, a] P^T[a, q]
        const __bf16* cV = sV + buf * STAGE;
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) accT[dt] = products_of_step(split_cols<D>(cV, col_base, half, dt), bp[half], accT[dt]);
        if (w0.st == w0.st_hi) {
            // the finished row: O^T[d, q] += Tv^T[d, q] * VB[b, d]   (register i of half g: d = 32 dt + c_row(g, i))
            if (row_ok) {
                const float* vb = sVb + (slot0 * NW + wave) * D + 4 * g;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int i = 0; i < 16; i += 4) {
                        const f32x4v v = *reinterpret_cast<const f32x4v*>(vb + 32 * dt + c_row(0, i));
#pragma unroll
                        for (int e = 0; e < 4; ++e) accO[dt][i + e] += accT[dt][i + e] * v[e];
                    }
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) accT[dt][i] = 0.f;
        }
        if (have1) {
            if (fresh2) store_rows(slot2);
            stream.complete();
            __syncthreads();
        }
        s = s1;
        buf ^= 1;
        slot0 = slot1; slot1 = slot2;
        w0 = w1; w1 = w2;
        fresh1 = fresh2;
        have = have1; have1 = have2;
    }

    // ---- merge the waves' partial results: each leaves its own, relative to the common maximum, in a [D][33] slice of LDS,
    // and the slices are added in a fixed order
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
        for (int i = 0; i < 16; ++i) sO[wave * D * 33 + (32 * dt + c_row(g, i)) * 33 + n] = accO[dt][i] * mine_scale;
    __syncthreads();
    auto merged = [&](int d, int r) {
        float v = sO[d * 33 + r];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += sO[(w * D + d) * 33 + r];
        return v;
    };
    auto sum_of = [&](int r, float& Mr) {
        Mr = kNegBig;
        float L = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) Mr = fmaxf(Mr, sM[w * 32 + r]);
#pragma unroll
        for (int w = 0; w < NW; ++w) L += sL[w * 32 + r] * fast_exp2(sM[w * 32 + r] - Mr);
        return L;
    };
    const bool split = p.deal.max_parts > 1;  // perhaps one of several workgroups of the tile (f32_merge_kernel)
    for (int idx = tid; idx < 32 * D; idx += NT) {
        const int r = idx / D, d = idx % D;
        if (q0 + r >= T) continue;
        if (split) {
            p.part[(((size_t)bh * T + q0 + r) * p.deal.max_parts + part) * (D + 4) + d] = merged(d, r);
        } else {
            float Mr;
            p.o[base + (size_t)(q0 + r) * D + d] = merged(d, r) / sum_of(r, Mr);
        }
    }
    if (wave == 0 && g == 0 && q < T) {
        float Mr;
        const float L = sum_of(n, Mr);
        if (split) {
            float* ml = p.part + (((size_t)bh * T + q) * p.deal.max_parts + part) * (D + 4) + D;
            ml[0] = Mr; ml[1] = L;
        } else {
            p.lse[(size_t)bh * T + q] = (Mr + fast_log2(L)) * kLn2;
        }
    }
}

template <int D, int NW>
constexpr size_t f32_split_fwd_smem() {
    constexpr size_t loop = sizeof(float) * 6 * NW * D + 2 * 2 * 3 * sizeof(__bf16) * split_plane<D>(), merge = sizeof(float) * NW * D * 33;
    return sizeof(float) * (2 * NW * 32 + 32 * f32_pitch<D>()) + (loop > merge ? loop : merge);
}

// ------------------------------------------------------------------------------------------ backward
// Two kinds of workgroups in one grid.  Both own 32 rows o (the columns of every tile), take rows b = k of (K2, V2), one per
// wave and round, and stream 32 rows a at a time:
//   queries:  o = q, a = j: own (Q, dO), streamed (K1, U):     dQ
//   keys:     o = j, a = q: own (K1, U), streamed (Q, dO):     dK1, dU, dK2, dV2
// With KO, VO the own and KA, VA the streamed tensors,
//   S^T[a, o] = KA[a] . (alpha log2(e) KO[o] (.) KB[b]),  dP^T[a, o] = VA[a] . (VO[o] (.) VB[b]),
//   P = exp2(S - LSE2[q]),  dS = P (dP - Delta[q]),
//   Z^T[d, o] += KA^T[d, a] dS^T[a, o],      keys: W^T[d, o] += VA^T[d, a] P^T[a, o]
// and when the row is finished
//   dKO[o] += Z KB[b],      keys: dVO[o] += W VB[b],  dKB[b] += sum_o Z KO[o],  dVB[b] += sum_o W VO[o]
// so the four row and key gradients take the two products Z and W: seven products in all, where launches that both own queries
// (streaming K1 and K2 in turn) execute eight.
// What is owned is summed in registers over the rounds and left in fp32, a place per part; the sums over own rows go to shared
// accumulators by row b (fixed point, or a tile's own fp32 ones: F32SplitBwdParams).
// What bounds it: vector work and latency beside the products.  A step of a key workgroup is 96 MFMAs (3072 cycles) at D = 64, of a
// query workgroup 72, but the four waves of a CU have a SIMD each (the accumulators, the held operands and the next step's
// scores take the 512 registers), so what is not interleaved with MFMAs in the instruction stream is not hidden: the first
// operand reads of a step, the operands and sums of a finished row (some 1100 vector instructions a round, which lasts T / 64
// steps on average).  Matrix pipe busy 45 % at T = 512.  fp32 MFMAs in two launches of eight products -> this, training step:
// B=2 H=4 T=500 D=64 4345 -> 2570 us, B=4 H=8 T=512 D=64 16.8 -> 10.1 ms, B=2 H=8 T=1000 D=32 32.1 -> 18.4 ms, B=2 H=4 T=500 D=128
// 8.5 -> 6.1 ms, B=1 H=2 T=2000 D=64 windows 128 / 64 1199 -> 694 us.  Of it: six bf16 products for one 16.8 -> 12.0, work pinned
// between the MFMAs -> 11.0, the sums over lanes by swaps and DPP -> 10.1.  D = 32 forms its scores in turn: two waves a SIMD
// fill each other's gaps (scores ahead need 212 B of scratch per lane there; 19.7 -> 18.4 ms).
// Scales of the fp32 tensors' row-gradient accumulators.  A gradient shrinks with every operand in it while dO stays, so the
// scale follows all of them: with the slice's largest finite |dO|, |Q|, |K1|, |V1|, |V2| (`maxima`, kScaleParts words per
// tensor and slice, [tensor][BH][parts]; |SiLU(x)| <= |x|) and sum P = 1,
//   |dV2| <= T max|dO| max|V1|       |dK2| <= alpha T max|Q| max|K1| 2 D max|dO| max|V1| max|V2|
// and a sum of that size is placed at 2^61.  A tensor with a few large elements makes this bound far too wide: the step is
// never coarser than 2^-36 of max |dO| (sums past 2^27 times it then set the row's poison word, common.hpp).
// B=4 H=8 T=128 D=64 with operands of 1 / 0.05 / 0.02 / 0.01, dK2 against 64 bits: 4.5e-7 / 1.4e-4 / 5.3e-3 / 8.1e-2 with the
// scale of dO alone, 4.5e-7 / 2.8e-7 / 3.1e-7 / 3.2e-7 with this one.  Kernel time of a training step, dO's scale -> this:
// B=2 H=4 T=500 D=64 4335 -> 4330 us, B=1 H=2 T=128 D=64 160.4 -> 159.8, B=4 H=8 T=128 D=64 531 -> 539.
constexpr int kF32FixedBias = 36;
enum { kMaxDO, kMaxQ, kMaxK1, kMaxV1, kMaxV2, kMaxima };
struct F32RowScale {
    const unsigned* maxima;      // null: one scale by max |dO| (or float accumulators)
    unsigned* fields;            // [BH][2] for the launch that converts: dK2, dV2
    int free_k, free_v;          // exponent field that a sum bounded by 1 would get, less what alpha, T and D take
};
__device__ __forceinline__ void f32_row_fields(const F32RowScale& s, int BH, int bh, int& field_k, int& field_v) {
    // lane t * kScaleParts + i holds part i of tensor t, and at the end an exponent that all of that tensor is below
    const int lane = threadIdx.x & 63, t = lane / kScaleParts;
    static_assert(kScaleParts == 8 && kMaxima * kScaleParts <= 64, "one word per lane");
    unsigned m = s.maxima[((size_t)min(t, kMaxima - 1) * BH + bh) * kScaleParts + lane % kScaleParts];
#pragma unroll
    for (int w = 1; w < kScaleParts; w *= 2) m = max(m, (unsigned)__shfl_xor((int)m, w, 64));
    const int e = (int)(m >> 23) - 126;
    auto exponent = [&](int tensor) { return __builtin_amdgcn_readlane(e, tensor * kScaleParts); };
    const int d_o = exponent(kMaxDO), v1 = exponent(kMaxV1), v2 = exponent(kMaxV2);
    const int least = max(min(kF32FixedBias + 254 - 126 - d_o, 254), 1);  // as fixed_scale_field
    field_v = s.free_v - d_o - v1;
    field_k = s.free_k - d_o - v1 - v2 - exponent(kMaxQ) - exponent(kMaxK1);
    field_k = max(least, min(field_k, 254));
    field_v = max(least, min(field_v, 254));
}

struct F32SplitBwdParams {
    const float *q, *d_o, *k1, *u, *k2, *v2;                     // dense [BH][T][D]
    const __bf16 *image_q, *image_do, *image_k1, *image_u;       // images of those that are streamed
    const float *lse, *delta;
    // queries: dQ / alpha of part y in part_q[((bh T + q) deal_q.max_parts + y) D], or dQ itself in dq (part_q null)
    float *dq, *part_q;
    float *part_k1, *part_u;  // keys: dK1 / alpha and dU, the same with deal_k
    void *acc_k, *acc_v;      // [BH][T][D] dK2 and dV2: fixed point (long long) or float
    size_t acc_tile;          // elements from one key tile's acc_k, acc_v to the next one's (0: all tiles add to the same)
    F32RowScale rows;         // fixed-point accumulators: their scales
    unsigned* poison;
    F32Deal deal_q, deal_k;
    int key_blocks;           // workgroups of the second kind: the first of the grid
    int T, BH, nqt;
    float alpha;
    TdpMask mask;             // in terms of a = j and b = k
};

// The waves' shares of what a tile owns, side by side in LDS and added in a fixed order; put(row, column, sum)
template <int D, int NW, typename F>
__device__ __forceinline__ void join_owned(float* s, const f32x16 (&acc)[D / 32], const F& put) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 31, g = lane >> 5;
    __syncthreads();
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[wave * D * 33 + (32 * dt + c_row(g, i)) * 33 + n] = acc[dt][i];
    __syncthreads();
    for (int idx = threadIdx.x; idx < 32 * D; idx += 64 * NW) {
        const int r = idx / D, d = idx % D;
        float v = s[d * 33 + r];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += s[(w * D + d) * 33 + r];
        put(r, d, v);
    }
}

template <int D, int NW, bool KEYS>
__device__ __forceinline__ void f32_split_bwd_body(const F32SplitBwdParams& p, const int block) {
    constexpr int DT = D / 32, KS = D / 16, LD = f32_pitch<D>(), NT = 64 * NW, STAGE = 3 * split_plane<D>();
    // D <= 64: the scores of the next step are formed beside the exponentials of this one (three stages in LDS) and the B operands
    // of the score products are held over a round; D = 128 has room for neither (registers; LDS)
    constexpr bool AHEAD = D == 64, HOLD = D <= 64;
    constexpr int NBUF = AHEAD ? 3 : 2;
    extern __shared__ __align__(16) float smem_f[];
    const LargeOperands<NW> large{reinterpret_cast<int*>(smem_f)};  // [NW]  not HOLD
    float* sKo = smem_f + NW;            // [32][LD]  own rows: KO * alpha * log2(e)
    float* sVo = sKo + 32 * LD;          // [32][LD]  VO
    float* sKb = sVo + 32 * LD;          // [3][NW][D]  rows of a round
    float* sVb = sKb + 3 * NW * D;       // [3][NW][D]
    float* sStat = sVb + 3 * NW * D;     // [NBUF][2][32]  keys: LSE2 and Delta of a stage's queries
    __bf16* sK = reinterpret_cast<__bf16*>(sStat + NBUF * 64);  // [NBUF][3][32][D]
    __bf16* sV = sK + NBUF * STAGE;                             // [NBUF][3][32][D]
    float* sO = sKb;                     // [NW][D][33] end of kernel (aliases everything from the rows on)

    const F32Deal& deal = KEYS ? p.deal_k : p.deal_q;
    int bh, order;
    if (!xcd_tile(p.BH, deal.items, block >> 3, block & 7, bh, order)) return;
    const F32Item item = f32_item(deal, p.mask, order, p.nqt, p.T, NW);
    const int part = item.part, step = item.parts;
    if (part >= step) return;

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int T = p.T;
    const size_t base = (size_t)bh * T * D;
    const float* __restrict__ KB = p.k2 + base;
    const float* __restrict__ VB = p.v2 + base;
    const TdpMask mask = p.mask;
    const float scale_log2 = p.alpha * kLog2e;
    const int o0 = item.qt * 32, o1 = min(T - 1, o0 + 31), o = o0 + n;
    const Range rows = own_row_range<KEYS>(mask, o0, o1, T);
    const int m_lo = rows.lo / NW + part, m_hi = rows.hi / NW;

    Walk w0{}, w1{}, w2{};
    auto next = [&](const Walk& w, Walk& to) {
        to = Walk{w.m, w.st + 1, w.st_hi};
        return w.st < w.st_hi || open_round<NW, KEYS>(to, mask, w.m + step, m_hi, step, o0, o1, T);
    };
    bool have = open_round<NW, KEYS>(w0, mask, m_lo, m_hi, step, o0, o1, T);
    bool have1 = have && next(w0, w1);

    SplitStream<D, NW, true> stream;
    const bool first = wave < NW / 2;
    stream.T = T;
    stream.silu = 0;
    stream.lds = first ? sK : sV;
    stream.src = (KEYS ? first ? p.image_q : p.image_do : first ? p.image_k1 : p.image_u) + (size_t)bh * p.nqt * STAGE;
    float stat = 0.f;
    auto fetch = [&](int st, int buf) {
        stream.fetch(st, buf);
        if (KEYS && tid < 64) {  // a query past the end of the sequence gets a huge LSE: its P is exactly 0
            const int q = st * 32 + (tid & 31);
            const float* src = tid < 32 ? p.lse : p.delta;
            stat = q < T ? src[(size_t)bh * T + q] : tid < 32 ? 1.0e30f : 0.f;
            if (tid < 32) stat *= kLog2e;
        }
    };
    auto complete = [&](int buf) {
        if (KEYS && tid < 64) sStat[buf * 64 + tid] = stat;
        stream.complete();
    };
    constexpr int kRowPer = (NW * D + NT - 1) / NT;
    float row_k[kRowPer], row_v[kRowPer];
    auto fetch_rows = [&](int m) {
#pragma unroll
        for (int i = 0; i < kRowPer; ++i) {
            const int idx = min(tid + i * NT, NW * D - 1);
            const size_t at = (size_t)min(m * NW + idx / D, T - 1) * D + idx % D;
            row_k[i] = KB[at];
            row_v[i] = VB[at];
        }
    };
    auto rows_most = [&] {
        float most = 0.f;
#pragma unroll
        for (int i = 0; i < kRowPer; ++i) most = fmaxf(most, fmaxf(fabsf(row_k[i]), fabsf(row_v[i])));
        return most;
    };
    auto store_rows = [&](int slot) {
#pragma unroll
        for (int i = 0; i < kRowPer; ++i)
            if (tid + i * NT < NW * D) {
                sKb[slot * NW * D + tid + i * NT] = row_k[i];
                sVb[slot * NW * D + tid + i * NT] = row_v[i];
            }
    };

    if (have) {
        fetch_rows(w0.m);
        fetch(w0.st, 0);
    }
    const float* KO = (KEYS ? p.k1 : p.q) + base;
    const float* VO = (KEYS ? p.u : p.d_o) + base;
    [[maybe_unused]] float most = 0.f;
    for (int idx = tid; idx < 32 * D; idx += NT) {
        const int r = idx / D, d = idx % D;
        const size_t at = (size_t)min(o0 + r, T - 1) * D + d;
        const float ko = KO[at] * scale_log2, vo = VO[at];
        sKo[r * LD + d] = ko;
        sVo[r * LD + d] = vo;
        if (!HOLD) most = fmaxf(most, fmaxf(fabsf(ko), fabsf(vo)));
    }
    float fscale_k = 0.f, fscale_v = 0.f;
    if (KEYS && p.rows.maxima) {
        int field_k, field_v;
        f32_row_fields(p.rows, p.BH, bh, field_k, field_v);
        fscale_k = fixed_scale_value(field_k);
        fscale_v = fixed_scale_value(field_v);
        if (o0 == 0 && part == 0 && tid == 0) {
            p.rows.fields[bh * 2] = field_k;
            p.rows.fields[bh * 2 + 1] = field_v;
        }
    }
    float lse2 = 1.0e30f, delta = 0.f;  // queries: this lane's
    if (!KEYS && o < T) {
        lse2 = p.lse[(size_t)bh * T + o] * kLog2e;
        delta = p.delta[(size_t)bh * T + o];
    }
    if (have) {
        store_rows(0);
        if (!HOLD) most = fmaxf(most, rows_most());
        complete(0);
    }
    if (!HOLD) large.start(most);
    bool fresh1 = have1 && w1.m != w0.m;  // w1 is the first step of its round
    if (AHEAD && have1) {
        fetch(w1.st, 1);
        if (fresh1) {
            fetch_rows(w1.m);
            store_rows(1);
        }
        complete(1);
    }
    __syncthreads();

    const int row_base = split_row_base<D>(lane), col_base = split_col_base<D>(lane);
    Split8 bq[HOLD ? KS : 1], bg[HOLD ? KS : 1];
    auto form_operands = [&](int slot) {
        if constexpr (HOLD) {
            const int at = (slot * NW + wave) * D + 8 * g;
            split_products(bq, sKo + n * LD + 8 * g, sKb + at);
            split_products(bg, sVo + n * LD + 8 * g, sVb + at);
        }
    };
    // the score products of the stage in `buf`; after MFMA i slots 2 i DT / 4 .. of other work (48 slots over 48 MFMAs at D = 64)
    auto scores = [&](int buf, f32x16& s, f32x16& dp, const auto& work) {
        using M = Mma<__bf16>;
        const __bf16 *tk = sK + buf * STAGE, *tv = sV + buf * STAGE;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = 0.f;
            dp[i] = 0.f;
        }
        Split8 ka[2] = {split_rows<D>(tk, row_base, 0), {}}, va[2] = {split_rows<D>(tv, row_base, 0), {}};
        bf16x8 kh[KS], vh[KS];
        auto tick = [&](auto at) {
            constexpr int I = decltype(at)::value;
            if constexpr (DT == 1) work(std::integral_constant<int, 2 * I>{});
            work(std::integral_constant<int, DT == 1 ? 2 * I + 1 : I>{});
            __builtin_amdgcn_sched_barrier(0);
        };
        auto step = [&](auto at) {
            constexpr int ks = decltype(at)::value;
            if constexpr (ks + 1 < KS) {
                ka[(ks + 1) & 1] = split_rows<D>(tk, row_base, ks + 1);
                va[(ks + 1) & 1] = split_rows<D>(tv, row_base, ks + 1);
            }
            const Split8 &a = ka[ks & 1], &v = va[ks & 1], &q = bq[HOLD ? ks : 0], &o = bg[HOLD ? ks : 0];
            s = M::mma(a.l, q.h, s); tick(std::integral_constant<int, 10 * ks>{});
            dp = M::mma(v.l, o.h, dp); tick(std::integral_constant<int, 10 * ks + 1>{});
            s = M::mma(a.h, q.l, s); tick(std::integral_constant<int, 10 * ks + 2>{});
            dp = M::mma(v.h, o.l, dp); tick(std::integral_constant<int, 10 * ks + 3>{});
            s = M::mma(a.m, q.m, s); tick(std::integral_constant<int, 10 * ks + 4>{});
            dp = M::mma(v.m, o.m, dp); tick(std::integral_constant<int, 10 * ks + 5>{});
            s = M::mma(a.m, q.h, s); tick(std::integral_constant<int, 10 * ks + 6>{});
            dp = M::mma(v.m, o.h, dp); tick(std::integral_constant<int, 10 * ks + 7>{});
            s = M::mma(a.h, q.m, s); tick(std::integral_constant<int, 10 * ks + 8>{});
            dp = M::mma(v.h, o.m, dp); tick(std::integral_constant<int, 10 * ks + 9>{});
            kh[ks] = a.h;
            vh[ks] = v.h;
        };
        auto large = [&](auto at) {
            constexpr int ks = decltype(at)::value;
            s = M::mma(kh[ks], bq[HOLD ? ks : 0].h, s); tick(std::integral_constant<int, 10 * KS + 2 * ks>{});
            dp = M::mma(vh[ks], bg[HOLD ? ks : 0].h, dp); tick(std::integral_constant<int, 10 * KS + 2 * ks + 1>{});
        };
        [&]<int... K>(std::integer_sequence<int, K...>) {
            (step(std::integral_constant<int, K>{}), ...);
            (large(std::integral_constant<int, K>{}), ...);
        }(std::make_integer_sequence<int, KS>{});
    };
    // the same without held operands
    auto scores_formed = [&](int buf, int slot, f32x16& s, f32x16& dp, auto any) {
        constexpr bool ANY = decltype(any)::value;
        const __bf16 *tk = sK + buf * STAGE, *tv = sV + buf * STAGE;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = 0.f;
            dp[i] = 0.f;
        }
        int own = n * LD + 8 * g, at = (slot * NW + wave) * D + 8 * g;
        asm volatile("" : "+v"(own), "+v"(at));  // (opaque: every read is one of them plus an immediate offset)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            s = products_of_step(split_rows<D>(tk, row_base, ks), split_value<ANY>(row_product(sKo + own, sKb + at, ks)), s);
            dp = products_of_step(split_rows<D>(tv, row_base, ks), split_value<ANY>(row_product(sVo + own, sVb + at, ks)), dp);
            __builtin_amdgcn_sched_barrier(0);  // one k-step's operands in registers at a time
        }
    };
    f32x16 accKo[DT], accVo[KEYS ? DT : 1], accZ[DT], accW[KEYS ? DT : 1], s, dp;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            accKo[dt][i] = 0.f;
            accZ[dt][i] = 0.f;
            if constexpr (KEYS) {
                accVo[dt][i] = 0.f;
                accW[dt][i] = 0.f;
            }
        }
    if constexpr (AHEAD)
        if (have) {
            form_operands(0);
            scores(0, s, dp, [](auto) {});
        }
    [[maybe_unused]] bool fresh = true;  // not AHEAD: w0 is the first step of its round
    int buf = 0, slot0 = 0, slot1 = fresh1 ? 1 : 0;
    while (have) {
        const int buf1 = buf + 1 == NBUF ? 0 : buf + 1, buf2 = buf1 + 1 == NBUF ? 0 : buf1 + 1;
        bool have2 = false, fresh2 = false;
        int slot2 = slot1;
        if constexpr (AHEAD) {
            have2 = have1 && next(w1, w2);
            fresh2 = have2 && w2.m != w1.m;
            if (fresh2) slot2 = slot1 == 2 ? 0 : slot1 + 1;
            if (have2) fetch(w2.st, buf2);
            if (fresh2) fetch_rows(w2.m);
            if (fresh1) form_operands(slot1);
        } else {
            if (fresh1) slot1 = slot0 == 2 ? 0 : slot0 + 1;
            if (have1) fetch(w1.st, buf1);
            if (fresh1) fetch_rows(w1.m);
            if (HOLD && fresh) form_operands(slot0);
            fresh = fresh1;
            if constexpr (HOLD) scores(buf, s, dp, [](auto) {});
            else if (__builtin_expect(large.any(), 0)) scores_formed(buf, slot0, s, dp, std::true_type{});
            else scores_formed(buf, slot0, s, dp, std::false_type{});
        }
        const int b = w0.m * NW + wave, a0 = w0.st * 32;
        const bool row_ok = b <= rows.hi && b >= rows.lo;
        if (!row_ok || !own_all_valid<KEYS>(mask, o0, a0, b, T)) {
            const Interval ok = own_interval<KEYS>(mask, o, b, T);
            const int x = a0 + 8 * g - ok.lo;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = row_ok && (unsigned)(x + key_of(0, i)) <= ok.span ? s[i] : -INFINITY;
        }
        f32x16 s1, dp1;
        const __bf16 *cK = sK + buf * STAGE, *cV = sV + buf * STAGE;
        f32x4v stat_l[KEYS ? 4 : 1], stat_d[KEYS ? 4 : 1];
        if constexpr (KEYS) {
            const float* at = sStat + buf * 64 + 8 * g;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                stat_l[i] = *reinterpret_cast<const f32x4v*>(at + 16 * (i / 2) + 4 * (i % 2));
                stat_d[i] = *reinterpret_cast<const f32x4v*>(at + 32 + 16 * (i / 2) + 4 * (i % 2));
            }
        }
        // P and dS, split: registers 8 half .. + 7 of a lane are its k-slots of streamed rows 16 half ..; slot I does a part of
        // the work on registers 2 (I / kSlots), + 1
        constexpr int kSlots = KEYS ? 6 : 4;
        Split8 bp[2], bs[2];
        f32x2 pv, ds;
        SplitPair rest;
        auto softmax = [&](auto slot) {
            constexpr int I = decltype(slot)::value, e = 2 * (I / kSlots), op = I % kSlots, half = (e / 8) & 1, k = e % 8;
            if constexpr (I < 8 * kSlots) {
                constexpr int last_op = kSlots - 2;
                if constexpr (op == 0) {
                    const float l0 = KEYS ? stat_l[KEYS ? e / 4 : 0][e % 4] : lse2, l1 = KEYS ? stat_l[KEYS ? e / 4 : 0][e % 4 + 1] : lse2;
                    pv = f32x2{fast_exp2(s[e] - l0), fast_exp2(s[e + 1] - l1)};
                } else if constexpr (op == 1) {
                    const float d0 = KEYS ? stat_d[KEYS ? e / 4 : 0][e % 4] : delta, d1 = KEYS ? stat_d[KEYS ? e / 4 : 0][e % 4 + 1] : delta;
                    ds = f32x2{pv[0] * (dp[e] - d0), pv[1] * (dp[e + 1] - d1)};
                } else if constexpr (op == last_op) {
                    split_pair_high(ds[0], ds[1], bs[half], k, rest);
                } else if constexpr (op == last_op + 1) {
                    split_pair_low(bs[half], k, rest);
                } else if constexpr (op == 2) {
                    split_pair_high(pv[0], pv[1], bp[half], k, rest);
                } else {
                    split_pair_low(bp[half], k, rest);
                }
            }
        };
        if constexpr (AHEAD) {
            scores(buf1, s1, dp1, softmax);  // of w1 (of no use after the last step)
        } else {
            [&]<int... I>(std::integer_sequence<int, I...>) { (softmax(std::integral_constant<int, I>{}), ...); }(std::make_integer_sequence<int, 8 * kSlots>{});
        }
        // W += VA^T P and Z += KA^T dS, a column tile at a time; the operands of one are read, and the sum of the one before is
        // taken up, beside the MFMAs of this one
        constexpr int kGroups = KEYS ? 2 * DT : DT;
        Split8 col[2][2];
        f32x16 sum[2];
        auto read_cols = [&](auto group) {
            constexpr int G = decltype(group)::value;
            if constexpr (G < kGroups) {
                const __bf16* tile = KEYS && G < DT ? cV : cK;
#pragma unroll
                for (int half = 0; half < 2; ++half) col[G & 1][half] = split_cols<D>(tile, col_base, half, G % DT);
            }
        };
        auto take_up = [&](auto group, auto slot) {  // registers of group G's sum, two a slot, where its MFMAs have drained
            constexpr int G = decltype(group)::value, I = decltype(slot)::value;
            if constexpr (G >= 0 && I >= 2 && I < 10) {
                f32x16& acc = KEYS && G < DT ? accW[KEYS ? G % DT : 0] : accZ[G % DT];
                acc[2 * (I - 2)] += sum[G & 1][2 * (I - 2)];
                acc[2 * (I - 2) + 1] += sum[G & 1][2 * (I - 2) + 1];
            }
        };
        read_cols(std::integral_constant<int, 0>{});
        auto product = [&](auto group) {
            constexpr int G = decltype(group)::value;
            if constexpr (G < kGroups) {
                read_cols(std::integral_constant<int, G + 1>{});
                sum[G & 1] = stage_product<0>(col[G & 1], KEYS && G < DT ? bp : bs, [&](auto slot) { take_up(std::integral_constant<int, G - 1>{}, slot); });
            }
        };
        [&]<int... G>(std::integer_sequence<int, G...>) { (product(std::integral_constant<int, G>{}), ...); }(std::make_integer_sequence<int, kGroups>{});
        [&]<int... I>(std::integer_sequence<int, I...>) { (take_up(std::integral_constant<int, kGroups - 1>{}, std::integral_constant<int, I>{}), ...); }(std::make_integer_sequence<int, 12>{});
        if (w0.st == w0.st_hi) {
            if (row_ok) {
                // register i of half g is column d = 32 dt + c_row(g, i)
                int at = (slot0 * NW + wave) * D + 4 * g, own = n * LD + 4 * g;
                asm volatile("" : "+v"(at), "+v"(own));
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int i = 0; i < 16; i += 4) {
                        const f32x4v kb = *reinterpret_cast<const f32x4v*>(sKb + at + 32 * dt + c_row(0, i));
#pragma unroll
                        for (int e = 0; e < 4; ++e) accKo[dt][i + e] += accZ[dt][i + e] * kb[e];
                        if constexpr (KEYS) {
                            const f32x4v vb = *reinterpret_cast<const f32x4v*>(sVb + at + 32 * dt + c_row(0, i));
#pragma unroll
                            for (int e = 0; e < 4; ++e) accVo[dt][i + e] += accW[dt][i + e] * vb[e];
                        }
                    }
                if constexpr (KEYS) {
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) {
                        f32x16 xk, xv;  // sKo holds KO * alpha * log2(e): alpha is wanted, log2(e) is not
#pragma unroll
                        for (int i = 0; i < 16; i += 4) {
                            const f32x4v ko = *reinterpret_cast<const f32x4v*>(sKo + own + 32 * dt + c_row(0, i));
                            const f32x4v vo = *reinterpret_cast<const f32x4v*>(sVo + own + 32 * dt + c_row(0, i));
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                xk[i + e] = accZ[dt][i + e] * ko[e];
                                xv[i + e] = accW[dt][i + e] * vo[e];
                            }
                        }
                        const float sum = half_sum_16x2(xk, xv);
                        const bool odd = n & 1;
                        const int d = 32 * dt + c_row(g, half_sum_register());
                        shared_add(odd ? p.acc_v : p.acc_k, (size_t)item.qt * p.acc_tile + base + (size_t)b * D + d, odd ? sum : sum * kLn2,
                                   odd ? fscale_v : fscale_k, p.poison + (size_t)bh * T + b, odd ? kPoisonDV2 : kPoisonDK2);
                        __builtin_amdgcn_sched_barrier(0);  // one tile's products and sums in registers at a time
                    }
                }
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    accZ[dt][i] = 0.f;
                    if constexpr (KEYS) accW[dt][i] = 0.f;
                }
        }
        if (have1) {
            if constexpr (AHEAD) {
                if (fresh2) store_rows(slot2);
                if (have2) complete(buf2);
            } else {
                if (fresh1) {
                    store_rows(slot1);
                    if (!HOLD) large.more(rows_most());
                }
                complete(buf1);
            }
            __syncthreads();
        }
        if constexpr (AHEAD) {
            s = s1;
            dp = dp1;
        }
        buf = buf1;
        slot0 = slot1; slot1 = slot2;
        w0 = w1;
        have = have1;
        if constexpr (AHEAD) {
            w1 = w2;
            fresh1 = fresh2;
            have1 = have2;
        } else {
            slot1 = slot0;
            if (have) {
                have1 = next(w0, w1);
                fresh1 = have1 && w1.m != w0.m;
            }
        }
    }

    auto place = [&](int r, int d) { return (((size_t)bh * T + o0 + r) * deal.max_parts + part) * D + d; };
    if constexpr (KEYS) {
        join_owned<D, NW>(sO, accKo, [&](int r, int d, float v) {
            if (o0 + r < T) p.part_k1[place(r, d)] = v;
        });
        join_owned<D, NW>(sO, accVo, [&](int r, int d, float v) {
            if (o0 + r >= T) return;
            p.part_u[place(r, d)] = v;
            // a non-finite element of dO is one of its column only here; the row is marked whole, as dV2's is
            if (p.rows.maxima && !(fabsf(v) < INFINITY)) atomicOr(p.poison + (size_t)bh * T + o0 + r, kPoisonDU);
        });
    } else if (p.part_q) {
        join_owned<D, NW>(sO, accKo, [&](int r, int d, float v) {
            if (o0 + r < T) p.part_q[place(r, d)] = v;
        });
    } else {
        join_owned<D, NW>(sO, accKo, [&](int r, int d, float v) {
            if (o0 + r < T) p.dq[base + (size_t)(o0 + r) * D + d] = v * p.alpha;
        });
    }
}

template <int D, int NW>
__global__ __launch_bounds__(64 * NW, D == 32 ? 2 : 1) void tdp_f32_split_bwd_kernel(F32SplitBwdParams p) {
    if ((int)blockIdx.x < p.key_blocks) f32_split_bwd_body<D, NW, true>(p, blockIdx.x);
    else f32_split_bwd_body<D, NW, false>(p, blockIdx.x - p.key_blocks);
}

template <int D, int NW>
constexpr size_t f32_split_bwd_smem() {
    constexpr int bufs = D == 64 ? 3 : 2;
    constexpr size_t loop = sizeof(float) * (6 * NW * D + bufs * 64) + bufs * 2 * 3 * sizeof(__bf16) * split_plane<D>(), merge = sizeof(float) * NW * D * 33;
    return sizeof(float) * (NW + 2 * 32 * f32_pitch<D>()) + (loop > merge ? loop : merge);
}

}  // namespace
}  // namespace tritt
