// The fp32 triple-dot kernels over whole problems (tdp_f32_mfma.hip launches them): fp32 operands, products as six bf16 products
// (f32_split.hpp).  Tiles, rounds, parts and masks as in tdp_f32_tiles.hpp.
#pragma once
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
    const Split8 s = split8(x);
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

// Images of two tensors, the second through SiLU when `silu`: one workgroup per 32-row tile (x), slice (y) and tensor (z)
template <int D>
__global__ __launch_bounds__(256) void f32_split_images_kernel(const float* __restrict__ x0, const float* __restrict__ x1,
                                                               __bf16* __restrict__ image0, __bf16* __restrict__ image1, int silu1, int T) {
    const int bh = blockIdx.y, tile = blockIdx.x;
    const float* src = (blockIdx.z ? x1 : x0) + (size_t)bh * T * D;
    __bf16* dst = (blockIdx.z ? image1 : image0) + ((size_t)bh * gridDim.x + tile) * (3 * split_plane<D>());
    const bool silu = blockIdx.z && silu1;
    for (int idx = threadIdx.x; idx < 32 * D / 8; idx += 256) {
        const int r = idx / (D / 8), c = idx % (D / 8), row = tile * 32 + r;
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

// B operand of a score product, k-step ks: columns 16 ks + 8 g .. + 7 of (query or key row n) times the round's row
__device__ __forceinline__ Split8 split_product(const float* own, const float* row, int ks) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
        const f32x4v a = *reinterpret_cast<const f32x4v*>(own + 16 * ks + e), b = *reinterpret_cast<const f32x4v*>(row + 16 * ks + e);
#pragma unroll
        for (int k = 0; k < 4; ++k) x[e + k] = a[k] * b[k];
    }
    return split8(x);
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
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) bq[ks] = split_product(sQ + n * LD + 8 * g, ob + 8 * g, ks);
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

}  // namespace
}  // namespace tritt
