// Triple-dot-product trittention for fp32 tensors on the matrix cores, D = 32, 64 or 128, every mask: fp32 operands and sums,
// every product as six bf16 products of three-way splits (f32_split.hpp; nearer to 64 bits than a chain of fp32 MFMAs, at up
// to 2.4 PFLOP/s / 6 instead of 157 TFLOP/s).  This file: the passes ahead and behind, the deal of tiles to workgroups and the
// launchers; tdp_f32_split.hpp: the forward and the backward kernel; tdp_f32_tiles.hpp: the deal's device side and the fp32
// query tiles of a 16-bit backward.
//
// All tensors here are fp32 [BH, T, D]; U = SiLU(V1) (see capi.hip).
//
// Formulation (the same virtual-query one as the 16-bit kernels).  A workgroup owns 32 consecutive rows (queries; the
// backward has workgroups that own keys as well); its waves take consecutive rows b of (K2, V2) per round, one per wave, and
// sweep the streamed index a in 32-row stages shared through LDS.  The rounds of a tile are dealt out over several workgroups
// by their cost (F32Deal): the forward's parts are joined by f32_merge_kernel and those of dQ, dK1 and dU by f32_finish_kernel;
// dK2 and dV2, sums over tiles, meet in fixed-point accumulators, or are left by each tile of a problem of a few tiles and
// joined like the others (f32_tile_slabs).
// For a fixed row b the scores of the 32 queries against 32 streamed rows are one 32x32 tile
//   S^T[a, q] = sum_d KA[a, d] * (scale * Q[q, d] * KB[b, d])
// The tile leaves the MFMA with lane <-> query and registers <-> streamed rows, which is (but for the order of the streamed
// rows) the B-operand layout of the next product
//   Tv^T[d, q] += sum_a VA^T[d, a] * P^T[a, q]
// so P is never moved between lanes, and every per-query quantity (running maximum, row sum, the merge of a
// finished row b into the output, O^T[d, q] += Tv^T[d, q] * VB[b, d]) is lane-local.
// One loop body serves every mask; only tiles on its edge evaluate it.
#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "kernels.hpp"
#include "mfma.hpp"
#include "tdp_f32_split.hpp"

namespace tritt {
namespace {

// One pass ahead of the backward kernels, 64 rows per workgroup: U = SiLU(V1) (u null: the caller has it), Delta =
// rowsum(dO * O), the accumulators cleared (`planes` times n words), the images of the streamed tensors and, for fixed-point
// accumulators (maxima not null), the partial maxima that fix a slice's scales (F32RowScale; V1's are U's where the caller has
// that) and the poison words cleared.  grid (64-row blocks, BH, 1 + the maxima's tensors + the images): one of them after the
// other in the blocks of z = 0 is 6 us longer, a launch for each 2-5 us.
struct F32PrepParams {
    const float *q, *k1, *v2, *u_in, *v1, *o, *d_o;
    float *u, *delta;
    unsigned* acc;
    int planes;
    size_t n;
    unsigned *maxima, *poison;
    __bf16* images[4];  // Q, dO, K1, U (null: not wanted)
    int T;
};
template <int D>
__global__ __launch_bounds__(256) void f32_prep_kernel(F32PrepParams p) {
    __shared__ unsigned red[4];
    constexpr int kPieces = D / 4;
    const int bh = blockIdx.y, j0 = blockIdx.x * 64, T = p.T;
    const size_t base = (size_t)bh * T * D;
    int z = blockIdx.z;
    if (z && p.maxima && z <= kMaxima) {  // part s of a slice: its 64-row blocks s, s + kScaleParts, ...
        const int t = z - 1;
        const float* src = (t == kMaxDO ? p.d_o : t == kMaxQ ? p.q : t == kMaxK1 ? p.k1 : t == kMaxV2 ? p.v2 : p.v1 ? p.v1 : p.u_in) + base;
        for (int part = blockIdx.x; part < kScaleParts; part += gridDim.x) {
            unsigned m = 0;
            for (int r0 = part * 64; r0 < T; r0 += kScaleParts * 64)
                m = max(m, block_absmax_bits<float>(src + (size_t)r0 * D, (size_t)min(64, T - r0) * kPieces, red));
            if (threadIdx.x == 0) p.maxima[((size_t)t * gridDim.y + bh) * kScaleParts + part] = m;
        }
        return;
    }
    if (z) {
        z -= p.maxima ? kMaxima + 1 : 1;
        const float* src = z == 0 ? p.q : z == 1 ? p.d_o : z == 2 ? p.k1 : p.v1 ? p.v1 : p.u_in;
        __bf16* dst = p.images[z];
        const int tiles = (T + 31) / 32;
        if (dst)
            for (int tile = 2 * blockIdx.x; tile < min(2 * (int)blockIdx.x + 2, tiles); ++tile)
                split_image_tile<D>(src + base, dst + ((size_t)bh * tiles + tile) * (3 * split_plane<D>()), tile * 32, T, z == 3 && p.v1);
        return;
    }
    if (p.maxima && threadIdx.x < 64 && j0 + threadIdx.x < T) p.poison[(size_t)bh * T + j0 + threadIdx.x] = 0;
    for (int idx = threadIdx.x; idx < 64 * kPieces; idx += 256) {  // whole waves: 64 kPieces is a multiple of 256
        const int j = j0 + idx / kPieces;
        const size_t off = base + (size_t)j * D + (idx % kPieces) * 4;
        float dot = 0.f;
        if (j < T) {
            if (p.u) {
                f32x4v x = *reinterpret_cast<const f32x4v*>(p.v1 + off);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = silu_f(x[e]);
                *reinterpret_cast<f32x4v*>(p.u + off) = x;
            }
            const f32x4v x = *reinterpret_cast<const f32x4v*>(p.o + off), y = *reinterpret_cast<const f32x4v*>(p.d_o + off);
            dot = x[0] * y[0] + x[1] * y[1] + (x[2] * y[2] + x[3] * y[3]);
            for (int t = 0; t < p.planes; ++t) *reinterpret_cast<uint4*>(p.acc + t * p.n + off) = make_uint4(0u, 0u, 0u, 0u);
        }
#pragma unroll
        for (int w = kPieces / 2; w > 0; w >>= 1) dot += __shfl_xor(dot, w, 64);
        if (idx % kPieces == 0 && j < T) p.delta[(size_t)bh * T + j] = dot;
    }
}
// The sums -> the gradients (null: not wanted), four elements per thread: dK2 and dV2 from fixed point (`slabs` > 0: from that
// many tiles' fp32 shares, in order); dQ, dK1 and dV1 = dU SiLU'(V1) are the sums of their tile's parts, in fp32 and in order: a
// gradient may lie many powers of two below what the scale of a fixed-point sum is set by.
struct F32FinishParams {
    const long long* acc;
    const unsigned *fields, *poison;
    const float *part_q, *part_k1, *part_u;
    F32Deal deal_q, deal_k;
    TdpMask mask;
    int nw, slabs;
    size_t n;
    int T, D;
    float alpha;
};
template <typename E>
__global__ __launch_bounds__(256) void f32_finish_kernel(F32FinishParams p, const E* __restrict__ v1, E* __restrict__ dq, E* __restrict__ dk1,
                                                         E* __restrict__ dk2, E* __restrict__ dv1, E* __restrict__ dv2) {
    typedef __attribute__((ext_vector_type(4))) E e4;
    for (size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4; i < p.n; i += (size_t)gridDim.x * 1024) {
        const size_t row = i / p.D;
        auto write = [&](E* out, const f32x4v& v) {
            e4 r;
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = (E)v[e];
            *reinterpret_cast<e4*>(out + i) = r;
        };
        auto shared = [&](E* out, int which, unsigned bit) {
            if (!out) return;
            if (p.slabs) {
                const float* src = reinterpret_cast<const float*>(p.acc) + (size_t)which * p.slabs * p.n + i;
                f32x4v sum = *reinterpret_cast<const f32x4v*>(src);
                for (int t = 1; t < p.slabs; ++t) sum += *reinterpret_cast<const f32x4v*>(src + t * p.n);
                write(out, sum);
                return;
            }
            const longlong2* src = reinterpret_cast<const longlong2*>(p.acc + which * p.n + i);
            const longlong2 lo = src[0], hi = src[1];
            const long long v[4] = {lo.x, lo.y, hi.x, hi.y};
            const double inv = fixed_scale_inverse(p.fields[row / p.T * 2 + which]);
            const bool bad = p.poison[row] & bit;
            f32x4v r;
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = bad ? __builtin_nanf("") : (float)((double)v[e] * inv);
            write(out, r);
        };
        shared(dk2, 0, kPoisonDK2);
        shared(dv2, 1, kPoisonDV2);
        const int tile = (int)(row % p.T) / 32, d = (int)(i % p.D);
        auto joined = [&](const float* part, const F32Deal& deal) {
            const float* src = part + row * deal.max_parts * p.D + d;
            const int parts = f32_tile_parts(deal, p.mask, tile, p.T, p.nw);
            f32x4v sum = *reinterpret_cast<const f32x4v*>(src);
#pragma unroll 4
            for (int s = 1; s < parts; ++s) sum += *reinterpret_cast<const f32x4v*>(src + s * p.D);
            return sum;
        };
        if (dq) write(dq, joined(p.part_q, p.deal_q) * p.alpha);
        if (dk1) write(dk1, joined(p.part_k1, p.deal_k) * p.alpha);
        if (dv1) {
            const e4 x = *reinterpret_cast<const e4*>(v1 + i);
            f32x4v v = joined(p.part_u, p.deal_k);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] *= silu_grad_f((float)x[e]);
            if (!p.slabs && (p.poison[row] & kPoisonDU)) v = f32x4v{NAN, NAN, NAN, NAN};
            write(dv1, v);
        }
    }
}

// waves per workgroup
constexpr int kSplitWaves = 4;
constexpr int f32_tile_waves(int D) { return D > 64 ? 8 : 4; }  // launch_f32_bwd_tiles

// Joins the parts of a split forward, four columns per thread.
__global__ __launch_bounds__(256) void f32_merge_kernel(const float* __restrict__ part, float* __restrict__ o,
                                                        float* __restrict__ lse, size_t rows, int T, int D, TdpMask mask,
                                                        F32Deal deal) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x, row = idx / (D / 4);
    const int d = (int)(idx % (D / 4)) * 4;
    if (row >= rows) return;
    const int parts = f32_tile_parts(deal, mask, (int)(row % T) / 32, T, kSplitWaves);
    const float* src = part + row * deal.max_parts * (D + 4);
    // four parts' loads in flight at a time (for a part beyond the last one that one's, not used: zero times an infinite output is NaN)
    float m = kNegBig, l = 0.f;
    f32x4v acc = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < parts; s0 += 4) {
        float ms[4], ls[4];
        f32x4v os[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float* at = src + min(s0 + k, parts - 1) * (D + 4);
            ms[k] = s0 + k < parts ? at[D] : kNegBig;
            ls[k] = at[D + 1];
            os[k] = *reinterpret_cast<const f32x4v*>(at + d);
        }
        const float top = fmaxf(fmaxf(fmaxf(ms[0], ms[1]), fmaxf(ms[2], ms[3])), m), keep = fast_exp2(m - top);
        l *= keep;
        acc *= keep;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float w = fast_exp2(ms[k] - top);
            l += w * ls[k];
            if (s0 + k < parts) acc += os[k] * w;
        }
        m = top;
    }
    *reinterpret_cast<f32x4v*>(o + row * D + d) = acc / l;
    if (d == 0) lse[row] = (m + fast_log2(l)) * kLn2;
}

// How the tiles of a problem are dealt out over workgroups.  `slots`: workgroups the chip holds at a time.  About six parts per
// slot even out a grid whose tiles differ by a factor of hundreds (B=4 H=8 T=512: one workgroup per tile 5.9 ms, a fixed
// count of 4 / 16 per tile 4.1 / 3.9, by cost 3.3); below sixteen steps per slot a part's own cost (prologue, merge: two
// or three steps' worth) asks for fewer, two per slot; a problem smaller than that gets one step per part (B=1 H=2 T=64
// D=32: 27 -> 9 us).  At most sixteen parts per tile: 32 gained nothing and double the scratch of a split forward.
// `share` of the chip: two kinds of tiles in one grid get half of those parts each.
F32Deal f32_deal(const TdpMask& mask, int BH, int T, int nw, int slots, int most, bool keys = false, double share = 1.0) {
    const int nqt = (T + 31) / 32;
    long long total = 0;
    int rounds;
    for (int qt = 0; qt < nqt; ++qt) {
        const int first = qt * 32, last = std::min(T - 1, qt * 32 + 31);
        total += keys ? f32_key_tile_steps(mask, first, last, T, nw, &rounds) : f32_tile_steps(mask, first, last, T, nw, &rounds);
    }
    const double per_slot = (double)total * BH / (slots * share);
    const double target = std::max({per_slot / 6.0, std::min(16.0, per_slot / 2.0), 1.0});
    F32Deal d{(float)(1.0 / target), most, 0, keys};
    int parts = 1;
    for (int qt = 0; qt < nqt; ++qt) parts = std::max(parts, f32_tile_parts(d, mask, qt, T, nw));
    d.max_parts = parts;
    for (int qt = 0; qt < nqt; ++qt) d.items += f32_tile_parts(d, mask, qt, T, nw);
    return d;
}
int f32_most_parts() { return knobs().bwd_splits > 0 ? std::min(knobs().bwd_splits, 16) : 16; }
F32Deal f32_tiles_deal(int BH, int T, int D, const TdpMask& mask) {  // launch_f32_bwd_tiles
    const int nw = f32_tile_waves(D);
    return f32_deal(mask, BH, T, nw, nw == 4 ? 512 : 256, f32_most_parts());
}
F32Deal f32_bwd_deal(int BH, int T, int D, const TdpMask& mask, bool keys) {
    return f32_deal(mask, BH, T, kSplitWaves, D == 32 ? 512 : 256, f32_most_parts(), keys, 0.5);
}

// Problems of less than eight query tiles: every tile has row-gradient accumulators of its own, fp32, where each element gets
// one share (a row belongs to one round, a round to one workgroup), and f32_finish_kernel adds the tiles'.  Nothing then has a
// step or a range of its own: in steps of 2^-36 max |dO| operands of 0.02 left dK1 2.5e-3 off (T = 64, D = 32), shares of fp32
// 4e-7 or less.  At most seven tiles' words, of at most 224 rows each.  Kernel time of a training step, fixed point -> this:
// B=1 H=2 T=64 D=32 50.0 -> 49.1 us, B=1 H=2 T=100 D=64 157.7 -> 160.2 (the last launch adds four tiles' words).
bool f32_tile_slabs(int BH, int T) { return (long long)BH * ((T + 31) / 32) < 8; }

// both launches of the backward over query tiles 0 .. nqt - 1
template <typename E, int D>
hipError_t launch_f32_bwd_tiles(F32BwdParams<E> p, const E* k1, const E* u, const E* k2, const E* v2, void* acc_k2,
                                void* acc_v2, void* acc_k1, void* acc_u, const TdpMask& natural, bool want_q,
                                bool want_k2, bool want_k1, hipStream_t st, const InputsAt& at, bool deal_out) {
    // a workgroup holds all D gradient columns and forms S and dP once (D = 128: dQ's running sum is kept in LDS)
    constexpr int DOUT = D;
    constexpr int NW = f32_tile_waves(D);
    auto kern_dq = tdp_f32_bwd_kernel<E, D, DOUT, true, NW>;
    auto kern_nodq = tdp_f32_bwd_kernel<E, D, DOUT, false, NW>;
    constexpr size_t smem = f32_bwd_smem<D, NW>();
    if (hipError_t e = ensure_dynamic_smem(reinterpret_cast<const void*>(kern_dq), smem); e != hipSuccess) return e;
    if (hipError_t e = ensure_dynamic_smem(reinterpret_cast<const void*>(kern_nodq), smem); e != hipSuccess) return e;
    // The rounds of a tile are dealt out to several workgroups (the launch with dQ: only when dQ's shares have a place).  The list
    // of parts belongs to the mask it was made for, and the second launch exchanges the two key indices.
    const TdpMask exchanged{natural.causal, natural.wb, natural.wa, natural.rab, natural.lab};
    const F32Deal whole{0.f, 1, p.nqt};
    auto deal_for = [&](const TdpMask& m) { return deal_out ? f32_tiles_deal(p.BH, p.T, D, m) : whole; };
    auto grid_of = [&](const F32Deal& d) { return dim3(8 * xcd_slots(p.BH, d.items), D / DOUT); };
    // rows = (K2, V2), streamed = (K1, U): dQ, dK2, dV2
    p.ka = k1; p.va = u; p.kb = k2; p.vb = v2;
    place_inputs(p, at, false);
    p.acc_k = acc_k2; p.acc_v = acc_v2; p.bit_k = kPoisonDK2; p.bit_v = kPoisonDV2;
    p.mask = natural;
    p.deal = want_q && !p.acc_q ? whole : deal_for(natural);
    if (want_q) hipLaunchKernelGGL(kern_dq, grid_of(p.deal), dim3(64 * NW), smem, st, p);
    else if (want_k2) hipLaunchKernelGGL(kern_nodq, grid_of(p.deal), dim3(64 * NW), smem, st, p);
    // rows = (K1, U), streamed = (K2, V2): dK1, dU (the mask with the two key indices exchanged)
    p.ka = k2; p.va = v2; p.kb = k1; p.vb = u;
    place_inputs(p, at, true);
    p.acc_k = acc_k1; p.acc_v = acc_u; p.bit_k = kPoisonDK1; p.bit_v = kPoisonDU;
    p.mask = exchanged;
    p.deal = deal_for(exchanged);
    if (want_k1) hipLaunchKernelGGL(kern_nodq, grid_of(p.deal), dim3(64 * NW), smem, st, p);
    return hipGetLastError();
}

// (a window beyond the sequence is no window; the workspace's query may name any)
TdpMask f32_mask(const GenericTdpArgs& a) {
    auto w = [&](int x) { return std::min(x, a.T); };
    return {a.causal, w(a.k1_window), w(a.k2_window), w(a.kk_left), w(a.kk_right)};
}

// Scratch of a backward: the accumulators of dK2 and dV2, with fixed-point ones the rows' poison words, the slices' partial
// maxima and exponent fields; the parts of dQ, dK1 and dU; the images of Q, dO, K1 and U.  base null: measuring (bytes = the end).
struct F32BwdScratch {
    F32Deal deal_q, deal_k;
    int slabs;
    long long* acc;
    unsigned *poison, *maxima, *fields;
    float *part_q, *part_k1, *part_u;
    __bf16* images;
    size_t image_elems, bytes;
};
template <int D>
F32BwdScratch f32_bwd_scratch(const GenericTdpArgs& a, void* base) {
    const TdpMask mask = f32_mask(a);
    const size_t rows = (size_t)a.BH * a.T, n = rows * D;
    F32BwdScratch s{};
    s.deal_q = f32_bwd_deal(a.BH, a.T, D, mask, false);
    s.deal_k = f32_bwd_deal(a.BH, a.T, D, mask, true);
    s.slabs = f32_tile_slabs(a.BH, a.T) ? (a.T + 31) / 32 : 0;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        char* p = base ? (char*)base + at : nullptr;
        at += (bytes + 255) & ~size_t(255);
        return p;
    };
    // (one or two tiles' own accumulators are smaller than the fixed-point ones: the size stays monotone in T)
    s.acc = (long long*)take(std::max((size_t)16 * n, (size_t)8 * s.slabs * n));
    s.poison = (unsigned*)take(4 * rows);
    s.maxima = (unsigned*)take((size_t)4 * a.BH * kScaleParts * kMaxima);
    s.fields = (unsigned*)take((size_t)8 * a.BH);
    s.part_q = (float*)take(4 * n * s.deal_q.max_parts);
    s.part_k1 = (float*)take(4 * n * s.deal_k.max_parts);
    s.part_u = (float*)take(4 * n * s.deal_k.max_parts);
    s.image_elems = split_image_elems<D>(a.BH, a.T);
    s.images = (__bf16*)take(4 * sizeof(__bf16) * s.image_elems);
    s.bytes = at;
    return s;
}

template <int D>
hipError_t launch_f32_bwd(const F32BwdCall& c, hipStream_t st) {
    const GenericTdpArgs& a = c.a;
    const size_t n = (size_t)a.BH * a.T * D;
    const bool want_q = c.dq != nullptr, want_keys = c.dk2 || c.dv2 || c.dk1 || c.dv1;
    const F32BwdScratch s = f32_bwd_scratch<D>(a, c.scratch);
    // a dQ of one part per tile needs no place of its own where the kernel can write the caller's type
    const bool direct_q = c.elem == 0 && s.deal_q.max_parts == 1;
    F32PrepParams prep{};
    prep.q = a.q; prep.k1 = a.k1; prep.v2 = a.v2; prep.u_in = a.u; prep.v1 = c.v1_f32; prep.o = c.o; prep.d_o = a.d_o;
    prep.u = c.v1_f32 ? c.u_out : nullptr; prep.delta = c.delta;
    prep.acc = reinterpret_cast<unsigned*>(s.acc); prep.planes = s.slabs ? 2 * s.slabs : 4; prep.n = n;
    prep.maxima = s.slabs ? nullptr : s.maxima; prep.poison = s.poison; prep.T = a.T;
    for (int i = 0; i < 4; ++i) prep.images[i] = (i < 2 ? want_keys : want_q) ? s.images + i * s.image_elems : nullptr;
    hipLaunchKernelGGL(f32_prep_kernel<D>, dim3((a.T + 63) / 64, a.BH, 1 + (s.slabs ? 0 : kMaxima) + 4), dim3(256), 0, st, prep);
    F32SplitBwdParams p{};
    p.q = a.q; p.d_o = a.d_o; p.k1 = a.k1; p.u = a.u; p.k2 = a.k2; p.v2 = a.v2;
    p.image_q = prep.images[0]; p.image_do = prep.images[1]; p.image_k1 = prep.images[2]; p.image_u = prep.images[3];
    p.lse = a.lse_in; p.delta = c.delta;
    p.dq = direct_q ? (float*)c.dq : nullptr; p.part_q = direct_q ? nullptr : s.part_q;
    p.part_k1 = s.part_k1; p.part_u = s.part_u;
    p.acc_k = s.acc;
    p.acc_v = s.slabs ? (void*)((float*)s.acc + s.slabs * n) : (void*)(s.acc + n);
    p.acc_tile = s.slabs ? n : 0;
    p.poison = s.poison;
    auto log2_above = [](float x) {  // x <= 2^this
        int e = 128;
        if (std::isfinite(x)) std::frexp(x, &e);
        return e;
    };
    p.rows.maxima = prep.maxima; p.rows.fields = s.fields;
    p.rows.free_v = 127 + 61 - log2_above((float)a.T);
    p.rows.free_k = p.rows.free_v - 1 - log2_above((float)D) - log2_above(a.alpha);
    p.T = a.T; p.BH = a.BH; p.nqt = (a.T + 31) / 32;
    p.alpha = a.alpha;
    p.mask = f32_mask(a);
    p.deal_q = s.deal_q; p.deal_k = s.deal_k;
    p.key_blocks = want_keys ? 8 * xcd_slots(a.BH, s.deal_k.items) : 0;
    const int query_blocks = want_q ? 8 * xcd_slots(a.BH, s.deal_q.items) : 0;
    auto kern = tdp_f32_split_bwd_kernel<D, kSplitWaves>;
    constexpr size_t smem = f32_split_bwd_smem<D, kSplitWaves>();
    if (hipError_t e = ensure_dynamic_smem(reinterpret_cast<const void*>(kern), smem); e != hipSuccess) return e;
    if (p.key_blocks + query_blocks)
        hipLaunchKernelGGL(kern, dim3(p.key_blocks + query_blocks), dim3(64 * kSplitWaves), smem, st, p);
    F32FinishParams f{};
    f.acc = s.acc; f.fields = s.fields; f.poison = s.poison; f.part_q = s.part_q; f.part_k1 = s.part_k1; f.part_u = s.part_u;
    f.deal_q = s.deal_q; f.deal_k = s.deal_k; f.mask = p.mask; f.nw = kSplitWaves; f.slabs = s.slabs;
    f.n = n; f.T = a.T; f.D = D; f.alpha = a.alpha;
    const dim3 grid((unsigned)std::min<size_t>((n / 4 + 255) / 256, 8192));
    auto finish = [&](auto zero) {
        using E = decltype(zero);
        hipLaunchKernelGGL(f32_finish_kernel<E>, grid, dim3(256), 0, st, f, (const E*)c.v1, direct_q ? nullptr : (E*)c.dq,
                           (E*)c.dk1, (E*)c.dk2, (E*)c.dv1, (E*)c.dv2);
    };
    if (c.elem == 0) finish(0.f);
    else if (c.elem == 1) finish((__bf16)0.f);
    else finish((_Float16)0.f);
    return hipGetLastError();
}

int f32_fwd_slots(int D) { return D > 64 ? 256 : 512; }
F32Deal f32_fwd_deal(const GenericTdpArgs& a, int most) {
    return f32_deal(f32_mask(a), a.BH, a.T, kSplitWaves, f32_fwd_slots(a.D), knobs().fwd_splits > 0 ? std::min(knobs().fwd_splits, most) : most);
}

template <int D>
hipError_t launch_f32_fwd(const GenericTdpArgs& a, hipStream_t st) {
    F32FwdParams p{};
    p.q = a.q; p.ka = a.k1; p.kb = a.k2; p.va = a.u; p.vb = a.v2;
    p.o = a.o; p.lse = a.lse;
    p.silu_va = a.u_is_v1;
    p.T = a.T; p.BH = a.BH; p.nqt = (a.T + 31) / 32;
    p.scale_log2 = a.alpha * kLog2e;
    p.mask = f32_mask(a);
    p.deal = a.part ? f32_fwd_deal(a, a.fwd_parts) : F32Deal{0.f, 1, p.nqt};
    p.part = a.part;
    constexpr int NW = kSplitWaves;
    if (a.images) {
        __bf16 *ka = (__bf16*)a.images, *va = ka + split_image_elems<D>(a.BH, a.T);
        hipLaunchKernelGGL(f32_split_images_kernel<D>, dim3(p.nqt, a.BH, 2), dim3(256), 0, st, a.k1, a.u, ka, va, a.u_is_v1, a.T);
        p.image_ka = ka; p.image_va = va;
    }
    auto kern = a.images ? tdp_f32_split_fwd_kernel<D, NW, true> : tdp_f32_split_fwd_kernel<D, NW, false>;
    constexpr size_t smem = f32_split_fwd_smem<D, NW>();
    if (hipError_t e = ensure_dynamic_smem(reinterpret_cast<const void*>(kern), smem); e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(8 * xcd_slots(a.BH, p.deal.items)), dim3(64 * NW), smem, st, p);
    if (p.deal.max_parts > 1) {
        const size_t rows = (size_t)a.BH * a.T;
        hipLaunchKernelGGL(f32_merge_kernel, dim3((unsigned)((rows * (D / 4) + 255) / 256)), dim3(256), 0, st, a.part, a.o,
                           a.lse, rows, a.T, D, p.mask, p.deal);
    }
    return hipGetLastError();
}

}  // namespace

// A short problem's streamed tensors are split, and V1 goes through SiLU, as their stages are put in LDS: 0.4 / 0.7 / 1.3 us a step at
// D = 32 / 64 / 128, every time a tile streams a row, where the launch that makes images takes 2-2.5 us.  `walk`: steps of the longest
// workgroup, or the average of a place on the chip where that is more.  Forward, split as staged against images, D = 32 / 64 / 128:
// B=1 H=2 T=64 (walk 2) 12.7 15.7 24.0 against 14.8 16.8 24.2 us, B=4 H=8 T=64 (2.5, D = 128: 5) 18.5 29.5 66.5 against 19.3 29.1 62.2,
// B=1 H=2 T=1000 windows 16 (3, 6) 22.0 33.9 79.1 against 23.5 35.0 76.8, B=1 H=2 T=128 (8) 22.9 30.8 52.8 against 22.1 27.3 43.7,
// T=256 (32) 59.8 87.5 161 against 49.0 65.3 114; T=72 (6) 19.7 26.2 43.3 against 19.8 24.1 37.3.
bool f32_fwd_takes_v1(const GenericTdpArgs& a) {
    const F32Deal d = f32_fwd_deal(a, std::max(1, a.fwd_parts));
    const TdpMask mask = f32_mask(a);
    double total = 0, walk = 0;
    for (int qt = 0; qt * 32 < a.T; ++qt) {
        int rounds;
        const int steps = f32_tile_steps(mask, qt * 32, std::min(a.T - 1, qt * 32 + 31), a.T, kSplitWaves, &rounds);
        total += steps;
        const int parts = f32_tile_parts(d, mask, qt, a.T, kSplitWaves);
        walk = std::max(walk, (double)((rounds + parts - 1) / parts) * steps / rounds);
    }
    walk = std::max(walk, total * a.BH / f32_fwd_slots(a.D));
    return walk * (a.D + 32) <= 330;
}
int f32_fwd_parts(const GenericTdpArgs& a) { return f32_fwd_deal(a, 16).max_parts; }
size_t f32_fwd_image_bytes(const GenericTdpArgs& a) {
    return 2 * sizeof(__bf16) * (a.D == 32 ? split_image_elems<32>(a.BH, a.T) : a.D == 64 ? split_image_elems<64>(a.BH, a.T) : split_image_elems<128>(a.BH, a.T));
}
size_t f32_fwd_part_floats(int D) { return D + 4; }

bool f32_mfma_tdp_supported(int D) { return D == 32 || D == 64 || D == 128; }

// The first query tiles of a 16-bit backward, in fp32 (see the comment above tdp_f32_bwd_kernel).
template <typename E, int D>
static hipError_t launch_stats(const FirstTileArgs& a, hipStream_t st) {
    F32StatsParams<E> p{};
    p.q = (const E*)a.q; p.ka = (const E*)a.k1; p.kb = (const E*)a.k2; p.va = (const E*)a.u; p.vb = (const E*)a.v2;
    place_inputs(p, inputs_of(a), false);
    p.lse = a.lse_f32; p.d_o = (const E*)a.d_o; p.delta = a.delta_f32;
    p.split_rounds = 0; p.zero_ptr = nullptr; p.zero_words = 0;
    p.T = a.T; p.BH = a.BH; p.nqt = a.tiles;
    p.scale_log2 = a.alpha * kLog2e;
    p.mask = TdpMask{a.causal, a.k1_window, a.k2_window, a.kk_left, a.kk_right};
    auto kern = tdp_f32_stats_kernel<E, D, kF32Waves>;
    constexpr size_t smem = f32_stats_smem<D, kF32Waves>();
    if (hipError_t e = ensure_dynamic_smem(reinterpret_cast<const void*>(kern), smem); e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(8 * xcd_slots(a.BH, p.nqt)), dim3(512), smem, st, p);
    return hipGetLastError();
}

// Query tile 0 alone, its rounds dealt out to workgroups (the launcher of the backward has run its STATS pass).
template <typename E, int D>
static hipError_t launch_tile0_split(const FirstTileArgs& a, hipStream_t st) {
    constexpr int DOUT = D > 64 ? 64 : D;
    F32BwdParams<E> r0, r1;
    int roles;
    const int rounds = tile0_rounds(a);
    tile0_backward<E, D>(a, r0, r1, roles);
    auto kern = tdp_f32_tile0_kernel<E, D, DOUT>;
    constexpr size_t smem = f32_bwd_smem<D>();
    if (hipError_t e = ensure_dynamic_smem(reinterpret_cast<const void*>(kern), smem); e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(8 * xcd_slots(a.BH, 1), D / DOUT, 2 * rounds), dim3(512), smem, st, r0, r1, roles);
    return hipGetLastError();
}

template <typename E>
static hipError_t first_tile_typed(const FirstTileArgs& a, hipStream_t st) {
    if (a.tiles == 1) {
        return a.D == 32 ? launch_tile0_split<E, 32>(a, st) : a.D == 64 ? launch_tile0_split<E, 64>(a, st)
             : a.D == 128 ? launch_tile0_split<E, 128>(a, st) : hipErrorInvalidValue;
    }
    // the rows' log-sum-exp and Delta once more, in fp32 from the same tensors: the saved LSE carries the 16-bit
    // rounding of the forward's scores and Delta that of the stored output, and nearly one-hot rows show both
    hipError_t es = a.D == 32 ? launch_stats<E, 32>(a, st) : a.D == 64 ? launch_stats<E, 64>(a, st)
                  : a.D == 128 ? launch_stats<E, 128>(a, st) : hipErrorInvalidValue;
    if (es != hipSuccess) return es;
    F32BwdParams<E> p{};
    p.q = (const E*)a.q; p.d_o = (const E*)a.d_o; p.lse = a.lse_f32; p.delta = a.delta_f32;
    p.dq = (E*)a.dq; p.acc_q = a.acc_q; p.acc_q_rows = 0; p.stats_part = nullptr; p.split_rounds = 0;
    p.scale_parts = a.scale_parts; p.poison = a.poison; p.scale_bias = a.scale_bias;
    p.T = a.T; p.BH = a.BH; p.nqt = a.tiles;
    p.alpha = a.alpha;
    const TdpMask natural{a.causal, a.k1_window, a.k2_window, a.kk_left, a.kk_right};
    const E *k1 = (const E*)a.k1, *u = (const E*)a.u, *k2 = (const E*)a.k2, *v2 = (const E*)a.v2;
    const bool wq = a.want_q, wk2 = a.want_k2, wk1 = a.want_k1;
    if (a.D == 32)
        return launch_f32_bwd_tiles<E, 32>(p, k1, u, k2, v2, a.acc_k2, a.acc_v2, a.acc_k1, a.acc_u, natural, wq, wk2, wk1, st, inputs_of(a), a.deal_out);
    if (a.D == 64)
        return launch_f32_bwd_tiles<E, 64>(p, k1, u, k2, v2, a.acc_k2, a.acc_v2, a.acc_k1, a.acc_u, natural, wq, wk2, wk1, st, inputs_of(a), a.deal_out);
    if (a.D == 128)
        return launch_f32_bwd_tiles<E, 128>(p, k1, u, k2, v2, a.acc_k2, a.acc_v2, a.acc_k1, a.acc_u, natural, wq, wk2, wk1, st, inputs_of(a), a.deal_out);
    return hipErrorInvalidValue;
}
hipError_t f32_mfma_tdp_bwd_first_tile(const FirstTileArgs& a, hipStream_t st) {
    return a.is_bf16 ? first_tile_typed<__bf16>(a, st) : first_tile_typed<_Float16>(a, st);
}

hipError_t f32_mfma_tdp_fwd(const GenericTdpArgs& a, hipStream_t st) {
    if (a.D == 32) return launch_f32_fwd<32>(a, st);
    if (a.D == 64) return launch_f32_fwd<64>(a, st);
    if (a.D == 128) return launch_f32_fwd<128>(a, st);
    return hipErrorInvalidValue;
}

size_t f32_mfma_tdp_bwd_scratch_bytes(const GenericTdpArgs& a) {
    return a.D == 32 ? f32_bwd_scratch<32>(a, nullptr).bytes : a.D == 64 ? f32_bwd_scratch<64>(a, nullptr).bytes : f32_bwd_scratch<128>(a, nullptr).bytes;
}

hipError_t f32_mfma_tdp_bwd(const F32BwdCall& c, hipStream_t st) {
    if (c.a.D == 32) return launch_f32_bwd<32>(c, st);
    if (c.a.D == 64) return launch_f32_bwd<64>(c, st);
    if (c.a.D == 128) return launch_f32_bwd<128>(c, st);
    return hipErrorInvalidValue;
}

}  // namespace tritt
