// Dot-product-sum trittention for fp32 tensors on the matrix cores, D = 32 or 64: fp32 operands and sums, every product as six
// bf16 products of three-way splits (f32_split.hpp).
//
// The same two chained attention passes as dps_kernels.hip (inner: lse1, R = softmax_s(alpha K1_s.K2_t) @ U;
// outer: softmax_t(alpha Q_q.K2_t + lse1[t]) @ (R * V2); backward = the two attention backwards chained through
// dR and dlse1): "attention with a per-key bias" forward, backward by owner rows and backward by owner columns, the
// last two in one launch.
//
// Tiling.  A workgroup owns 32 rows (one per MFMA column = lane % 32) in all of its waves; the 32-row tiles of the other
// operand are dealt out to the waves in turn, each wave sums its own share and the shares are joined through LDS at the
// end: a call of a few hundred owner tiles waits for the serial chain of steps of one wave.  Streamed operands come from L2
// straight into registers as floats (16 KB per step and wave), without LDS and without a barrier inside the loop, and are split
// there; a register set is loaded again as soon as the product that reads it has been issued.
//
// What bounds it: vector issue.  A SIMD issues one vector or matrix instruction per five cycles or so, and a step has 11 of the
// former for one MFMA of 32 cycles (a split takes 11 per pair of floats; the streamed rows are split once as rows and once as
// columns).  Placing the splits between the MFMAs by hand or wave priorities around them changed nothing.  fp32 MFMAs -> this, training
// step: B=2 H=8 T=1000 D=64 k_diff 128 192 -> 150 us, B=4 H=8 T=1024 D=64 424 -> 327, B=4 H=16 T=2048 D=64 2708 -> 2356, B=4 H=8 T=1024
// D=32 229 -> 183; gradients against 64 bits at the first 5.4-6.1e-7 -> 3.7-4.8e-7.
//
// A 32x32 score tile S^T[a, r] = Ka[a] . Xr[r] takes the streamed row key_of_row(n) in A row n, so that it leaves the MFMAs with
// lane <-> owner row and registers <-> streamed rows key_of(g, i): registers 8 h .. + 7 are the k-slots of rows 16 h .. of the
// output products
//   O^T[d, r] += sum_a V^T[d, a] P^T[a, r]                            (A: loads along a row, B = the P registers)
// so P never moves between lanes and every per-owner quantity (running maximum, sums, LSE, Delta) is lane-local.
// MFMA row n of output tile dt is column d = (D / 32) n + dt, so that a lane's loads are as wide as D allows.
// One owner per output element: no atomics, bitwise reproducible.
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "f32_split.hpp"
#include "mfma.hpp"

namespace tritt {
namespace {

__device__ __forceinline__ void pin_order() { __builtin_amdgcn_sched_barrier(0); }

constexpr int kWaves = 4;  // per workgroup; every wave walks each kWaves-th tile of the workgroup's range

// valid pair (owner-like row r attends key-like row a)
__device__ __forceinline__ bool pair_valid(int causal, int k_diff, int r, int a) {
    return !causal || ((a <= r) & (r - a <= k_diff));
}

// Rows row0 .. row0 + 31 of a head's row-major [T][D] operand (row0 is uniform).  A buffer resource of the rows that
// exist: rows past T read as zeros, the loads share their lane offsets, and no 64-bit address is kept per lane.  Every
// offset stands in the lane offset or the instruction: the scalar offset has no part in the range check, so a row reached
// through it would be read from whatever lies behind the tensor, and a NaN there outlives its zero weight.
template <int D>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rows(const float* src, int row0, int T) {
    row0 = __builtin_amdgcn_readfirstlane(row0);
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src) + (size_t)row0 * D, 0, min(32, T - row0) * D * 4, 0x00020000);
}
// operand of a score product: lane (n, g) holds columns 16 ks + 8 g .. + 7 of row `row`, which is n for the owner's rows (B) and
// key_of_row(n) for the streamed ones (A)
template <int D>
__device__ __forceinline__ void load_rows(float (&reg)[D / 2], const float* src, int row0, int T, int row, int g) {
    const __amdgpu_buffer_rsrc_t rows = tile_rows<D>(src, row0, T);
#pragma unroll
    for (int j = 0; j < D / 8; ++j) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rows, (row * D + 8 * g) * 4 + 64 * (j / 2) + 16 * (j % 2), 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) reg[4 * j + e] = __uint_as_float(v[e]);
    }
}
// A operand of an output product: lane n holds columns DT n .. DT n + DT - 1 of rows key_of(g, 0 .. 15)
template <int D>
__device__ __forceinline__ void load_cols(float (&reg)[D / 2], const float* src, int row0, int T, int n, int g) {
    const __amdgpu_buffer_rsrc_t rows = tile_rows<D>(src, row0, T);
    // rows 0 .. 15 and 16 .. 31; opaque, so that the rows of a half are one register plus the instruction's offset
    int lower = (8 * g * D + D / 32 * n) * 4, upper = lower + 16 * D * 4;
    asm volatile("" : "+v"(lower), "+v"(upper));
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int at = i < 8 ? lower : upper, row = i % 8 * D * 4;
        if constexpr (D == 64) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(rows, at + row, 0, 0);
            reg[2 * i] = __uint_as_float(v[0]);
            reg[2 * i + 1] = __uint_as_float(v[1]);
        } else {
            reg[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rows, at + row, 0, 0));
        }
    }
}
// one value per streamed row, lane n <-> row row0 + n (0 past T)
__device__ __forceinline__ float load_vec(const float* src, int row0, int T, int n) {
    const __amdgpu_buffer_rsrc_t rows = tile_rows<1>(src, row0, T);
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rows, 4 * n, 0, 0));
}
// ANY: the values may be infinite.  Testing every value of a step for that would cost a tenth of its vector instructions, so a wave
// forms its share with split8, whose third plane is NaN for such a value, and forms it again if a NaN came out of it
// (B=2 H=8 T=300 D=64 forward 23.6 -> 24.0, backward 48.3 -> 48.8 us, B=4 H=8 T=512 k_diff 100 34.2 -> 33.1 and 89.5 -> 89.7; the branch
// taken for unlikely: D = 32 backward of T=300 33.9 -> 33.2).
template <bool ANY>
__device__ __forceinline__ Split8 split_at(const float* x) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = x[e];
    return split_value<ANY>(v);
}
template <int DT>
__device__ __forceinline__ bool any_nan(const f32x16 (&acc)[DT]) {
    float sum[4] = {0.f, 0.f, 0.f, 0.f};  // (infinities that cancel are taken for one: the share is formed again for nothing)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) sum[i % 4] += acc[dt][i];
    const float all = sum[0] + sum[1] + (sum[2] + sum[3]);
    return __any(all != all);
}
// S^T of a tile; own(ks): the owner's operand of k-step ks.  The small products of all k-steps come first, and the split of a
// k-step's streamed operand stands beside the products of the one before.
template <int D, bool ANY, typename F>
__device__ __forceinline__ f32x16 score_tile(const float (&rows)[D / 2], const F& own) {
    constexpr int KS = D / 16;
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    Split8 a = split_at<ANY>(rows);
    bf16x8 h[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        Split8 next = a;
        if (ks + 1 < KS) next = split_at<ANY>(rows + 8 * (ks + 1 < KS ? ks + 1 : 0));
        s = small_products(a, own(ks), s);
        h[ks] = a.h;
        a = next;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) s = large_product(h[ks], own(ks).h, s);
    return s;
}
// acc^T[d, owner] += sum over the 32 streamed rows of cols[row, d] * w[row, owner]   (w in score-tile layout)
template <int D, bool ANY>
__device__ __forceinline__ void output_tile(f32x16 (&acc)[D / 32], const float (&cols)[D / 2], const f32x16& w) {
    constexpr int DT = D / 32;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = w[8 * half + e];
        const Split8 b = split_value<ANY>(x);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = cols[(8 * half + e) * DT + dt];
            acc[dt] = products_of_step(split_value<ANY>(v), b, acc[dt]);
        }
    }
}
template <int D>
__device__ __forceinline__ void clear(f32x16 (&acc)[D / 32]) {
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;
}

// The waves' shares of a 32 x D result, joined in wave order.
template <int D>
struct Shares {
    static constexpr int LD = D + 4, kPieces = 32 * D / 4;  // 16-byte pieces of the result: thread t takes t, t + 256, ...
    alignas(16) float part[kWaves][32 * LD];
    float row[kWaves][32], row2[kWaves][32];  // per owner row and wave
    alignas(16) float vec[kWaves][2][32];                 // one value per streamed row of a wave's step, on its way into the registers
    // the backward's owner rows, split: the scaled X or K, and G or V.  Rows of 16 (D / 8 + 1) bytes: a wave's 16-byte reads of 32
    // rows fall on distinct bank groups
    static constexpr int kOwnLD = D + 8;
    alignas(16) __bf16 own[2][3][32 * kOwnLD];
    __device__ __forceinline__ Split8 own_operand(int which, int ks, int n, int g) const {
        const int at = n * kOwnLD + 16 * ks + 8 * g;
        return {*reinterpret_cast<const bf16x8*>(own[which][0] + at), *reinterpret_cast<const bf16x8*>(own[which][1] + at),
                *reinterpret_cast<const bf16x8*>(own[which][2] + at)};
    }

    // lane n's values of the wave's 32 streamed rows, in score-tile order (registers 4 i4 .. + 3: rows key_of(g, 4 i4) .. + 3).  Only the wave
    // itself writes and reads its slots and its LDS accesses stay in order.
    __device__ __forceinline__ void vec_put(int which, float v, int wave, int n) {
        vec[wave][which][n] = v;
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ float4 vec_get(int which, int wave, int g, int i4) const {
        return *reinterpret_cast<const float4*>(&vec[wave][which][key_of(0, 4 * i4) + 8 * g]);
    }
    // this wave's registers, scaled per owner row
    __device__ __forceinline__ void put(const f32x16 (&acc)[D / 32], float f, int wave, int n, int g) {
        float* mine = part[wave] + n * LD;
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            const int i = 4 * i4;
            if constexpr (D == 64) {  // registers i .. i + 3 of both tiles are eight consecutive columns
                float* p = mine + 16 * i4 + 8 * g;
                *reinterpret_cast<float4*>(p) = make_float4(acc[0][i] * f, acc[1][i] * f, acc[0][i + 1] * f, acc[1][i + 1] * f);
                *reinterpret_cast<float4*>(p + 4) =
                    make_float4(acc[0][i + 2] * f, acc[1][i + 2] * f, acc[0][i + 3] * f, acc[1][i + 3] * f);
            } else {
                *reinterpret_cast<float4*>(mine + 8 * i4 + 4 * g) =
                    make_float4(acc[0][i] * f, acc[0][i + 1] * f, acc[0][i + 2] * f, acc[0][i + 3] * f);
            }
        }
    }
    __device__ __forceinline__ float4 sum(int piece) const {
        const int at = piece / (D / 4) * LD + piece % (D / 4) * 4;
        float4 o = *reinterpret_cast<const float4*>(part[0] + at);
#pragma unroll
        for (int w = 1; w < kWaves; ++w) {
            const float4 e = *reinterpret_cast<const float4*>(part[w] + at);
            o.x += e.x; o.y += e.y; o.z += e.z; o.w += e.w;
        }
        return o;
    }
};

// Attention forward with an optional per-key bias (log2 units):
//   out[r] = softmax_a(scale X[r].K[a] + bias[a]) @ V ;  lse_out[r] = lse_scale * log2-sum-exp2
//   out_mul[r] = out[r] * mul[r]   (when mul != nullptr; out may then be null)
struct FwdP {
    const float *X, *K, *V, *bias, *mul;
    float *out, *out_mul, *lse_out;
    float lse_scale, scale_log2;
    int BH, T, causal, k_diff;
};
template <int D>
__global__ __launch_bounds__(64 * kWaves, 2) void attn_fwd_f32m_kernel(FwdP p) {
    constexpr int DT = D / 32, KS = D / 16;
    __shared__ Shares<D> sh;
    const int T = p.T, ntiles = (T + 31) / 32;
    int bh, order;
    if (!xcd_tile(p.BH, ntiles, blockIdx.x >> 3, blockIdx.x & 7, bh, order)) return;
    const size_t base = (size_t)bh * T * D, vbase = (size_t)bh * T;
    const float *X = p.X + base, *K = p.K + base, *V = p.V + base;
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // heavy first: under a causal mask the last owner tiles stream the most rows.  A grid that the CUs take whole, two workgroups
    // each, goes in the other direction from the middle on, so that a heavy tile shares its CU with a light one
    const bool whole = p.BH * ntiles <= 512 && order >= (ntiles + 1) / 2;
    const int r0 = (!p.causal ? order : whole ? order - (ntiles + 1) / 2 : ntiles - 1 - order) * 32, r = r0 + n;
    const int a_lo = p.causal ? max(0, r0 - p.k_diff) & ~31 : 0, a_hi = p.causal ? min(T - 1, r0 + 31) : T - 1;

    f32x16 acc[DT];
    float m, l;
    auto share = [&](auto any) {  // this wave's
        constexpr bool ANY = decltype(any)::value;
        clear<D>(acc);
        m = -INFINITY;
        l = 0.f;
        int a0 = a_lo + 32 * wave;
        if (a0 <= a_hi) {
            float bias = p.bias ? load_vec(p.bias + vbase, a0, T, n) : 0.f;
            float x[D / 2], rows[D / 2], cols[D / 2];
            load_rows<D>(x, X, r0, T, n, g);
            load_rows<D>(rows, K, a0, T, key_of_row(n), g);
            load_cols<D>(cols, V, a0, T, n, g);
            Split8 own[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = x[8 * ks + e] * p.scale_log2;
                own[ks] = split_value<ANY>(v);
            }
            for (; a0 <= a_hi; a0 += 32 * kWaves) {
                const int next = min(a0 + 32 * kWaves, a_hi & ~31);  // (past the end: in bounds, not used)
                if (p.bias) sh.vec_put(0, bias, wave, n);
                f32x16 s = score_tile<D, ANY>(rows, [&](int ks) -> const Split8& { return own[ks]; });
                pin_order();
                load_rows<D>(rows, K, next, T, key_of_row(n), g);
                if (p.bias) bias = load_vec(p.bias + vbase, next, T, n);
                pin_order();
                if (p.bias) {
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        const float4 b = sh.vec_get(0, wave, g, i4);
                        s[4 * i4] += b.x; s[4 * i4 + 1] += b.y; s[4 * i4 + 2] += b.z; s[4 * i4 + 3] += b.w;
                    }
                }
                if (a0 + 32 > T || (p.causal && (a0 + 31 > r0 || r0 + 31 - a0 > p.k_diff))) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int a = a0 + key_of(g, i);
                        s[i] = ((a < T) & pair_valid(p.causal, p.k_diff, r, a)) ? s[i] : -INFINITY;
                    }
                }
                float mx = s[0];
#pragma unroll
                for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
                mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
                const float m_new = fmaxf(m, mx);
                const float f = m_new == -INFINITY ? 1.f : fast_exp2(m - m_new);  // nothing seen yet: keep the zeros
                float ps = 0.f;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    s[i] = s[i] == -INFINITY ? 0.f : fast_exp2(s[i] - m_new);
                    ps += s[i];
                }
                ps += __shfl_xor(ps, 32, 64);
                l = l * f + ps;
                m = m_new;
                if (__any(f != 1.f)) {
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[dt][i] *= f;
                }
                output_tile<D, ANY>(acc, cols, s);
                pin_order();
                load_cols<D>(cols, V, next, T, n, g);
                pin_order();
            }
        }
    };
    share(std::false_type{});
    if (__builtin_expect(any_nan(acc), 0)) share(std::true_type{});
    if (g == 0) sh.row[wave][n] = m;
    __syncthreads();
    float M = sh.row[0][n];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) M = fmaxf(M, sh.row[w][n]);
    const float f = m == -INFINITY ? 0.f : fast_exp2(m - M);  // a share without a valid pair is zeros
    sh.put(acc, f, wave, n, g);
    if (g == 0) sh.row2[wave][n] = l * f;
    __syncthreads();
#pragma unroll
    for (int piece = tid; piece < Shares<D>::kPieces; piece += 64 * kWaves) {
        const int row = piece / (D / 4), c = piece % (D / 4) * 4;
        float L = sh.row2[0][row], Mr = sh.row[0][row];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) {
            L += sh.row2[w][row];
            Mr = fmaxf(Mr, sh.row[w][row]);
        }
        if (r0 + row < T) {
            const float inv = 1.0f / L;
            float4 o = sh.sum(piece);
            o.x *= inv; o.y *= inv; o.z *= inv; o.w *= inv;
            const size_t off = base + (size_t)(r0 + row) * D + c;
            if (p.out) *reinterpret_cast<float4*>(p.out + off) = o;
            if (p.mul) {
                const float4 mm = *reinterpret_cast<const float4*>(p.mul + off);
                *reinterpret_cast<float4*>(p.out_mul + off) = make_float4(o.x * mm.x, o.y * mm.y, o.z * mm.z, o.w * mm.w);
            }
            if (c == 0) p.lse_out[vbase + r0 + row] = (Mr + fast_log2(L)) * p.lse_scale;
        }
    }
}

// Attention backward.  P = exp2(scale X[r].K[a] + bias[a] - lse2[r]);  dS = P (G[r].V[a] - delta[r]).
//   owner = query-like row r:  dX[r] = alpha * sum_a dS K[a]  (+ addend[r])
//   owner = key-like row a:    dK[a] = alpha * sum_r dS X[r];  dV[a] = sum_r P G[r];  dbias[a] = sum_r dS
// Both directions are one launch (neither reads what the other writes); odd places of the grid's order take rows.
// What becomes of dV is the caller's choice:
//   mid != nullptr  the outer pass: dV is dW, the gradient of W = R * V2:  mid_out = dW * R,  dR = dW * V2 and
//                   delta1 = rowsum(dR * R) - dbias
//   v1 != nullptr   the inner pass of fp32 tensors: dV = the gradient of SiLU(V1), times SiLU'(V1)
struct BwdP {
    const float *X, *G, *K, *V, *bias, *lse, *delta, *addend;
    float *dX, *dK, *dV;
    const float *mid_r, *mid_v2, *v1;
    float *dR, *delta1;
    float lse_to_log2, alpha;
    int BH, T, causal, k_diff;
};

// In the backward the owner's two operands are read from LDS in every step, by all waves: in registers beside the accumulators,
// two operand sets and the score tiles they do not fit.
template <int D>
__device__ __forceinline__ void own_put(Shares<D>& sh, const float* src0, const float* src1, int row0, int T, float scale0, int tid) {
    for (int piece = tid; piece < 32 * D / 8; piece += 64 * kWaves) {
        const int row = piece / (D / 8), c = piece % (D / 8) * 8;
        const size_t at = (size_t)min(row0 + row, T - 1) * D + c;
        float v[2][8];  // (both loaded ahead of the first split, which branches)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[0][e] = src0[at + e] * scale0;
            v[1][e] = src1[at + e];
        }
#pragma unroll
        for (int which = 0; which < 2; ++which) {
            const Split8 x = split8_any(v[which]);
            *reinterpret_cast<bf16x8*>(sh.own[which][0] + row * Shares<D>::kOwnLD + c) = x.h;
            *reinterpret_cast<bf16x8*>(sh.own[which][1] + row * Shares<D>::kOwnLD + c) = x.m;
            *reinterpret_cast<bf16x8*>(sh.own[which][2] + row * Shares<D>::kOwnLD + c) = x.l;
        }
    }
}
template <int D, bool ANY>
__device__ __forceinline__ f32x16 score_tile(const float (&rows)[D / 2], const Shares<D>& sh, int which, int n, int g) {
    asm volatile("" ::: "memory");  // (the reads stay inside the caller's loop)
    return score_tile<D, ANY>(rows, [&](int ks) { return sh.own_operand(which, ks, n, g); });
}

template <int D>
__device__ __forceinline__ void bwd_rows(const BwdP& p, Shares<D>& sh, int bh, int tile, int tid, int wave, int n, int g) {
    constexpr int DT = D / 32;
    const int T = p.T;
    const size_t base = (size_t)bh * T * D, vbase = (size_t)bh * T;
    const float *X = p.X + base, *G = p.G + base, *K = p.K + base, *V = p.V + base;
    const int r0 = tile * 32, r = r0 + n, rc = min(r, T - 1);
    const int a_lo = p.causal ? max(0, r0 - p.k_diff) & ~31 : 0, a_hi = p.causal ? min(T - 1, r0 + 31) : T - 1;
    const float scale_log2 = p.alpha * kLog2e;
    f32x16 acc[DT];
    own_put<D>(sh, X, G, r0, T, scale_log2, tid);
    __syncthreads();
    auto share = [&](auto any) {
        constexpr bool ANY = decltype(any)::value;
        clear<D>(acc);
        int a0 = a_lo + 32 * wave;
        if (a0 <= a_hi) {
            float bias = p.bias ? load_vec(p.bias + vbase, a0, T, n) : 0.f;
            const int nk = key_of_row(n);
            float ra[D / 2], rb[D / 2];
            load_rows<D>(ra, K, a0, T, nk, g);
            load_rows<D>(rb, V, a0, T, nk, g);
            const float lse2 = p.lse[vbase + rc] * p.lse_to_log2, dl = p.delta[vbase + rc];
            // two operand sets in turn: the K rows of the next step take the set the V rows are in now
            auto step = [&](float (&A)[D / 2], float (&B)[D / 2]) {
                const int next = min(a0 + 32 * kWaves, a_hi & ~31);
                if (p.bias) sh.vec_put(0, bias, wave, n);
                f32x16 s = score_tile<D, ANY>(A, sh, 0, n, g);
                pin_order();
                load_cols<D>(A, K, a0, T, n, g);
                if (p.bias) bias = load_vec(p.bias + vbase, next, T, n);
                pin_order();
                const f32x16 dp = score_tile<D, ANY>(B, sh, 1, n, g);
                pin_order();
                load_rows<D>(B, K, next, T, nk, g);
                pin_order();
                if (p.bias) {
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        const float4 b = sh.vec_get(0, wave, g, i4);
                        s[4 * i4] += b.x; s[4 * i4 + 1] += b.y; s[4 * i4 + 2] += b.z; s[4 * i4 + 3] += b.w;
                    }
                }
                const bool edge = a0 + 32 > T || (p.causal && (a0 + 31 > r0 || r0 + 31 - a0 > p.k_diff));
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = fast_exp2(s[i] - lse2) * (dp[i] - dl);
                if (edge) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int a = a0 + key_of(g, i);
                        s[i] = ((a < T) & pair_valid(p.causal, p.k_diff, r, a)) ? s[i] : 0.f;
                    }
                }
                output_tile<D, ANY>(acc, A, s);
                pin_order();
                load_rows<D>(A, V, next, T, nk, g);
                pin_order();
            };
            while (true) {
                step(ra, rb);
                a0 += 32 * kWaves;
                if (a0 > a_hi) break;
                step(rb, ra);
                a0 += 32 * kWaves;
                if (a0 > a_hi) break;
            }
        }
    };
    share(std::false_type{});
    if (__builtin_expect(any_nan(acc), 0)) share(std::true_type{});
    sh.put(acc, p.alpha, wave, n, g);
    __syncthreads();
#pragma unroll
    for (int piece = tid; piece < Shares<D>::kPieces; piece += 64 * kWaves) {
        const int row = piece / (D / 4), c = piece % (D / 4) * 4;
        if (r0 + row >= T) continue;
        float4 o = sh.sum(piece);
        const size_t off = base + (size_t)(r0 + row) * D + c;
        if (p.addend) {
            const float4 e = *reinterpret_cast<const float4*>(p.addend + off);
            o.x += e.x; o.y += e.y; o.z += e.z; o.w += e.w;
        }
        *reinterpret_cast<float4*>(p.dX + off) = o;
    }
}

template <int D>
__device__ __forceinline__ void bwd_cols(const BwdP& p, Shares<D>& sh, int bh, int tile, int tid, int wave, int n, int g) {
    constexpr int DT = D / 32;
    const int T = p.T;
    const size_t base = (size_t)bh * T * D, vbase = (size_t)bh * T;
    const float *X = p.X + base, *G = p.G + base, *K = p.K + base, *V = p.V + base;
    const int c0 = tile * 32, a = c0 + n;
    const int r_lo = p.causal ? c0 : 0, r_hi = p.causal ? (int)min((long)T - 1, (long)c0 + 31 + p.k_diff) : T - 1;
    const float scale_log2 = p.alpha * kLog2e;
    f32x16 accK[DT], accV[DT];
    float db;
    own_put<D>(sh, K, V, c0, T, scale_log2, tid);
    __syncthreads();
    auto share = [&](auto any) {
        constexpr bool ANY = decltype(any)::value;
        clear<D>(accK);
        clear<D>(accV);
        db = 0.f;
        int rr0 = r_lo + 32 * wave;
        if (rr0 <= r_hi) {
            float lse = load_vec(p.lse + vbase, rr0, T, n), delta = load_vec(p.delta + vbase, rr0, T, n);
            const int nk = key_of_row(n);
            float ra[D / 2], rb[D / 2];
            load_rows<D>(ra, X, rr0, T, nk, g);
            load_rows<D>(rb, G, rr0, T, nk, g);
            const float b = p.bias ? p.bias[vbase + min(a, T - 1)] : 0.f;
            for (; rr0 <= r_hi; rr0 += 32 * kWaves) {
                const int next = min(rr0 + 32 * kWaves, r_hi & ~31);
                sh.vec_put(0, lse * p.lse_to_log2, wave, n);
                sh.vec_put(1, delta, wave, n);
                f32x16 s = score_tile<D, ANY>(ra, sh, 0, n, g);  // rows = streamed r, columns = owner a
                pin_order();
                load_cols<D>(ra, X, rr0, T, n, g);
                lse = load_vec(p.lse + vbase, next, T, n);
                delta = load_vec(p.delta + vbase, next, T, n);
                pin_order();
                f32x16 dp = score_tile<D, ANY>(rb, sh, 1, n, g);
                pin_order();
                load_cols<D>(rb, G, rr0, T, n, g);
                pin_order();
                const bool edge = rr0 + 32 > T || (p.causal && (rr0 < c0 + 31 || rr0 + 31 - c0 > p.k_diff));
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    const float4 l2 = sh.vec_get(0, wave, g, i4), dl = sh.vec_get(1, wave, g, i4);
                    const float l2s[4] = {l2.x, l2.y, l2.z, l2.w}, dls[4] = {dl.x, dl.y, dl.z, dl.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int i = 4 * i4 + e;
                        const float pr = fast_exp2(s[i] + b - l2s[e]);
                        s[i] = pr * (dp[i] - dls[e]);
                        dp[i] = pr;
                    }
                }
                if (edge) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int rr = rr0 + key_of(g, i);
                        const bool ok = (rr < T) & pair_valid(p.causal, p.k_diff, rr, a);
                        s[i] = ok ? s[i] : 0.f;
                        dp[i] = ok ? dp[i] : 0.f;
                    }
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) db += s[i];
                output_tile<D, ANY>(accK, ra, s);
                pin_order();
                load_rows<D>(ra, X, next, T, nk, g);
                pin_order();
                output_tile<D, ANY>(accV, rb, dp);
                pin_order();
                load_rows<D>(rb, G, next, T, nk, g);
                pin_order();
            }
        }
    };
    share(std::false_type{});
    if (__builtin_expect(any_nan(accK) || any_nan(accV), 0)) share(std::true_type{});
    db += __shfl_xor(db, 32, 64);
    if (g == 0) sh.row[wave][n] = db;
    sh.put(accK, p.alpha, wave, n, g);
    __syncthreads();
#pragma unroll
    for (int piece = tid; piece < Shares<D>::kPieces; piece += 64 * kWaves) {
        const int row = piece / (D / 4), c = piece % (D / 4) * 4;
        if (c0 + row < T) *reinterpret_cast<float4*>(p.dK + base + (size_t)(c0 + row) * D + c) = sh.sum(piece);
    }
    __syncthreads();
    sh.put(accV, 1.f, wave, n, g);
    __syncthreads();
#pragma unroll
    for (int piece = tid; piece < Shares<D>::kPieces; piece += 64 * kWaves) {
        const int row = piece / (D / 4), c = piece % (D / 4) * 4;
        const bool in = c0 + row < T;
        const size_t off = base + (size_t)(in ? c0 + row : 0) * D + c;
        float4 o = sh.sum(piece);
        if (p.mid_r) {
            const float4 R = *reinterpret_cast<const float4*>(p.mid_r + off), v2 = *reinterpret_cast<const float4*>(p.mid_v2 + off);
            const float4 dr = make_float4(o.x * v2.x, o.y * v2.y, o.z * v2.z, o.w * v2.w);
            float dot = dr.x * R.x + dr.y * R.y + dr.z * R.z + dr.w * R.w;  // over the D / 4 lanes of the row
#pragma unroll
            for (int d = D / 8; d > 0; d >>= 1) dot += __shfl_xor(dot, d, 64);
            if (in) {
                *reinterpret_cast<float4*>(p.dR + off) = dr;
                if (c == 0) {
                    float dbias = sh.row[0][row];
#pragma unroll
                    for (int w = 1; w < kWaves; ++w) dbias += sh.row[w][row];
                    p.delta1[vbase + c0 + row] = dot - dbias;
                }
            }
            o = make_float4(o.x * R.x, o.y * R.y, o.z * R.z, o.w * R.w);
        } else if (p.v1) {
            const float4 v1 = *reinterpret_cast<const float4*>(p.v1 + off);
            o.x *= silu_grad_f(v1.x); o.y *= silu_grad_f(v1.y); o.z *= silu_grad_f(v1.z); o.w *= silu_grad_f(v1.w);
        }
        if (in) *reinterpret_cast<float4*>(p.dV + off) = o;
    }
}

template <int D>
__global__ __launch_bounds__(64 * kWaves, 2) void attn_bwd_f32m_kernel(BwdP p) {
    __shared__ Shares<D> sh;
    const int ntiles = (p.T + 31) / 32;
    int bh, order;
    if (!xcd_tile(p.BH, 2 * ntiles, blockIdx.x >> 3, blockIdx.x & 7, bh, order)) return;
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // heavy first: under a causal mask the first owner columns see the most rows, the last owner rows the most columns
    if (order & 1)
        bwd_rows<D>(p, sh, bh, p.causal ? ntiles - 1 - (order >> 1) : order >> 1, tid, wave, n, g);
    else
        bwd_cols<D>(p, sh, bh, order >> 1, tid, wave, n, g);
}

// what the backward needs ahead of its passes: u = SiLU(v1) and delta = rowsum(dO * O); w = r * v2 where the forward's r is at
// hand (r not null).  D / 4 lanes a row
template <int D>
__global__ __launch_bounds__(256) void dps_prep_f32m_kernel(const float* __restrict__ v1, float* __restrict__ u,
                                                            const float* __restrict__ d_o, const float* __restrict__ o,
                                                            float* __restrict__ delta, const float* __restrict__ r,
                                                            const float* __restrict__ v2, float* __restrict__ w,
                                                            size_t rows) {
    const size_t piece = (size_t)blockIdx.x * 256 + threadIdx.x, row = piece / (D / 4);
    if (row >= rows) return;
    const float4 x = reinterpret_cast<const float4*>(v1)[piece];
    reinterpret_cast<float4*>(u)[piece] = make_float4(silu_f(x.x), silu_f(x.y), silu_f(x.z), silu_f(x.w));
    const float4 a = reinterpret_cast<const float4*>(d_o)[piece], b = reinterpret_cast<const float4*>(o)[piece];
    float dot = a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w;
#pragma unroll
    for (int d = D / 8; d > 0; d >>= 1) dot += __shfl_xor(dot, d, 64);
    if (piece % (D / 4) == 0) delta[row] = dot;
    if (r) {
        const float4 p = reinterpret_cast<const float4*>(r)[piece], q = reinterpret_cast<const float4*>(v2)[piece];
        reinterpret_cast<float4*>(w)[piece] = make_float4(p.x * q.x, p.y * q.y, p.z * q.z, p.w * q.w);
    }
}

template <int D>
void launch_fwd(const FwdP& p, hipStream_t st) {
    hipLaunchKernelGGL(attn_fwd_f32m_kernel<D>, dim3(xcd_slots(p.BH, (p.T + 31) / 32) * 8), dim3(64 * kWaves), 0, st, p);
}
template <int D>
void launch_bwd(const BwdP& p, hipStream_t st) {
    hipLaunchKernelGGL(attn_bwd_f32m_kernel<D>, dim3(xcd_slots(p.BH, 2 * ((p.T + 31) / 32)) * 8), dim3(64 * kWaves), 0, st, p);
}

// rows = K2[t], keys K1, values U; outputs R (the backward reads it), W = R * V2, lse1 (log2 units)
FwdP inner_fwd(const DpsArgs& a, float* r) {
    return {a.k2, a.k1, a.u, nullptr, a.v2, r, a.w, a.lse1, 1.0f, a.alpha * kLog2e, a.BH, a.T, a.causal, a.k_diff};
}

template <int D>
hipError_t fwd_impl(const DpsArgs& a, hipStream_t st) {
    launch_fwd<D>(inner_fwd(a, a.r), st);  // r: null, or kept for the backward
    // outer: rows = Q[q], keys K2 with bias lse1, values W; outputs O, LSE (natural log)
    launch_fwd<D>({a.q, a.k2, a.w, a.lse1, nullptr, a.o, nullptr, a.lse, kLn2, a.alpha * kLog2e, a.BH, a.T, a.causal, a.T}, st);
    return hipGetLastError();
}

template <int D>
hipError_t bwd_impl(const DpsArgs& a, hipStream_t st) {
    if (a.v1) {
        const size_t rows = (size_t)a.BH * a.T;
        hipLaunchKernelGGL(dps_prep_f32m_kernel<D>, dim3((unsigned)((rows * (D / 4) + 255) / 256)), dim3(256), 0, st, a.v1,
                           const_cast<float*>(a.u), a.d_o, a.o_in, a.delta, a.kept ? a.r : (const float*)nullptr, a.v2, a.w,
                           rows);
    }
    // kept: 205 -> 193 us for the training step of B=2 H=8 T=1000 D=64 k_diff 128
    if (!a.kept) launch_fwd<D>(inner_fwd(a, a.r), st);
    // outer pass: dQ; dK2 part, dV2, dR, delta1
    BwdP o{};
    o.X = a.q; o.G = a.d_o; o.K = a.k2; o.V = a.w; o.bias = a.lse1; o.lse = a.lse; o.lse_to_log2 = kLog2e;
    o.delta = a.delta; o.dX = a.dq; o.dK = a.dk2_part; o.dV = a.dv2;
    o.mid_r = a.r; o.mid_v2 = a.v2; o.dR = a.dr; o.delta1 = a.delta1;
    o.alpha = a.alpha; o.BH = a.BH; o.T = a.T; o.causal = a.causal; o.k_diff = a.T;
    launch_bwd<D>(o, st);
    // inner pass: dK2 (total); dK1, dU (dV1 for fp32 tensors)
    BwdP i{};
    i.X = a.k2; i.G = a.dr; i.K = a.k1; i.V = a.u; i.lse = a.lse1; i.lse_to_log2 = 1.0f;
    i.delta = a.delta1; i.addend = a.dk2_part; i.dX = a.dk2; i.dK = a.dk1; i.dV = a.du; i.v1 = a.v1;
    i.alpha = a.alpha; i.BH = a.BH; i.T = a.T; i.causal = a.causal; i.k_diff = a.k_diff;
    launch_bwd<D>(i, st);
    return hipGetLastError();
}

}  // namespace

bool f32_mfma_dps_supported(int D) { return D == 32 || D == 64; }

hipError_t f32_mfma_dps_fwd(const DpsArgs& a, hipStream_t st) {
    if (a.D == 32) return fwd_impl<32>(a, st);
    if (a.D == 64) return fwd_impl<64>(a, st);
    return hipErrorInvalidValue;
}
hipError_t f32_mfma_dps_bwd(const DpsArgs& a, hipStream_t st) {
    if (a.D == 32) return bwd_impl<32>(a, st);
    if (a.D == 64) return bwd_impl<64>(a, st);
    return hipErrorInvalidValue;
}

}  // namespace tritt
