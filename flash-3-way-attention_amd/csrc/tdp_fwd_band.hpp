// Triple-dot-product trittention forward for NARROW windowed causal masks (gfx950, 16-bit tensors):
// the band-resident kernel.  Included by tdp_fwd_mfma.hip (FwdParams, kLazyThreshold).
//
// Under a windowed mask a query q only sees keys j in [q - wa, q] and k in [q - wb, q].  When the
// windows are narrow, every key row a tile of 32 queries can touch (at most max(wa, wb) + 32 + 31 rows
// of K1, U^T, K2 and V2) fits in LDS at once.  The workgroup loads that band ONCE, synchronises once,
// and from then on its eight or sixteen waves run independently with no barrier and no global load: each
// wave walks its four or two queries one after another, per query the k-tiles of 32 inside [q - wb, q], per k-tile
// the 32-key steps of j inside the band of that tile.  Same formulation as the streaming kernel (virtual
// rows (q, k), transposed scores, P fed back as the A operand); what changes is that a k-tile of a narrow
// band has only a handful of steps, so everything per k-tile is kept cheap:
//   * FAST sweep first (P = exp2(S), reference 0, no maximum tracking); a wave whose sweep left the
//     safe exponent range repeats it by itself with the CAREFUL online softmax.
//   * masks of the k-j band come from a table in LDS: the pattern of a 32x32 step depends only on
//     (first key j - first key k), and at most four such offsets straddle an edge of the band; the
//     table holds them in the MFMA C layout (0 or -3e4), read as the C operand of the score product.
//     Steps cut by j <= q or j >= q - wa add another table's entries (by j - limit, the same for every row), k-tiles
//     cut by the k window a penalty per row.
//   * with reference 0 everywhere the merge of a k-tile into the running output needs no maximum, no
//     rescaling and no row weights (masked rows have P = 0 exactly): O += V2[k] (.) Tv[(q,k)].
// What bounds it: vector issue, one vector or matrix instruction per five cycles and SIMD, with 13-18 of the former for an MFMA:
// exponentials, the operand of a k-tile (80 for 24 MFMAs) and its merge.  B=2 H=8 T=2048 D=64 fp16, windows 128 / 32 (a call): 176 us;
// with the step loop on the scalar unit and V2 by transposed reads 167, with the limits' masks from a table 164, with K2 as floats
// 155 (B=4 H=8 T=1024 windows 64 / 16: 109 -> 94; D = 32 B=4 H=8 T=2048 windows 300 / 100 953 -> 845).
#pragma once

namespace tritt {

constexpr int kBandQ = 32;  // queries per workgroup
constexpr int kCutRow = 72;  // entries of a limit's mask, j - limit = -32 .. 31 and what a copy is shifted by

// rows of the resident band: everything queries q0 .. q0+31 can touch (q0 is a multiple of 32, and so is the
// first resident row)
inline int band_rows(int wa, int wb) { return ((wa > wb ? wa : wb) + 31) / 32 * 32 + kBandQ; }

template <int D, int kW>
constexpr size_t band_smem_bytes(int nr, bool k2_float = false) {
    return (k2_float ? sizeof(float) * nr * (D + 4) - sizeof(uint16_t) * nr * (D + 8) : 0) + sizeof(uint16_t) * ((size_t)3 * nr * (D + 8) + (size_t)D * (nr + 8)) + sizeof(float) * (kBandQ * D + kW * 32 + 5 * 16 * 64 + 2 * 4 * kCutRow);
}

// kW: waves per workgroup (band_waves16).  K2F: K2 lies in LDS as floats, converted once per workgroup and not once per query and
// k-tile (32 of a k-tile's 340 vector instructions at D = 64)
template <typename E, int D, int kW, bool MV = false, bool K2F = false>
__global__ __launch_bounds__(64 * kW, kW / 4) void tdp_fwd_band_kernel(FwdParams<E> p, int NR) {
    using M = Mma<E>;
    using v8 = typename M::v8;
    using v2 = typename M::v2;
    constexpr int KS = D / 16, DT = D / 32, LDK = D + 8, kThreads = 64 * kW;
    const int LDU = NR + 8;

    extern __shared__ __align__(16) char smem[];
    E* sK1 = reinterpret_cast<E*>(smem);  // [NR][LDK]
    E* sK2 = sK1 + NR * LDK;                // [NR][LDK], K2F: floats, [NR][D + 4]
    E* sV2 = K2F ? reinterpret_cast<E*>(reinterpret_cast<float*>(sK2) + NR * (D + 4)) : sK2 + NR * LDK;
    E* sUT = sV2 + NR * LDK;               // [D][LDU]
    float* sQ = reinterpret_cast<float*>(sUT + D * LDU);  // [32][D]  Q * alpha*log2(e), fp32
    float* sW = sQ + kBandQ * D;                                // [kW][32] per-wave scratch
    float* sTab = sW + kW * 32;  // [5 slots][4][64 lanes][4]  band masks in the MFMA C layout; slot 4: zeros
    // [2][4][kCutRow]  masks of the limits j <= q and j >= q - wa by j - limit (0 or -3e4); copy c is shifted by c entries, so that
    // four consecutive ones are an aligned read whatever the limit
    float* sCut = sTab + 5 * 16 * 64;

    int bh, order;
    if (!xcd_tile(p.BH, p.nqt, blockIdx.x >> 3, blockIdx.x & 7, bh, order)) return;
    const int qt = p.nqt - 1 - order;

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int T = p.T;
    const size_t base = (size_t)bh * T * D;  // of the outputs
    const size_t in_base = (size_t)(bh / p.H) * p.in_sb + (size_t)(bh % p.H) * p.in_sh;
    const unsigned in_st = p.in_st;
    const E* __restrict__ Q = p.q + in_base;
    const int wa = p.wa, wb = p.wb, lab = p.lab, rab = p.rab;
    const int q0 = qt * kBandQ;
    const int rlo = max(0, q0 - max(wa, wb)) & ~31;  // first resident key row

    // ---- load the band ---------------------------------------------------------------------------
    {
        auto slice = [&](const E* t, const TensorAt& at) {
            return MV ? t + (size_t)(bh / p.H) * at.sb + (size_t)(bh % p.H) * at.sh : t + in_base;
        };
        const E* __restrict__ K1 = slice(p.k1, p.at_k1);
        const E* __restrict__ K2 = slice(p.k2, p.at_k2);
        const E* __restrict__ V2 = slice(p.v2, p.at_v2);
        const unsigned st_k1 = MV ? p.at_k1.st : in_st, st_k2 = MV ? p.at_k2.st : in_st, st_v2 = MV ? p.at_v2.st : in_st;
        const E* __restrict__ UT = p.ut + (size_t)bh * D * p.Tp;
        // Q, and two 16-byte chunks of each of the four tensors, are asked for before any of them is waited for: nothing else runs
        // under the round trips of a workgroup that has a CU to itself (165.2 -> 160.2 us at B2 H8 T2048 D64 fp16, bands 128 and 32).
        // Every tensor has NR D / 8 chunks.
        static_assert(kBandQ * D % kThreads == 0, "every thread takes as many elements of Q");
        constexpr int kQ = kBandQ * D / kThreads;
        E qv[kQ];
#pragma unroll
        for (int i = 0; i < kQ; ++i) {
            const int idx = tid + i * kThreads;
            qv[i] = Q[(size_t)((unsigned)min(q0 + idx / D, T - 1) * in_st) + idx % D];
        }
        const int chunks = NR * (D / 8);
        struct Chunk {
            uint4 k1, k2, v2, ut;
        };
        auto load = [&](int c) {
            const int r = c / (D / 8), ch = c % (D / 8);
            const unsigned row = (unsigned)min(rlo + r, T - 1);
            Chunk x;
            x.k1 = *reinterpret_cast<const uint4*>(K1 + (size_t)(row * st_k1) + ch * 8);
            x.k2 = *reinterpret_cast<const uint4*>(K2 + (size_t)(row * st_k2) + ch * 8);
            x.v2 = *reinterpret_cast<const uint4*>(V2 + (size_t)(row * st_v2) + ch * 8);
            const int d = c / (NR / 8), j0 = rlo + c % (NR / 8) * 8;
            x.ut = uint4{0u, 0u, 0u, 0u};
            if (j0 + 8 <= p.Tp) x.ut = *reinterpret_cast<const uint4*>(UT + (size_t)d * p.Tp + j0);
            return x;
        };
        auto store = [&](int c, const Chunk& x) {
            const int r = c / (D / 8), ch = c % (D / 8);
            *reinterpret_cast<uint4*>(sK1 + r * LDK + ch * 8) = x.k1;
            if constexpr (K2F) {
                const v8 k = __builtin_bit_cast(v8, x.k2);
                float* at = reinterpret_cast<float*>(sK2) + r * (D + 4) + ch * 8;
                *reinterpret_cast<float4*>(at) = make_float4((float)k[0], (float)k[1], (float)k[2], (float)k[3]);
                *reinterpret_cast<float4*>(at + 4) = make_float4((float)k[4], (float)k[5], (float)k[6], (float)k[7]);
            } else {
                *reinterpret_cast<uint4*>(sK2 + r * LDK + ch * 8) = x.k2;
            }
            *reinterpret_cast<uint4*>(sV2 + r * LDK + ch * 8) = x.v2;
            *reinterpret_cast<uint4*>(sUT + c / (NR / 8) * LDU + c % (NR / 8) * 8) = x.ut;
        };
        for (int c = tid; c < chunks; c += 2 * kThreads) {
            const Chunk x = load(c), y = load(min(c + kThreads, chunks - 1));
            store(c, x);
            if (c + kThreads < chunks) store(c + kThreads, y);
        }
#pragma unroll
        for (int i = 0; i < kQ; ++i) sQ[tid + i * kThreads] = (float)qv[i] * p.scale_log2;
    }
    // ---- band mask table: slot -> offset m = (jb - k0) / 32 ----------------------------------------
    const int mlo = -((lab + 31) / 32), mhi = (rab + 31) / 32;
    if (tid < 320) {
        const int sl = tid >> 6, m = sl < 2 ? mlo + sl : mhi - (sl - 2);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int dlt = 32 * m + key_of(g, i) - n;  // j - k
            sTab[((sl * 4 + i / 4) * 64 + lane) * 4 + (i % 4)] = (sl == 4 || (dlt >= -lab && dlt <= rab)) ? 0.f : -3.0e4f;
        }
    }
    for (int idx = tid; idx < 2 * 4 * kCutRow; idx += kThreads) {
        const int x = idx % kCutRow + idx / kCutRow % 4 - 32;
        sCut[idx] = (idx < 4 * kCutRow ? x <= 0 : x >= 0) ? 0.f : -3.0e4f;
    }
    __syncthreads();
    // from here on the waves never meet again

    // (the compiler takes the maximum of three on the vector ALU and then keeps the loop that starts from it there, under exec
    // masks: 20 of 56 vector instructions per step)
    auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
    float* sWw = sW + wave * 32;
    const int krow_off = key_of_row(n);
    auto rows_of = [&](float v, float (&out)[16]) {
        if (g == 0) sWw[n] = v;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const float4 f4 = *reinterpret_cast<const float4*>(sWw + 8 * b + 4 * g);
            out[4 * b] = f4.x; out[4 * b + 1] = f4.y; out[4 * b + 2] = f4.z; out[4 * b + 3] = f4.w;
        }
        __builtin_amdgcn_wave_barrier();
    };

    for (int qi = 0; qi < kBandQ / kW; ++qi) {
        const int q = q0 + wave + kW * qi;  // interleaved: the waves' loads stay even at the start of a sequence
        if (q >= T) break;
        const float* sQw = sQ + (wave + kW * qi) * D;

        float Mrun = -INFINITY, Lrun = 0.f, Orun[DT];  // Lrun, Orun: per-lane partial sums
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) Orun[dt] = 0.f;

        // k >= q - wb, and some j with q - wa <= j <= k + rab
        const int kt_a = uniform(max(0, max(q - wb, q - wa - rab)) / 32), kt_b = q / 32;
        for (int kt = kt_a; kt <= kt_b; ++kt) {
            const int k0 = kt * 32, k = k0 + n;
            // window of keys j of the virtual row (q, k); empty: hi < lo
            int wlo = max(q - wa, k - lab), whi = min(q, k + rab);
            if (k > q || q > k + wb || whi < wlo) { wlo = 0; whi = -1; }
            const bool kval = whi >= 0;
            // all 32 rows of the tile are inside the k window
            const bool rows_clean = (k0 + 31 <= q) && (q <= k0 + wb);
            const int jlo_t = uniform(max(0, max(q - wa, k0 - lab))), jhi_t = min(q, k0 + 31 + rab);
            const int jb_lo = jlo_t & ~31;
            if (jlo_t > jhi_t) continue;  // no (j, k) of this tile is inside the band of q

            v8 bq[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                float kf[8];
                if constexpr (K2F) {
                    const float* at = reinterpret_cast<const float*>(sK2) + (k0 - rlo + n) * (D + 4) + ks * 16 + g * 8;
                    const float4 lo = *reinterpret_cast<const float4*>(at), hi = *reinterpret_cast<const float4*>(at + 4);
                    kf[0] = lo.x; kf[1] = lo.y; kf[2] = lo.z; kf[3] = lo.w;
                    kf[4] = hi.x; kf[5] = hi.y; kf[6] = hi.z; kf[7] = hi.w;
                } else {
                    const v8 kv = *reinterpret_cast<const v8*>(sK2 + (k0 - rlo + n) * LDK + ks * 16 + g * 8);
#pragma unroll
                    for (int e = 0; e < 8; ++e) kf[e] = (float)kv[e];
                }
                const float* qp = sQw + ks * 16 + g * 8;
                const float4 qa = *reinterpret_cast<const float4*>(qp), qb = *reinterpret_cast<const float4*>(qp + 4);
                const float qf[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
                v8 r;
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const v2 pr = M::pack(kf[e] * qf[e], kf[e + 1] * qf[e + 1]);
                    r[e] = pr[0];
                    r[e + 1] = pr[1];
                }
                bq[ks] = r;
            }

            f32x16 acc[DT];
            float mref = 0.f, lsum = 0.f;
            auto clear = [&] {
                mref = 0.f;
                lsum = 0.f;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;
            };
            auto value_product = [&](const v8 (&pa)[2], int jb) {
                const E* utp = sUT + n * LDU + (jb - rlo) + g * 8;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        acc[dt] = M::mma(pa[h], *reinterpret_cast<const v8*>(utp + dt * 32 * LDU + h * 16), acc[dt]);
            };

            // ---- FAST sweep ---------------------------------------------------------------------
            // C operand of the score product = the mask, all of it additive: the k-j band from the table
            // (slot 4: all zeros), a per-lane penalty for rows outside the k window, and, on the steps the
            // limits j <= q / j >= q - wa cut through, the limits' tables.  The first step starts the
            // value accumulators from a zero C operand instead of cleared registers.
            const float row_pen = kval ? 0.f : -3.0e4f;
            auto fast_step = [&](int jb, auto first_tag) {
                constexpr bool FIRST = decltype(first_tag)::value;
                const E* k1p = sK1 + (jb - rlo + krow_off) * LDK + g * 8;
                const int m = (jb - k0) >> 5;
                const bool partial = 32 * m - 31 < -lab || 32 * m + 31 > rab;  // straddles an edge of the band
                const int sl = !partial ? 4 : (m - mlo < 2) ? m - mlo : 2 + (mhi - m);
                f32x16 s;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const float4 f4 = *reinterpret_cast<const float4*>(sTab + ((sl * 4 + b) * 64 + lane) * 4);
                    s[4 * b] = f4.x; s[4 * b + 1] = f4.y; s[4 * b + 2] = f4.z; s[4 * b + 3] = f4.w;
                }
                if (!rows_clean) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) s[i] += row_pen;
                }
                auto cut = [&](const float* masks, int limit) {  // |jb - limit| <= 31
                    const int x = jb - limit + 32, c = x & 3;
                    const float* at = masks + c * kCutRow + (x - c) + 8 * g;
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        const float4 f4 = *reinterpret_cast<const float4*>(at + key_of(0, 4 * b));
                        s[4 * b] += f4.x; s[4 * b + 1] += f4.y; s[4 * b + 2] += f4.z; s[4 * b + 3] += f4.w;
                    }
                };
                if (jb + 31 > q) cut(sCut, q);
                if (jb < q - wa) cut(sCut + 4 * kCutRow, q - wa);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) s = M::mma(*reinterpret_cast<const v8*>(k1p + ks * 16), bq[ks], s);
                v8 pa[2];
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int e = 0; e < 8; e += 2) {
                        const v2 pr = M::pack(fast_exp2(s[h * 8 + e]), fast_exp2(s[h * 8 + e + 1]));
                        lsum = M::add_pair(pr, lsum);
                        pa[h][e] = pr[0];
                        pa[h][e + 1] = pr[1];
                    }
                const E* utp = sUT + n * LDU + (jb - rlo) + g * 8;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    f32x16 c;
                    if constexpr (FIRST) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) c[i] = 0.f;
                    } else {
                        c = acc[dt];
                    }
                    c = M::mma(pa[0], *reinterpret_cast<const v8*>(utp + dt * 32 * LDU), c);
                    acc[dt] = M::mma(pa[1], *reinterpret_cast<const v8*>(utp + dt * 32 * LDU + 16), c);
                }
            };
            mref = 0.f;
            lsum = 0.f;
            fast_step(jb_lo, std::true_type{});
            for (int jb = jb_lo + 32; jb <= jhi_t; jb += 32) fast_step(jb, std::false_type{});
            bool fast_ok;
            {
                // P <= its row sum, so a row sum inside this range keeps the value accumulators finite as well
                const float lk = lsum + __shfl_xor(lsum, 32, 64);
                fast_ok = !__any(kval && !(lk > fast_row_sum_floor<E>() && lk < 1e25f));
            }
            if (!fast_ok) {
                // ---- CAREFUL sweep: online softmax, reference raised lazily; a row may meet its first
                // valid key late, until then its reference sits at a finite floor
                clear();
                bool started = false;
                for (int jb = jb_lo; jb <= jhi_t; jb += 32) {
                    const E* k1p = sK1 + (jb - rlo + krow_off) * LDK + g * 8;
                    f32x16 s;
#pragma unroll
                    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks) s = M::mma(*reinterpret_cast<const v8*>(k1p + ks * 16), bq[ks], s);
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int j = jb + key_of(g, i);
                        s[i] = (j >= wlo && j <= whi) ? s[i] : -INFINITY;
                    }
                    float mx = fmaxf(s[0], s[1]);
#pragma unroll
                    for (int i = 2; i < 16; i += 2) mx = fmaxf(fmaxf(mx, s[i]), s[i + 1]);
                    const bool begin = !started;
                    started = true;
                    if (begin || __any(mx - mref > kLazyThreshold)) {
                        const float rmax = fmaxf(fmaxf(mx, __shfl_xor(mx, 32, 64)), -1.0e30f);
                        const float newref = begin ? rmax : fmaxf(rmax, mref);
                        const float f = fast_exp2(mref - newref);
                        mref = newref;
                        if (!begin) {
                            lsum *= f;
                            float fr[16];
                            rows_of(f, fr);
#pragma unroll
                            for (int i = 0; i < 16; ++i)
#pragma unroll
                                for (int dt = 0; dt < DT; ++dt) acc[dt][i] *= fr[i];
                        }
                    }
                    v8 pa[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int e = 0; e < 8; e += 2) {
                            const v2 pr = M::pack(fast_exp2(s[h * 8 + e] - mref), fast_exp2(s[h * 8 + e + 1] - mref));
                            lsum = M::add_pair(pr, lsum);
                            pa[h][e] = pr[0];
                            pa[h][e + 1] = pr[1];
                        }
                    value_product(pa, jb);
                }
            }

            // ---- merge the 32 virtual rows (q, k) into the running output ---------------------------
            // V2 of rows c_row(g, i), column dt 32 + n: four rows of a column per transposed read (in every group of 16 lanes
            // ds_read_b64_tr_b16 gives lane l element l % 4 of what lanes l / 4, 4 + l / 4, ... address)
            const E* v2p = sV2 + (k0 - rlo + 4 * g + (lane & 15) / 4) * LDK + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
            auto v2_rows = [&](int dt, int b, float (&v)[4]) {  // registers 4 b .. + 3
                typedef __attribute__((ext_vector_type(4))) short s4;
                typedef __attribute__((ext_vector_type(4))) E e4;
                const e4 x = __builtin_bit_cast(e4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4*)(v2p + 8 * b * LDK + dt * 32)));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = (float)x[e];
            };
            if (fast_ok && (Mrun == 0.f || Mrun == -INFINITY)) {
                // everything so far is relative to reference 0 and masked rows hold exact zeros
                Mrun = 0.f;
                Lrun += lsum;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    float part = 0.f;
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        float v[4];
                        v2_rows(dt, b, v);
#pragma unroll
                        for (int e = 0; e < 4; ++e) part += v[e] * acc[dt][4 * b + e];
                    }
                    Orun[dt] += part;
                }
            } else {
                float mt = kval ? mref : -INFINITY;
#pragma unroll
                for (int off = 16; off > 0; off >>= 1) mt = fmaxf(mt, __shfl_xor(mt, off, 64));
                const float mnew = fmaxf(Mrun, mt);
                const float f = (mnew == -INFINITY) ? 1.f : fast_exp2(Mrun - mnew);
                const float w = kval ? fast_exp2(mref - mnew) : 0.f;
                Lrun = Lrun * f + w * lsum;
                Mrun = mnew;
                float wr[16];
                rows_of(w, wr);
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    float part = 0.f;
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        float v[4];
                        v2_rows(dt, b, v);
#pragma unroll
                        for (int e = 0; e < 4; ++e) part += wr[4 * b + e] * v[e] * acc[dt][4 * b + e];
                    }
                    Orun[dt] = Orun[dt] * f + part;
                }
            }
        }

        // ---- this query is done --------------------------------------------------------------------
        float L = Lrun;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) L += __shfl_xor(L, off, 64);
        const float inv = 1.0f / L;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const float o = (Orun[dt] + __shfl_xor(Orun[dt], 32, 64)) * inv;
            if (g == 0) p.o[base + (size_t)q * D + dt * 32 + n] = (E)o;
        }
        if (lane == 0) p.lse[(size_t)bh * T + q] = (Mrun + fast_log2(L)) * kLn2;
    }
}

}  // namespace tritt
