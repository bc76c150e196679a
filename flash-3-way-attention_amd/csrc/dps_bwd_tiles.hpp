// Included by dps_mfma.hip inside namespace tritt::{anonymous}: the backward attention-with-bias passes at D = 32 and 64.
//
// A workgroup of four waves owns 32 * kOT rows (row pass: query-like rows -> dX; column pass: key-like rows -> dK, dV,
// dbias), kOT tiles of 32, and kSH waves share an owner tile: the streamed 32-row tiles are dealt out to them in turn and
// their sums are joined through LDS at the end.  The streamed tensors (two of them: K, V or X, dO) come as packing P1 in
// groups of kSH tiles, fetched straight into an LDS ring three groups ahead; the scores read the packed rows as they lie, the
// gradient products read the same bytes transposed in the LDS unit (ds_read_b64_tr_b16), so nothing else is fetched or packed.
//
// What bounds it: vector issue (80 instructions beside 16 MFMAs per tile of a column pass: 16 each of fused multiply-add,
// exp2, multiply, accumulate, and pack) and two waves per SIMD that seldom use both pipes at once; a column tile takes about
// 1260 cycles of a SIMD where its MFMAs take 512.  Timing-only ablations (B=1 H=8 T=8192, outer columns 168 us): no loads
// 148, no barriers 153, no exp2 152, no transposed reads 157.  Reading the next rows a barrier earlier (246 registers instead
// of 202) changed nothing.  Against one 32-row tile per workgroup with operands fetched per wave and the passes as launches of
// their own (four-wave workgroups of 128 rows on large grids), training steps in turn, bf16, D = 64: B=4 H=8 T=1024 142 -> 110 us,
// B=1 H=8 T=8192 k_diff 2048 795 -> 622 (both in workgroups of 64 rows); the three passes that depend on nothing of each other in one
// grid instead of one after the other, and half the bytes per tile, are most of it.
#pragma once

template <int D, int kOT, int kSH>
struct BwdTiles {
    static constexpr int KS = D / 16, DT = D / 32, kW = kOT * kSH, kNS = 4;
    static constexpr int kTensor = KS * 1024, kTile = 2 * kTensor;  // bytes of a streamed tile: two tensors
    static constexpr int LW = 2 * KS * kSH / kW;                    // 1 KB blocks a wave fetches per stage, of one tensor and tile
    static constexpr int kVec = 256;                                // bytes of a stage's per-row vector: 64 floats
    static constexpr int kStage = kSH * kTile + 2 * kVec;
    static constexpr int kMerge = 4 * (kW * D * kLdr + kW * 32 + 2 * kW * 32);
    static constexpr int smem = kNS * kStage > kMerge ? kNS * kStage : kMerge;
    static_assert(kW == 4 && kSH <= 2 && LW >= 1 && KS % LW == 0, "a wave fetches blocks of one tensor and tile");
};

// transposed operand (d-tile, half) of a packed tile: lane (g, n) receives rows 16 kk + 8 g .. + 7 of column 32 dt + n.
// ds_read_b64_tr_b16: in every group of 16 lanes, lane i addresses four consecutive elements and lane l receives element
// l % 4 of what lanes l / 4, 4 + l / 4, 8 + l / 4, 12 + l / 4 address; so lane i addresses row i / 4 and columns 4 (i % 4) ..
// of the group's 16 columns.  This is the offset for the first four rows, ^ 128 that for the other four; the packing's swizzle gives 32 lanes 32
// different 8-byte slots of the 256 bytes that LDS serves at once.
__device__ __forceinline__ int tr_offset(int lane) {
    const int i = lane & 15, h = (lane >> 4) & 1, g = lane >> 5, gp = (i >> 1) & 1;
    return h * (1024 + 128) + gp * 512 + (g ^ gp) * 64 + (i >> 2) * 16 + (i & 1) * 8;
}
// What a backward's exponents are multiplied with: alpha log2(e), kept away from zero because the streamed terms are
// divided by it (scores that small do not change an exponent).
__host__ __device__ __forceinline__ float bwd_scale(float alpha) {
    const float s = alpha * kLog2e;
    return s < 0.f ? fminf(s, -0x1p-100f) : fmaxf(s, 0x1p-100f);
}

// One pass over an owner block.  COL: column pass (streams X and dO and two values per row), else row pass (streams K and V
// and, with BIAS, a value per key).  LINK: the outer column pass, whose epilogue holds the element-wise link.
//
// The exponent of a pair is score * scale + (a term of the owner) + (a term of the streamed row: -LSE[row] or bias[key]).
// The streamed term comes divided by the scale and is what the score product starts from (the C operand, read from LDS
// straight into the accumulator), so an exponent is one fused multiply-add; -Delta is what the dP product starts from.
// NEG: the vector holds +LSE / scale; the owner's score operand and the scale are taken negative instead.
// An exponent is thereby rounded two or three times at its terms' size where a sum formed ahead of the score is once or twice.  P's 16
// bits hide that up to |LSE| of 2^12: against 64 bits errors are those of such a sum with operands 16 times normal ones, and with
// one element of 1e4 in Q, K1 or K2 in bf16; in fp16 that element makes dV1 4.0e-4 instead of 3.4e-4, one of 6e4 1.8e-3 instead of
// 0.9e-3 (a rounded LSE).  Forming the score products of such tiles once more from zero gives the latter figures; telling them apart
// costs every workgroup a pass over the terms, 1 us and 1 to 5 % of a call of this package's sizes, and was taken back.
template <typename E, int D, int kOT, int kSH, bool COL, bool BIAS, bool LINK, bool NEG, bool SV>
__device__ __forceinline__ void attn_bwd_tiles_body(const AttnBwdP<E, SV>& p, int bh, int tile) {
    using M = Mma<E>;
    using v8 = typename M::v8;
    using v2 = typename M::v2;
    using S = BwdTiles<D, kOT, kSH>;
    constexpr int KS = S::KS, DT = S::DT, LW = S::LW, kW = S::kW, NS = S::kNS;
    constexpr bool kVectors = COL || BIAS;
    constexpr int kLoads = LW + (kVectors ? 1 : 0);
    extern __shared__ __align__(16) char smem_raw[];

    const int n_owner = (p.Tp / 32 + kOT - 1) / kOT;
    const int o0 = (COL ? tile : n_owner - 1 - tile) * 32 * kOT;  // longest blocks first
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ot = wave % kOT, sh = wave / kOT;
    const int T = p.T, Tp = p.Tp;
    const size_t base = (size_t)bh * T * D, tb = (size_t)bh * D * Tp, vb = (size_t)bh * Tp;
    const int ow0 = o0 + 32 * ot, own = ow0 + n, ownc = min(own, T - 1);
    const float scale = bwd_scale(p.alpha) * (NEG ? -1.f : 1.f);
    const int2 at = slice_at<SV>(bh, p.H);

    // streamed tiles of the workgroup, of this wave's owner tile, and those of them that need no element-wise mask
    const int last_own = min(T - 1, o0 + 32 * kOT - 1), wlast_own = min(T - 1, ow0 + 31);
    int t_first = 0, t_last = (T - 1) / 32, tw_first = 0, tw_last = t_last, ti_first = 0, ti_last = T / 32 - 1;
    if (p.causal) {
        if constexpr (COL) {
            t_first = o0 / 32;
            t_last = (int)min((long)T - 1, (long)last_own + p.k_diff) / 32;
            tw_first = ow0 / 32;
            tw_last = (int)min((long)T - 1, (long)wlast_own + p.k_diff) / 32;
            ti_first = ow0 / 32 + 1;
            ti_last = min(ti_last, p.k_diff < 31 ? -1 : (int)(((long)ow0 + p.k_diff - 31) / 32));
        } else {
            t_first = max(0, o0 - p.k_diff) / 32;
            t_last = last_own / 32;
            tw_first = max(0, ow0 - p.k_diff) / 32;
            tw_last = wlast_own / 32;
            ti_first = (max(0, ow0 + 31 - p.k_diff) + 31) / 32;
            ti_last = min(ti_last, ow0 / 32 - 1);
        }
    }
    if (ow0 + 31 >= T) ti_last = -1;
    if (ow0 >= T) tw_last = -1;
    const int steps = (t_last - t_first) / kSH + 1;

    // ---- stage loader: wave w fetches LW blocks of one tensor of one tile of every stage, and 64 floats of a vector
    // (a stage's vectors are read for kSH * 32 rows; kSH = 1 leaves the second half unused)
    const E* first = COL ? p.xp : p.kp;
    const E* second = COL ? p.gp : p.vp;
    constexpr int kPer = KS / LW;  // waves per (tensor, tile)
    const int unit = wave / kPer, l_tile = unit >> 1, l_tensor = unit & 1, l_block = (wave % kPer) * LW;
    const char* gsrc = reinterpret_cast<const char*>(uniform_ptr((l_tensor ? second : first) + tb)) + l_block * 1024;
    const int gdst = l_tile * S::kTile + l_tensor * S::kTensor + l_block * 1024;
    const int vec = COL ? wave & 1 : 0;
    const float* vsrc = nullptr;
    if constexpr (COL) vsrc = uniform_ptr((vec ? p.delta : p.term) + vb);
    else if constexpr (BIAS) vsrc = uniform_ptr(p.term + vb);
    int f_tile = t_first;
    auto fetch = [&](int slot) {  // the next stage -> slot; tiles past t_last are fetched as t_last once more, and masked
        char* dst = smem_raw + slot * S::kStage;
        const char* src = uniform_ptr(gsrc + (unsigned)min(f_tile + l_tile, t_last) * (size_t)S::kTensor);
#pragma unroll
        for (int j = 0; j < LW; ++j) direct_load_16(src + j * 1024, lane * 16, dst + gdst + j * 1024);
        if constexpr (kVectors)
            direct_load_4(vsrc, (unsigned)min(f_tile * 32 + lane, Tp - 1) * 4, dst + kSH * S::kTile + vec * S::kVec);
        f_tile += kSH;
    };

    // ---- the owner tile's operands; everything the loop reads from registers has arrived before the first stage is asked
    // for, so that no wait inside the loop has to reach past the stages in flight
    v8 xb[KS], gb[KS];
    {
        const View<E, SV>&first_own = COL ? p.k : p.x, &second_own = COL ? p.v : p.g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            xb[ks] = ld8<E>(first_own.row(at, ownc, T, D) + 16 * ks + 8 * g);
            if constexpr (NEG) xb[ks] = -xb[ks];
            gb[ks] = ld8<E>(second_own.row(at, ownc, T, D) + 16 * ks + 8 * g);
        }
    }
    float own_term = 0.f, own_delta = 0.f;
    if constexpr (COL) own_term = p.bias ? p.bias[vb + ownc] : 0.f;
    else { own_term = -p.lse2[vb + ownc]; own_delta = p.delta[vb + ownc]; }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(xb[ks]), "+v"(gb[ks]));
    asm volatile("" : "+v"(own_term), "+v"(own_delta));
#pragma unroll
    for (int u = 0; u < NS - 1; ++u) fetch(u);

    // streamed rows that pair with this lane's own one: lo .. lo + span
    int lo, span;
    if (own >= T) {
        lo = 1 << 30; span = 0;
    } else if (!p.causal) {
        lo = 0; span = T - 1;
    } else if (COL) {
        lo = own; span = (int)min((long)T - 1 - own, (long)p.k_diff);
    } else {
        lo = max(0, own - p.k_diff); span = own - lo;
    }
    const float dead = -1.0e30f / scale;  // a score whose exponent no other term brings back above any exp2 can return

    f32x16 acca[DT], accb[COL ? DT : 1];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            acca[dt][i] = 0.f;
            if constexpr (COL) accb[dt][i] = 0.f;
        }
    float db = 0.f;
    f32x16 minus_delta;
    if constexpr (!COL) {
#pragma unroll
        for (int i = 0; i < 16; ++i) minus_delta[i] = own_delta;
        asm volatile("" : "+v"(minus_delta));
    }

    // packed rows of a tile in MFMA order (the packing's swizzle is the same for all even and for all odd k-steps)
    const char* row_even = smem_raw + sh * S::kTile + (lane ^ (g << 2)) * 16;
    const char* row_odd = smem_raw + sh * S::kTile + ((lane ^ (g << 2)) * 16 ^ 128);
    const char* tr = smem_raw + sh * S::kTile + tr_offset(lane);
    const char* tr4 = smem_raw + sh * S::kTile + (tr_offset(lane) ^ 128);
    const float* vecs = reinterpret_cast<const float*>(smem_raw + kSH * S::kTile + sh * 128);
    v8 ra[KS], rb[KS];
    f32x16 s, dp;
    auto load_rows = [&](int slot) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const char* r = ((ks & 1) ? row_odd : row_even) + slot * S::kStage + ks * 1024;
            ra[ks] = *reinterpret_cast<const v8*>(r);
            rb[ks] = *reinterpret_cast<const v8*>(r + S::kTensor);
        }
        float x[16];
        if constexpr (kVectors) {
            tile_vector(vecs + slot * (S::kStage / 4), g, x);
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = x[i];
        }
        if constexpr (COL) {
            tile_vector(vecs + (slot * S::kStage + S::kVec) / 4, g, x);
#pragma unroll
            for (int i = 0; i < 16; ++i) dp[i] = x[i];
        }
    };
    barrier_keep_loads<kLoads * (NS - 2)>();  // stage 0 has landed for everyone
    load_rows(0);

    int t = t_first + sh;
    auto step = [&](auto slot_c) {
        constexpr int slot = decltype(slot_c)::value, next = (slot + 1) % NS;
        // this step's barrier: the next stage has landed for everyone and the previous one has been read by everyone, so
        // that its slot can be fetched into
        auto cross = [&]() {
            barrier_keep_loads<kLoads * (NS - 3)>();
            fetch((slot + NS - 1) % NS);
        };
        v8 ta[DT][2], tb2[COL ? DT : 1][2];
        auto transposed = [&](const char* z, int dt, int kk) {
            typedef __attribute__((ext_vector_type(4))) short s4;
            const int off = slot * S::kStage + dt * 2048 + kk * 256 + (int)(z - tr);
            const s4 lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4*)(tr + off));
            const s4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4*)(tr4 + off));
            return __builtin_bit_cast(v8, __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
        };
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!kVectors) {
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = 0.f;
        }
        if constexpr (!COL) dp = minus_delta;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            s = M::mma(ra[ks], xb[ks], s);
            dp = M::mma(rb[ks], gb[ks], dp);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                ta[dt][kk] = transposed(tr, dt, kk);
                if constexpr (COL) tb2[dt][kk] = transposed(tr + S::kTensor, dt, kk);
            }
        __builtin_amdgcn_sched_barrier(0);
        // only tiles on an edge of the band (or past the end of the sequence) need the element-wise mask: a pair that
        // does not take part gets P = dS = 0 whatever its scores hold.  A tile that another owner tile of the workgroup
        // needs and this one does not goes through the same code (a branch around it would have the accumulators copied),
        // with operands that are zero: no infinity of its rows meets a zero weight
        if (t < ti_first || t > ti_last) {
            const int off = t * 32 + 8 * g - lo;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const bool ok = (unsigned)(off + key_of(0, i)) <= (unsigned)span;
                s[i] = ok ? s[i] : dead;
                dp[i] = ok ? dp[i] : 0.f;
            }
            if (t < tw_first || t > tw_last) {
                const v8 zero = {};
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk) {
                        ta[dt][kk] = zero;
                        if constexpr (COL) tb2[dt][kk] = zero;
                    }
            }
        }
        v8 pa[2], da[2];
        auto softmax_pair = [&](int r) {  // elements 2 r, 2 r + 1: P and dS = P (dP - Delta), packed to 16 bit
            const int h = r >> 2, e = 2 * (r & 3), i = h * 8 + e;
            const float p0 = fast_exp2(fmaf(s[i], scale, own_term)), p1 = fast_exp2(fmaf(s[i + 1], scale, own_term));
            const float d0 = p0 * dp[i], d1 = p1 * dp[i + 1];
            const v2 dd = M::pack(d0, d1);
            da[h][e] = dd[0]; da[h][e + 1] = dd[1];
            if constexpr (COL) {
                const v2 pp = M::pack(p0, p1);
                pa[h][e] = pp[0]; pa[h][e + 1] = pp[1];
            }
            if constexpr (LINK) { db += d0; db += d1; }
        };
        // dX^T[d][r] += K^T[d][a] dS^T[a][r]  |  dK^T[d][a] += X^T[d][r] dS[r][a],  dV^T[d][a] += dO^T[d][r] P[r][a]
        auto product = [&](int kk, int j) {
            if constexpr (COL) {
                if (j & 1) accb[j >> 1] = M::mma(tb2[j >> 1][kk], pa[kk], accb[j >> 1]);
                else acca[j >> 1] = M::mma(ta[j >> 1][kk], da[kk], acca[j >> 1]);
            } else acca[j] = M::mma(ta[j][kk], da[kk], acca[j]);
        };
        constexpr int NP = COL ? 2 * DT : DT;  // products per half
#pragma unroll
        for (int r = 0; r < 4; ++r) softmax_pair(r);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (NP == 4) product(0, r);
            else if (NP == 2 && (r & 1) == 0) product(0, r >> 1);
            else if (NP == 1 && r == 0) product(0, 0);
            __builtin_amdgcn_sched_barrier(0);
            softmax_pair(4 + r);
            __builtin_amdgcn_sched_barrier(0);
        }
        cross();
        load_rows(next);  // (the last step reads a slot nobody needs)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NP; ++j) product(1, j);
        __builtin_amdgcn_sched_barrier(0);
        t += kSH;
    };
    for (int u = 0; u < steps; u += NS) {  // a step per ring slot: the slots' addresses are constants
        step(std::integral_constant<int, 0>{});
        if (u + 1 < steps) step(std::integral_constant<int, 1>{});
        if (u + 2 < steps) step(std::integral_constant<int, 2>{});
        if (u + 3 < steps) step(std::integral_constant<int, 3>{});
    }
    barrier_keep_loads<0>();  // every stage has landed and been read: the ring becomes the merge tiles

    // ---- join the kSH shares of every owner tile: thread (rr, owner tile mo, dg) takes 16-byte pieces dg, dg + 2 kSH, ... of a row
    float* sO = reinterpret_cast<float*>(smem_raw);  // [kW][D][kLdr]
    float* sB = sO + kW * D * kLdr;                  // [kW][32]     dbias shares
    float* sR = sB + kW * 32;                        // [2 kW][32]   delta1 partials
    const int rr = tid & 31, mo = (tid >> 5) % kOT, dg = (tid >> 5) / kOT, row = o0 + 32 * mo + rr;
    auto joined = [&](int d) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < kSH; ++w) v += sO[((w * kOT + mo) * D + d) * kLdr + rr];
        return v;
    };
    if constexpr (!COL) {
        spill_tiles<D>(sO, wave, acca, n, g);
        __syncthreads();
        if (row >= T) return;
#pragma unroll
        for (int c = dg; c < D / 8; c += 2 * kSH) {
            const int d0 = 8 * c;
            const size_t off = base + (size_t)row * D + d0;
            v8 ov;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                float v = joined(d0 + j) * p.alpha;
                if (p.addend) v += p.addend[off + j];
                ov[j] = (E)v;
            }
            *reinterpret_cast<v8*>(p.dx + off) = ov;
        }
    } else {
        if constexpr (LINK) {
            db += __shfl_xor(db, 32, 64);
            if (g == 0) sB[wave * 32 + n] = db;
        }
        spill_tiles<D>(sO, wave, acca, n, g);
        __syncthreads();
        if (row < T) {
#pragma unroll
            for (int c = dg; c < D / 8; c += 2 * kSH) {
                const int d0 = 8 * c;
                const size_t off = base + (size_t)row * D + d0;
                float o[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = joined(d0 + j) * p.alpha;
                if constexpr (LINK) {
                    *reinterpret_cast<float4*>(p.dk_f32 + off) = make_float4(o[0], o[1], o[2], o[3]);
                    *reinterpret_cast<float4*>(p.dk_f32 + off + 4) = make_float4(o[4], o[5], o[6], o[7]);
                } else {
                    v8 ov;
#pragma unroll
                    for (int j = 0; j < 8; ++j) ov[j] = (E)o[j];
                    *reinterpret_cast<v8*>(p.dk + off) = ov;
                }
            }
        }
        __syncthreads();
        spill_tiles<D>(sO, wave, accb, n, g);
        __syncthreads();
        [[maybe_unused]] float part = 0.f;
#pragma unroll
        for (int c = dg; c < D / 8; c += 2 * kSH) {
            const int d0 = 8 * c;
            const size_t off = base + (size_t)row * D + d0;
            if constexpr (!LINK) {
                if (row < T) {
                    const v8 x = ld8<E>(p.v1.row(at, row, T, D) + d0);
                    v8 ov;
#pragma unroll
                    for (int j = 0; j < 8; ++j) ov[j] = (E)(joined(d0 + j) * silu_grad_f((float)x[j]));
                    *reinterpret_cast<v8*>(p.dv + off) = ov;
                }
            } else if (row < Tp) {
                v8 dv2, dr;
#pragma unroll
                for (int j = 0; j < 8; ++j) dr[j] = (E)0.f;
                if (row < T) {
                    const v8 x = ld8<E>(p.v2.row(at, row, T, D) + d0);
                    const float4 r0 = *reinterpret_cast<const float4*>(p.r_f32 + off);
                    const float4 r1 = *reinterpret_cast<const float4*>(p.r_f32 + off + 4);
                    const float rv[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const float o = joined(d0 + j), drj = o * (float)x[j];
                        dv2[j] = (E)(o * rv[j]);
                        dr[j] = (E)drj;
                        part += drj * rv[j];
                    }
                    *reinterpret_cast<v8*>(p.dv2 + off) = dv2;
                    *reinterpret_cast<v8*>(p.dr + off) = dr;
                }
                *reinterpret_cast<v8*>(p.dr_p1 + tb + p1_index<D>(row, d0)) = dr;  // zeros for the padding rows
            }
        }
        if constexpr (LINK) {
            // -delta1 = dbias - rowsum(dR R)
            sR[(mo * 2 * kSH + dg) * 32 + rr] = part;
            __syncthreads();
            if (dg == 0 && row < Tp) {
                float d1 = 0.f;
#pragma unroll
                for (int j = 0; j < 2 * kSH; ++j) d1 -= sR[(mo * 2 * kSH + j) * 32 + rr];
#pragma unroll
                for (int w = 0; w < kSH; ++w) d1 += sB[(w * kOT + mo) * 32 + rr];
                p.delta1[vb + row] = row < T ? d1 : 0.f;
            }
        }
    }
}

// The outer column pass: dK2 (its share), and through the link dV2, dR, delta1 that the inner passes stream.
template <typename E, int D, int kOT, int kSH, bool SV>
__global__ __launch_bounds__(256, 2) void attn_bwd_link_kernel(AttnBwdP<E, SV> outer) {
    // Two workgroups fit a CU (D = 32: three).  A grid that is resident at once is not levelled by the order of its workgroups: the
    // second one that a CU gets (slots 32 .. of an XCD) is then the lighter, the heavier the first.  The backward with and without,
    // bf16: B=4 H=8 T=1024 79.3 / 80.6 us, B=3 H=8 T=1300 k_diff 300 80.2 / 82.2; at D = 32 49.8 / 50.1 and 50.9 / 51.1.
    const int n_owner = (outer.Tp / 32 + kOT - 1) / kOT, slots = xcd_slots(outer.BH, n_owner);
    int bh, tile, slot = blockIdx.x >> 3;
    if (slots <= 64 && slot >= 32) slot = slots - 1 - (slot - 32);
    if (!xcd_tile(outer.BH, n_owner, slot, blockIdx.x & 7, bh, tile)) return;
    attn_bwd_tiles_body<E, D, kOT, kSH, true, false, true, false, SV>(outer, bh, tile);
}
// The other three passes depend on nothing of each other: outer rows (dQ), inner rows (dK2) and inner columns (dK1, dV1) in one grid.
template <typename E, int D, int kOT, int kSH, bool SV>
__global__ __launch_bounds__(256, 2) void attn_bwd_rest_kernel(AttnBwdP<E, SV> outer, AttnBwdP<E, SV> inner) {
    int bh, tile;
    const int slot = blockIdx.x >> 3, pass = slot % 3;
    if (!xcd_tile(outer.BH, (outer.Tp / 32 + kOT - 1) / kOT, slot / 3, blockIdx.x & 7, bh, tile)) return;
    if (pass == 0) attn_bwd_tiles_body<E, D, kOT, kSH, false, true, false, false, SV>(outer, bh, tile);
    else if (pass == 1) attn_bwd_tiles_body<E, D, kOT, kSH, true, false, false, true, SV>(inner, bh, tile);
    else attn_bwd_tiles_body<E, D, kOT, kSH, false, false, false, false, SV>(inner, bh, tile);
}
