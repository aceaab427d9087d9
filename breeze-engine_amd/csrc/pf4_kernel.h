// pf4_kernel.h -- the INT4 prefill GEMM on the scaled FP6 matrix instructions, and
// its launcher, instantiated per activation mode by pf_w4_{hp,lp}.hip.
#pragma once

#include "qmm_common.h"

namespace bq {

// Bound: VALU and MFMA issue.  A step (a block's 32 rows by 32 columns) is two
// matrix instructions (18 ns each on one SIMD) and 32 vector instructions
// (24 ns with two waves issuing); on this GPU the two overlap little, and a
// copy of the compute alone takes 74-85 ns a step whatever the order of its
// instructions, 120 us at K=5120 N=17408 and 512 rows.  The call takes 161
// there, 5 of them the record quantizer: operand loads (vector memory issue,
// 16 cycles of the CU per 1 KB load), the expansion of the weights and the
// stores (4 us a round, the rate that memory takes writes at) add the rest.
// On INT8 matrix instructions (64 vector instructions a step) it took 209.
//
// Split: wave (rp, part) takes 32 rows and its part of the workgroup's column
// groups.  The rows' operands go from L2 straight to registers, reused over
// the wave's groups (through LDS they would cost as much as the weights do);
// weights are expanded once a workgroup, through LDS, a stage (four blocks)
// ahead.  Every load has a stage to land: loads complete in order, so a short
// prefetch of the rows would wait for the weights' latency (163 us against
// 176 with the rows one block ahead).
//
// The row scale enters as a DPP operand (fma_rows8): one register instead of
// 16 a block.

// One block's A operands of a wave (32 rows): the base-16 digits of q, two
// digits a matrix instruction.
template <bool HP>
struct F6Rows {
    v8i a0, a1;
};

template <bool HP, bool ZP, int CT, int RP>
__global__ __launch_bounds__((Pf4Shape<CT, RP>::kThreads)) void pf4_kernel(Pf4Args a) {
    using L = Pf4Shape<CT, RP>;
    extern __shared__ __align__(16) char pf4_lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int rp = wave % RP, part = wave / RP;
    const int t0 = blockIdx.x * CT;
    const int rpair = blockIdx.y * RP + rp;
    const bool active = rpair * 32 < a.M;
    const int nst = a.nbg;
    const int c32 = lane & 31, kh = lane >> 5;

    // ---- weights: lane (column ec, block ej) of a tile's chunk
    const int ec = lane & 15, ej = lane >> 4;
    // TPW tile slots a wave, and one more for CT % kWaves waves: the first, or,
    // where these are all (five tiles), the last, whose part has fewer column
    // groups (K=5120 N=17408, 128 rows, INT8 activations 67.0 -> 63.4 us).
    constexpr int TPW = CT / L::kWaves, REM = CT % L::kWaves;
    constexpr int SLOTS = TPW + (REM > 0), REM0 = TPW == 0 ? L::kWaves - REM : 0;
    const bool has_rem = wave >= REM0 && wave < REM0 + REM;
    // The tile of slot i (the last slot of a wave without one: any tile).
    auto slot_tile = [&](int i) { return L::kWaves * i + (i < TPW ? wave : max(wave - REM0, 0)); };
    uint4 raw[SLOTS];
    float rsc[SLOTS];
    int rzp[SLOTS];
    const uint32_t soff = a.s_col * ec + a.s_blk * ej;
    // The tile slots' weights (scales, zero points).
    gptr wt[SLOTS], stp[SLOTS], zt[SLOTS];
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
        const int t = min(t0 + slot_tile(i), a.ntiles - 1), k = a.find(t);
        const size_t ts = t - a.first(k);
        wt[i] = uniform_ptr(a.seg[k].W + ts * a.nbg * 1024);
        stp[i] = uniform_ptr(a.seg[k].S + ts * a.s_tile);
        zt[i] = ZP ? uniform_ptr(a.seg[k].Z + ts * a.nbg * 64) : nullptr;
    }
    auto load_raw = [&](int i, int g) __attribute__((always_inline)) {
        const uint32_t gc = (uint32_t)min(g, nst - 1);
        raw[i] = __builtin_bit_cast(uint4, gload<v4u>(wt[i] + (size_t)uniform_offset(gc) * 1024 + (uint32_t)(16 * lane)));
        rsc[i] = gload<float>(stp[i] + (size_t)uniform_offset((4 * gc) >> a.sc_shift) * a.s_grp + soff);
        if (ZP) rzp[i] = gload<int8_t>(zt[i] + (size_t)uniform_offset(gc) * 64 + (uint32_t)(4 * ec + ej));
    };
    // Expands tile slot i of a stage into the operand buffer eb: two 16-byte
    // planes per (column group, block), so sixteen lanes write and read 256
    // contiguous bytes.
    auto expand = [&](int i, char* eb) __attribute__((always_inline)) {
        const int u = slot_tile(i);
        uint32_t w[4], d[6];
        octets_of_block(raw[i], w);
        f6_pack(w, d);
        char* p = eb + (u >> 1) * 4096 + ej * 1024 + ((u & 1) * 16 + ec) * 16;
        *reinterpret_cast<uint4*>(p) = make_uint4(d[0], d[1], d[2], d[3]);
        *reinterpret_cast<uint4*>(p + 512) =
            make_uint4(d[4], d[5], __float_as_uint(rsc[i]), ZP ? __float_as_uint((float)rzp[i]) : 0u);
    };

    // ---- activations
    // Rows r32 = lane & 31 of the row pair, digits kh and 2 + kh.
    const char* rec = a.R + (size_t)rpair * 2 * a.nblk * kF6Rec;
    const uint32_t tile_off = (uint32_t)a.nblk * kF6Rec;  // second 16-row tile
    const uint32_t row_off = (lane & 16 ? tile_off : 0) + 16 * ((lane & 15) + 16 * kh);
    auto load_rows = [&](F6Rows<HP>& f, int blk) __attribute__((always_inline)) {
        const char* q = rec + uniform_offset((uint32_t)min(blk, a.nblk - 1) * kF6Rec);
        const uint4 x0 = *reinterpret_cast<const uint4*>(q + row_off);
        const uint2 y0 = *reinterpret_cast<const uint2*>(q + row_off + kF6Plane);
        f.a0 = v8i{(int)x0.x, (int)x0.y, (int)x0.z, (int)x0.w, (int)y0.x, (int)y0.y, 0, 0};
        if (HP) {
            const uint4 x1 = *reinterpret_cast<const uint4*>(q + row_off + 512);
            const uint2 y1 = *reinterpret_cast<const uint2*>(q + row_off + 512 + kF6Plane);
            f.a1 = v8i{(int)x1.x, (int)x1.y, (int)x1.z, (int)x1.w, (int)y1.x, (int)y1.y, 0, 0};
        }
    };
    // Row scales and sums of a stage's blocks: wave (rp, part) moves blocks
    // part, part + kParts, ... of its row pair to LDS, in the order of a
    // lane's results: result j of half kh is row (j & 3) + 8 (j >> 2) + 4 kh.
    // Lane l takes value l >> 5 (scale or sum) of result l & 15, half
    // (l >> 4) & 1.
    constexpr int MPW = (4 + L::kParts - 1) / L::kParts;
    uint32_t meta[MPW];
    const int mrow = (lane & 3) + 8 * ((lane >> 2) & 3) + 4 * ((lane >> 4) & 1);
    const uint32_t meta_off = (mrow & 16 ? tile_off : 0) + kF6Plane +
                              16 * ((mrow & 3) + 16 * ((mrow >> 2) & 3)) + 8 + 4 * (lane >> 5);
    const uint32_t lane4 = 4 * lane;
    auto load_meta = [&](int g) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MPW; ++i) {
            const int b = min(part + i * L::kParts, 3);
            const char* q = rec + uniform_offset((uint32_t)min(4 * g + b, a.nblk - 1) * kF6Rec);
            meta[i] = *reinterpret_cast<const uint32_t*>(q + meta_off);
        }
    };
    auto store_meta = [&](char* eb) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MPW; ++i) {
            const int b = min(part + i * L::kParts, 3);
            *reinterpret_cast<uint32_t*>(eb + L::kMeta + (b * RP + rp) * 256 + lane4) = meta[i];
        }
    };

    // The stage's blocks; each is reloaded a stage ahead once used.  The first
    // loads go out before the wait for the first weights (K=5120 N=17408, 64
    // rows: 61.7 -> 58.1 us), but not where two runs of column groups share
    // registers that are full: 26 spilled registers become 79 there.
    F6Rows<HP> ab[4];
    constexpr bool kEarlyRows = !HP || L::kGroupRem == 0;
    auto load_first = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < 4; ++b) load_rows(ab[b], b);
    };

    // ---- one wave's column groups
    auto run = [&](auto ng_tag, int g0) {
        constexpr int NG = decltype(ng_tag)::value;
        // Scale exponents: operand codes are value / 8; digit i weighs 16^i.
        const int sc0 = 127 + 3 + 4 * kh, sc1 = sc0 + 8, scb = 127 + 3;
        float acc[NG][16];
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[g][j] = 0.0f;
        v16f dp = {}, ci = {};
        float sap = 0.0f, nqv[16] = {};
        float scp = 0.0f, zp = 0.0f;

        // Epilogue of results 8 H .. 8 H + 7 of the previous step (column group g).
        auto epi = [&](int g, float sv, auto ht) __attribute__((always_inline)) {
            constexpr int H = decltype(ht)::value;
            float f[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                float v = dp[8 * H + j];
                if (ZP) v = __builtin_fmaf(zp, nqv[8 * H + j], v);
                f[j] = v * scp;
            }
            fma_rows8<8 * H>(&acc[g][8 * H], sv, f);
        };
        // The 16 row values of this lane's results (part 0 scales, 1 sums) of
        // block b: uniform over the lanes of a half.
        auto meta_at = [&](const char* eb, int b, int what) __attribute__((always_inline)) {
            return reinterpret_cast<const float4*>(eb + L::kMeta + (b * RP + rp) * 256 + what * 128 + 64 * kh);
        };
        auto read_meta = [&](float (&v)[16], const char* eb, int b, int what) __attribute__((always_inline)) {
            const float4* m = meta_at(eb, b, what);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 x = m[q];
                v[4 * q] = x.x;
                v[4 * q + 1] = x.y;
                v[4 * q + 2] = x.z;
                v[4 * q + 3] = x.w;
            }
        };
        auto read_c = [&](const char* eb, int b) __attribute__((always_inline)) {
            const float4* m = meta_at(eb, b, 1);
            const float4 x = m[0], y = m[1], z = m[2], w = m[3];
            ci = v16f{x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w, z.x, z.y, z.z, z.w, w.x, w.y, w.z, w.w};
        };
        const char* bp0 = pf4_lds + g0 * 4096 + c32 * 16;
        auto read_b = [&](const char* q) __attribute__((always_inline)) {
            const uint4 x = *reinterpret_cast<const uint4*>(q);
            const uint2 y = *reinterpret_cast<const uint2*>(q + 512);
            return v8i{(int)x.x, (int)x.y, (int)x.z, (int)x.w, (int)y.x, (int)y.y, 0, 0};
        };
        // Step (block A, group gg): the previous step's epilogue runs between
        // and behind this step's two matrix instructions.
        auto step = [&](const F6Rows<HP>& A, const v8i& bc, const char* q, int gprev, float sv) __attribute__((always_inline)) {
            v16f d = mfma_f6(A.a0, bc, ci, sc0, scb);
            epi(gprev, sv, std::integral_constant<int, 0>{});
            __builtin_amdgcn_sched_barrier(0);
            if (HP) d = mfma_f6(A.a1, bc, d, sc1, scb);
            epi(gprev, sv, std::integral_constant<int, 1>{});
            dp = d;
            scp = *reinterpret_cast<const float*>(q + 520);
            if (ZP) zp = *reinterpret_cast<const float*>(q + 524);
            __builtin_amdgcn_sched_barrier(0);
        };
        // This lane's row scale (result slot lane & 15) of block b.
        auto read_sa = [&](const char* eb, int b) __attribute__((always_inline)) {
            return *reinterpret_cast<const float*>(eb + L::kMeta + (b * RP + rp) * 256 + 64 * kh + 4 * (lane & 15));
        };
        // One full stage (four blocks) from operand buffer g & 1; the next
        // stage's weights are expanded into the other one.
        auto stage = [&](int g) __attribute__((always_inline)) {
            const char* eb = pf4_lds + (g & 1) * L::kStage;
            const char* bp = bp0 + (g & 1) * L::kStage;
            char* en = pf4_lds + ((g & 1) ^ 1) * L::kStage;
            if (!ZP) read_c(eb, 0);
            v8i bq = read_b(bp);
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const float sa = read_sa(eb, b);
#pragma unroll
                for (int gg = 0; gg < NG; ++gg) {
                    const v8i bc = bq;
                    if (gg + 1 < NG) bq = read_b(bp + (gg + 1) * 4096 + b * 1024);
                    else if (b < 3) bq = read_b(bp + (b + 1) * 1024);
                    step(ab[b], bc, bp + gg * 4096 + b * 1024, gg == 0 ? NG - 1 : gg - 1, gg == 0 ? sap : sa);
                    if (!ZP && gg == NG - 1 && b < 3) read_c(eb, b + 1);
                    if (ZP && gg == 0) read_meta(nqv, eb, b, 1);
                }
                sap = sa;
                load_rows(ab[b], 4 * (g + 1) + b);
                if (b < TPW) {
                    expand(b, en);
                    load_raw(b, g + 2);
                }
                if (b == 3) {
                    store_meta(en);
                    load_meta(g + 2);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // At the stage's end: a branch inside it would split the block of
            // instructions that the pipeline above is scheduled in.
            if (REM > 0 && has_rem) {
                expand(TPW, en);
                load_raw(TPW, g + 2);
            }
        };
        const int nfull = a.nblk >> 2;
        if (!kEarlyRows) load_first();
        for (int g = 0; g < nfull; ++g) {
            stage(g);
            lds_barrier();
        }
        // The last one to three blocks.
        for (int b = 4 * nfull; b < a.nblk; ++b) {
            const char* eb = pf4_lds + (nfull & 1) * L::kStage;
            load_rows(ab[0], b);
            if (!ZP) read_c(eb, b & 3);
            const float sa = read_sa(eb, b & 3);
#pragma unroll
            for (int gg = 0; gg < NG; ++gg) {
                const char* q = bp0 + (nfull & 1) * L::kStage + (b & 3) * 1024 + gg * 4096;
                step(ab[0], read_b(q), q, gg == 0 ? NG - 1 : gg - 1, gg == 0 ? sap : sa);
                if (ZP && gg == 0) read_meta(nqv, eb, b & 3, 1);
            }
            sap = sa;
        }
        epi(NG - 1, sap, std::integral_constant<int, 0>{});
        epi(NG - 1, sap, std::integral_constant<int, 1>{});
        // Stores.  The two tiles of a group have uniform numbers, and what is
        // read of their segments stays in scalar registers: loads and stores
        // share a counter, so a vector load ahead of a store makes it wait for
        // every store before it (K=512 N=17408, 1024 rows: 59.0 -> 48.9 us
        // without).
        const int m0 = rpair * 32 + 4 * kh;
        const bool odd = c32 & 16, whole = rpair * 32 + 32 <= a.M;
        auto column0 = [&](int t, int& n) __attribute__((always_inline)) {
            const int k = a.find(t);
            n = __builtin_amdgcn_readfirstlane(a.seg[k].N);
            return (gfptr)uniform_ptr(a.seg[k].C + (t - a.first(k)) * 16);
        };
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int ct = 2 * (g0 + g), t = t0 + ct;
            int na, nb;
            const gfptr ca = column0(min(t, a.ntiles - 1), na), cb = column0(min(t + 1, a.ntiles - 1), nb);
            const ptrdiff_t n = odd ? nb : na;
            gfptr c = (odd ? cb : ca) + (c32 & 15) + m0 * n;
            if (ct + odd >= CT || t + odd >= a.ntiles) continue;
            if (whole) {
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    *c = acc[g][j];
                    c += (j & 3) == 3 ? 5 * n : n;
                }
            } else {
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    if (m0 + (j & 3) + 8 * (j >> 2) < a.M) *c = acc[g][j];
                    c += (j & 3) == 3 ? 5 * n : n;
                }
            }
        }
    };

    const int nfull = a.nblk >> 2;
    // Stage g's tiles are expanded during stage g - 1, from registers loaded a
    // stage earlier still.
    auto expand_all = [&](int g, char* eb) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            expand(i, eb);
            load_raw(i, g + 1);
        }
        if (REM > 0 && has_rem) {
            expand(TPW, eb);
            load_raw(TPW, g + 1);
        }
    };
#pragma unroll
    for (int i = 0; i < TPW; ++i) load_raw(i, 0);
    if (REM > 0 && has_rem) load_raw(TPW, 0);
    if (active) {
        load_meta(0);
        if (kEarlyRows) load_first();
    }
    expand_all(0, pf4_lds);
    if (active) {
        store_meta(pf4_lds);
        load_meta(1);
    }
    lds_barrier();
    if (!active) {
        // A wave past the last row only expands its tiles.
        for (int g = 0; g < nfull; ++g) {
            expand_all(g + 1, pf4_lds + ((g & 1) ^ 1) * L::kStage);
            lds_barrier();
        }
        return;
    }
    if constexpr (L::kGroupRem > 0) {
        if (part < L::kGroupRem) {
            run(std::integral_constant<int, L::kGroupBase + 1>{}, part * (L::kGroupBase + 1));
            return;
        }
    }
    run(std::integral_constant<int, L::kGroupBase>{}, part * L::kGroupBase + L::kGroupRem);
}

template <bool HP, bool ZP, int CT, int RP>
hipError_t launch_pf4_t(bool* attr, const Pf4Args& p, dim3 grid, hipStream_t st) {
    using L = Pf4Shape<CT, RP>;
    auto kern = pf4_kernel<HP, ZP, CT, RP>;
    int slot = 0;
    while (kPfCfgs[slot].rp != RP || kPfCfgs[slot].ct != CT) ++slot;
    const int key = 128 | (HP ? 1 : 0) | (ZP ? 2 : 0) | slot << 3;
    if (!attr[key]) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 2 * L::kStage);
        if (e != hipSuccess) return e;
        attr[key] = true;
    }
    kern<<<grid, L::kThreads, 2 * L::kStage, st>>>(p);
    return hipGetLastError();
}

template <bool HP, bool ZP>
hipError_t launch_pf4_zp(bool* attr, const Pf4Args& p, int rp, int ct, dim3 grid, hipStream_t st) {
    switch (rp * 100 + ct) {
        case 417: return launch_pf4_t<HP, ZP, 17, 4>(attr, p, grid, st);
        case 416: return launch_pf4_t<HP, ZP, 16, 4>(attr, p, grid, st);
        case 413: return launch_pf4_t<HP, ZP, 13, 4>(attr, p, grid, st);
        case 412: return launch_pf4_t<HP, ZP, 12, 4>(attr, p, grid, st);
        case 409: return launch_pf4_t<HP, ZP, 9, 4>(attr, p, grid, st);
        case 408: return launch_pf4_t<HP, ZP, 8, 4>(attr, p, grid, st);
        case 405: return launch_pf4_t<HP, ZP, 5, 4>(attr, p, grid, st);
        case 404: return launch_pf4_t<HP, ZP, 4, 4>(attr, p, grid, st);
        case 216: return launch_pf4_t<HP, ZP, 16, 2>(attr, p, grid, st);
        case 208: return launch_pf4_t<HP, ZP, 8, 2>(attr, p, grid, st);
        case 204: return launch_pf4_t<HP, ZP, 4, 2>(attr, p, grid, st);
        case 116: return launch_pf4_t<HP, ZP, 16, 1>(attr, p, grid, st);
        case 108: return launch_pf4_t<HP, ZP, 8, 1>(attr, p, grid, st);
        default: return hipErrorInvalidValue;
    }
}

template <bool HP>
hipError_t launch_pf4(bool* attr, const Pf4Args& p, bool zp, int rp, int ct, dim3 grid, hipStream_t st) {
    return zp ? launch_pf4_zp<HP, true>(attr, p, rp, ct, grid, st)
              : launch_pf4_zp<HP, false>(attr, p, rp, ct, grid, st);
}

}  // namespace bq
