// pf16_w8_kernel.h -- the INT8 GEMM for few output tiles: independent waves of
// 16 rows by one 16-column tile.
#pragma once

#include "qmm_common.h"

namespace bq {

// Bound: one wave's chain per block (two matrix instructions, sixteen
// dependent vector instructions) and the CU's vector memory issue.  Weights
// are the matrix operand as they lie in memory and records are written in
// operand order (r16_rec_bytes), so a block is three 1 KB loads a wave (its half of
// the weight chunk and of its sums and scales among them) and there is no LDS
// and no barrier.  The workgroups of prefill_kernel (32 RP rows) leave most
// CUs without one here.
template <bool HP, int SCM>
__global__ __launch_bounds__(kPf16Waves * 64, 4) void pf16_w8_kernel(PfArgs a, int row_waves) {
    constexpr int PD = 4;  // chunks (two blocks) in flight
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // The row tiles of a column tile are neighbouring waves: they share the
    // weights through the caches.
    const int id = blockIdx.x * kPf16Waves + wave;
    const int tile = id / row_waves, rt = id - tile * row_waves;
    if (tile >= a.ntiles) return;
    const int c16 = lane & 15, q4 = lane >> 4;
    const int nch = a.nch;

    struct Chunk {
        uint4 w, a0, a1;
        float2 sa;
        int2 ws;
        float2 sc;
    };
    const char* wp = a.W + (size_t)tile * nch * 1024 + 16 * lane;
    const char* wsp = a.WS + (size_t)tile * nch * 128 + 8 * c16;
    const char* sp = SCM == 2 ? a.S + (size_t)tile * nch * 128 + 8 * c16 : a.S + (size_t)tile * a.ngrp * 64 + 4 * c16;
    const char* rec = a.R + (size_t)rt * nch * r16_rec_bytes(HP);
    const uint32_t lane16 = 16 * lane, lane8 = 8 * lane;
    const float sc0 = *reinterpret_cast<const float*>(sp);
    auto load = [&](Chunk& k, int c) __attribute__((always_inline)) {
        const size_t cc = uniform_offset((uint32_t)min(c, nch - 1));
        k.w = *reinterpret_cast<const uint4*>(wp + cc * 1024);
        const char* r = rec + cc * r16_rec_bytes(HP);
        k.a0 = *reinterpret_cast<const uint4*>(r + lane16);
        if (HP) k.a1 = *reinterpret_cast<const uint4*>(r + 1024 + lane16);
        k.sa = *reinterpret_cast<const float2*>(r + (HP ? 2048 : 1024) + lane8);
        if (HP) k.ws = *reinterpret_cast<const int2*>(wsp + cc * 128);
        if (SCM == 2) {
            k.sc = *reinterpret_cast<const float2*>(sp + cc * 128);
        } else if (SCM == 1) {
            const size_t g = uniform_offset((uint32_t)(2 * cc) >> a.sc_shift);
            k.sc.x = k.sc.y = *reinterpret_cast<const float*>(sp + g * 64);
        } else {
            k.sc.x = k.sc.y = sc0;
        }
    };

    v4f acc = {};
    v4i dp = {0, 0, 0, 0};
    float sap = 0.0f, scp = 0.0f;
    auto epi = [&]() __attribute__((always_inline)) {
        fma_rows4(acc, sap, v4f{(float)dp[0] * scp, (float)dp[1] * scp, (float)dp[2] * scp, (float)dp[3] * scp});
    };
    auto u64 = [](uint32_t lo, uint32_t hi) __attribute__((always_inline)) { return (uint64_t)hi << 32 | lo; };
    // One block: cs = 256 H + L + 128 S (two-pass), then the previous block's
    // epilogue behind the matrix instructions.
    auto block = [&](uint64_t ah, uint64_t al, uint64_t b, int s128, float sa, float sc) __attribute__((always_inline)) {
        v4i d = mfma16(ah, b);
        epi();
        if (HP) {
            const v4i ci = {(d[0] << 8) + s128, (d[1] << 8) + s128, (d[2] << 8) + s128, (d[3] << 8) + s128};
            d = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)al, (long)b, ci, 0, 0, 0);
        }
        dp = d;
        sap = sa;
        scp = sc;
    };
    auto block0 = [&](const Chunk& k) __attribute__((always_inline)) {
        block(u64(k.a0.x, k.a0.y), u64(k.a0.z, k.a0.w), u64(k.w.x, k.w.y), k.ws.x, k.sa.x, k.sc.x);
    };
    auto block1 = [&](const Chunk& k) __attribute__((always_inline)) {
        if (HP) block(u64(k.a1.x, k.a1.y), u64(k.a1.z, k.a1.w), u64(k.w.z, k.w.w), k.ws.y, k.sa.y, k.sc.y);
        else block(u64(k.a0.z, k.a0.w), 0, u64(k.w.z, k.w.w), 0, k.sa.y, k.sc.y);
    };

    Chunk ring[PD];
#pragma unroll
    for (int i = 0; i < PD; ++i) load(ring[i], i);
    const int nfull = a.nblk >> 1;  // whole chunks
    int c = 0;
    for (; c + PD <= nfull; c += PD) {
#pragma unroll
        for (int i = 0; i < PD; ++i) {
            block0(ring[i]);
            block1(ring[i]);
            load(ring[i], c + i + PD);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int i = 0; i < PD; ++i) {
        if (c + i < nfull) {
            block0(ring[i]);
            block1(ring[i]);
        } else if (c + i == nfull && (a.nblk & 1)) {
            block0(ring[i]);  // the last, odd block
        }
    }
    epi();
    const int n = tile * 16 + c16;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int m = 16 * rt + 4 * q4 + j;
        if (m < a.M) a.C[(size_t)m * a.N + n] = acc[j];
    }
}

}  // namespace bq
