// pf16_kernel.h -- the INT4 GEMM for few output tiles on the scaled FP6 matrix
// instructions: independent waves of 16 rows by one 16-column tile.
#pragma once

#include "qmm_common.h"

namespace bq {

// Bound: with up to a few waves a SIMD, one wave's chain per block (an operand
// read, the matrix instruction, eight dependent vector instructions) and the
// CU's vector memory issue (16 cycles per 1 KB load: a record is two, a chunk
// of weights one per four blocks).  A tile of 32 rows by 32 columns a wave
// (pf4_kernel) needs a quarter of the loads but leaves most SIMDs without a
// wave: K=5120 N=5120 takes 46 us at 64 rows there and 29 here, 61 on the
// INT8 matrix instructions (record quantizer included).
//
// No barriers: a wave expands its own weights in its own LDS.  AHEAD chunks
// of weights are in flight in registers: four while the waves are few, two
// past that (107 registers, 110 with zero points: four waves a SIMD).
constexpr int kPf16Stage = 2048;  // LDS of one stage (four blocks) of a wave: 64 operands of 32 B

template <bool ZP, int AHEAD>
__global__ __launch_bounds__(kPf16Waves * 64, AHEAD == 2 ? 4 : 3) void pf16_kernel(Pf4Args a, int row_waves) {
    __shared__ __align__(16) char pf16_lds[kPf16Waves * 2 * kPf16Stage];
    static_assert(AHEAD % 2 == 0, "a register slot keeps its buffer's parity");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // The row tiles of a column tile are neighbouring waves: they share the
    // weights through the caches.
    const int id = blockIdx.x * kPf16Waves + wave;
    const int tile = id / row_waves, rt = id - tile * row_waves;
    if (tile >= a.ntiles) return;
    char* lds = pf16_lds + wave * 2 * kPf16Stage;
    const int c16 = lane & 15, q4 = lane >> 4;
    const int nst = a.nbg;
    const int sk = a.find(tile), st = tile - a.first(sk);  // segment, and the tile within it
    const Pf4Seg& sg = a.seg[sk];

    // Weights: after the transpose, lane (column c16, block q4) of the chunk.
    uint4 raw[AHEAD];
    float rsc[AHEAD];
    int rzp[AHEAD];
    const gptr wp = uniform_ptr(sg.W + (size_t)st * a.nbg * 1024);
    const gptr sp = uniform_ptr(sg.S + (size_t)st * a.s_tile);
    const uint32_t soff = a.s_col * c16 + a.s_blk * q4;
    const gptr zpp = ZP ? uniform_ptr(sg.Z + (size_t)st * a.nbg * 64) : nullptr;
    auto load_raw = [&](int r, int g) __attribute__((always_inline)) {
        const int gc = min(g, nst - 1);
        raw[r] = __builtin_bit_cast(uint4, gload<v4u>(wp + (size_t)uniform_offset((uint32_t)gc) * 1024 + (uint32_t)(16 * lane)));
        rsc[r] = gload<float>(sp + (size_t)uniform_offset((uint32_t)((4 * gc) >> a.sc_shift)) * a.s_grp + soff);
        if (ZP) rzp[r] = gload<int8_t>(zpp + (size_t)uniform_offset((uint32_t)gc) * 64 + (uint32_t)(4 * c16 + q4));
    };
    auto expand = [&](int r, char* eb) __attribute__((always_inline)) {
        uint32_t w[4], d[6];
        octets_of_block(raw[r], w);
        f6_pack(w, d);
        char* p = eb + q4 * 512 + c16 * 16;
        *reinterpret_cast<uint4*>(p) = make_uint4(d[0], d[1], d[2], d[3]);
        *reinterpret_cast<uint4*>(p + 256) =
            make_uint4(d[4], d[5], __float_as_uint(rsc[r]), ZP ? __float_as_uint((float)rzp[r]) : 0u);
    };

    // Activations.
    struct Rows {
        v8i a;
        float sa, nq;
    };
    const char* rec = a.R + (size_t)rt * a.nblk * kF6Rec + 16 * lane;
    auto load_rows = [&](Rows& f, int blk) __attribute__((always_inline)) {
        const char* q = rec + (size_t)uniform_offset((uint32_t)min(blk, a.nblk - 1)) * kF6Rec;
        const uint4 x = *reinterpret_cast<const uint4*>(q);
        const uint4 y = *reinterpret_cast<const uint4*>(q + kF6Plane);
        f.a = v8i{(int)x.x, (int)x.y, (int)x.z, (int)x.w, (int)y.x, (int)y.y, 0, 0};
        f.sa = __uint_as_float(y.z);
        f.nq = __uint_as_float(y.w);
    };

    const int sca = 127 + 3 + 4 * q4, scb = 127 + 3;  // digit i weighs 16^i; codes are value / 8
    v4f acc = {}, dp = {};
    float sap = 0.0f, nqp = 0.0f, scp = 0.0f, zp = 0.0f;
    Rows ab[4];  // the stage's blocks; each is reloaded a stage ahead once used
    auto epi = [&]() __attribute__((always_inline)) {
        v4f v = dp;
        if (ZP) {
            v[0] = __builtin_fmaf(row_bcast<0>(nqp), zp, v[0]);
            v[1] = __builtin_fmaf(row_bcast<1>(nqp), zp, v[1]);
            v[2] = __builtin_fmaf(row_bcast<2>(nqp), zp, v[2]);
            v[3] = __builtin_fmaf(row_bcast<3>(nqp), zp, v[3]);
        }
        fma_rows4(acc, sap, v4f{v[0] * scp, v[1] * scp, v[2] * scp, v[3] * scp});
    };
    const char* bp0 = lds + 16 * c16;
    // Block b of the stage in buffer eb with the rows in f: this block's
    // matrix instruction, then the previous block's epilogue.
    auto block = [&](const char* eb, int b, const Rows& f) __attribute__((always_inline)) {
        const uint4 x = *reinterpret_cast<const uint4*>(eb + b * 512);
        const uint4 y = *reinterpret_cast<const uint4*>(eb + b * 512 + 256);
        const v8i bq = v8i{(int)x.x, (int)x.y, (int)x.z, (int)x.w, (int)y.x, (int)y.y, 0, 0};
        v4f c = {};
        if (!ZP) c = v4f{row_bcast<0>(f.nq), row_bcast<1>(f.nq), row_bcast<2>(f.nq), row_bcast<3>(f.nq)};
        const v4f d = mfma_f6_16(f.a, bq, c, sca, scb);
        epi();
        dp = d;
        sap = f.sa;
        scp = __uint_as_float(y.z);
        if (ZP) {
            nqp = f.nq;
            zp = __uint_as_float(y.w);
        }
    };

#pragma unroll
    for (int r = 0; r < AHEAD; ++r) load_raw(r, r);
#pragma unroll
    for (int b = 0; b < 4; ++b) load_rows(ab[b], b);
    expand(0, lds);
    load_raw(0, AHEAD);
    const int nfull = a.nblk >> 2;
    // Stage g computes from buffer g & 1 while the next stage's weights (in
    // register slot (g + 1) % AHEAD) are expanded into the other.  A wave's
    // own LDS accesses stay in order.
    auto stage = [&](int g, int r) __attribute__((always_inline)) {
        const char* eb = bp0 + (r & 1) * kPf16Stage;
        const int rn = (r + 1) % AHEAD;
        expand(rn, lds + ((r & 1) ^ 1) * kPf16Stage);
        load_raw(rn, g + 1 + AHEAD);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            block(eb, b, ab[b]);
            load_rows(ab[b], 4 * (g + 1) + b);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int g = 0;
    for (; g + AHEAD <= nfull; g += AHEAD) {
#pragma unroll
        for (int r = 0; r < AHEAD; ++r) stage(g + r, r);
    }
#pragma unroll
    for (int r = 0; r + 1 < AHEAD; ++r)
        if (g + r < nfull) stage(g + r, r);
    // The last one to three blocks.
    for (int b = 4 * nfull; b < a.nblk; ++b) {
        load_rows(ab[0], b);
        block(bp0 + (nfull & 1) * kPf16Stage, b & 3, ab[0]);
    }
    epi();
    const int n = st * 16 + c16;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int m = 16 * rt + 4 * q4 + j;
        if (m < a.M) sg.C[(size_t)m * sg.N + n] = acc[j];
    }
}

}  // namespace bq
