// nslm_mv_dev.h - device pieces of the seed matvec shared by the stand-alone kernels (nslm_mv.hip) and the fused MoE
// decode kernel (nslm_fused.hip): a chunk's records, the chunk x activations product, the generic block decoder.
#pragma once
#include "nslm_dev.h"

namespace nslm {

struct Chunk {
    uint4 sd, cw;
    uint32_t codes;
};

// A chunk's records: 16 bytes of seeds, 16 of coefficient (nibble) words, 4 of exponent codes.  The streams of a slice may start
// at any 2-byte (codes: 1-byte) boundary - the loads are typed with that alignment, and the target reads a misaligned
// unit in one instruction all the same - so there is one code path and no branch on the alignment.  The loads are
// unconditional (callers clamp `unit` to a chunk that exists): after a load under a condition the compiler no longer knows how
// many loads are in flight and waits for all of them before the next use of any loaded value - the activations' staging then
// waited for the records.
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32_a1 __attribute__((aligned(1)));
template <int P>
__device__ __forceinline__ Chunk load_chunk(const WSlice& w, uint32_t unit) {
    Chunk c;
    c.codes = 0;
    // In pieces, in the order the blocks are decoded - the codes, then seeds and coefficient words of blocks 0..3, then of blocks
    // 4..7: a wave's loads return in the order they went out, and so do the whole launch's requests to the memory, so when every
    // wave asks for its records at once the first pieces of all of them arrive before any last piece does.  A thread starts
    // on its first blocks when 20 of its 36 bytes are there.
    typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
    const NSLM_GLOBAL uint8_t* ps = gp<uint8_t>(w.p[0]) + (size_t) unit * 16;
    const NSLM_GLOBAL uint8_t* pc = gp<uint8_t>(w.p[1]) + (size_t) unit * 16;
    if (P == 4) c.codes = *(const NSLM_GLOBAL u32_a1*) (gp<uint8_t>(w.p[3]) + (size_t) unit * 4);
    const u32x2_a2 s0 = *(const NSLM_GLOBAL u32x2_a2*) ps, c0 = *(const NSLM_GLOBAL u32x2_a2*) pc;
    asm volatile("" ::: "memory");   // (keeps the halves apart: left alone, the compiler joins them into 16-byte loads again)
    const u32x2_a2 s1 = *(const NSLM_GLOBAL u32x2_a2*) (ps + 8), c1 = *(const NSLM_GLOBAL u32x2_a2*) (pc + 8);
    c.sd = make_uint4(s0.x, s0.y, s1.x, s1.y);
    c.cw = make_uint4(c0.x, c0.y, c1.x, c1.y);
    return c;
}
__device__ __forceinline__ bool streams_aligned(int P, const WSlice& w) {
    return (((uintptr_t) w.p[0] | (uintptr_t) w.p[1]) & 15u) == 0 && (P != 4 || ((uintptr_t) w.p[3] & 3u) == 0);
}

__device__ __forceinline__ uint32_t word_of(const uint4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// ---- activations as the matvec reads them: in LDS, LDS floats per 64-weight chunk (8 blocks + 4): 16-byte reads of 8 consecutive lanes land on 32
// distinct banks (68 is 4 mod 32) ----
#define XPAD 68
// block `blk` of a row into its place of a chunk-padded LDS row
__device__ __forceinline__ void store_block(float* row, int blk, const float (&x)[8]) {
    float* dst = row + (blk >> 3) * XPAD + (blk & 7) * 8;
    *(float4*) dst = make_float4(x[0], x[1], x[2], x[3]);
    *(float4*) (dst + 4) = make_float4(x[4], x[5], x[6], x[7]);
}

// Block b of a chunk: its weights as isum 2^-22 and the block's scale 2^(eb + code); ebase: sums_e2 of the slice
template <int P>
__device__ __forceinline__ float block_of(const Chunk& ck, int b, uint32_t ebase, const uint32_t* tab, float (&w)[8]) {
    const uint32_t ss = word_of(ck.sd, b >> 1), cc = word_of(ck.cw, b >> 1);
    const uint32_t g = stream_of(tab, (b & 1) ? ss >> 16 : ss & 0xFFFFu);
    const SumCoefs sc = sum_coefs<P>(cc, b & 1, tab + 512 + sum_tab_at<P>(cc, b & 1));
    uint32_t y[8];
    sums_of<P>((b & 1) ? ss : ss << 16, g, sc, y, [](int) {});
    sums_float<P>(y, sc.k, w);
    const uint32_t code = P == 4 ? code_of<P>(ck.codes, b) : code_of<P>(cc, 4 * (b & 1));
    return __uint_as_float((code << 23) + ebase);
}
// a block's products with 8 activations, in order.  REGS: they are in registers, else in LDS
template <bool REGS = false>
__device__ __forceinline__ float block_dot(const float (&w)[8], const float* xb) {
    float x[8];
    if constexpr (REGS) {
#pragma unroll
        for (int c = 0; c < 8; ++c) x[c] = xb[c];
    } else {
        const float4 a = *(const float4*) xb, b = *(const float4*) (xb + 4);
        x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w; x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
    }
    float d = w[0] * x[0];
#pragma unroll
    for (int c = 1; c < 8; ++c) d = fmaf(w[c], x[c], d);
    return d;
}
// One chunk (8 blocks) against NT tokens.  xr: this chunk's staged activations, token t at xr + t * xstride (registers when
// NT == 1 and the caller copied them, LDS otherwise).  acc[t] accumulates 2^e * (block . x) per block (NSLM_SUM_R32 is applied to the row sum).
template <int P, int NT, bool REGS = false>
__device__ __forceinline__ void chunk_dot(const Chunk& ck, int eb, const uint32_t* tab, const float* xr, int xstride, float (&acc)[NT]) {
    const uint32_t ebase = sums_e2(eb);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        float w[8];
        const float e2 = block_of<P>(ck, b, ebase, tab, w);
        // Every token of the pass is computed (rows past its tokens hold whatever the LDS holds; their sums are never stored):
        // an early exit on the run-time count would make each token's LDS reads wait for the one before.
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = fmaf(block_dot<REGS>(w, xr + t * xstride + 8 * b), e2, acc[t]);
    }
}
// The same in two halves, for a caller that has a chunk's records before it has the activations: the weights (64 registers), then the products -
// the same operations in the same order, so the same bits.
template <int P>
__device__ __forceinline__ void chunk_pre(const Chunk& ck, const uint32_t* tab, float (&w)[8][8]) {
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        (void) block_of<P>(ck, b, 0u, tab, w[b]);
        __builtin_amdgcn_sched_barrier(0);   // (a block at a time: 64 registers of results leave little room for eight blocks' temporaries)
    }
}
template <int P>
__device__ __forceinline__ void chunk_post(const Chunk& ck, const float (&w)[8][8], int eb, const float* xr, float& acc) {
    const uint32_t ebase = sums_e2(eb);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const uint32_t code = P == 4 ? code_of<P>(ck.codes, b) : code_of<P>(word_of(ck.cw, b >> 1), 4 * (b & 1));
        acc = fmaf(block_dot(w[b], xr + 8 * b), __uint_as_float((code << 23) + ebase), acc);
    }
}

// A chunk's sum by 2^ls adjacent lanes (ls = 1 .. 3), lane s of the group taking blocks [s nb, (s + 1) nb), nb = 8 >> ls: each
// block's product with the activations as chunk_dot forms it, then its chain of multiply-adds over the blocks in block
// order, handed from lane to lane (lane s holds its final value after step s).  The group's last lane returns chunk_dot's bits.  P = 3.
__device__ __forceinline__ float chunk_dot_split(const Chunk& ck, int eb, const uint32_t* tab, const float* xr, int s, int ls) {
    constexpr int P = 3;
    const int nb = 8 >> ls, b0 = s * nb;
    const uint32_t ebase = sums_e2(eb);
    float d[4] = {0.0f, 0.0f, 0.0f, 0.0f}, e2[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i < nb) {
            const int b = b0 + i;
            // (the lane's block, brought to the even place of a pair: which half of a word it takes is no constant here)
            const uint32_t sh = 16u * (uint32_t) (b & 1), seed = (word_of(ck.sd, b >> 1) >> sh) & 0xFFFFu, cc = word_of(ck.cw, b >> 1) >> sh;
            const SumCoefs sc = sum_coefs<P>(cc, 0, tab + 512 + sum_tab_at<P>(cc, 0));
            uint32_t y[8];
            sums_of<P>(seed << 16, stream_of(tab, seed), sc, y, [](int) {});
            float w[8];
            sums_float<P>(y, sc.k, w);
            d[i] = block_dot(w, xr + 8 * b);
            e2[i] = __uint_as_float(((cc & 15u) << 23) + ebase);
        }
    }
    float acc = 0.0f;
    for (int step = 0; step < (1 << ls); ++step) {
        // (the lane below, by a row shift of the wave's data path: the groups lie inside rows of 16 lanes)
        const float in = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, acc), 0x111, 0xF, 0xF, false));
        float v = s == 0 ? 0.0f : in;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i < nb) v = fmaf(d[i], e2[i], v);
        acc = v;
    }
    return acc;
}

// The 8 weights of block j of row r as f32: seeds unscaled integers with *sc = 2^e R32; BF16 / Q8 as BF16 values; Q4 in
// MLX's matvec form s * q + b unrounded (reference engine/kernels_moe.cu:91-107, 171-189).
__device__ __forceinline__ void block_weights(int fmt, const WSlice& w, const uint32_t* tab, int r, int K, int j, float (&o)[8],
                                              float* sc) {
    const int nbk = K / 8;
    *sc = 1.0f;
    if (fmt == MF_SEED4P4 || fmt == MF_SEED4) {
        const size_t g = (size_t) r * nbk + j;
        const uint32_t seed = gp<uint16_t>(w.p[0])[g], word = gp<uint16_t>(w.p[1])[g];
        int is[8], code;
        if (fmt == MF_SEED4P4) {
            block_isum<4>(tab, seed, word, is);
            code = (gp<uint8_t>(w.p[3])[g >> 1] >> ((g & 1) * 4)) & 15;
        } else {
            block_isum<3>(tab, seed, word, is);
            code = (int) (word & 15u);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) o[c] = (float) is[c];
        *sc = pow2f(w.eb + code) * NSLM_R32;
    } else if (fmt == MF_BF16) {
        const NSLM_GLOBAL uint16_t* v = gp<uint16_t>(w.p[0]) + (size_t) r * K + (size_t) j * 8;
#pragma unroll
        for (int c = 0; c < 8; ++c) o[c] = bf(v[c]);
    } else {
        const size_t e0 = (size_t) r * K + (size_t) j * 8, gi = e0 >> group_shift(w);
        const float s = bf(gp<uint16_t>(w.p[1])[gi]), b = bf(gp<uint16_t>(w.p[2])[gi]);
        if (fmt == MF_Q8) {
            const NSLM_GLOBAL uint32_t* q = gp<uint32_t>(w.p[0]) + e0 / 4;
#pragma unroll
            for (int c = 0; c < 8; ++c) o[c] = bfr(s * (float) ((q[c >> 2] >> (8 * (c & 3))) & 255u) + b);
        } else {
            const uint32_t q = gp<uint32_t>(w.p[0])[e0 / 8];
#pragma unroll
            for (int c = 0; c < 8; ++c) o[c] = s * (float) ((q >> (4 * c)) & 15u) + b;
        }
    }
}


}   // namespace nslm
