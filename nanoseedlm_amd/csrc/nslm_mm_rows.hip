// nslm_mm_rows.hip - the GEMM for few tokens a matrix: Y[n][r] = sum_k W[r][k] X[n][k], dense or grouped by expert.
//
// With few tokens what a launch takes is the decode of the weights (about 70 vector instructions a seed block, four clocks each), and the
// chip has to be filled from R / 16 row tiles.  The streamed kernel's workgroups take 64 rows and decode with one wave a SIMD: 64
// workgroups for 4096 rows, each decoding alone.  Here
//   * a lane's decoded 8-weight block never leaves its registers: eight BF16 weights of one row are exactly a lane's operand of
//     v_mfma_f32_16x16x32_bf16 (lane l: row l % 16, K block l / 16), so nothing is handed over or waited for between the decode and the
//     matrix core, and every wave decodes, independently of the others until their sums meet;
//   * the waves of a workgroup share its rows and split K: 64-weight chunk c belongs to segment c % 8, and a segment's sum is one
//     chain of MFMAs.  8 waves a workgroup: a segment each; 4 waves (grouped launches, whose many workgroups overlap): two each,
//     y = sum over w < 4 of (segment w + segment w + 4).  So a token's bits depend on K alone, not on the launch's shape, the tile or its
//     other tokens, in every dense launch of this file and in grouped passes of up to 32 pairs.  Passes of more have no registers for two
//     sums a pair: a wave's two segments are one chain there, and k_mm_wide's sum is one chain over all of K.
// Measured (us, streamed kernel -> this one, when both decoded by four multiply-adds a weight): P = 4, 4096 x 4096: 9 tokens 40.1 -> 9.7, 48 tokens
// 42.8 -> 11.1, 200 tokens 51.8 -> 23.0; 1024 x 4096, 100 tokens 44.7 -> 11.2; Q4 2880 x 2880, 301 tokens 43.0 -> 17.8; BF16 151936 x 2048, 16 tokens
// 155.7 -> 115.3 (5.5 TB/s).  By one multiply-add a weight 48 tokens take 9.4, by Q4's scales 16 lanes a row tile 301 tokens 15.9, by bytes that
// the conversion selects 15.2.
// What bounds it: vector issue of the decode for the seed formats, the activations' way from L2 for Q4 / Q8 / BF16 at many tokens,
// HBM for BF16 at few.
#include "nslm_mm_dev.h"

using namespace nslm;

namespace {

// ---- a step: 64 K (one chunk) of a wave's 16 RT rows and 16 NT tokens, staged in the wave's own part of the LDS ------------------------
// Loads in an MFMA operand's layout (consecutive lanes in different rows) cost the address unit a cycle a lane; staged by
// global_load_lds, consecutive lanes take consecutive 16-byte pieces of a row.  The wave reads a step into registers at once and
// requests the next one into the same place, so the LDS holds one step a wave and its decode covers the latency.
//   activations  [16 NT][64] BF16, the 16-byte pieces of a row swizzled (x_swizzle16) so that a fragment read spreads over the banks
//   seeds        per row tile: 16 rows x 16 bytes of seeds, 16 x 16 of coefficient words; then 16 x 4 of codes
//   Q4 / Q8      16 rows x 32 / 64 bytes a row tile (Q8: pieces swizzled); scales and biases a dword each (SL), or they stay in registers
//   BF16         like the activations
template <int FMT>
constexpr int row_bytes() { return seed_fmt<FMT>() || FMT == MF_Q4 ? 32 : FMT == MF_Q8 ? 64 : 128; }   // of weights, a chunk
// SL: the scales and biases of Q4 / Q8 in the LDS, too.  A load of them by every lane for its own row takes the address unit as many cycles as
// there are lanes, and 2 RT of them a step were a fifth to a third of the launch; where a chunk has one scale and one bias a row, 16 lanes load
// those of a row tile, and the others read what they landed.  In registers that gained half as much: the compiler waited for the loads
// where the two cases met.  Q4, 301 tokens, 2880 x 2880 18.3 -> 16.0 us; 26 tokens, 8513 x 4800 18.3 -> 14.7; Q8, 12 tokens, 6309 x 9792
// 17.7 -> 14.9.  (Only the dense kernel: the grouped ones have no LDS left for it.)
template <int FMT, int RT, int NT, bool PACKED, bool SL = false>
constexpr int step_bytes() {
    return 16 * RT * (row_bytes<FMT>() + (FMT == MF_SEED4P4 ? 4 : SL && (FMT == MF_Q4 || FMT == MF_Q8) ? 32 : 0)) + (PACKED ? NT * 2048 : 0);
}

__device__ __forceinline__ void to_lds2(const void* src, uint8_t* dst) {   // two bytes a lane, at dst + 4 l
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*) src, (__attribute__((address_space(3))) void*) dst, 2, 0, 0);
}
__device__ __forceinline__ void to_lds4(const void* src, uint8_t* dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*) src, (__attribute__((address_space(3))) void*) dst, 4, 0, 0);
}

// Block `odd` of the pair of seeds u and words v as BF16 weights.  hook(0 .. 5) is called between the phases (sums_of), hook(6) and hook(7) behind the last.
template <int FMT, class Hook>
__device__ __forceinline__ bf16x8 seed_weights(uint32_t u, uint32_t v, int odd, uint32_t codes, const uint32_t* tab, Hook hook) {
    constexpr int P = seed_p<FMT>();
    const uint32_t g = stream_of(tab, odd ? u >> 16 : u & 0xFFFFu);
    const SumCoefs sc = sum_coefs<P>(v, odd, tab + 512 + sum_tab_at<P>(v, odd));
    hook(0);
    uint32_t y[8];
    sums_of<P>(odd ? u : u << 16, g, sc, y, [&](int i) { hook(1 + i); });
    float f[8];
    sums_scaled<P>(y, sc.k, P == 4 ? code_of<P>(codes, odd) : code_of<P>(v, 4 * odd), f);
    hook(5);
    bf16x8 w = __builtin_bit_cast(bf16x8, make_uint4(cvt_pk_bf16(f[0], f[1]), cvt_pk_bf16(f[2], f[3]), cvt_pk_bf16(f[4], f[5]), cvt_pk_bf16(f[6], f[7])));
    hook(6);
    hook(7);
    return w;
}
// eight Q4 (q.x) or Q8 weights
template <int FMT>
__device__ __forceinline__ bf16x8 affine_weights(uint2 q, float scale, float bias) {
    float f[8];
    affine8<FMT>(q.x, q.y, scale, bias, f);
    return __builtin_bit_cast(bf16x8, make_uint4(cvt_pk_bf16(f[0], f[1]), cvt_pk_bf16(f[2], f[3]), cvt_pk_bf16(f[4], f[5]), cvt_pk_bf16(f[6], f[7])));
}

// A wave's weights: 16 RT rows from r0 (with gu: 8 RT gate rows of m0 and the same 8 RT rows of up, m1), a chunk a step, staged in the wave's
// own part of the LDS.
template <int FMT, int RT, bool SL = false>
struct Weights {
    static constexpr bool SEED = seed_fmt<FMT>(), AFFINE = FMT == MF_Q4 || FMT == MF_Q8;
    static constexpr int RB = row_bytes<FMT>(), CODES = 16 * RT * RB;
    static constexpr int NA = SEED || FMT == MF_Q4 ? (RT + 1) / 2 : FMT == MF_Q8 ? RT : 2 * RT;   // 16-byte loads a step
    const WSlice &m0, &m1;
    const bool gu;
    const int K, R, r0, lane, t, g;
    const uint8_t *pa[NA], *pcode;   // the lane's addresses in chunk 0
    uint32_t sc[RT], bi[RT];         // Q4 / Q8: scale and bias bits of the step that is staged
    // SL: value k = scales of row tiles 0 .. RT - 1, then biases.  `whole` (groups of 64 or more): 16 lanes a value, four values a load
    static constexpr int NS = (2 * RT + 3) / 4;
    const uint8_t* ps[NS];
    size_t g0;        // the row that the lane loads for, in groups of 64 weights
    int gsh, read0, read1;   // its matrix's group in those, as a shift; the LDS bytes from a lane's first value, and from a value to the next
    bool whole;
    bool aligned;
    // what a step's decode reads.  u, v, cd: two seeds, two words, their codes; Q4 / Q8: scale and bias.  raw: BF16: the two blocks; Q8: [0]; Q4: [0].xy
    struct Step {
        uint32_t u[RT], v[RT], cd[RT];
        uint4 raw[RT][2];
    };

    __device__ __forceinline__ int row_of(int i) const { return min(r0 + (gu ? i % (8 * RT) : i), R - 1); }   // rows past R: the last one again, never stored
    __device__ __forceinline__ bool second(int rt) const { return gu && rt >= RT / 2; }
    __device__ __forceinline__ const uint8_t* stream(int rt, int s) const { return (const uint8_t*) (second(rt) ? m1.p[s] : m0.p[s]); }

    __device__ __forceinline__ Weights(const WSlice& a_, const WSlice& b_, bool gu_, int K_, int R_, int r0_, int lane_)
        : m0(a_), m1(b_), gu(gu_), K(K_), R(R_), r0(r0_), lane(lane_), t(lane_ & 15), g(lane_ >> 4) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            if constexpr (SEED) {   // groups of 16 lanes: seeds, words of row tile 2i, the same of 2i + 1
                const int rt = min(2 * i + (g >> 1), RT - 1);
                pa[i] = ((g & 1) ? stream(rt, 1) : stream(rt, 0)) + (size_t) row_of(16 * rt + t) * (size_t) (K / 4);
            } else {
                const int at = 1024 * i + 16 * lane, r = min(at / RB, 16 * RT - 1), piece = (at % RB) / 16;
                const int sw = FMT == MF_BF16 ? piece ^ x_swizzle16(r & 15) : FMT == MF_Q8 ? piece ^ (r >> 3 & 1) * 3 : piece;
                pa[i] = stream(r >> 4, 0) + (size_t) row_of(r) * (size_t) (K / 64 * RB) + 16 * sw;
            }
        }
        if constexpr (FMT == MF_SEED4P4) {
            const int rt = min(g, RT - 1);
            pcode = stream(rt, 3) + (size_t) row_of(16 * rt + t) * (size_t) (K / 16);
        }
        if constexpr (AFFINE && SL) {
            const int rt = RT == 4 ? g : RT == 2 ? g & 1 : 0;
#pragma unroll
            for (int i = 0; i < NS; ++i) ps[i] = (4 * i + g) / RT & 1 ? stream(rt, 2) : stream(rt, 1);
            g0 = (size_t) row_of(16 * rt + t) * (size_t) (K / 64);
            whole = group_shift(m0) >= 6 && group_shift(m1) >= 6;
            gsh = (second(rt) ? group_shift(m1) : group_shift(m0)) - 6;
            read0 = CODES + 4 * (whole ? t : lane);
            read1 = whole ? 64 : 256;
        }
        // streams may start at any 2-byte (codes: any) boundary; those that are not aligned go through registers
        auto low = [&](const WSlice& m) { return (uintptr_t) m.p[0] | (SEED ? (uintptr_t) m.p[1] : 0) | (FMT == MF_SEED4P4 ? ((uintptr_t) m.p[3] & 3u) << 2 : 0); };
        aligned = ((low(m0) | (gu ? low(m1) : 0)) & 15u) == 0;
    }
    __device__ __forceinline__ void request(int c, uint8_t* ws) {   // chunk c -> the LDS at ws
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const uint8_t* src = pa[i] + (size_t) c * (SEED ? 16 : RB);
            if (!((SEED || FMT == MF_Q4) && 2 * i + 1 == RT) || lane < 32) {   // (an odd row tile: half a load)
                if (aligned) to_lds16(src, ws + 1024 * i);
                else *(u32x4*) (ws + 1024 * i + 16 * lane) = *(const NSLM_GLOBAL u32x4_a2*) src;
            }
        }
        if constexpr (FMT == MF_SEED4P4) {
            if (RT >= 4 || lane < 16 * RT) {
                if (aligned) to_lds4(pcode + 4 * (size_t) c, ws + CODES);
                else *(uint32_t*) (ws + CODES + 4 * lane) = *(const NSLM_GLOBAL u32_a1*) (pcode + 4 * (size_t) c);
            }
        }
        if (AFFINE && SL && whole) {
            const size_t gi = (g0 + (size_t) c) >> gsh;
#pragma unroll
            for (int i = 0; i < NS; ++i)
                if (RT > 1 || lane < 32) to_lds2(ps[i] + 2 * gi, ws + CODES + 256 * i);
        } else if constexpr (AFFINE) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const size_t gi = ((size_t) row_of(16 * rt + t) * K + (size_t) c * 64 + 16 * g) >> (second(rt) ? group_shift(m1) : group_shift(m0));
                if constexpr (SL) {
                    to_lds2(stream(rt, 1) + 2 * gi, ws + CODES + 256 * rt);
                    to_lds2(stream(rt, 2) + 2 * gi, ws + CODES + 256 * (RT + rt));
                } else {
                    sc[rt] = gp<uint16_t>(stream(rt, 1))[gi];
                    bi[rt] = gp<uint16_t>(stream(rt, 2))[gi];
                }
            }
        }
    }
    __device__ __forceinline__ void read(const uint8_t* ws, Step& s) const {   // a step that has landed, into registers
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            if constexpr (SEED) {
                s.u[rt] = *(const uint32_t*) (ws + 512 * rt + 16 * t + 4 * g);
                s.v[rt] = *(const uint32_t*) (ws + 512 * rt + 256 + 16 * t + 4 * g);
                if (FMT == MF_SEED4P4) s.cd[rt] = ws[CODES + 64 * rt + 4 * t + g];
            } else if constexpr (FMT == MF_BF16) {
#pragma unroll
                for (int h = 0; h < 2; ++h) s.raw[rt][h] = *(const uint4*) (ws + 2048 * rt + t * 128 + 16 * ((2 * g + h) ^ x_swizzle16(t)));
            } else {
                s.u[rt] = SL ? *(const uint16_t*) (ws + read0 + rt * read1) : sc[rt];
                s.v[rt] = SL ? *(const uint16_t*) (ws + read0 + (RT + rt) * read1) : bi[rt];
                if (FMT == MF_Q8) s.raw[rt][0] = *(const uint4*) (ws + 1024 * rt + 64 * t + 16 * (g ^ (t >> 3) * 3));
                else {
                    const uint2 b = *(const uint2*) (ws + 512 * rt + 32 * t + 8 * g);
                    s.raw[rt][0] = make_uint4(b.x, b.y, 0, 0);
                }
            }
        }
    }
    template <class Hook>
    __device__ __forceinline__ bf16x8 block(const Step& s, int rt, int h, const uint32_t* tab, Hook hook) const {   // the lane's block 2 g + h of the chunk's eight
        if constexpr (SEED) {
            return seed_weights<FMT>(s.u[rt], s.v[rt], h, FMT == MF_SEED4P4 ? s.cd[rt] : 0u, tab, hook);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) hook(i);
            const uint4& r = s.raw[rt][0];
            if constexpr (FMT == MF_BF16) return __builtin_bit_cast(bf16x8, s.raw[rt][h]);
            else return affine_weights<FMT>(FMT == MF_Q8 ? (h ? make_uint2(r.z, r.w) : make_uint2(r.x, r.y)) : make_uint2(h ? r.y : r.x, 0), bf(s.u[rt]), bf(s.v[rt]));
        }
    }
    __device__ __forceinline__ bf16x8 block(const Step& s, int rt, int h, const uint32_t* tab) const { return block(s, rt, h, tab, [](int) {}); }
};

template <int FMT>
__device__ __forceinline__ f32x4 scaled(const f32x4& s, int eb) {
    return (f32x4) {mm_scale<FMT>(s[0], eb), mm_scale<FMT>(s[1], eb), mm_scale<FMT>(s[2], eb), mm_scale<FMT>(s[3], eb)};
}
// four sums of pair / token dst, rows orow .. orow + 3 (those below R)
__device__ __forceinline__ void store_rows(const MmArgs& a, float* Y, int dst, int orow, const f32x4& s) {
    float* yo = Y + (size_t) dst * a.ys + orow;
    if ((a.ys & 3) == 0 && orow + 4 <= a.R && !a.add && !a.f32out && ((uintptr_t) yo & 15u) == 0) *(f32x4*) yo = (f32x4) {bfr(s[0]), bfr(s[1]), bfr(s[2]), bfr(s[3])};
    else
        for (int j = 0; j < 4 && orow + j < a.R; ++j) store_y(yo + j, s[j], a.add, a.f32out);
}
// the values the two GEMMs would have stored (rounded to BF16), then SwiGLU and its rounding, stored as BF16 bits
__device__ __forceinline__ void store_swiglu(const MmArgs& a, int dst, int orow, const f32x4& gate, const f32x4& up) {
    uint32_t v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = __float_as_uint(bfr(silu_bf(bfr(gate[j])) * bfr(up[j]))) >> 16;
    uint16_t* ao = a.a16 + (size_t) dst * a.ys + orow;
    if ((a.ys & 3) == 0 && orow + 4 <= a.R && ((uintptr_t) ao & 7u) == 0) *(uint2*) ao = make_uint2(v[0] | v[1] << 16, v[2] | v[3] << 16);
    else
        for (int j = 0; j < 4 && orow + j < a.R; ++j) ao[j] = (uint16_t) v[j];
}

// The 16 RT rows from r0 (with a.a16: 8 RT gate rows and the same 8 RT up rows) x the 16 NT tokens n0 .. of a workgroup of NW waves.
// lds: NW x max(step, RT NT KB).  meet: the decode tables are requested, and the workgroup has not met since.
template <int FMT, int RT, int NT, int NW, bool PACKED, bool GROUPED>
__device__ __forceinline__ void rows_tile(const MmArgs& a, const WSlice& m0, const WSlice& m1, const void* X, float* Y, const int32_t* perm, int start, int count,
                                          int n0, int r0, const uint32_t* tab, uint8_t* lds, bool meet) {
    const int tid = threadIdx.x & (64 * NW - 1), lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), t = lane & 15, g = lane >> 4;
    const bool gu = GROUPED && a.a16 != nullptr;
    const int nch = a.K / 64;
    constexpr bool SL = NW == 8;
    Weights<FMT, RT, SL> W(m0, m1, gu, a.K, a.R, r0, lane);
    uint8_t* const ws = lds + w * step_bytes<FMT, RT, NT, PACKED, SL>();
    uint8_t* const wx = ws + step_bytes<FMT, RT, NT, false, SL>();   // activations
    auto src_of = [&](int i) {   // token i of the tile's 16 NT (past the end: the last one again, never stored)
        const int n = start + min(n0 + i, count - 1);
        return (size_t) (GROUPED ? perm[n] / a.xdiv : n) * (size_t) a.xs;
    };
    uint32_t px[PACKED ? 2 * NT : NT];   // in 16-byte pieces
    if constexpr (PACKED) {
#pragma unroll
        for (int i = 0; i < 2 * NT; ++i) {
            const int n = 8 * i + (lane >> 3);
            px[i] = (uint32_t) (src_of(n) >> 3) + (uint32_t) ((lane & 7) ^ x_swizzle16(n & 15));
        }
    } else {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) px[nt] = (uint32_t) (src_of(16 * nt + t) >> 2) + 4u * (uint32_t) g;
    }
    auto request = [&](int c) {
        W.request(c, ws);
        if constexpr (PACKED) {
#pragma unroll
            for (int i = 0; i < 2 * NT; ++i) to_lds16((const uint8_t*) X + (size_t) (px[i] + 8u * (uint32_t) c) * 16, wx + 1024 * i);
        }
    };
    constexpr bool SEGS = NW == 4 && NT < 4;   // (four token tiles: one chain a wave, and half a step's activations at a time - the registers)
    f32x4 acc[RT][NT], tot[SEGS ? RT : 1][SEGS ? NT : 1];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            acc[rt][nt] = (f32x4) {0.0f, 0.0f, 0.0f, 0.0f};
            if (SEGS) tot[rt][nt] = acc[rt][nt];
        }
    const int n = (nch - w + NW - 1) / NW;   // this wave's chunks: those of segment w, then (4 waves) of segment w + 4
    int c = w;
    auto next = [&](int at) { at += 8; if (NW == 4 && at >= nch) at = at % 8 >= 4 ? nch : w + 4; return at; };
    if (n > 0) request(c);
    if (seed_fmt<FMT>() && meet) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int s = 0; s < n; ++s) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        constexpr bool HALVES = NW == 4 && NT >= 4;
        bf16x8 xb[HALVES ? 1 : 2][NT];
        auto read_x = [&](int h) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if constexpr (PACKED) {
                    xb[HALVES ? 0 : h][nt] = *(const bf16x8*) (wx + nt * 2048 + t * 128 + 16 * ((2 * g + h) ^ x_swizzle16(t)));
                } else {
                    const NSLM_GLOBAL uint8_t* xp = gp<uint8_t>(X) + (size_t) (px[nt] + 16u * (uint32_t) c + 2u * h) * 16;
                    const uint4 va = ldg16(xp), vb = ldg16(xp + 16);
#define F(w) __uint_as_float(w)
                    xb[HALVES ? 0 : h][nt] = __builtin_bit_cast(bf16x8, make_uint4(cvt_pk_bf16(F(va.x), F(va.y)), cvt_pk_bf16(F(va.z), F(va.w)),
                                                                                   cvt_pk_bf16(F(vb.x), F(vb.y)), cvt_pk_bf16(F(vb.z), F(vb.w))));
#undef F
                }
            }
        };
        read_x(0);
        if (!HALVES) read_x(1);
        typename Weights<FMT, RT, SL>::Step st;
        W.read(ws, st);
        const int cn = next(c);
        auto go_on = [&]() {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the step is in registers: its place is free
            if (s + 1 < n) request(cn);
            loads_issued();
        };
        if (!HALVES) go_on();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (HALVES && h) {
                read_x(1);
                go_on();
            }
            bf16x8 wb[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) wb[rt] = W.block(st, rt, h, tab);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) acc[rt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[rt], xb[HALVES ? 0 : h][nt], acc[rt][nt], 0, 0, 0);
        }
        if (SEGS && c < nch && c + 8 >= nch) {   // the segment is complete
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    tot[rt][nt] += acc[rt][nt];
                    acc[rt][nt] = (f32x4) {0.0f, 0.0f, 0.0f, 0.0f};
                }
        }
        c = cn;
    }
    __syncthreads();
    // accumulator element i of lane l: token l % 16, row 4 (l / 16) + i
    f32x4* red = (f32x4*) lds;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) red[((w * RT + rt) * NT + nt) * 64 + lane] = SEGS ? tot[rt][nt] : acc[rt][nt];
    __syncthreads();
    auto sum = [&](int tile, int l, int eb) {
        f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f32x4 p = red[(i * RT * NT + tile) * 64 + l];
            if (NW == 8) p = ((f32x4) {0.0f, 0.0f, 0.0f, 0.0f} + p) + red[((i + 4) * RT * NT + tile) * 64 + l];
            s += p;
        }
        return scaled<FMT>(s, eb);
    };
    const int nout = (gu ? RT / 2 : RT) * NT * 64;
    for (int i = tid; i < nout; i += 64 * NW) {
        const int tile = i >> 6, l = i & 63, rt = tile / NT, nt = tile % NT, tok = n0 + 16 * nt + (l & 15), orow = r0 + 16 * rt + 4 * (l >> 4);
        if (tok >= count || orow >= a.R) continue;
        const int dst = GROUPED ? perm[start + tok] : start + tok;
        if (gu) store_swiglu(a, dst, orow, sum(tile, l, m0.eb), sum(tile + RT / 2 * NT, l, m1.eb));
        else store_rows(a, Y, dst, orow, sum(tile, l, m0.eb));
    }
}

// ---- fuller tiles of a grouped launch -----------------------------------------------------------------------------------------------
// Up to 256 pairs of an expert - two table tiles - against 128 weight rows (64 gate and 64 up) a workgroup, so that an expert's weights are
// decoded once.  Each of the 8 waves decodes its own 16 rows into operands and multiplies them with every pair; the pairs' activations of a step
// sit once a workgroup in one of two LDS buffers, and the waves meet at one barrier a step, where the buffer before the last is free.
// Two workgroups a CU, four waves a SIMD: 16 rows a wave leave the registers for that (64 of accumulators at 256 pairs), and the decode
// needs them - with 32 rows and two waves a SIMD a block took 650 clocks instead of 430.
template <int FMT, int NT>
constexpr int wide_lds() { return 2 * (NT * 2048 + 8 * step_bytes<FMT, 1, NT, false>()); }
template <int FMT, int NT>
__device__ __forceinline__ void wide_tile(const MmArgs& a, const WSlice& m, const uint16_t* X, float* Y, const int32_t* perm, int start, int count,
                                          int r0, const uint32_t* tab, uint8_t* lds) {
    static_assert(NT % 2 == 0, "half the sums fit the activations' LDS");
    constexpr int SB = step_bytes<FMT, 1, NT, false>(), NS = (NT + 3) / 4;   // NS: 64 pairs each
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // (an item's own: kept out of the loop over items, whose registers it would take)
    const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), t = lane & 15, g = lane >> 4;
    const bool gu = a.a16 != nullptr;   // waves 0 - 3: gate rows, 4 - 7: the same rows of up
    const int nch = a.K / 64, rw = r0 + 16 * (gu ? w & 3 : w);
    Weights<FMT, 1> W(m, m, false, a.K, a.R, rw, lane);
    uint8_t* const ws = lds + 2 * NT * 2048 + w * 2 * SB;
    uint32_t px[NS];   // in 16-byte pieces: the wave stages eight pairs' rows of every 64
#pragma unroll
    for (int i = 0; i < NS; ++i) {
        const int n = 64 * i + 8 * w + (lane >> 3);
        px[i] = (uint32_t) (((size_t) (perm[start + min(n, count - 1)] / a.xdiv) * (size_t) a.xs) >> 3) + (uint32_t) ((lane & 7) ^ x_swizzle16(n & 15));
    }
    auto request_x = [&](int c) {
#pragma unroll
        for (int i = 0; i < NS; ++i)
            if (NT % 4 == 0 || i + 1 < NS || w < 2 * (NT % 4)) to_lds16((const uint8_t*) X + (size_t) (px[i] + 8u * (uint32_t) c) * 16, lds + (c & 1) * NT * 2048 + 1024 * (8 * i + w));
    };
    f32x4 acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = (f32x4) {0.0f, 0.0f, 0.0f, 0.0f};
    // The matrix instructions of half a chunk are issued among the vector instructions that decode the next half.  A wave's records run a chunk
    // ahead of its activations.
    constexpr int NG = (NT + 7) / 8;   // token tiles a hook, at most: hook i has tiles i NT / 8 and up
    // Hooks a fragment is read ahead of its use.  P = 3 at 256 pairs has registers for one: with two the loop kept values in scratch memory, whose loads wait
    // for all of the wave's requests (757 rows, E 16, top-4, d 2752, ff 1984 223 -> 213 us; P = 4, with fewer such loads, gains nothing).
    constexpr int XD = NT > 12 && FMT == MF_SEED4 ? 1 : 2;
    typename Weights<FMT, 1>::Step st;
    bf16x8 wb, xq[XD][NG];
    auto half = [&](int c, int h) {   // multiplies (c, h) while the next half's weights are formed
        const uint8_t* const xt = lds + (c & 1) * NT * 2048 + t * 128 + 16 * ((2 * g + h) ^ x_swizzle16(t));
        auto fetch = [&](int i) {
#pragma unroll
            for (int j = 0; j < NG; ++j)
                if (i < 8 && i * NT / 8 + j < (i + 1) * NT / 8) xq[i % XD][j] = *(const bf16x8*) (xt + (i * NT / 8 + j) * 2048);
        };
#pragma unroll
        for (int i = 0; i < XD; ++i) fetch(i);
        wb = W.block(st, 0, h ^ 1, tab, [&](int i) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NG; ++j) {
                const int nt = i * NT / 8 + j;
                if (nt < (i + 1) * NT / 8) acc[nt < NT ? nt : 0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb, xq[i % XD][j], acc[nt < NT ? nt : 0], 0, 0, 0);
            }
            fetch(i + XD);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    W.request(0, ws);
    request_x(0);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (and the decode tables)
    W.read(ws, st);
    wb = W.block(st, 0, 0, tab, [](int) {});
    if (nch > 1) W.request(1, ws + SB);
    for (int c = 0; c < nch; ++c) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the activations of chunk c have landed, those of c - 1 are read
        if (c + 1 < nch) request_x(c + 1);
        half(c, 0);
        if (c + 1 < nch) W.read(ws + ((c + 1) & 1) * SB, st);
        if (c + 2 < nch) W.request(c + 2, ws + (c & 1) * SB);
        loads_issued();
        half(c, 1);   // (past the end: some block again)
    }
    // The sums go to the LDS of the activations, and from there to their pairs in a loop: 64 or 128 rows of a pair side by side, by all waves.  (Out of
    // the registers, a pass's code was 10 to 50 KB that ran once an item, as fast as it could be fetched: 13K of an item's 120K clocks; 1917 rows, E 16,
    // top-8, d 1792, ff 384, P = 3: 181 -> 168 us.)  Row group q of four, token t: slot t ^ mix(q) of the group's 16, so that the reads, of many groups'
    // same token, reach all banks as the writes do.
    auto mix = [](int q) { return (q ^ (q >> 4)) & 15; };
    const int q = 4 * (gu ? w & 3 : w) + g, slot = 16 * g + (t ^ mix(q));
    __syncthreads();
    if (gu || a.f32out == OUT_BF16) {   // as the BF16 that is stored, or that SwiGLU reads
        uint2* const red = (uint2*) lds;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const f32x4 s = scaled<FMT>(acc[nt], m.eb);
            red[(w * NT + nt) * 64 + slot] = make_uint2(pack_bf2(s[0], s[1]), pack_bf2(s[2], s[3]));
        }
        __syncthreads();
        const int lg = gu ? 4 : 5, oq = tid & ((1 << lg) - 1), orow = r0 + 4 * oq, step = 512 >> lg;
        if (orow >= a.R) return;
        const uint2* const own = red + (oq >> 2) * NT * 64 + 16 * (oq & 3);
        int n = tid >> lg, dst = perm[start + min(n, count - 1)];
#pragma unroll 1
        for (; n < count; n += step) {
            const int next = perm[start + min(n + step, count - 1)], at = (n >> 4) * 64 + ((n & 15) ^ mix(oq));
            const uint2 v = own[at];
            const f32x4 s = {bf(v.x & 0xFFFFu), bf(v.x >> 16), bf(v.y & 0xFFFFu), bf(v.y >> 16)};
            if (gu) {
                const uint2 u = own[4 * NT * 64 + at];
                store_swiglu(a, dst, orow, s, (f32x4) {bf(u.x & 0xFFFFu), bf(u.x >> 16), bf(u.y & 0xFFFFu), bf(u.y >> 16)});
            } else {
                uint16_t* const o = (uint16_t*) Y + (size_t) dst * a.ys + orow;
                if ((a.ys & 3) == 0 && orow + 4 <= a.R && ((uintptr_t) o & 7u) == 0) *(uint2*) o = v;
                else
                    for (int j = 0; j < 4 && orow + j < a.R; ++j) o[j] = (uint16_t) (__float_as_uint(s[j]) >> 16);
            }
            dst = next;
        }
        return;
    }
    f32x4* const red = (f32x4*) lds;
    const int oq = tid & 31, orow = r0 + 4 * oq;
#pragma unroll
    for (int part = 0; part < 2; ++part) {   // (half the pairs' fit)
        if (8 * NT * part >= count) return;
        if (part) __syncthreads();
#pragma unroll
        for (int nt = 0; nt < NT / 2; ++nt) red[(w * (NT / 2) + nt) * 64 + slot] = scaled<FMT>(acc[part * (NT / 2) + nt], m.eb);
        __syncthreads();
#pragma unroll 1
        for (int n = tid >> 5; n < min(8 * NT, count - 8 * NT * part); n += 16)
            if (orow < a.R)
                store_rows(a, Y, perm[start + 8 * NT * part + n], orow, red[((oq >> 2) * (NT / 2) + (n >> 4)) * 64 + 16 * (oq & 3) + ((n & 15) ^ mix(oq))]);
    }
}

// Who computes a tile of a grouped launch, whatever table the host made: k_mm_wide takes every tile of more than `least` pairs, alone or together
// with one that joins it, and k_mm_rows_grouped beside it takes what is left: the tiles of up to `least` pairs that join none.  A tile can join
// the one before it where that one is k_mm_wide's and both are a slice's adjoining pairs (an empty tile, too), and does if that one did not
// join another itself: the parity of the run of tiles that can, up to the last one that cannot.  A wave looks at 64 tiles at once (a
// token's experts by the thousand make runs of hundreds of tiles, and a walk tile by tile is a chain of as many loads).
// Beside k_mm_rows_grouped every tile can join: which kernel computes a tile, and with it its sums' order, is then a matter of the table alone,
// not of the matrices in the launch.  Alone k_mm_wide pairs full tiles where their workgroups are more than 5/8 of two a CU, of which P = 3, P = 4 and Q4 run as many at once: a
// pair saves a decode and leaves half the workgroups.  us for so many workgroups of a full tile, and for half as many of a pair (K 2048, P = 4):
// 256 44 and 56, 320 63 and 57, 512 69 and 64, 768 97 and 94, 1024 134 and 105, 1536 210 and 149.  36 layer steps of 140 to 620 pairs an expert:
// geometric mean 0.917 of the time of a workgroup a tile, with one round as the line 0.925, with two 0.941.  (25 other steps, K 256 to 4096, against the line at 5/8: with one
// round P = 4 0.998, P = 3 0.999, Q4 1.002 of the time, with two 1.030, 1.026, 1.039.  BF16, with the line at 5/16, 5/8, one and two
// times two a CU: E 32, top-4, d 512, ff 256, 2048 rows 36.6, 31.0, 31.2, 31.4; E 16, top-2, d 2048, ff 1024, two experts in all 83, 84, 107, 107; E 16, top-4, d 2048,
// ff 1024, 1024 rows 120, 119, 119, 112.)  A tile of up to FEW pairs joins at any number: it adds a pass's step to a full one's, no decode (E 16, top-8,
// d 3584, ff 384, 325 rows - about 162 pairs an expert - with FEW 32, 48, 64: 149, 138, 138).
// Where workgroups are started a tile each (Q8) a pair's second one is an empty one: there full tiles stay alone up to a round and in a second that they
// fill (E 16, top-2, d 2048, ff 1024, 2048 rows on the same two experts, 512 workgroups: 171 alone, 222 in pairs; 576: 299 and 269).
#define FEW 64
struct JoinAt {   // tile counts: full tiles go in pairs from [2] on, and between [0] and [1]
    int n[3];
    JoinAt(int blocks, int round, bool dealt) {   // a tile's workgroups; two a CU
        n[0] = dealt ? 0 : round / blocks;
        n[1] = dealt ? 0 : (5 * round / 4 + blocks - 1) / blocks;
        n[2] = dealt ? 5 * round / 8 / blocks + 1 : (2 * round + blocks - 1) / blocks;
    }
    __device__ __forceinline__ bool pairs(int nt) const { return nt >= n[2] || (nt > n[0] && nt < n[1]); }
};
struct Join {
    int least, few;   // k_mm_wide's tiles; the pairs of a tile that can join one
    __device__ __forceinline__ bool can(const MmTile& t, const MmTile& before) const {
        return before.count > least && t.count <= few && t.slice == before.slice && t.start == before.start + before.count;
    }
    __device__ __forceinline__ bool joins(const MmTile* tiles, int y) const {   // all 64 lanes, the same y: tile y goes with tile y - 1
        if (y < 1 || !can(tiles[y], tiles[y - 1])) return false;   // (most: by scalar loads)
        for (int n = 0;; n += 64) {
            const int i = y - n - (int) (threadIdx.x & 63);
            const unsigned long long stop = ~__ballot(i > 0 && can(tiles[max(i, 0)], tiles[max(i - 1, 0)]));
            if (stop) return (__ffsll(stop) - 1) & 1;   // (i <= 0 stops)
        }
    }
};

constexpr int max_of(int a, int b) { return a > b ? a : b; }
template <int FMT, int RT, int NT, int NW, bool PACKED>
constexpr size_t rows_lds() { return (size_t) NW * max_of(step_bytes<FMT, RT, NT, PACKED, NW == 8>(), RT * NT * 1024); }
constexpr size_t MOST_LDS = 156 * 1024;   // beside the decode tables

template <int FMT, int RT, int NT, bool PACKED>
__global__ void __launch_bounds__(512, 2) k_mm_rows(MmArgs a, WSlice w, const void* X, float* Y) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ __attribute__((aligned(8))) uint32_t tab[mm_tab_words<FMT>()];
    if constexpr (seed_fmt<FMT>()) {
        load_sum_tables<seed_p<FMT>()>(tab);
        __syncthreads();
    }
    rows_tile<FMT, RT, NT, 8, PACKED, false>(a, w, w, X, Y, nullptr, 0, a.T, (int) blockIdx.y * 16 * NT, (int) blockIdx.x * 16 * RT, tab, lds, false);
}

#define GRT 2   // row tiles of the grouped kernel's workgroups
// MOST: token tiles a pass.  Two or four: four waves a SIMD, with four tiles also what the LDS holds.  Six: registers for three; the LDS
// holds three workgroups a CU of Q4 (52 KB), two of the other formats (56 to 64 KB).
template <int FMT, int MOST, bool PACKED>
__global__ void __launch_bounds__(256, MOST > 4 ? 3 : 4) k_mm_rows_grouped(MmArgs a, const WSlice* ws, const void* X, float* Y, const int32_t* perm,
                                                                           const MmTile* tiles, const int32_t* ntiles, int limit, int few) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ __attribute__((aligned(16))) uint32_t tab[mm_tab_words<FMT>()];
    // The grid has a workgroup row for as many tiles as the host's table holds.  Of fewer than `few` tiles, whose own workgroups do not fill the
    // chip, those past *ntiles take the later passes over 16 MOST pairs: pass 1 of every tile, then pass 2, .. (row nt + e: pass 1 + e / nt of
    // tile e % nt); the passes that they do not reach are the tile's own workgroups', after pass 0.  Tokens that agree on a few experts make
    // few and full tiles (E 128, top-2, d 2048, ff 768, 100 rows on the same two experts: 66 -> 47 us a layer step).
    constexpr int PASS = 16 * MOST;
    const int nt = ntiles ? *ntiles : (int) gridDim.y, extra = (int) blockIdx.y - nt;
    int y = (int) blockIdx.y, first = 0, next = PASS;   // the first pair, and that of the pass after it
    if (nt >= few) {
        if (extra >= 0) return;
    } else if (extra < 0) {
        next = PASS * (1 + (max((int) gridDim.y - nt - y, 0) + nt - 1) / nt);
    } else {
        if (nt < 1) return;
        y = extra % nt;
        first = PASS * (1 + extra / nt);
        next = 2 * MMT_BN;   // (none)
    }
    const bool gu = a.a16 != nullptr;
    const int rows = gu ? 8 * GRT : 16 * GRT, r0 = (int) blockIdx.x * rows;
    const MmTile tl = tiles[y];
    if (tl.count > a.most || tl.count <= first) return;                  // another launch's, or no such pass
    if (a.paired && Join {a.least, MMT_BN}.joins(tiles, y)) return;   // another launch's
    if (blockIdx.z) {   // the launch's second matrix: same tiles and activations, its own slices and output
        ws = a.ws2;
        Y = a.y2;
    }
    const WSlice m0 = ws[tl.slice], m1 = gu ? a.ws2[tl.slice] : m0;
    if (tl.count > limit)   // a broken promise is made visible: pairs beyond the launch's bound are stored as NaN, not left stale
        for (int i = limit * rows + (int) threadIdx.x; i < tl.count * rows; i += 256) {
            const int orow = r0 + i % rows;
            const size_t at = (size_t) perm[tl.start + i / rows] * a.ys + orow;
            if (orow < a.R) {
                if (gu) a.a16[at] = 0x7FC0u;
                else Y[at] = __uint_as_float(0x7FC00000u);
            }
        }
    const int count = min(tl.count, limit);
    if constexpr (seed_fmt<FMT>()) tables_to_lds<seed_p<FMT>()>(tab);
    for (int n0 = first; n0 < count; n0 = next, next += PASS) {
        if (n0 != first) __syncthreads();   // the sums of the tokens before are read
        const int left = count - n0;
#define T(NT) rows_tile<FMT, GRT, NT, 4, PACKED, true>(a, m0, m1, X, Y, perm, tl.start, count, n0, r0, tab, lds, n0 == first)
        if (left <= 16) T(1);
        else if (MOST == 2 || left <= 32) T(2);
        else if constexpr (MOST == 4) T(4);
        else if constexpr (MOST == 6) {
            if (left <= 64) T(4);
            else T(6);
        }
#undef T
    }
}

// A grouped launch's tiles of more than a.least pairs, each with the tile that joins it (Join).  The grid is what runs at once, two workgroups a CU (of BF16, whose steps take
// more LDS, one: in a grid of two the second half began behind the first one's lists; 1762 rows, E 128, top-4, d 512, ff 256: 44.8 -> 41.6 us, geometric mean of 25 steps 0.978), and a
// workgroup takes items blockIdx.x, + gridDim.x, .. of (matrix, tile, block of rows): with a workgroup an item, the ones that found nothing to do between
// them, they were started in turn over the shader engines, and an engine that was full kept the free places of the others waiting, 20 to 40 us of an
// item's 75 (2048 rows, E 128, top-8, d 2048, ff 768: 54 to 58 of an XCD's 64 places taken; 435 us a
// layer step, 415 so).  Its tiles are found 64 a wave at once and listed in LDS: an item is then two dependent loads from its slice, as it was.
// Passes of 64, 96, 128, 160, 192 and 256 pairs: an expert's share of a step spreads round its mean, and of 128 pairs on average half have a few more,
// joined to the full tile (in passes of 64, 128, 192 and 256, of which the middle two met: 6 % of that step).  Passes of 144 and 224 gave nothing more.
// Fuller items come first: what a workgroup has more than another is then one of the smallest (E 16, top-4, d 2048, ff 1600, 1152 rows, experts of
// 256 and 32 pairs: 259 us a layer step in the table's order, 229 so).  Two workgroups' LDS of Q8 leave no room for the list: there a workgroup has the tile of its row.
#define WIDE_TILES 1024   // of the table, looked at together
template <int FMT>
constexpr bool wide_deals() { return FMT != MF_Q8; }
template <int FMT>
constexpr int wide_at_once() { return FMT == MF_BF16 ? 1 : 2; }   // workgroups a CU
template <int FMT>
__global__ void __launch_bounds__(512, 4) k_mm_wide(MmArgs a, const WSlice* ws, const uint16_t* X, float* Y, const int32_t* perm, const MmTile* tiles,
                                                    const int32_t* ntiles, int grid_tiles, JoinAt at) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ __attribute__((aligned(16))) uint32_t tab[mm_tab_words<FMT>()];
    const int nt = ntiles ? min(*ntiles, grid_tiles) : grid_tiles;
    const Join join = {a.least, a.least > 0 || at.pairs(nt) ? MMT_BN : FEW};
    const bool gu = a.a16 != nullptr;
    const int blocks = (a.R + (gu ? 63 : 127)) / (gu ? 64 : 128);
    if constexpr (seed_fmt<FMT>()) tables_to_lds<seed_p<FMT>()>(tab);
    const int wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
    const WSlice* const mine_ws = gu && wave >= 4 ? a.ws2 : ws;   // waves 4 - 7: up
    auto item = [&](int y, bool second, int r0) {   // second: the launch's second matrix: same tiles and activations, its own slices and output
        const MmTile tl = tiles[y];
        const WSlice m = (second ? a.ws2 : mine_ws)[tl.slice];
        int count = tl.count;
        if (y + 1 < nt && join.can(tiles[y + 1], tl)) count += tiles[y + 1].count;
        __syncthreads();   // the item before has read the LDS
#define W(NT) wide_tile<FMT, NT>(a, m, X, second ? a.y2 : Y, perm, tl.start, count, r0, tab, lds)
        if (count <= 64) W(4);
        else if (count <= 96) W(6);
        else if (count <= 128) W(8);
        else if (count <= 160) W(10);
        else if (count <= 192) W(12);
        else W(16);
#undef W
    };
    if constexpr (!wide_deals<FMT>()) {
        const int y = (int) blockIdx.y;
        if (y < nt && tiles[y].count > a.least && !join.joins(tiles, y)) item(y, blockIdx.z, (int) blockIdx.x * (gu ? 64 : 128));
        return;
    }
    __shared__ uint16_t list[WIDE_TILES];   // the launch's tiles: those of more than 64 pairs from the front, the others from the back
    __shared__ uint64_t cans[WIDE_TILES / 64], large[WIDE_TILES / 64], fuller[WIDE_TILES / 64];
    __shared__ int2 found;
    int run = 0;   // (wave 0) of tiles that can join the one before them, up to the last one looked at
    for (int base = 0;; base += WIDE_TILES) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));   // (as in wide_tile: nothing of this is kept)
        for (int g = wave; g < WIDE_TILES / 64 && base + 64 * g < nt; g += 8) {   // (the table need not have grid_tiles rows: none past *ntiles is read)
            const int y = base + 64 * g + lane, at_y = min(y, nt - 1);
            const MmTile t = tiles[at_y], before = tiles[max(at_y - 1, 0)];
            const uint64_t c = __ballot(y > 0 && y < nt && join.can(t, before)), l = __ballot(y < nt && t.count > a.least), f = __ballot(t.count > 64);
            if (lane == 0) {
                cans[g] = c;
                large[g] = l;
                fuller[g] = f;
            }
        }
        __syncthreads();
        if (wave == 0) {
            int n = 0, few = 0;
            for (int g = 0; g < WIDE_TILES / 64 && base + 64 * g < nt; ++g) {
                const uint64_t can = cans[g], stop = ~can & (~0ull >> (63 - lane));
                const uint64_t next = can >> 1 | (g + 1 < WIDE_TILES / 64 && base + 64 * (g + 1) < nt ? cans[g + 1] << 63 : 0);   // (the tile after it can join it)
                const int len = stop ? lane - (63 - __clzll((long long) stop)) : run + lane + 1;
                const uint64_t mine = large[g] & __ballot(!(len & 1)), m = mine & (fuller[g] | next), under = ~(~0ull << lane);
                if ((m >> lane) & 1) list[n + __popcll(m & under)] = (uint16_t) (64 * g + lane);
                else if ((mine >> lane) & 1) list[WIDE_TILES - 1 - (few + __popcll(mine & ~m & under))] = (uint16_t) (64 * g + lane);
                n += __popcll(m);
                few += __popcll(mine & ~m);
                run = __builtin_amdgcn_readlane(len, 63);
            }
            if (lane == 0) found = make_int2(n, few);
        }
        __syncthreads();
        const int full = __builtin_amdgcn_readfirstlane(found.x), n = full + __builtin_amdgcn_readfirstlane(found.y), items = n * blocks * (a.ws2 && !gu ? 2 : 1);
        for (int i = (int) blockIdx.x; i < items; i += (int) gridDim.x) {
            const int ti = i / blocks, second = ti >= n, of = second ? ti - n : ti;
            item(base + __builtin_amdgcn_readfirstlane((int) list[of < full ? of : WIDE_TILES - 1 - (of - full)]), second, (i - ti * blocks) * (gu ? 64 : 128));
        }
        if (base + WIDE_TILES >= nt) return;
    }
}

template <int FMT, int RT, int NT, bool PACKED>
void launch(hipStream_t st, const MmArgs& a, const WSlice& w, const void* X, float* Y) {
    constexpr size_t lds = rows_lds<FMT, RT, NT, 8, PACKED>();
    static_assert(lds <= MOST_LDS, "a step of every wave fits the CU's LDS");
    allow_big_lds<k_mm_rows<FMT, RT, NT, PACKED>>(lds);
    const dim3 grid((unsigned) (a.R + 16 * RT - 1) / (16 * RT), (unsigned) (a.T + 16 * NT - 1) / (16 * NT));
    hipLaunchKernelGGL((k_mm_rows<FMT, RT, NT, PACKED>), grid, dim3(512), lds, st, a, w, X, Y);
    host_note_launch();
}

// The workgroup's shape: what a CU spends on a workgroup's step is RT decodes + NT token tiles' loads and MFMAs (beta: a token
// tile's share against a row tile's decode, from the times of matrices of 300 .. 14336 rows at 9 .. 1024 tokens), and the launch
// takes as many workgroups one after the other as the fullest CU gets.
struct Shape {
    int rt, nt;
    double cost;
};
double beta_of(int fmt) { return fmt == MF_BF16 ? 1.0 : fmt == MF_Q8 || fmt == MF_Q4 ? 0.3 : 0.13; }
bool fits(int fmt, int rt, int nt) { return !(fmt == MF_BF16 && rt + nt > 9); }   // (BF16 weights: 2 KB of LDS a wave and tile)
Shape shape_of(int fmt, int R, int T, bool packed) {
    static const int rts[][2] = {{1, 1}, {1, 2}, {1, 3}, {1, 4}, {1, 6}, {1, 8}, {2, 1}, {2, 2}, {2, 3}, {2, 4}, {2, 6}, {2, 8}, {4, 1}, {4, 2}, {4, 4}};
    const int cus = host_cu_count();
    Shape best = {0, 0, 1e30};
    for (const auto& s : rts) {
        const int rt = s[0], nt = s[1];
        if (!fits(fmt, rt, nt) || (!packed && !(rt == 1 && (nt == 1 || nt == 4)) && !(rt == 4 && nt == 4))) continue;
        const long long wgs = (long long) ((R + 16 * rt - 1) / (16 * rt)) * ((T + 16 * nt - 1) / (16 * nt));
        const double cost = (double) ((wgs + cus - 1) / cus) * (rt + nt * beta_of(fmt));
        if (cost < best.cost) best = {rt, nt, cost};
    }
    return best;
}

template <int FMT, bool PACKED>
void dense(hipStream_t st, const MmArgs& a, const WSlice& w, const void* X, float* Y) {
    const Shape s = shape_of(FMT, a.R, a.T, PACKED);
#define C(RT, NT) case 10 * RT + NT: launch<FMT, RT, NT, PACKED>(st, a, w, X, Y); return;
    if constexpr (PACKED) {
        switch (10 * s.rt + s.nt) { C(1, 1) C(1, 2) C(1, 3) C(1, 4) C(1, 6) C(1, 8) C(2, 1) C(2, 2) C(2, 3) C(2, 4) C(2, 6) C(4, 1) C(4, 2) C(4, 4) }
        if constexpr (FMT != MF_BF16) launch<FMT, 2, 8, PACKED>(st, a, w, X, Y);
    } else {
        switch (10 * s.rt + s.nt) { C(1, 1) C(1, 4) C(4, 4) }
    }
#undef C
}
template <int FMT, int MOST, bool PACKED>
void grouped(hipStream_t st, const MmArgs& a, const WSlice* ws, const void* X, float* Y, const int32_t* perm, const MmTile* tiles, const int32_t* ntiles,
             int grid_tiles, int limit) {
    const int rows = a.a16 ? 8 * GRT : 16 * GRT;
    const dim3 grid((unsigned) (a.R + rows - 1) / rows, (unsigned) grid_tiles, a.ws2 && !a.a16 ? 2u : 1u);
    constexpr size_t lds = rows_lds<FMT, GRT, MOST, 4, PACKED>();
    allow_big_lds<k_mm_rows_grouped<FMT, MOST, PACKED>>(lds);
    // Passes of 64: four workgroups a CU run at once; passes of 96, of which a CU holds two or three, have the same line.
    // (Passes of 32: half of that; most tiles there have one pass, and the rows that find none cost small matrices
    // more than they give: E 128, top-2, d 512, ff 256, 96 rows 28 -> 32 us.  Passes of 64, E 16, top-2, d 2688, ff 384, 1010 rows: 135 and 121.)
    const int few = (limit < a.most ? limit : a.most) > 16 * MOST ? (MOST > 2 ? 4 : 2) * host_cu_count() / (int) (grid.x * grid.z) + 1 : 0;
    hipLaunchKernelGGL((k_mm_rows_grouped<FMT, MOST, PACKED>), grid, dim3(256), lds, st, a, ws, X, Y, perm, tiles, ntiles, limit, few);
    host_note_launch();
}
// tile_rows: what the caller says of its tiles' pairs.  The fewer token tiles a pass, the more the kernel's registers leave the decode
template <int FMT, bool PACKED>
void grouped_any(hipStream_t st, const MmArgs& a, const WSlice* ws, const void* X, float* Y, const int32_t* perm, const MmTile* tiles, const int32_t* ntiles,
                 int grid_tiles, int tile_rows) {
    const int limit = tile_rows <= 32 ? 32 : MMT_BN;
    if constexpr (PACKED) {
        if (a.most > 64 && tile_rows > 64) { grouped<FMT, 6, true>(st, a, ws, X, Y, perm, tiles, ntiles, grid_tiles, limit); return; }
        if (a.most > 32 && tile_rows > 48) { grouped<FMT, 4, true>(st, a, ws, X, Y, perm, tiles, ntiles, grid_tiles, limit); return; }
    }
    grouped<FMT, 2, PACKED>(st, a, ws, X, Y, perm, tiles, ntiles, grid_tiles, limit);
}
template <int FMT>
void wide(hipStream_t st, const MmArgs& a, const WSlice* ws, const uint16_t* X, float* Y, const int32_t* perm, const MmTile* tiles, const int32_t* ntiles,
          int grid_tiles) {
    const int rows = a.a16 ? 64 : 128;
    const int blocks = (a.R + rows - 1) / rows, mats = a.ws2 && !a.a16 ? 2 : 1, once = wide_at_once<FMT>() * host_cu_count();
    const long long most = (long long) blocks * grid_tiles * mats;
    const dim3 grid = wide_deals<FMT>() ? dim3((unsigned) (most < once ? most : once)) : dim3((unsigned) blocks, (unsigned) grid_tiles, (unsigned) mats);
    constexpr size_t lds = wide_lds<FMT, 16>();
    constexpr size_t all = lds + (seed_fmt<FMT>() ? 4 * mm_tab_words<FMT>() : 0) + (wide_deals<FMT>() ? 2 * WIDE_TILES + 3 * WIDE_TILES / 8 + 16 : 0);
    static_assert(wide_at_once<FMT>() == 160 * 1024 / ((all + 1279) / 1280 * 1280), "as many fit a CU's LDS, given out in pieces of 1280 bytes");
    allow_big_lds<k_mm_wide<FMT>>(lds);
    hipLaunchKernelGGL((k_mm_wide<FMT>), grid, dim3(512), lds, st, a, ws, X, Y, perm, tiles, ntiles, grid_tiles, JoinAt(blocks * mats, 2 * host_cu_count(), wide_deals<FMT>()));
    host_note_launch();
}

}   // namespace

namespace nslm {

#define BY_FORMAT(CALL)                                        \
    switch (fmt) {                                             \
        case MF_SEED4P4: CALL(MF_SEED4P4); break;              \
        case MF_SEED4: CALL(MF_SEED4); break;                  \
        case MF_BF16: CALL(MF_BF16); break;                    \
        case MF_Q8: CALL(MF_Q8); break;                        \
        default: CALL(MF_Q4); break;                           \
    }

// Against the kernel of 64 rows x up to 512 tokens a workgroup - for packed activations the streamed one, for f32 the first-generation one -, which
// spends on a step, in row decodes, what `step` says: that one wins where its workgroups fill the chip.  The streamed kernel was timed with 64 ..
// 224 workgroups, one a CU; BF16 of more than 128 tokens again, on both and on every shape of this file (521 tokens, 17758 x 8000: 395 us with the
// line where it was, streamed 276; 415 tokens, 7690 x 768 29.7 and 18.1; 132 tokens, 71938 x 448 69 and 52; none slower).  f32: 290 matrices of
// 300 .. 32000 rows at 9 .. 2048 tokens on both kernels; the lines lie where the faster one changes (up to 128 tokens, and for Q4, Q8 and BF16 up to
// 256, it never does), and the kernel taken is 0.1 % off the faster one on average, 16 % at worst
// (4096 x 4096, 1000 tokens, P = 4: first generation 236 us, this 165; 14336 x 4096, 400 tokens: 216 and 270).
bool mm_rows_better(int fmt, int R, int T, bool packed) {
    static const double step[2][3][3] = {{{6.2, 7.5, 8.8}, {8.4, 12.7, 14.5}, {13.7, 19.5, 27.0}},
                                         {{16.0, 16.0, 24.0}, {24.0, 24.0, 31.6}, {32.0, 40.0, 60.0}}};
    const int q = T <= 128 ? 0 : T <= 256 ? 1 : 2, f = fmt == MF_BF16 ? 2 : fmt == MF_Q8 || fmt == MF_Q4 ? 1 : 0, cus = host_cu_count();
    const long long wgs = (long long) ((R + 63) / 64) * ((T + 511) / 512);
    return shape_of(fmt, R, T, packed).cost < (double) ((wgs + cus - 1) / cus) * step[packed ? 0 : 1][f][q];
}
void mm_rows_dense(hipStream_t st, int fmt, const MmArgs& a, const WSlice& w, const void* X, bool packed, float* Y) {
#define D(F) packed ? dense<F, true>(st, a, w, X, Y) : dense<F, false>(st, a, w, X, Y)
    BY_FORMAT(D)
#undef D
}
void mm_rows_grouped(hipStream_t st, int fmt, const MmArgs& a, const WSlice* ws, const void* X, bool packed, float* Y, const int32_t* perm,
                     const MmTile* tiles, const int32_t* ntiles, int grid_tiles, int tile_rows) {
#define G(F)                                                                                                 \
    packed ? grouped_any<F, true>(st, a, ws, X, Y, perm, tiles, ntiles, grid_tiles, tile_rows)             \
           : grouped_any<F, false>(st, a, ws, X, Y, perm, tiles, ntiles, grid_tiles, tile_rows)
    BY_FORMAT(G)
#undef G
}

void mm_wide_grouped(hipStream_t st, int fmt, const MmArgs& a, const WSlice* ws, const uint16_t* X, float* Y, const int32_t* perm, const MmTile* tiles,
                     const int32_t* ntiles, int grid_tiles) {
#define G(F) wide<F>(st, a, ws, X, Y, perm, tiles, ntiles, grid_tiles)
    BY_FORMAT(G)
#undef G
}

}   // namespace nslm
