// nslm_dev.h - device-side building blocks shared by the gfx950 kernels: BF16 rounding, the LFSR stream basis, and the
// exact integer decode of one 8-weight SeedLM block on 16-bit integer dot products.
//
// Arithmetic contract (reference: nslm/lfsr.h:4-10, nslm/search4.h:4-6): state_k of seed s is bits k..k+15 of the bit
// stream s | g(s) << 16, where g(s) is GF(2)-linear in s; weight c of a block is
//   isum_c = sum_p (state_(P*c+p+1) - 32768) * q_p   (exact, |isum| < 2^20),   w_c = (float) isum_c * fl(R32 * 2^e).
// Everything up to isum_c is done in integers here, so regenerated weights are bit-exact by construction.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels_hip.h"

namespace nslm {

// ---- global-memory pointers ---------------------------------------------------------------------------------------------
// Stream pointers arrive inside structs (WSlice), where the compiler cannot tell that they address global memory and would
// emit flat loads.  A flat load also counts against the LDS counter, so every LDS wait - and every barrier built on one -
// would wait for the HBM latency of loads issued steps ahead on purpose.  gp<T>(p) states the address space.
#define NSLM_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ const NSLM_GLOBAL T* gp(const void* p) { return (const NSLM_GLOBAL T*) p; }
// 16- and 8-byte global loads (uint4 / uint2 are class types and cannot be read through a qualified pointer directly)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <typename P>
__device__ __forceinline__ uint4 ldg16(P p) {
    const u32x4 v = *(const NSLM_GLOBAL u32x4*) p;
    return make_uint4(v.x, v.y, v.z, v.w);
}
template <typename P>
__device__ __forceinline__ uint2 ldg8(P p) {
    const u32x2 v = *(const NSLM_GLOBAL u32x2*) p;
    return make_uint2(v.x, v.y);
}

// ---- BF16 (round to nearest even; reference engine/kernels_moe.cu:17-31) ---------------------------------------------
__device__ __forceinline__ float bfr(float x) {
    uint32_t u = __float_as_uint(x);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return __uint_as_float(u & 0xFFFF0000u);
}
__device__ __forceinline__ uint32_t tobf(float x) {
    uint32_t u = __float_as_uint(x);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return u >> 16;
}
__device__ __forceinline__ float bf(uint32_t h) { return __uint_as_float(h << 16); }
// Eight Q4 (x) or Q8 weights, unrounded.  Q4: even and odd nibbles as bytes, which the conversion selects by itself; the compiler, left to it, takes
// each nibble out of x first, an instruction of half rate a weight (301 tokens, 2880 x 2880: 17.2 -> 16.5 us; 12, 6309 x 9792: 14.2 -> 13.0;
// one, 14336 x 4096: 12.0 -> 11.4).
template <int FMT>
__device__ __forceinline__ void affine8(uint32_t x, uint32_t y, float scale, float bias, float (&f)[8]) {
    uint32_t a = FMT == MF_Q8 ? x : x & 0x0F0F0F0Fu, b = FMT == MF_Q8 ? y : x >> 4 & 0x0F0F0F0Fu;
    if constexpr (FMT == MF_Q4) asm("" : "+v"(a), "+v"(b));
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t v = FMT == MF_Q8 ? (i < 4 ? a : b) >> (8 * (i & 3)) & 255u : (i & 1 ? b : a) >> (8 * (i >> 1)) & 255u;
        f[i] = scale * (float) v + bias;
    }
}
__device__ __forceinline__ uint32_t pack_bf2(float a, float b) { return tobf(a) | (tobf(b) << 16); }
// nn.silu on a BF16 tensor: the sigmoid and the product are each rounded to BF16
__device__ __forceinline__ float silu_bf(float g) {
    const float s = bfr(1.0f / (1.0f + expf(-g)));
    return bfr(g * s);
}
// y = bf16(acc), or the residual form bf16(y + bf16(acc)); f32out keeps the unrounded sum (a switch of this backend)
__device__ __forceinline__ void store_y(float* yo, float s, int add, int f32out) {
    if (f32out) *yo = add ? *yo + s : s;
    else *yo = add ? bfr(*yo + bfr(s)) : bfr(s);
}

// ---- the stream basis -------------------------------------------------------------------------------------------------
// g(s) = the 32 stream bits that follow seed s: bit k = top bit of state k+1.  g is linear over GF(2), so
// g(s) = lo[s & 0xFF] ^ hi[s >> 8] with two 256-entry tables, built here at compile time from the LFSR definition
// (taps 0, 1, 3, 12; shift right; feedback into bit 15).  The P = 3 format reads the low 24 bits of the same table.
struct alignas(16) StreamBasis {
    uint32_t v[512];
};
constexpr uint32_t stream32_of(uint32_t s) {
    uint32_t g = 0;
    for (int k = 0; k < 32; ++k) {
        const uint32_t fb = (s ^ (s >> 1) ^ (s >> 3) ^ (s >> 12)) & 1u;
        s = (s >> 1) | (fb << 15);
        g |= (s >> 15) << k;
    }
    return g;
}
constexpr StreamBasis make_basis(uint32_t flip) {   // flip: exclusive-or on the sum
    StreamBasis b{};
    for (uint32_t i = 0; i < 256; ++i) {
        b.v[i] = stream32_of(i);
        b.v[256 + i] = stream32_of(i << 8) ^ flip;
    }
    return b;
}
// Pairs of sign-extended int4 coefficients as packed int16: entry b = { sext4(b & 15), sext4(b >> 4) }.
struct CoefPairs {
    uint32_t v[256];
};
constexpr CoefPairs make_pairs() {
    CoefPairs t{};
    for (uint32_t b = 0; b < 256; ++b) {
        const int lo = (int) (b & 15u) - (int) ((b & 8u) << 1), hi = (int) (b >> 4) - (int) (((b >> 4) & 8u) << 1);
        t.v[b] = ((uint32_t) lo & 0xFFFFu) | ((uint32_t) hi << 16);
    }
    return t;
}
__device__ const StreamBasis kBasis = make_basis(0);
__device__ const CoefPairs kPairs = make_pairs();

// LDS copy of both tables: [0,512) stream basis, [512,768) coefficient pairs
#define NSLM_TAB_WORDS 768
__device__ __forceinline__ void load_tables(uint32_t* tab) {
    for (int i = threadIdx.x; i < 512; i += blockDim.x) tab[i] = kBasis.v[i];
    for (int i = threadIdx.x; i < 256; i += blockDim.x) tab[512 + i] = kPairs.v[i];
}
// keeps the loads written above this line above it: left alone, the compiler moves a load down to its first use, and a load
// whose use sits in a conditional block becomes a load, a wait and a branch - one round trip per load instead of one for all
__device__ __forceinline__ void loads_issued() { asm volatile("" ::: "memory"); }
template <int N>
__device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void to_lds16(const void* src, uint8_t* dst) {   // dst: the wave's base, lane l lands at dst + 16 l; both 16-byte aligned
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*) src, (__attribute__((address_space(3))) void*) dst, 16, 0, 0);
}
__device__ __forceinline__ uint32_t stream_of(const uint32_t* tab, uint32_t seed16) {
    return tab[seed16 & 0xFFu] ^ tab[256 + (seed16 >> 8)];
}

// ---- exact block decode -----------------------------------------------------------------------------------------------
// Written as the three-source encoding: left to itself the compiler prefers the accumulating two-source form, whose
// destination is tied to the addend, and pays a register move whenever the addend has another use or a different home.
__device__ __forceinline__ int dot2(uint32_t a, uint32_t b, int c) {
    int d;
    asm("v_dot2_i32_i16 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}
// the same with a zero addend: the three-source encoding takes the constant inline, where the accumulating two-source
// form the compiler picks for dot2(a, b, 0) would first spend a move on zeroing its destination
__device__ __forceinline__ int dot2z(uint32_t a, uint32_t b) {
    int d;
    asm("v_dot2_i32_i16 %0, %1, %2, 0" : "=v"(d) : "v"(a), "v"(b));
    return d;
}
// { word X's half hx, word Y's half hy } as one packed pair
__device__ __forceinline__ uint32_t halves(uint32_t X, int hx, uint32_t Y, int hy) {
    const uint32_t sel = (uint32_t) (2 * hx) | ((uint32_t) (2 * hx + 1) << 8) | ((uint32_t) (4 + 2 * hy) << 16) |
                         ((uint32_t) (5 + 2 * hy) << 24);
    return __builtin_amdgcn_perm(Y, X, sel);
}

// The 16 windows of a block's stream.  `up` is any word whose upper 16 bits are the seed, g the 32 bits that follow.
// A[k], k = 1..16: low half = state_k - 32768, high half = state_(k+16) - 32768 as int16 (state ^ 0x8000).
__device__ __forceinline__ void windows(uint32_t up, uint32_t g, uint32_t (&A)[17]) {
#pragma unroll
    for (int k = 1; k <= 15; ++k) A[k] = __builtin_amdgcn_alignbit(g, up, 16 + k) ^ 0x80008000u;
    A[16] = g ^ 0x80008000u;
}

// P = 4: weight c reads states 4c+1..4c+4; q01 = {q0,q1}, q23 = {q2,q3} as packed int16 (reference nslm/lib_search4.c:22-31)
__device__ __forceinline__ void isum_p4(uint32_t up, uint32_t g, uint32_t q01, uint32_t q23, int (&is)[8]) {
    uint32_t A[17];
    windows(up, g, A);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int k = 4 * c + 1;
        is[c] = dot2(halves(A[k], 0, A[k + 1], 0), q01, dot2z(halves(A[k + 2], 0, A[k + 3], 0), q23));
        is[c + 4] = dot2(halves(A[k], 1, A[k + 1], 1), q01, dot2z(halves(A[k + 2], 1, A[k + 3], 1), q23));
    }
}
// P = 3: weight c reads states 3c+1..3c+3; q01 = {q0,q1}, q2 = {q2,0} (reference nslm/lfsr.h:116-128)
__device__ __forceinline__ void isum_p3(uint32_t up, uint32_t g, uint32_t q01, uint32_t q2, int (&is)[8]) {
    uint32_t A[17];
    windows(up, g, A);
    const uint32_t q2hi = q2 << 16;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int k0 = 3 * c + 1, k1 = k0 + 1, k2 = k0 + 2;   // state k lives in A[k] low (k <= 16) or A[k-16] high
        const uint32_t pr = halves(A[k0 <= 16 ? k0 : k0 - 16], k0 > 16, A[k1 <= 16 ? k1 : k1 - 16], k1 > 16);
        const int third = k2 <= 16 ? dot2z(A[k2], q2) : dot2z(A[k2 - 16], q2hi);
        is[c] = dot2(pr, q01, third);
    }
}

#define NSLM_R32 (1.0f / 32767.0f)

// ---- the eight sums by one multiply-add each (the matvecs' and the GEMMs' form) -----------------------------------------------------------------
// The P states of a weight are one window of the stream, shifted: all but the few bits at its two ends are the same bits.  So one state times
// one multiplier, and two small corrections that depend on the end bits alone, give the whole sum:
//   P = 4, weight c, T = state_(4c+4), l = the three stream bits below it, h = the three above it:  state_(4c+1+p) = 2^(3-p) T + (l >> p) - 65536 (h >> p), so
//     isum_c = M (T - 32768) + H(l) - 65536 H(h) + 32768 L,   M = 8 q0 + 4 q1 + 2 q2 + q3,   H(b) = q0 b + q1 (b >> 1) + q2 (b >> 2),   L = H(7);
//   P = 3, T = state_(3c+1), l = its two lowest bits, h = the two stream bits above it:  state_(3c+1+p) = (T - T mod 2^p + 65536 (h mod 2^p)) / 2^p, so
//     4 isum_c = M (T - 32768) - H(l) + 65536 H(h) - 32768 L,  M = 4 q0 + 2 q1 + q2,   H(b) = 2 q1 (b & 1) + q2 b,   L = H(3).
// H has 8 (4) entries of a byte: two registers, looked up by v_perm.  P = 4: l and h are bits 4i + 1 .. 4i + 3 of the stream, i = c and c + 4, so
// one v_perm looks up four of them, and one more a weight joins the two corrections.  H is antisymmetric, H(7 - b) = L - H(b), so a
// flipped index changes the sign; -M comes from one dot product over the nibbles (8 is no int4, -8 is), and everything is formed negated.
// The bytes are offset to be positive, so what a multiply-add leaves is an integer 0 < y < 2^24, y = k - isum (P = 3: k + 4 isum):
//   P = 4: k = 32769 L + 88 * 65537, 1.8e6 <= y <= 9.4e6;   P = 3: k = 32768 L + 40 + 80 * 65536, 0.8e6 <= y <= 9.6e6.
// Such an integer is a float's bits: y * 2^-149, subnormal or of the first binade, so no convert is needed and k goes by an exact subtraction.
// A block is about 70 vector instructions as BF16 weights, records and all (four multiply-adds a weight, a convert and a multiply: about 95);
// as one token's products about 68 (P = 4 by eleven sums of nibble columns, a convert and a multiply-add each: 78; P = 3 by windows paired
// for dot products: 76).  us a pass, before and after: layer step of 64 tokens (E 128, top-8, d 2048, ff 768, P = 4) 239 -> 200, of 8 tokens
// 95 -> 86.5, of one 19.7 -> 18.3; of 3 tokens, E 64, top-4, d 2880, ff 2880, P = 3, 147 -> 134; 2880 x 2880, P = 3, 6 tokens 10.9 -> 10.2.
struct alignas(16) SumTab4 {
    uint32_t v[256];
};
struct alignas(16) SumTab3 {
    uint32_t v[512];
};
constexpr int sext4(uint32_t n) { return (int) (n & 15u) - (int) ((n & 8u) << 1); }
constexpr SumTab4 make_sumtab4() {   // entry { q0, q1 }: H(0..3) + 88
    SumTab4 t{};
    for (uint32_t b = 0; b < 256; ++b) {
        const int q0 = sext4(b), q1 = sext4(b >> 4);
        t.v[b] = 88u | (uint32_t) (88 + q0) << 8 | (uint32_t) (88 + 2 * q0 + q1) << 16 | (uint32_t) (88 + 3 * q0 + q1) << 24;
    }
    return t;
}
constexpr SumTab3 make_sumtab3() {   // entry { q1, q2 }: 40 - H(0..3), 80 + H(0..3)
    SumTab3 t{};
    for (uint32_t b = 0; b < 256; ++b) {
        const int q1 = sext4(b), q2 = sext4(b >> 4), H[4] = {0, 2 * q1 + q2, 2 * q2, 2 * q1 + 3 * q2};
        for (int i = 0; i < 4; ++i) {
            t.v[2 * b] |= (uint32_t) (40 - H[i]) << (8 * i);
            t.v[2 * b + 1] |= (uint32_t) (80 + H[i]) << (8 * i);
        }
    }
    return t;
}
static_assert(alignof(StreamBasis) >= 16 && alignof(SumTab4) >= 16 && alignof(SumTab3) >= 16, "to_lds16 reads 16 bytes a lane");
__device__ const StreamBasis kBasis3 = make_basis(0x8000u);   // sums_of's for P = 3: bit 15 flipped
__device__ const SumTab4 kSumTab4 = make_sumtab4();
__device__ const SumTab3 kSumTab3 = make_sumtab3();
template <int P>
__device__ __forceinline__ const uint32_t* sum_basis() { return P == 4 ? kBasis.v : kBasis3.v; }
template <int P>
constexpr int sum_tab_words() { return P == 4 ? 768 : 1024; }   // LDS: [0, 512) the stream basis, then the table above
template <int P>
__device__ __forceinline__ void load_sum_tables(uint32_t* tab) {
    for (int i = threadIdx.x; i < 512; i += blockDim.x) tab[i] = sum_basis<P>()[i];
    for (int i = threadIdx.x; i < sum_tab_words<P>() - 512; i += blockDim.x) tab[512 + i] = P == 4 ? kSumTab4.v[i] : kSumTab3.v[i];
}
// The same, requested into the LDS (16-byte aligned) by the workgroup's first four waves: beside the kernel's other first loads they cost no
// round trip of their own, where the loop above waits for each of its loads.  The waves wait for vmcnt(0) before the workgroup meets.
// (Grouped GEMM, E 128, top-8, d 2048, ff 768, 64 rows 196 -> 189 us a layer step, 32 rows 172 -> 166; wide, 2048 rows 428 -> 424.  The dense GEMM
// for few tokens, whose waves went on at once after its loop, lost 2 % by meeting with their first weights.)
template <int P>
__device__ __forceinline__ void tables_to_lds(uint32_t* tab) {
    const int w = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t* const rest = P == 4 ? kSumTab4.v : kSumTab3.v;
    if (256 * w < sum_tab_words<P>()) to_lds16((w < 2 ? sum_basis<P>() + 256 * w : rest + 256 * (w - 2)) + 4 * lane, (uint8_t*) (tab + 256 * w));
}
// The same for a workgroup of exactly NTHR threads (256, 512 or 1024), in two halves: a thread's loads are requested in
// tables_fetch() (put it beside the kernel's other first loads), and tables_store() writes them to LDS once they are needed -
// the loop above waits for every load in turn, one memory round trip each.
template <int P>
__device__ __forceinline__ uint32_t sum_tab_word(int i) { return i < 512 ? sum_basis<P>()[i] : P == 4 ? kSumTab4.v[i - 512] : kSumTab3.v[i - 512]; }
template <int P, int NTHR>
struct TableWords {
    uint32_t w[(sum_tab_words<P>() + NTHR - 1) / NTHR];
};
template <int P, int NTHR>
__device__ __forceinline__ TableWords<P, NTHR> tables_fetch() {
    TableWords<P, NTHR> t;
#pragma unroll
    for (int j = 0; j < (sum_tab_words<P>() + NTHR - 1) / NTHR; ++j)
        t.w[j] = sum_tab_word<P>(min((int) threadIdx.x + NTHR * j, sum_tab_words<P>() - 1));   // clamped: the loads stay unconditional
    return t;
}
template <int P, int NTHR>
__device__ __forceinline__ void tables_store(uint32_t* tab, const TableWords<P, NTHR>& t) {
#pragma unroll
    for (int j = 0; j < (sum_tab_words<P>() + NTHR - 1) / NTHR; ++j) {
        const int i = (int) threadIdx.x + NTHR * j;
        if (i < sum_tab_words<P>()) tab[i] = t.w[j];
    }
}
// half ha of a x half hb of b, int16, + c (ha, hb: constants once unrolled)
#define NSLM_MAD16(HA, HB) asm("v_mad_i32_i16 %0, %1, %2, %3 op_sel:[" #HA "," #HB ",0,0]" : "=v"(d) : "v"(a), "v"(b), "v"(c))
__device__ __forceinline__ int mad16(uint32_t a, int ha, uint32_t b, int hb, int c) {
    int d;
    if (ha && hb) { NSLM_MAD16(1, 1); }
    else if (ha) { NSLM_MAD16(1, 0); }
    else if (hb) { NSLM_MAD16(0, 1); }
    else { NSLM_MAD16(0, 0); }
    return d;
}
// the nibbles of w x the int4 constants of C, + 0
template <uint32_t C>
__device__ __forceinline__ int dot8c(uint32_t w) {
    int d;
    asm("v_dot8_i32_i4 %0, %1, %2, 0" : "=v"(d) : "v"(w), "s"(C));
    return d;
}
// A block's exponent code: nibble n of w (constant once unrolled).  P = 3: spelled out, for left to itself the compiler moves the shift by 23 in front, and
// code << 23 plus a constant is three instructions instead of two.
template <int P>
__device__ __forceinline__ uint32_t code_of(uint32_t w, int n) {
    if constexpr (P == 4) return (w >> (4 * n)) & 15u;
    uint32_t c;
    asm("v_bfe_u32 %0, %1, %2, 4" : "=v"(c) : "v"(w), "n"(4 * n));
    return c;
}
struct SumCoefs {
    uint32_t lo, hi;   // the tables
    uint32_t m;        // the multiplier, int16
    uint32_t k;
};
// cc: a packed pair of coefficient (nibble) words, of which block `odd` (0 / 1) is taken; t: its entry of the LDS table (sum_tab_at)
template <int P>
__device__ __forceinline__ uint32_t sum_tab_at(uint32_t cc, int odd) {
    return P == 4 ? (odd ? (cc >> 16) & 0xFFu : cc & 0xFFu) : 2u * (odd ? cc >> 24 : (cc >> 8) & 0xFFu);
}
template <int P>
__device__ __forceinline__ SumCoefs sum_coefs(uint32_t cc, int odd, const uint32_t* t) {
    SumCoefs s;
    s.lo = t[0];
    if constexpr (P == 4) {
        const int h = odd ? dot8c<0x01240000u>(cc) : dot8c<0x0124u>(cc), l = odd ? dot8c<0x01370000u>(cc) : dot8c<0x0137u>(cc);
        uint32_t t3;   // H(b + 4) = H(b) + h, h = 4 q0 + 2 q1 + q2 (three bytes, then the fourth: left to itself the compiler takes a 64-bit multiply)
        asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(t3) : "v"(h), "s"(0x010101), "v"(s.lo));
        s.hi = t3 + ((uint32_t) h << 24);
        s.m = (uint32_t) (odd ? dot8c<0xFEC80000u>(cc) : dot8c<0xFEC8u>(cc));
        s.k = (uint32_t) (__mul24(l, 32769) + 88 * 65537);
    } else {
        s.hi = t[1];
        s.m = (uint32_t) (odd ? dot8c<0x12400000u>(cc) : dot8c<0x1240u>(cc));
        s.k = ((uint32_t) (odd ? dot8c<0x32000000u>(cc) : dot8c<0x3200u>(cc)) << 15) + (uint32_t) (40 + 80 * 65536);
    }
    return s;
}
// A constant that the compiler keeps in a vector register: an instruction of three operands takes one scalar of them, and with both constants known the
// compiler makes two instructions of it instead.  (P = 3: a window's selector in one instruction instead of two, 78 -> 68.5 a block in the GEMMs with the flipped
// bit and the code below.  us a layer step: 3 tokens, E 64, top-4, d 2880, ff 2880 115.3 -> 109.3; 4 tokens, E 128, top-8, d 2048, ff 768 52.7 -> 48.8; 106, E 64, top-2,
// d 3840, ff 576 155.8 -> 147.6; dense, 6 tokens, 2880 x 2880 10.2 -> 9.9.  The same for P = 4, one instruction of 69 less, is no gain: grouped GEMMs
// - 1.5 %, dense matrices of few tokens + 1 to + 4 %.)
template <uint32_t C>
__device__ __forceinline__ uint32_t vconst() {
    uint32_t v;
    asm("v_mov_b32 %0, %1" : "=v"(v) : "i"(C));
    return v;
}
// The eight y of N blocks.  up: any word whose upper 16 bits are the seed; g: stream_of its table (the 32 stream bits that follow; P = 3: bit 15 flipped, as a
// signed product wants the top bit of one of its windows).  hook(0 .. 3) is called between the phases: a
// caller with matrix instructions to issue puts them there, where the vector ALU has work beside them, and one whose wave has a SIMD's vector issue to itself
// holds the scheduler to the phases, in which every operand of several blocks is a dozen instructions old.
template <int P, int N, class Hook>
__device__ __forceinline__ void sums_of(const uint32_t (&up)[N], const uint32_t (&g)[N], const SumCoefs (&s)[N], uint32_t (&y)[N][8], Hook hook) {
    if constexpr (P == 4) {
        uint32_t xl[N][2], xh[N][2], A[N][4];
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const uint32_t le = __builtin_amdgcn_alignbit(g[n], up[n], 17), lo = __builtin_amdgcn_alignbit(g[n], up[n], 21);   // bits 1 .., 5 ..: fields 0, 2, 4, 6; 1, 3, 5, 7
            const uint32_t he = g[n] >> 1, ho = g[n] >> 5;                                                                   // bits 17 .., 21 ..: fields 4, 6, 8, 10; 5, 7, 9, 11
            xl[n][0] = __builtin_amdgcn_perm(s[n].hi, s[n].lo, ~le & 0x07070707u);
            xl[n][1] = __builtin_amdgcn_perm(s[n].hi, s[n].lo, ~lo & 0x07070707u);
            xh[n][0] = __builtin_amdgcn_perm(s[n].hi, s[n].lo, he & 0x07070707u);
            xh[n][1] = __builtin_amdgcn_perm(s[n].hi, s[n].lo, ho & 0x07070707u);
        }
        hook(0);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int n = 0; n < N; ++n) A[n][c] = (c < 3 ? __builtin_amdgcn_alignbit(g[n], up[n], 20 + 4 * c) : g[n]) ^ 0x80008000u;   // states 4c + 4, 4c + 20
        hook(1);
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int n = 0; n < N; ++n) y[n][c] = __builtin_amdgcn_perm(xh[n][c & 1], xl[n][c & 1], 0x0C040C00u + 0x00010001u * (uint32_t) (c >> 1));
        hook(2);
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int n = 0; n < N; ++n) y[n][c] = (uint32_t) mad16(A[n][c & 3], c >> 2, s[n].m, 0, (int) y[n][c]);
        hook(3);
    } else {
        uint32_t W[N][8];
        const uint32_t q = vconst<0x0C040C00u>();
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int n = 0; n < N; ++n) W[n][c] = c < 5 ? __builtin_amdgcn_alignbit(g[n], up[n], 17 + 3 * c) : g[n] >> (3 * c - 15);   // state 3c + 1 and the bits above it
        hook(0);
        // (state - 32768: bit 15 flipped.  In g it comes flipped, which is window 5's, bit 12 of window 6 and bit 9 of window 7; bits 18 and up of the others,
        // where nothing reads it)
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int n = 0; n < N; ++n)
                if (c != 5) W[n][c] ^= c < 5 ? 0x8000u : c == 6 ? 0x9000u : 0x8200u;
        hook(1);
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int n = 0; n < N; ++n) y[n][c] = __builtin_amdgcn_perm(s[n].hi, s[n].lo, __builtin_amdgcn_bitop3_b32(W[n][c], 0x00030003u, q, 0xEA));   // (W & ..) | q
        hook(2);
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int n = 0; n < N; ++n) y[n][c] = (uint32_t) mad16(W[n][c], 0, s[n].m, 0, (int) y[n][c]);
        hook(3);
    }
}
template <int P, class Hook>
__device__ __forceinline__ void sums_of(uint32_t up, uint32_t g, const SumCoefs& s, uint32_t (&y)[8], Hook hook) {
    const uint32_t u1[1] = {up}, g1[1] = {g};
    const SumCoefs s1[1] = {s};
    uint32_t y1[1][8];
    sums_of<P, 1>(u1, g1, s1, y1, hook);
#pragma unroll
    for (int c = 0; c < 8; ++c) y[c] = y1[0][c];
}
// isum_c 2^-22 (exact): what a matvec multiplies with the activations; a row's sum is then multiplied by R32 2^22.  So a sum of blocks is kept 2^-22 low:
// where base + code lie below about -120 it is subnormal, and an addition to it rounds by up to 2^-150, 2^-143 of the row's sum (at -126, the lowest, about one
// part in 2^18 of a block's; bases of real packs are about -22).  Kept 22 binades higher it would leave the f32 range at the other end.
#define NSLM_SUM_R32 (NSLM_R32 * 4194304.0f)
template <int P>
__device__ __forceinline__ void sums_float(const uint32_t (&y)[8], uint32_t k, float (&f)[8]) {
    const float s = __uint_as_float((P == 4 ? 254u : 252u) << 23), d = __uint_as_float(k) * s;   // 2^127, P = 3: a quarter
#pragma unroll
    for (int c = 0; c < 8; ++c) f[c] = P == 4 ? fmaf(__uint_as_float(y[c]), -s, d) : fmaf(__uint_as_float(y[c]), s, -d);
}
// 2^eb as f32 bits: a block's scale is this plus its code in the exponent field
__device__ __forceinline__ uint32_t sums_e2(int eb) { return (uint32_t) (eb + 127) << 23; }
// The weights times 2^(-eb - 22): y as a float's bits, k off (exact), times the block's scale (one rounding).  The products' sums are these of
// the weights themselves to the last bit once sums_scale has put the power of two back.
template <int P>
__device__ __forceinline__ void sums_scaled(const uint32_t (&y)[8], uint32_t k, uint32_t code, float (&f)[8]) {
    const float s = __uint_as_float((code << 23) + ((P == 4 ? 239u : 237u) << 23 | 0x100u));   // R32 = 2^-15 (1 + 2^-15); 2^(149 + 15 - 15 - 37 + code)
#pragma unroll
    for (int c = 0; c < 8; ++c) f[c] = P == 4 ? __uint_as_float(k) - __uint_as_float(y[c]) : __uint_as_float(y[c]) - __uint_as_float(k);
#pragma unroll
    for (int c = 0; c < 8; ++c) f[c] *= s;
}
__device__ __forceinline__ float sums_scale(float v, int eb) { return ldexpf(v, eb + 22); }

// One block of either seed format from its raw fields.  seed16 / word16: the 16-bit seed and coefficient (P = 4) or
// nibble (P = 3) word, zero-extended.  Returns the integer sums and the block's exponent e = eb + code.
template <int P>
__device__ __forceinline__ void block_isum(const uint32_t* tab, uint32_t seed16, uint32_t word16, int (&is)[8]) {
    const uint32_t g = stream_of(tab, seed16), up = seed16 << 16;
    if (P == 4) isum_p4(up, g, tab[512 + (word16 & 0xFFu)], tab[512 + (word16 >> 8)], is);
    else isum_p3(up, g, tab[512 + ((word16 >> 4) & 0xFFu)], tab[512 + (word16 >> 12)], is);
}
// 2^e as f32 bits; e in the normal range
__device__ __forceinline__ float pow2f(int e) { return __uint_as_float((uint32_t) (e + 127) << 23); }

__device__ __forceinline__ int group_shift(const WSlice& w) { return w.gs ? w.gs : 6; }

// process-wide switches and launch-error bookkeeping (defined in nslm_mv.hip)
int host_store_f32();
int host_cu_count();
void host_note_launch();
void host_note_unsupported();   // a launcher refused its arguments: kc_last_error() reports an invalid value

// the sum of v over the workgroup's 256 threads, the same value in every thread (every thread must call)
__device__ __forceinline__ float wg_sum(float v, float* red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();   // red may still be read from a previous call
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}
// rsqrt(mean(x^2) + eps) of a row of g <= 256 NSLM_NORM_NR values, bit for bit as the RMSNorm kernel forms it (thread tid
// sums k = tid, tid + 256, .. in order, then the workgroup tree), so a consumer that normalises its own input,
// xn_k = x_k * r * (1 + w_k), computes what the separate kernel would have stored.  256 threads, every thread calls.
#define NSLM_NORM_NR 16
__device__ __forceinline__ float row_rnorm(const float* xi, int g, float eps, float* red) {
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < NSLM_NORM_NR; ++j) {
        const int k = (int) threadIdx.x + j * 256;
        const float xv = xi[min(k, g - 1)];   // unconditional (a conditional load waits for the loads before it)
        const float v = k < g ? xv : 0.0f;
        ss = fmaf(v, v, ss);
    }
    return rsqrtf(wg_sum(ss, red) / (float) g + eps);
}

}   // namespace nslm
