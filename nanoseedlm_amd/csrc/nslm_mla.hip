// nslm_mla.hip - decode attention over a latent KV cache (absorbed MLA) and what feeds it: per-head maps, RoPE with the
// cache write, the FP8 (E4M3 codes, one E8M0 scale per 32 values) cache codec, split-key latent attention and its reduce.
// Replaces the reference's k_heads_mv, k_mla_rope, k_mla_attn / k_mla_reduce, k_kv_f32 and the FP8 half of kvq_put /
// kvq_get8 (engine/kernels_moe.cu:955-1118,1147-1176,1177-1208,1217-1323; the codec's definition is nslm/kvq.h:19-80)
// behind the same launchers.  BF16 and FP8 caches; the FP4 cache format is not built.
//
// Per cached position the kernel reads r + rope values once for ALL heads of a workgroup (multi-query over the shared
// latent): 660 bytes at r = 512, rope 128, FP8 - so the attention of a 4096-token context moves 2.7 MB per row, and what
// it costs is the 2 x (r + rope) multiply-adds per (key, head).  Latent 512 + RoPE 64 runs them on the matrix cores
// (k_mla_attn_mfma: exact BF16 products, f32 sums, P as BF16 hi + lo, which holds the reference tests' bound of one BF16
// ulp + 2e-6 of a double-precision softmax); other shapes stay in f32 on the vector ALUs (k_mla_attn_any).
#include "nslm_mv_dev.h"

using namespace nslm;

namespace {

// ---- the FP8 codec (nslm/kvq.h) ----------------------------------------------------------------------------------------
__device__ __forceinline__ float e4m3_dec(uint32_t c) {
    const int e = (int) ((c >> 3) & 15u), m = (int) (c & 7u);
    const float v = e ? ldexpf(1.0f + (float) m / 8.0f, e - 7) : ldexpf((float) m, -9);
    return (c & 0x80u) ? -v : v;
}
// a >= 0: the E4M3 code of a, rounded to nearest even, saturated at 448
__device__ __forceinline__ uint32_t e4m3_enc_abs(float a) {
    if (!(a < 448.0f)) return 0x7Eu;
    if (a < 0.015625f) return (uint32_t) rintf(a * 512.0f);   // subnormals (8: the smallest normal)
    int e;
    const float f = frexpf(a, &e);   // a = 2f 2^(e - 1), 2f in [1, 2)
    int E = e - 1, m = (int) rintf((2.0f * f - 1.0f) * 8.0f);
    if (m == 8) { ++E; m = 0; }
    const int c = ((E + 7) << 3) | m;
    return (uint32_t) (c > 0x7E ? 0x7E : c);
}
// the E8M0 scale byte of a block with max |x| = amax
__device__ __forceinline__ uint32_t fp8_scale(float amax) {
    if (!(amax > 0.0f)) return 127u;
    int k;
    (void) frexpf(amax, &k);   // amax in [2^(k-1), 2^k); 448 2^(k-9) = 0.875 2^k
    int e = amax <= ldexpf(448.0f, k - 9) ? k - 9 : k - 8;
    e = e < -126 ? -126 : e > 127 ? 127 : e;
    return (uint32_t) (e + 127);
}
// one cached value as the f32 of its BF16 bits (a code times its scale is exact; truncation as the reference packs it)
__device__ __forceinline__ float fp8_value(uint32_t code, uint32_t sc) {
    return __uint_as_float(__float_as_uint(e4m3_dec(code) * ldexpf(1.0f, (int) sc - 127)) & 0xFFFF0000u);
}
// Store value v at dim d of FP8 row `row` (n values) when `store`: the 32 dims of a block are 32 consecutive lanes, which
// share the block's max |v|.  Every lane of the wave calls it.
__device__ __forceinline__ void fp8_put(bool store, float v, uint8_t* C, uint8_t* S, size_t row, int n, int d) {
    float a = fabsf(v);
    for (int o = 1; o < 32; o <<= 1) a = fmaxf(a, __shfl_xor(a, o));
    const uint32_t sc = fp8_scale(a);
    const uint32_t c = e4m3_enc_abs(ldexpf(fabsf(v), 127 - (int) sc));
    if (!store) return;
    C[row * (size_t) n + d] = (uint8_t) (c && v < 0.0f ? c | 0x80u : c);
    if (d % 32 == 0) S[row * (size_t) (n / 32) + d / 32] = (uint8_t) sc;
}

__device__ __forceinline__ KvSeg kv_seg(const KvView& kv, int pos, int* row) {
    if (pos < kv.nv) { *row = pos; return kv.a; }
    *row = pos - kv.nv;
    return kv.b;
}
// dims d .. d + 7 of a cache row (the RoPE key or the latent, n values a row) as f32
__device__ __forceinline__ void cache_get8(int fmt, const void* codes, const void* scales, size_t row, int n, int d, float (&o)[8]) {
    if (fmt == KV_BF16) {
        const uint4 q = ldg16(gp<uint16_t>(codes) + row * (size_t) n + d);
        const uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) { o[2 * i] = __uint_as_float(u[i] << 16); o[2 * i + 1] = __uint_as_float(u[i] & 0xFFFF0000u); }
    } else {
        const uint2 q = ldg8(gp<uint8_t>(codes) + row * (size_t) n + d);
        const uint32_t sc = gp<uint8_t>(scales)[row * (size_t) (n / 32) + d / 32];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[i] = fp8_value((q.x >> (8 * i)) & 255u, sc);
            o[4 + i] = fp8_value((q.y >> (8 * i)) & 255u, sc);
        }
    }
}

// softplus(x, beta = ln 2) in f32, then BF16 (engine/kernels_moe.cu:215-218)
__device__ __forceinline__ float softplus_gate(float g) {
    const float gx = g * 0.69314718055994531f;
    return bfr((fmaxf(gx, 0.0f) + logf(1.0f + expf(-fabsf(gx)))) / 0.69314718055994531f);
}

// ---- per-head maps: y[t][h][o] = bf16(W_h[o] . x[t * xs + h * hs ..]), optionally times bf16(softplus_ln2(g)) ----------
// LPR lanes per output row (a power of two, the row's blocks rounded up), 64 / LPR rows a wave; the lane's blocks and the
// FMA chain per block are k_mv_any's.  Seed maps take head h's exponent bias from W.p[2][h].
__global__ void __launch_bounds__(256) k_heads_mv(HmvArgs a, int fmt, WSlice W, const float* x, const float* g, float* y, int lpr) {
    __shared__ uint32_t tab[NSLM_TAB_WORDS];
    if (fmt == MF_SEED4P4 || fmt == MF_SEED4) {
        load_tables(tab);
        __syncthreads();
    }
    const int tid = threadIdx.x, rpw = 64 / lpr, sub = (tid & 63) / lpr, ln = tid & (lpr - 1);
    const int o = ((int) blockIdx.x * 4 + (tid >> 6)) * rpw + sub, h = (int) blockIdx.y, t = (int) blockIdx.z;
    const bool live = o < a.O;
    const float* xv = x + (size_t) t * a.xs + (size_t) h * a.hs;
    WSlice ws = W;
    if (fmt == MF_SEED4P4) ws.eb = gp<int32_t>(W.p[2])[h];
    float acc = 0.0f;
    if (live)
        for (int j = ln; j < a.I / 8; j += lpr) {
            float w[8], sc;
            block_weights(fmt, ws, tab, h * a.O + o, a.I, j, w, &sc);
            const float* xb = xv + (size_t) j * 8;
            float d = w[0] * xb[0];
#pragma unroll
            for (int c = 1; c < 8; ++c) d = fmaf(w[c], xb[c], d);
            acc = fmaf(d, sc, acc);
        }
    for (int s = lpr >> 1; s > 0; s >>= 1) acc += __shfl_xor(acc, s);
    if (live && ln == 0) {
        const size_t yi = ((size_t) t * a.H + h) * a.O + o;
        float v = bfr(acc);
        if (a.gate) v = bfr(v * softplus_gate(g[yi]));
        y[yi] = v;
    }
}

// ---- RoPE of the query RoPE parts (in place) and of the RoPE key into the cache; the latent into the cache -------------
// The work of a row is cut into jobs of one wave each: job 0 rotates the RoPE key and writes it, job 1 + j writes latent
// dims [64 j, 64 j + 64).  An FP8 block is 32 consecutive values, so it always sits in 32 consecutive lanes of one job and
// its maximum is five shuffles.  (The reference gives thread i latent dim i and, at once, rotation pair i % half of head
// i / half, engine/kernels_moe.cu:1177-1208; here the query heads are a loop of their own over a table of the row's
// sines and cosines, computed once instead of once per head.)
__device__ __forceinline__ void rotate(float x0, float x1, float cs, float sn, float* y0, float* y1) {
    *y0 = __fsub_rn(__fmul_rn(x0, cs), __fmul_rn(x1, sn));   // spelled out: the same bits wherever it is inlined
    *y1 = __fadd_rn(__fmul_rn(x1, cs), __fmul_rn(x0, sn));
}
__device__ __forceinline__ void cache_job(int job, const MlaArgs& a, int rope, const float* kr, const float* c, const KvView& kv, const RowInfo* ri,
                                          const float* inv, int t) {
    const int lane = threadIdx.x & 63, pos = ri[t].pos, half = rope / 2;
    int row;
    const KvSeg sg = kv_seg(kv, ri[t].kv0 + pos, &row);
    if (job == 0) {   // the key: lane p < half holds the pair (p, p + half)
        const bool on = lane < half;
        float y0 = 0.0f, y1 = 0.0f;
        if (on) {
            float sn, cs;
            sincosf((float) pos * inv[lane], &sn, &cs);
            rotate(kr[(size_t) t * rope + lane], kr[(size_t) t * rope + lane + half], cs, sn, &y0, &y1);
        }
        if (kv.fmt == KV_BF16) {
            if (on) {
                uint16_t* kc = (uint16_t*) sg.k + (size_t) row * rope;
                kc[lane] = (uint16_t) tobf(y0);
                kc[lane + half] = (uint16_t) tobf(y1);
            }
        } else {   // every lane runs the shuffles
            fp8_put(on, bfr(y0), (uint8_t*) sg.k, (uint8_t*) sg.ks, (size_t) row, rope, on ? lane : 0);
            fp8_put(on, bfr(y1), (uint8_t*) sg.k, (uint8_t*) sg.ks, (size_t) row, rope, on ? lane + half : 0);
        }
        return;
    }
    const int i = (job - 1) * 64 + lane;
    const bool on = i < a.r;
    const float v = on ? c[(size_t) t * a.r + i] : 0.0f;
    if (kv.fmt == KV_BF16) {
        if (on) ((uint16_t*) sg.v)[(size_t) row * a.r + i] = (uint16_t) tobf(v);
    } else {
        fp8_put(on, bfr(v), (uint8_t*) sg.v, (uint8_t*) sg.vs, (size_t) row, a.r, on ? i : 0);
    }
}
// one workgroup a row: the cache jobs dealt to the four waves, then every query head's pairs
__global__ void __launch_bounds__(256) k_mla_rope(MlaArgs a, int rope, float* qr, const float* kr, const float* c, KvView kv,
                                                  const RowInfo* ri, const float* inv) {
    __shared__ float cs_s[ATT_HD / 2], sn_s[ATT_HD / 2];
    const int t = (int) blockIdx.x, tid = threadIdx.x, half = rope / 2;
    if (tid < half) sincosf((float) ri[t].pos * inv[tid], &sn_s[tid], &cs_s[tid]);
    for (int job = tid >> 6; job < 1 + (a.r + 63) / 64; job += 4) cache_job(job, a, rope, kr, c, kv, ri, inv, t);
    __syncthreads();
    for (int i = tid; i < a.n_head * half; i += 256) {
        const int h = i / half, p = i - h * half;
        float* qh = qr + ((size_t) t * a.n_head + h) * rope;
        float y0, y1;
        rotate(qh[p], qh[p + half], cs_s[p], sn_s[p], &y0, &y1);
        qh[p] = bfr(y0);
        qh[p + half] = bfr(y1);
    }
}

// ---- the two maps of the query, its RoPE, and the cache write as ONE launch -----------------------------------------------
// Grid (1 + r / 64, n_head + 1, rows).  Head h < n_head: block 0 computes the `rope` rows of the RoPE mix
// (k_heads_mv's arithmetic), rotates them (k_mla_rope's) and stores them; block b > 0 computes latent-query rows
// [64 (b - 1), 64 b).  "Head" n_head: the blocks' waves take the cache jobs (the rotated key, the latent).
// The same bits as kc_heads_mv x 2 + kc_mla_rope.
__global__ void __launch_bounds__(256) k_qmaps_rope(MlaArgs a, int rope, HmvArgs hq, HmvArgs hl, int fmt, WSlice Wq, WSlice Wl, const float* q,
                                                   float* qr, float* ql, const float* kr, const float* c, KvView kv, const RowInfo* ri,
                                                   const float* inv, int lpr) {
    __shared__ uint32_t tab[NSLM_TAB_WORDS];
    __shared__ float qs[ATT_HD];
    const int tid = threadIdx.x, h = (int) blockIdx.y, t = (int) blockIdx.z, b = (int) blockIdx.x;
    if (h == a.n_head) {   // uniform over the block: cache jobs 4 b .. 4 b + 3
        const int job = b * 4 + (tid >> 6);
        if (job < 1 + (a.r + 63) / 64) cache_job(job, a, rope, kr, c, kv, ri, inv, t);
        return;
    }
    if (fmt == MF_SEED4P4 || fmt == MF_SEED4) {
        load_tables(tab);
        __syncthreads();
    }
    const bool mix = b == 0;
    const HmvArgs& hm = mix ? hq : hl;
    const int O = hm.O, o0 = mix ? 0 : 64 * (b - 1), o1 = mix ? O : min(o0 + 64, O);
    const int rpw = 64 / lpr, sub = (tid & 63) / lpr, ln = tid & (lpr - 1);
    const float* xv = q + (size_t) t * hm.xs + (size_t) h * hm.hs;
    WSlice ws = mix ? Wq : Wl;
    if (fmt == MF_SEED4P4) ws.eb = gp<int32_t>(ws.p[2])[h];
    for (int ob = o0; ob < o1; ob += 4 * rpw) {
        const int o = ob + (tid >> 6) * rpw + sub;
        const bool live = o < o1;
        float acc = 0.0f;
        if (live)
            for (int j = ln; j < hm.I / 8; j += lpr) {
                float w[8], sc;
                block_weights(fmt, ws, tab, h * O + o, hm.I, j, w, &sc);
                const float* xb = xv + (size_t) j * 8;
                float d = w[0] * xb[0];
#pragma unroll
                for (int cc = 1; cc < 8; ++cc) d = fmaf(w[cc], xb[cc], d);
                acc = fmaf(d, sc, acc);
            }
        for (int sft = lpr >> 1; sft > 0; sft >>= 1) acc += __shfl_xor(acc, sft);
        if (live && ln == 0) {
            if (mix) qs[o] = bfr(acc);
            else ql[((size_t) t * hl.H + h) * O + o] = bfr(acc);
        }
    }
    if (!mix) return;
    __syncthreads();
    const int half = rope / 2;
    if (tid < half) {
        float sn, cs;
        sincosf((float) ri[t].pos * inv[tid], &sn, &cs);
        float y0, y1;
        rotate(qs[tid], qs[tid + half], cs, sn, &y0, &y1);
        float* qh = qr + ((size_t) t * a.n_head + h) * rope;
        qh[tid] = bfr(y0);
        qh[tid + half] = bfr(y1);
    }
}

// ---- latent attention, any shape (f32 on the vector ALUs) ---------------------------------------------------------------------
// Workgroup (split, group of GA_HW heads, row), one query head a wave.  A tile of GA_KT keys (latent, then RoPE key) is decoded
// to f32 in LDS once for the workgroup's heads.
//   scores   lane (key u = lane / 4, quarter q = lane % 4) forms the part of s_u = q . k_u that falls into its quarter of the
//            r + rope dims - sequential reads of the key's LDS row and of the wave's staged query - and two quad shuffles add
//            the quarters: GA_KT scores a wave are ready at once (no wave-wide reduction per key);
//   softmax  the tile's maximum and its sum of exp over the 16 quads: four shuffles each, once a tile;
//   P c      lane l owns latent dims l, l + 64, ...; exp(s_u - m) reaches it as the broadcast of lane 4 u.
// n_splits > 1: partials (m, l, acc[r]) for the reduce; n_splits == 1: olat[row][head] = bf16(acc / l).
#define GA_KT 16
#define GA_HW 4
#define MLA_MAXL 16    // latent dims a lane (r <= 1024)
#define MLA_SPLITS_SHORT 32
// The splits of a row at position pos: the keys of 0..pos in `first` equal runs at most, as few as `chunk` keys a run allow.  Where first is less than the caller's
// n_splits (k_mla_attn_mfma: as many as fill the chip) and a run would be twice cap() or longer, it is cap() keys, and the rest goes in further splits of `rest` keys.
struct MlaSplits {
    int n, first, run, rest;   // (n: splits with keys; run, rest: keys)
    __device__ __forceinline__ void range(int split, int pos, int* p0, int* p1) const {
        *p0 = split < first ? split * run : first * run + (split - first) * rest;
        *p1 = split < n ? min(pos + 1, *p0 + (split < first ? run : rest)) : *p0;
    }
};
#define MLA_REST 512   // keys of a further split, and of a cut run, at least
__device__ __forceinline__ int mla_most(const MlaArgs& a) { return a.pad[2] > 0 && a.n_splits > MLA_SPLITS_SHORT ? MLA_SPLITS_SHORT : a.n_splits; }
template <class Cap>
__device__ __forceinline__ MlaSplits mla_splits(const MlaArgs& a, int first, int pos, Cap cap) {
    const int most = mla_most(a), want = (pos + a.chunk) / a.chunk;
    const int used = max(min(min(first, most), want), 1);
    MlaSplits s = {0, first, max((pos + used) / used, 1), 0};
    s.n = (pos + s.run) / s.run;
    if (__builtin_expect(first < most && s.run >= 2 * MLA_REST, 0)) {
        const int c = cap();
        if (s.run >= 2 * c) {   // (used is first: no run is longer than chunk otherwise)
            const int left = pos + 1 - first * c;   // (at least as long as the cut runs)
            s.run = c;
            s.rest = max(MLA_REST, (left + most - first - 1) / (most - first));
            s.n = first + (left + s.rest - 1) / s.rest;
        }
    }
    return s;
}
// Inclusive sums over the lanes
__device__ __forceinline__ int wave_scan(int v) {
#define STEP(ctrl, rows) v += __builtin_amdgcn_update_dpp(0, v, ctrl, rows, 0xF, false)
    STEP(0x111, 0xF);   // from the lane before, 2, 4, 8 before, of 16
    STEP(0x112, 0xF);
    STEP(0x114, 0xF);
    STEP(0x118, 0xF);
    STEP(0x142, 0xA);   // lane 15 to lanes 16 - 31, 47 to 48 - 63
    STEP(0x143, 0xC);   // lane 31 to lanes 32 - 63
#undef STEP
    return v;
}
// What a run may be twice of before it is cut: the rows' mean length over `first`, doubled; the mean of 64 rows spread over the launch where it has more.
// mla_sample: a lane's one of them, its position, requested before anything else
__device__ __forceinline__ int mla_sample(const RowInfo* ri, int T, int lane) { return ri[T > 64 ? (int) ((long long) lane * T >> 6) : min(lane, T - 1)].pos; }
__device__ __forceinline__ int mla_cap(const MlaArgs& a, int first, int sample, int T, int lane) {
    const int rows = min(T, 64), sum = __builtin_amdgcn_readlane(wave_scan(lane < rows ? max(sample + 1, 0) >> 5 : 0), 63);
    return max(max(MLA_REST, a.chunk), (int) (64.0f * (float) sum / (float) (rows * first)));
}
// part: [row][head][split][r] accumulators, then [row][head][split] (m, l); splits without keys are neither written nor read
__device__ __forceinline__ size_t part_ml(const MlaArgs& a, int T) { return (size_t) T * a.n_head * a.n_splits * a.r; }
__global__ void __launch_bounds__(64 * GA_HW) k_mla_attn_any(MlaArgs a, int rope, const float* ql, const float* qr, KvView kv, const RowInfo* ri,
                                                            float* out) {
    extern __shared__ __attribute__((aligned(16))) float sm[];   // [GA_KT keys][ld] then [GA_HW queries][ld]
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, u = lane >> 2, qt = lane & 3;
    const int split = (int) blockIdx.x, t = (int) blockIdx.z, r = a.r, kw = r + rope, ld = kw + 4, nl = (r + 63) / 64;
    const int h = (int) blockIdx.y * GA_HW + wv;
    const bool live = h < a.n_head;
    float* keys = sm;
    float* qs = sm + GA_KT * ld + wv * ld;
    for (int i = lane; i < kw; i += 64) {   // the wave's query, scaled (its own rows of LDS: no barrier needed before the wave reads them)
        const int hh = live ? h : 0;
        qs[i] = a.scale * (i < r ? ql[((size_t) t * a.n_head + hh) * r + i] : qr[((size_t) t * a.n_head + hh) * rope + (i - r)]);
    }
    int p0, p1;
    mla_splits(a, a.n_splits, ri[t].pos, [] { return 0; }).range(split, ri[t].pos, &p0, &p1);
    if (p0 >= p1 && a.n_splits > 1) return;   // uniform; nobody reads its partials (one split: a row without keys is written, as 0 / 0)
    const int q0 = qt * (kw / 4), q1 = q0 + kw / 4;   // kw % 8 == 0: whole pairs
    float acc[MLA_MAXL];
#pragma unroll
    for (int j = 0; j < MLA_MAXL; ++j) acc[j] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    for (int p = p0; p < p1; p += GA_KT) {
        const int nk = min(GA_KT, p1 - p);
        __syncthreads();
        for (int e = tid; e < nk * (kw / 8); e += 64 * GA_HW) {   // 8 dims a thread (r and rope are multiples of 8)
            const int ku = e / (kw / 8), d = (e - ku * (kw / 8)) * 8;
            int row;
            const KvSeg sg = kv_seg(kv, ri[t].kv0 + p + ku, &row);
            float v[8];
            if (d < r) cache_get8(kv.fmt, sg.v, sg.vs, (size_t) row, r, d, v);
            else cache_get8(kv.fmt, sg.k, sg.ks, (size_t) row, rope, d - r, v);
            float* dst = keys + ku * ld + d;
            *(float4*) dst = make_float4(v[0], v[1], v[2], v[3]);
            *(float4*) (dst + 4) = make_float4(v[4], v[5], v[6], v[7]);
        }
        __syncthreads();
        float sc = 0.0f;
        if (u < nk) {
            const float* kr_ = keys + u * ld;
            for (int i = q0; i < q1; i += 2) {
                const float2 kk = *(const float2*) (kr_ + i), qq = *(const float2*) (qs + i);
                sc = fmaf(qq.x, kk.x, sc);
                sc = fmaf(qq.y, kk.y, sc);
            }
        }
        sc += __shfl_xor(sc, 1);
        sc += __shfl_xor(sc, 2);
        if (u >= nk) sc = -INFINITY;
        float mx = sc;
        for (int o = 4; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        mx = fmaxf(mx, m);
        const float cor = expf(m - mx), e = expf(sc - mx);   // exp(-inf) = 0: keys past the run, and the first tile's m
        float es = e;
        for (int o = 4; o < 64; o <<= 1) es += __shfl_xor(es, o);
        l = fmaf(l, cor, es);
        m = mx;
#pragma unroll
        for (int j = 0; j < MLA_MAXL; ++j) acc[j] *= cor;
#pragma unroll
        for (int ku = 0; ku < GA_KT; ++ku) {
            const float ek = __shfl(e, 4 * ku);
            if (ku >= nk) break;   // uniform
            const float* kr_ = keys + ku * ld;
#pragma unroll
            for (int j = 0; j < MLA_MAXL; ++j)
                if (j < nl && lane + 64 * j < r) acc[j] = fmaf(ek, kr_[lane + 64 * j], acc[j]);
        }
    }
    if (!live) return;
    if (a.n_splits == 1) {
        float* o = out + ((size_t) t * a.n_head + h) * r;
#pragma unroll
        for (int j = 0; j < MLA_MAXL; ++j)
            if (j < nl && lane + 64 * j < r) o[lane + 64 * j] = bfr(acc[j] / l);
    } else {
        const size_t at = ((size_t) t * a.n_head + h) * a.n_splits + split;
        float *pp = out + at * r, *ml = out + part_ml(a, (int) gridDim.z) + 2 * at;
        if (lane == 0) { ml[0] = m; ml[1] = l; }
#pragma unroll
        for (int j = 0; j < MLA_MAXL; ++j)
            if (j < nl && lane + 64 * j < r) pp[lane + 64 * j] = acc[j];
    }
}

// ---- latent attention on the matrix cores ---------------------------------------------------------------------------------
// Absorbed MLA is multi-query attention over the latent: the 16 heads of a group read the same keys, so a tile of keys is
// one MFMA operand for all of them (the reference's default path does the same on its tensor cores,
// engine/kernels_moe.cu:1388-1397, with the same rounding points: queries are BF16 values, products exact, f32 sums,
// f32 online softmax, P entering the second product as two BF16 terms hi + lo).
// Workgroup (split, group of 16 heads, row) of 8 waves, a round = 128 keys, 16 a wave.  Per round:
//   keys    a wave's cache bytes come by loads of whole 128-byte lines (8 lanes a key FP8, 16 BF16: a load whose adjacent lanes are 16 keys, as the MFMA
//           wants them, saves the way through LDS but costs a look-up a lane: one BF16 row of 12 k positions 7 us more), are decoded in
//           registers and go to LDS once, key by key;
//   scores  S^T[key][head] = K Q^T by v_mfma_f32_16x16x32_bf16, the wave's own 16 keys, all r + rope dims: no barrier; Q fragments stay in registers;
//   softmax the waves' maxima meet in LDS (barrier), every wave forms the same reference score and its own keys' P, hi + lo terms, to LDS (barrier);
//   P c     O^T[dim][head] += V P^T, wave w owns latent dims 64 w .. 64 w + 63 over the round's 128 keys.  MFMA contracts over the index that is
//           contiguous in a lane's fragment, here the keys: ds_read_b64_tr_b16 hands a lane four keys of one latent dim, so the same LDS copy serves.
// The next round's cache bytes are requested as soon as this round's are decoded.  FP8 -> BF16 is v_cvt_scalef32_pk_bf16_fp8 (E4M3 code x
// E8M0 scale, exact); the codes 0x7F / 0xFF (never written by the encoder; the reference's decoder reads them as +-480, the instruction as
// NaN) show as a NaN score of their key, and with scales outside [2^-95, 2^96] they send the wave's keys through the arithmetic decoder, so
// every byte decodes as in nslm/kvq.h.
// What bounds it: with all CUs at work the first rounds' bytes come at the rate of a large copy; then a round is 7000 clocks of phases (writes to LDS 1500,
// the scores' chain of reads and MFMAs 1500, two barriers with the softmax 1000, P c 1500), none of the units a third busy.  Tried: workgroups of four
// waves, two a CU (16 rows of 2 to 4 k positions + 6 %, one row of 12 k + 23 %); two rounds' bytes in registers (they spill).  us with the reduce, back to back, FP8 / BF16,
// against tiles of 32 keys decoded twice into LDS by four waves: 16 rows of 2 to 4 k positions 24.0 -> 17.5 / 22.7 -> 20.2, one of 12 k 25.5 -> 16.8 / 23.1 -> 17.0, 32 of 3
// to 6 k 49.0 -> 32.3 / 50.0 -> 39.0, 32 of 0.5 to 1 k 38.0 -> 15.6 / 34.5 -> 17.9, one of 76 13.3 -> 10.1 / 12.5 -> 10.3.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));   // partial results: the caller's buffer promises no more
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u32x2u __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(1)));   // cache rows and scales: at whatever address the caller's views have them
typedef short i16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint32_t bf2(float lo, float hi) {   // v_cvt_pk_bf16_f32: both round to nearest even
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
#define MA_NW 8
#define MA_KEYS (16 * MA_NW)
// A wave's keys in LDS: 16 rows of r values, then 16 of the RoPE key.  A latent row's 16-byte slots are permuted by exclusive or with mla_swz(key): the 16 lanes that
// a 16-byte access serves together ({0-3, 12-15, 20-23, 24-27} and so on) and the 8 keys x 32 bytes of a transposing read then fall on distinct banks.  The RoPE rows'
// slots, with key & 7 (two rows share the banks), serve the writes; their reads, the queries' and the stores of P, 8 bytes of every 16, meet two ways: a third
// of the LDS's active cycles are conflicts.
__device__ __forceinline__ int mla_swz(int key) { return 2 * (key & 7) + (key >> 3); }
template <int R, int ROPE>
constexpr int mla_mfma_lds() { return MA_NW * 16 * 2 * (R + ROPE) + (MA_NW / 2) * 2048 + 2 * 16 * MA_NW * 4; }

template <int R, int ROPE, int FMT, bool CUT, bool AGAIN>
__device__ __forceinline__ void mla_run(const MlaArgs& a, int first, const float* ql, const float* qr, const KvView& kv, const RowInfo* __restrict__ ri, float* part,
                                        float* olat, int T, uint8_t* mla_lds, int t, int split, int sample) {
    static_assert(R == 512 && ROPE == 64, "eight 64-dim slices of the latent, one of the RoPE key, four dim tiles a wave");
    constexpr int KW = R + ROPE, QLD = KW + 8, NS = R / 64, MT = R / 16 / MA_NW, ES = FMT == KV_FP8 ? 1 : 2;
    constexpr int LK = FMT == KV_FP8 ? 8 : 16, KL = 16 * LK / 64, NL = R * ES / (16 * LK);   // lanes a key, keys a lane, 16-byte loads a key and lane
    uint32_t* const Ps = (uint32_t*) (mla_lds + MA_NW * 32 * KW);   // [pair of waves][hi, lo][lane][4]
    float* const mxs = (float*) (Ps + MA_NW / 2 * 512);             // [head][wave]
    float* const ls = mxs + 16 * MA_NW;
    int tid = (int) threadIdx.x;
    if (AGAIN) asm volatile("" : "+v"(tid));   // (a run's own: kept out of the loop over runs, whose registers it would take)
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, g = lane >> 4, h = (int) blockIdx.y * 16 + c;
    const int pos = ri[t].pos, kv0 = ri[t].kv0;
    const size_t th = (size_t) t * a.n_head + h;

    // the group's queries: heads past n_head read head 0 and are zeroed
    constexpr int NQ4 = 16 * KW / 4, QV = (NQ4 + 64 * MA_NW - 1) / (64 * MA_NW);   // float4 in all, and a thread
    u32x4 qv[QV];
#pragma unroll
    for (int i = 0; i < QV; ++i) {
        const int e = min(tid + 64 * MA_NW * i, NQ4 - 1), hh = e < 16 * R / 4 ? e / (R / 4) : (e - 16 * R / 4) / (ROPE / 4);
        const int hq = (int) blockIdx.y * 16 + hh;
        const size_t tq = (size_t) t * a.n_head + (hq < a.n_head ? hq : 0);
        const NSLM_GLOBAL uint32_t* src = e < 16 * R / 4 ? gp<uint32_t>(ql) + tq * R + 4 * (e % (R / 4)) : gp<uint32_t>(qr) + tq * ROPE + 4 * ((e - 16 * R / 4) % (ROPE / 4));
        qv[i] = *(const NSLM_GLOBAL u32x4*) src;
    }
    int p0, p1;
    const MlaSplits sp = mla_splits(a, CUT ? first : a.n_splits, pos, [&] { return mla_cap(a, first, sample, T, lane); });
    sp.range(split, pos, &p0, &p1);
    const bool partial = !olat || sp.n > 1 || (a.n_splits > 1 && first > 1);   // (else the row's one split writes its result)
    if (p0 >= p1) {   // a split without keys (uniform over the workgroup): the reduce does not read it; a row without any is 0 / 0
        if (!partial && h < a.n_head)
            for (int d = 4 * w + g; d < R / 4; d += 4 * MA_NW) *(f32x4u*) (olat + th * R + 4 * d) = f32x4u{NAN, NAN, NAN, NAN};
        return;
    }

    // the keys of a lane's loads, i < KL (of its RoPE loads, i < 2); keys 8 apart lie on adjacent lanes
    const int kr = lane / LK, kj = lane % LK, rr = lane >> 3, rj = lane & 7;
    auto key_of = [&](int i) { return FMT == KV_FP8 ? 8 * (kr & 1) + (kr >> 1) + 4 * i : kr + 4 * i; };
    auto rkey_of = [&](int i) { return 8 * (rr & 1) + (rr >> 1) + 4 * i; };
    struct Raw {
        u32x4 v[KL][NL], vs[2], k[2];   // (k, FP8: two words)
        uint32_t ks[2];
    } raw;
    // Keys past the split's end read its last key (finite values; their scores are masked), so no load is conditional.  A split inside one of the
    // view's segments reads at 32-bit offsets from its first row (two instructions an address), one across both by each key's own segment.
    const bool front = kv0 + p0 < kv.nv, one = front == (kv0 + p1 <= kv.nv) && p1 - p0 <= 1 << 21;
    const size_t row0 = (size_t) (front ? kv0 + p0 : kv0 + p0 - kv.nv);
    const NSLM_GLOBAL uint8_t* const vb0 = gp<uint8_t>(front ? kv.a.v : kv.b.v) + row0 * (R * ES);
    const NSLM_GLOBAL uint8_t* const kb0 = gp<uint8_t>(front ? kv.a.k : kv.b.k) + row0 * (ROPE * ES);
    const NSLM_GLOBAL uint8_t* const vsb0 = gp<uint8_t>(front ? kv.a.vs : kv.b.vs) + row0 * (R / 32);
    const NSLM_GLOBAL uint8_t* const ksb0 = gp<uint8_t>(front ? kv.a.ks : kv.b.ks) + row0 * (ROPE / 32);
    auto row_at = [&](int p, int key, const void* pa, const void* pb, int bytes) {
        const int at = kv0 + min(p + 16 * w + key, p1 - 1);
        const bool f = at < kv.nv;
        return gp<uint8_t>(f ? pa : pb) + (size_t) (f ? at : at - kv.nv) * bytes;
    };
    auto load_keys = [&](Raw& r, int p) {
        if (one) {
            auto row = [&](int key) { return (uint32_t) min(p - p0 + 16 * w + key, p1 - p0 - 1); };
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t u = row(rkey_of(i));
                if constexpr (FMT == KV_FP8) {
                    const u32x2 x = *(const NSLM_GLOBAL u32x2u*) (kb0 + (u * (uint32_t) ROPE + 8u * (uint32_t) rj));
                    r.k[i][0] = x[0];
                    r.k[i][1] = x[1];
                    r.ks[i] = ksb0[u * (uint32_t) (ROPE / 32) + (uint32_t) (rj >> 2)];
                    r.vs[i] = *(const NSLM_GLOBAL u32x4u*) (vsb0 + u * (uint32_t) (R / 32));   // (FP8: the same keys)
                } else r.k[i] = *(const NSLM_GLOBAL u32x4u*) (kb0 + (u * (uint32_t) (2 * ROPE) + 16u * (uint32_t) rj));
            }
#pragma unroll
            for (int i = 0; i < KL; ++i) {
                const uint32_t o = row(key_of(i)) * (uint32_t) (R * ES) + 16u * (uint32_t) kj;
#pragma unroll
                for (int s = 0; s < NL; ++s) r.v[i][s] = *(const NSLM_GLOBAL u32x4u*) (vb0 + (size_t) o + 16 * LK * s);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const NSLM_GLOBAL uint8_t* kb = row_at(p, rkey_of(i), kv.a.k, kv.b.k, ROPE * ES) + 8 * ES * rj;
            if constexpr (FMT == KV_FP8) {
                const u32x2 x = *(const NSLM_GLOBAL u32x2u*) kb;
                r.k[i][0] = x[0];
                r.k[i][1] = x[1];
                r.ks[i] = row_at(p, rkey_of(i), kv.a.ks, kv.b.ks, ROPE / 32)[rj >> 2];
                r.vs[i] = *(const NSLM_GLOBAL u32x4u*) row_at(p, key_of(i), kv.a.vs, kv.b.vs, R / 32);
            } else r.k[i] = *(const NSLM_GLOBAL u32x4u*) kb;
        }
#pragma unroll
        for (int i = 0; i < KL; ++i) {
            const NSLM_GLOBAL uint8_t* vb = row_at(p, key_of(i), kv.a.v, kv.b.v, R * ES) + 16 * kj;
#pragma unroll
            for (int s = 0; s < NL; ++s) r.v[i][s] = *(const NSLM_GLOBAL u32x4u*) (vb + 16 * LK * s);
        }
    };
    auto cvt8 = [&](uint32_t x0, uint32_t x1, float f) {   // 8 codes x the scale
        return u32x4{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x0, f, false)), __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x0, f, true)),
                     __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x1, f, false)), __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x1, f, true))};
    };
    auto cvt8_exact = [&](uint32_t x0, uint32_t x1, uint32_t sc) {
        u32x4 d;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t wd = (i < 2 ? x0 : x1) >> (16 * (i & 1));
            d[i] = (__float_as_uint(fp8_value(wd & 255u, sc)) >> 16) | (__float_as_uint(fp8_value((wd >> 8) & 255u, sc)) & 0xFFFF0000u);
        }
        return d;
    };
    uint8_t *const Vw = mla_lds + w * 32 * R, *const Kw = mla_lds + MA_NW * 32 * R + w * 32 * ROPE;   // the wave's keys
    // (a latent slot's low four bits and the sixteens of slots apart: the permutation reaches the first alone, the second is an instruction's offset)
    auto vslot = [&](int key, int low, int high) { return (u32x4*) (Vw + 2 * R * key + 16 * (low ^ mla_swz(key)) + 256 * high); };
    auto kslot = [&](int key, int slot) { return (u32x4*) (Kw + 2 * ROPE * key + 16 * (slot ^ (key & 7))); };

    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f;
    load_keys(raw, p0);
    bf16x8 qf[NS + 1][2];
    {   // queries -> BF16 rows in LDS (over the keys, which the first round stores after the barrier below) -> the wave's B fragments
        uint16_t* Qs = (uint16_t*) mla_lds;
#pragma unroll
        for (int i = 0; i < QV; ++i) {
            const int e = tid + 64 * MA_NW * i, hh = e < 16 * R / 4 ? e / (R / 4) : (e - 16 * R / 4) / (ROPE / 4);
            const int d = e < 16 * R / 4 ? 4 * (e % (R / 4)) : R + 4 * ((e - 16 * R / 4) % (ROPE / 4));
            const uint32_t keep = (int) blockIdx.y * 16 + hh < a.n_head ? 0xFFFFFFFFu : 0u;
            if (e < NQ4)
                *(u32x2*) &Qs[hh * QLD + d] = u32x2{bf2(__uint_as_float(qv[i][0]), __uint_as_float(qv[i][1])) & keep,
                                                    bf2(__uint_as_float(qv[i][2]), __uint_as_float(qv[i][3])) & keep};
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s <= NS; ++s)
#pragma unroll
            for (int i = 0; i < 2; ++i) qf[s][i] = *(const bf16x8*) &Qs[c * QLD + 64 * s + 16 * g + 8 * i];
        __syncthreads();
    }
    // the wave's 16 keys x 16 heads, from its own rows in LDS; dims 64 s + 16 g + 8 i of key c are lane (c, g)'s
    auto scores = [&]() {
        f32x4 s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = s0;   // two chains
#pragma unroll
        for (int s = 0; s <= NS; ++s) {
            const bf16x8 k0 = *(const bf16x8*) (s < NS ? vslot(c, 8 * (s & 1) + 2 * g, s >> 1) : kslot(c, 2 * g));
            const bf16x8 k1 = *(const bf16x8*) (s < NS ? vslot(c, 8 * (s & 1) + 2 * g + 1, s >> 1) : kslot(c, 2 * g + 1));
            s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, qf[s][0], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, qf[s][1], s1, 0, 0, 0);
        }
        return s0 + s1;
    };
    // Online softmax against a reference score m per head that is raised only when a round's maximum exceeds it by more than
    // MLA_LAZY (so P <= e^MLA_LAZY and the accumulators are rescaled on few rounds); l and acc are in the scale e^-m.
    constexpr float MLA_LAZY = 8.0f;
    // lane (c, g) of a transposing read: key 4 g + c / 4, four dims from 4 (c % 4) of a tile
    const int vkey = 4 * g + (c >> 2), vx = ((c >> 1) & 1) ^ mla_swz(vkey);
    const uint8_t* const vrow = mla_lds + 2 * R * vkey + 8 * (c & 1) + 256 * (w >> 1);   // (tile 4 w + mt: slots 8 w + 2 mt, + 1)
    for (int p = p0; p < p1; p += MA_KEYS) {
        Raw& r = raw;
        const int n = p1 - p;                       // keys left
        const bool mine = 32 * (w >> 1) < n;        // (a pair of waves shares a fragment of P: both or none)
        float sv[4], mx = -INFINITY;
        if (mine) {
            bool odd = false;
            if constexpr (FMT == KV_FP8) {   // scale bytes in [32, 223]: b + 32 has one of its two top bits (a byte that overflows shows itself)
                uint32_t ok = 0x80808080u;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
#pragma unroll
                    for (int j = 0; j < 5; ++j) {
                        const uint32_t x = (j < 4 ? r.vs[i][j & 3] : r.ks[i] | 0x7F7F7F00u) + 0x20202020u;
                        ok &= x | (x << 1);
                    }
                }
                odd = (ok & 0x80808080u) != 0x80808080u;
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
                *kslot(rkey_of(i), rj) = FMT == KV_FP8 ? cvt8(r.k[i][0], r.k[i][1], __uint_as_float(r.ks[i] << 23)) : r.k[i];
#pragma unroll
            for (int i = 0; i < KL; ++i)
#pragma unroll
                for (int s = 0; s < NL; ++s) {
                    if constexpr (FMT == KV_FP8) {   // dims 128 s + 16 kj ..: scale byte 4 s + kj / 2
                        const float f = __uint_as_float(r.vs[i][s] >> (8 * (kj >> 1)) << 23 & 0x7F800000u);
                        *vslot(key_of(i), 2 * kj, s) = cvt8(r.v[i][s][0], r.v[i][s][1], f);
                        *vslot(key_of(i), 2 * kj + 1, s) = cvt8(r.v[i][s][2], r.v[i][s][3], f);
                    } else *vslot(key_of(i), kj, s) = r.v[i][s];
                }
            load_keys(r, p + MA_KEYS);
            f32x4 s0 = scores();
            if constexpr (FMT == KV_FP8) {
                odd |= s0[0] != s0[0] || s0[1] != s0[1] || s0[2] != s0[2] || s0[3] != s0[3];
                if (__any(odd)) {   // the arithmetic decoder for the wave's keys
#pragma unroll 1
                    for (int i = 0; i < 2; ++i) {
                        const u32x2 x = *(const NSLM_GLOBAL u32x2u*) (row_at(p, rkey_of(i), kv.a.k, kv.b.k, ROPE) + 8 * rj);
                        *kslot(rkey_of(i), rj) = cvt8_exact(x[0], x[1], row_at(p, rkey_of(i), kv.a.ks, kv.b.ks, ROPE / 32)[rj >> 2]);
#pragma unroll 1
                        for (int s = 0; s < NL; ++s) {
                            const u32x4 y = *(const NSLM_GLOBAL u32x4u*) (row_at(p, key_of(i), kv.a.v, kv.b.v, R) + 16 * kj + 128 * s);
                            const uint32_t sc = row_at(p, key_of(i), kv.a.vs, kv.b.vs, R / 32)[4 * s + (kj >> 1)];
                            *vslot(key_of(i), 2 * kj, s) = cvt8_exact(y[0], y[1], sc);
                            *vslot(key_of(i), 2 * kj + 1, s) = cvt8_exact(y[2], y[3], sc);
                        }
                    }
                    s0 = scores();
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sv[j] = 16 * w + 4 * g + j < n ? s0[j] * a.scale : -INFINITY;
                mx = fmaxf(mx, sv[j]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
        }
        if (g == 0) mxs[c * MA_NW + w] = mx;
        __syncthreads();
        {
            const f32x4 a0 = *(const f32x4*) (mxs + c * MA_NW), a1 = *(const f32x4*) (mxs + c * MA_NW + 4);
            mx = fmaxf(fmaxf(fmaxf(a0[0], a0[1]), fmaxf(a0[2], a0[3])), fmaxf(fmaxf(a1[0], a1[1]), fmaxf(a1[2], a1[3])));
        }
        const bool up = mx > m + MLA_LAZY;   // true on the first round (m = -inf; every round has a key, so mx is finite); the same in every wave
        if (__any(up)) {
            const float cor = up ? __expf(m - mx) : 1.0f;
            m = up ? mx : m;
            l *= cor;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[mt] *= cor;
        }
        if (mine) {
            uint32_t* const pd = Ps + (w >> 1) * 512 + 4 * lane + 2 * (w & 1);
            u32x2 bh, bl;
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
                const float e0 = __expf(sv[j] - m), e1 = __expf(sv[j + 1] - m);   // masked keys: exp(-inf) = 0
                l += e0 + e1;
                bh[j >> 1] = bf2(e0, e1);
                bl[j >> 1] = bf2(e0 - __uint_as_float(bh[j >> 1] << 16), e1 - __uint_as_float(bh[j >> 1] & 0xFFFF0000u));
            }
            *(u32x2*) pd = bh;
            *(u32x2*) (pd + 256) = bl;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < MA_NW / 2; ++q) {
            if (32 * q >= n) break;   // uniform
            const bf16x8 ph = *(const bf16x8*) (Ps + q * 512 + 4 * lane), pl = *(const bf16x8*) (Ps + q * 512 + 256 + 4 * lane);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const uint8_t* const v = vrow + 2 * q * 32 * R + 16 * ((8 * (w & 1) + 2 * mt) ^ vx);
                const i16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*) v);
                const i16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*) (v + 32 * R));
                const bf16x8 vt = __builtin_bit_cast(bf16x8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
                acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt, ph, acc[mt], 0, 0, 0);
                acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt, pl, acc[mt], 0, 0, 0);
            }
        }
        if (n > MA_KEYS) __syncthreads();   // the next round writes V
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (g == 0) ls[c * MA_NW + w] = l;
    __syncthreads();
    {
        const f32x4 a0 = *(const f32x4*) (ls + c * MA_NW), a1 = *(const f32x4*) (ls + c * MA_NW + 4);
        l = ((a0[0] + a0[1]) + (a0[2] + a0[3])) + ((a1[0] + a1[1]) + (a1[2] + a1[3]));
    }
    if (h >= a.n_head) return;
    if (!partial) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int d = 16 * (MT * w + mt) + 4 * g;
            *(f32x4u*) (olat + th * R + d) = f32x4u{bfr(acc[mt][0] / l), bfr(acc[mt][1] / l), bfr(acc[mt][2] / l), bfr(acc[mt][3] / l)};
        }
    } else {
        const size_t at = th * a.n_splits + split;
        if (w == 0 && g == 0) *(f32x2u*) (part + part_ml(a, T) + 2 * at) = f32x2u{m, l};
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int d = 16 * (MT * w + mt) + 4 * g;
            *(f32x4u*) (part + at * R + d) = acc[mt];
        }
    }
}
// Workgroup (split of the first ones, 16 heads, row).  CUT: where first is less than n_splits, the further splits of rows much longer than the others are then dealt
// to all workgroups of a head group, one after the other.  The host does not know the rows' lengths; the kernel looks for such rows behind a workgroup's own
// run, which is another copy of the code: in one loop with the further ones it took 11 % longer, and a list of all the launch's keys dealt evenly,
// made before the first load, 1.6 us (16 rows of 2 to 4 k positions 17.3 -> 19.3).  us with as many splits of every row -> this, FP8: one row of 16 k positions
// among 31 of 200 55 -> 34 (BF16 59 -> 35), among 128 of 500 357 -> 54; 4 of 8 k among 60 of 300 57 -> 44, 20 among 180 of 500 186 -> 124.  Rows alike: the same,
// but where there are more than half as many as CUs (first 1) the reduce, with nothing to do, adds 3 us: 129 of 2 to 4 k 95 -> 98.
template <int R, int ROPE, int FMT, bool CUT>
__global__ void __launch_bounds__(64 * MA_NW) k_mla_attn_mfma(MlaArgs a, int first, const float* ql, const float* qr, KvView kv, const RowInfo* __restrict__ ri,
                                                             float* part, float* olat, int T) {
    extern __shared__ __attribute__((aligned(16))) uint8_t mla_lds[];
    const int tid = (int) threadIdx.x, lane = tid & 63, sample = CUT ? mla_sample(ri, T, lane) : 0;
    int t = (int) blockIdx.z, split = (int) blockIdx.x, pos = CUT ? ri[min(T > 64 ? tid : lane, T - 1)].pos : 0;   // (no branch: it would wait for the loads)
    mla_run<R, ROPE, FMT, CUT, false>(a, first, ql, qr, kv, ri, part, olat, T, mla_lds, t, split, sample);
    if constexpr (!CUT) return;
    if (T <= 64 && !__any(pos >= (2 * MLA_REST - 1) * first)) return;
    const int cap = mla_cap(a, first, sample, T, lane), from = (2 * cap - 1) * first;   // (where runs of 2 cap keys begin)
    if (T <= 64) {
        if (!__any(pos >= from)) return;
    } else {
        bool some = pos >= from;
        for (int i = tid + 64 * MA_NW; i < T; i += 64 * MA_NW) some |= ri[i].pos >= from;
        int* const flags = (int*) mla_lds;   // (the keys: read for the last time before a run's last barrier)
        if (lane == 0) flags[tid >> 6] = 0;
        if (__any(some) && lane == 0) flags[tid >> 6] = 1;
        __syncthreads();
        if (!__any(flags[lane & 7])) return;
        __syncthreads();
    }
    for (int blk = 0, base = 0, item = first * t + split; blk < T;) {   // rows blk + lane; the further splits of the rows before; the next to do
        pos = ri[min(blk + lane, T - 1)].pos;
        const MlaSplits s = mla_splits(a, first, pos, [&] { return cap; });
        const int more = blk + lane < T ? max(s.n - first, 0) : 0, upto = base + wave_scan(more);
        const uint64_t past = __ballot(upto > item);
        if (!past) {
            base = __builtin_amdgcn_readlane(upto, 63);
            blk += 64;
            continue;
        }
        const int l = __builtin_ctzll(past);
        t = blk + l;
        split = first + item - __builtin_amdgcn_readlane(upto - more, l);
        item += (int) gridDim.x * T;
        mla_run<R, ROPE, FMT, true, true>(a, first, ql, qr, kv, ri, part, olat, T, mla_lds, t, split, sample);
    }
}

// The splits of a (row, head) summed, a workgroup of 256 threads: o[i] = bf16(acc / l) of latent dims d0 + i, i < 256 NQ, as far as r reaches.  Wave w takes
// splits w, w + 4, ... (of whole quads of dims, 16 bytes a load) and the four sums meet in LDS; every wave forms the splits' weights exp(m_s - m) itself, a
// split a lane, and takes them from there by v_readlane.  The loads of the first 32 splits, as far as every row may have
// them, are requested before anything waits, the row's position included: what a split without keys left in the buffer is not used.
#define MLA_RED_MAXS 256
template <int NQ, bool CUT>
__device__ __forceinline__ void mla_reduce(const MlaArgs& a, int n1, int T, int t, int h, int d0, const RowInfo* ri, int sample, const float* part, f32x4 (&sum)[4][64 * NQ], float* o) {
    constexpr int PF = 8, NM = MLA_RED_MAXS / 64;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r = a.r;
    const size_t th = (size_t) t * a.n_head + h;
    const NSLM_GLOBAL float* pa = gp<float>(part) + th * a.n_splits * r;
    const NSLM_GLOBAL float* pm = gp<float>(part) + part_ml(a, T) + 2 * th * a.n_splits;
    const int pos = ri[t].pos, first = CUT ? n1 : a.n_splits;
    int q[NQ];
#pragma unroll
    for (int k = 0; k < NQ; ++k) q[k] = min(d0 + 4 * (lane + 64 * k), r - 4);
    f32x2 ml[NM];
    f32x4 pv[NQ][PF];
#pragma unroll
    for (int i = 0; i < NM; ++i) ml[i] = *(const NSLM_GLOBAL f32x2u*) (pm + 2 * min(lane + 64 * i, a.n_splits - 1));
#pragma unroll
    for (int j = 0; j < PF; ++j)
#pragma unroll
        for (int k = 0; k < NQ; ++k) pv[k][j] = *(const NSLM_GLOBAL f32x4u*) (pa + (size_t) min(w + 4 * j, first - 1) * r + q[k]);
    loads_issued();
    const int ns = mla_splits(a, first, pos, [&] { return mla_cap(a, first, sample, T, lane); }).n;
    float m = -INFINITY, l = 0.0f, c[NM];
#pragma unroll
    for (int i = 0; i < NM; ++i) m = fmaxf(m, lane + 64 * i < ns ? ml[i][0] : -INFINITY);
    for (int s = 32; s > 0; s >>= 1) m = fmaxf(m, __shfl_xor(m, s));
#pragma unroll
    for (int i = 0; i < NM; ++i) {
        const bool on = lane + 64 * i < ns;
        c[i] = on && ml[i][0] != -INFINITY ? expf(ml[i][0] - m) : 0.0f;
        l = on ? fmaf(ml[i][1], c[i], l) : l;
    }
    for (int s = 32; s > 0; s >>= 1) l += __shfl_xor(l, s);
    f32x4 acc[NQ];
#pragma unroll
    for (int k = 0; k < NQ; ++k) acc[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto add = [&](const f32x4 (&v)[NQ], float wt) {
#pragma unroll
        for (int k = 0; k < NQ; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[k][i] = fmaf(v[k][i], wt, acc[k][i]);
    };
#pragma unroll
    for (int i = 0; i < NM; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int s = 64 * i + w + 4 * j;
            if (s >= ns) break;   // uniform
            const float wt = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c[i]), s & 63));
            f32x4 v[NQ];
#pragma unroll
            for (int k = 0; k < NQ; ++k)
                v[k] = i == 0 && j < PF && (!CUT || s < first) ? pv[k][j < PF ? j : 0] : *(const NSLM_GLOBAL f32x4u*) (pa + (size_t) s * r + q[k]);
            add(v, wt);
        }
#pragma unroll
    for (int k = 0; k < NQ; ++k) sum[w][lane + 64 * k] = acc[k];
    __syncthreads();
    const float* sf = (const float*) sum;
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
        const int i = tid + 256 * k;
        const float v = (sf[i] + sf[256 * NQ + i]) + (sf[512 * NQ + i] + sf[768 * NQ + i]);
        if (d0 + i < r) o[i] = bfr(v / l);
    }
}
// olat[t][h][d] = bf16(acc / l).  Workgroup (head, row, 256 latent dims).  FEW (first 1: most rows' one split has written their results): heads blockIdx.x, + gridDim.x, ..
template <bool CUT, bool FEW>
__global__ void __launch_bounds__(256) k_mla_reduce(MlaArgs a, int first, const RowInfo* ri, const float* part, float* olat) {
    __shared__ f32x4 sum[4][64];
    int h = (int) blockIdx.x;
    const int t = (int) blockIdx.y, d0 = (int) blockIdx.z * 256, T = (int) gridDim.y, lane = (int) threadIdx.x & 63, sample = CUT ? mla_sample(ri, T, lane) : 0;
    if (FEW && mla_splits(a, first, ri[t].pos, [&] { return mla_cap(a, first, sample, T, lane); }).n <= 1) return;
    for (;;) {
        mla_reduce<1, CUT>(a, first, T, t, h, d0, ri, sample, part, sum, olat + ((size_t) t * a.n_head + h) * a.r + d0);
        h += (int) gridDim.x;
        if (!FEW || h >= a.n_head) return;
        __syncthreads();
    }
}

// The splits' reduce and the value-up map of a head in ONE launch: workgroup (row group, head, row) reduces the head's
// latent output into LDS (k_mla_reduce's arithmetic, 512 dims a pass: the map needs them all) and computes rows
// [RG g, RG (g + 1)) of y[t][h] = bf16(W_h . olat[t][h]) (k_heads_mv's arithmetic).  The same bits as the two kernels.
#define MLA_RV_GROUPS 16   // row groups a head at most: fewer when there are many (row, head) pairs, each group re-reads the partials
template <bool CUT>
__global__ void __launch_bounds__(256) k_mla_reduce_vup(MlaArgs a, int first, const RowInfo* ri, const float* part, HmvArgs hv, int fmt, WSlice W, float* y,
                                                       int lpr) {
    __shared__ uint32_t tab[NSLM_TAB_WORDS];
    __shared__ f32x4 sum[4][128];
    __shared__ __attribute__((aligned(16))) float ol[64 * MLA_MAXL];
    constexpr int NP = 2;   // map passes whose loads are issued before anything waits
    const int g = (int) blockIdx.x, h = (int) blockIdx.y, t = (int) blockIdx.z, r = a.r, tid = threadIdx.x, sample = CUT ? mla_sample(ri, (int) gridDim.z, tid & 63) : 0;
    const int rg = (hv.O + (int) gridDim.x - 1) / (int) gridDim.x, o0 = g * rg, o1 = min(o0 + rg, hv.O);
    const int rpw = 64 / lpr, sub = (tid & 63) / lpr, ln = tid & (lpr - 1);
    // BF16 maps, one block a lane: the map rows of the first NP passes are in flight beside the splits
    const bool pre = fmt == MF_BF16 && hv.I / 8 == lpr && (((uintptr_t) W.p[0] | (uintptr_t) (2 * hv.I)) & 15u) == 0;
    uint4 wq[NP];
    if (pre) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int o = min(o0 + i * 4 * rpw + (tid >> 6) * rpw + sub, hv.O - 1);
            wq[i] = ldg16(gp<uint16_t>(W.p[0]) + ((size_t) h * hv.O + o) * hv.I + (size_t) ln * 8);
        }
    }
    if (fmt == MF_SEED4P4 || fmt == MF_SEED4) load_tables(tab);
    for (int d0 = 0; d0 < r; d0 += 512) {
        mla_reduce<2, CUT>(a, first, (int) gridDim.z, t, h, d0, ri, sample, part, sum, ol + d0);
        __syncthreads();
    }
    WSlice ws = W;
    if (fmt == MF_SEED4P4) ws.eb = gp<int32_t>(W.p[2])[h];
    auto finish = [&](int o, bool live, float acc) {
        for (int sft = lpr >> 1; sft > 0; sft >>= 1) acc += __shfl_xor(acc, sft);
        if (live && ln == 0) y[((size_t) t * hv.H + h) * hv.O + o] = bfr(acc);
    };
    int ob = o0;
    if (pre) {   // one block a lane from the prefetched rows: the same products and sums as the loop below
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            if (ob >= o1) break;
            const int o = ob + (tid >> 6) * rpw + sub;
            const uint4 q = wq[i];
            const float* xb = ol + (size_t) ln * 8;
            float d = bf(q.x & 0xFFFFu) * xb[0];
            d = fmaf(bf(q.x >> 16), xb[1], d);
            d = fmaf(bf(q.y & 0xFFFFu), xb[2], d);
            d = fmaf(bf(q.y >> 16), xb[3], d);
            d = fmaf(bf(q.z & 0xFFFFu), xb[4], d);
            d = fmaf(bf(q.z >> 16), xb[5], d);
            d = fmaf(bf(q.w & 0xFFFFu), xb[6], d);
            d = fmaf(bf(q.w >> 16), xb[7], d);
            finish(o, o < o1, fmaf(d, 1.0f, 0.0f));
            ob += 4 * rpw;
        }
    }
    for (; ob < o1; ob += 4 * rpw) {
        const int o = ob + (tid >> 6) * rpw + sub;
        const bool live = o < o1;
        float acc = 0.0f;
        if (live)
            for (int j = ln; j < hv.I / 8; j += lpr) {
                float wv[8], sc;
                block_weights(fmt, ws, tab, h * hv.O + o, hv.I, j, wv, &sc);
                const float* xb = ol + (size_t) j * 8;
                float d = wv[0] * xb[0];
#pragma unroll
                for (int cc = 1; cc < 8; ++cc) d = fmaf(wv[cc], xb[cc], d);
                acc = fmaf(d, sc, acc);
            }
        finish(o, live, acc);
    }
}

// y = `rows` FP8 cache rows of n values, decoded (8 values a thread; for tests)
__global__ void k_kv_f32(int fmt, const uint8_t* C, const uint8_t* S, int n, int rows, float* y) {
    const int i = ((int) blockIdx.x * (int) blockDim.x + threadIdx.x) * 8;
    if (i >= n * rows) return;
    float v[8];
    cache_get8(fmt, C, S, (size_t) (i / n), n, i % n, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) y[i + j] = v[j];
}

int rope_of(const MlaArgs& a) { return a.pad[0] > 0 ? a.pad[0] : ATT_HD; }

}   // namespace

extern "C" {

void kc_heads_mv(kc_stream_t s, HmvArgs a, int fmt, WSlice W, const uint32_t* G, const float* x, const float* g, float* y, int T) {
    (void) G;
    if (T < 1 || a.H < 1 || a.O < 1 || a.I < 8) return;
    int lpr = 1;
    while (lpr < 64 && lpr < a.I / 8) lpr <<= 1;
    const int rows_wg = 4 * (64 / lpr);
    hipLaunchKernelGGL(k_heads_mv, dim3((unsigned) (a.O + rows_wg - 1) / rows_wg, (unsigned) a.H, (unsigned) T), dim3(256), 0, (hipStream_t) s,
                       a, fmt, W, x, g ? g : x, y, lpr);
    host_note_launch();
}
void kc_mla_rope(kc_stream_t s, MlaArgs a, float* qr, const float* kr, const float* c, KvView kv, const RowInfo* ri, const float* inv,
                 int T) {
    const int rope = rope_of(a);
    if (T < 1 || (kv.fmt != KV_BF16 && kv.fmt != KV_FP8) || (rope != 64 && rope != 128) || a.r % 32) { host_note_unsupported(); return; }
    hipLaunchKernelGGL(k_mla_rope, dim3((unsigned) T), dim3(256), 0, (hipStream_t) s, a, rope, qr, kr, c, kv, ri, inv);
    host_note_launch();
}
int kc_mla_qmaps_rope(kc_stream_t s, MlaArgs a, HmvArgs hq, HmvArgs hl, int fmt, WSlice Wq, WSlice Wl, const float* q, float* qr, float* ql,
                      const float* kr, const float* c, KvView kv, const RowInfo* ri, const float* inv, int T) {
    const int rope = rope_of(a);
    int lpr = 1;
    while (lpr < 64 && lpr < hq.I / 8) lpr <<= 1;
    if (T < 1 || (kv.fmt != KV_BF16 && kv.fmt != KV_FP8) || (rope != 64 && rope != 128) || a.r % 64 || hq.O != rope || hl.O != a.r || hq.I != hl.I ||
        hq.I % 8 || hq.I / 8 > 64 || lpr != hq.I / 8 || hq.H != a.n_head || hl.H != a.n_head || hq.gate || hl.gate || hq.xs != hl.xs || hq.hs != hl.hs)
        return -1;
    const int bx = 1 + a.r / 64;   // >= the cache jobs' blocks: (1 + r / 64 + 3) / 4
    hipLaunchKernelGGL(k_qmaps_rope, dim3((unsigned) bx, (unsigned) a.n_head + 1, (unsigned) T), dim3(256), 0, (hipStream_t) s, a, rope, hq, hl, fmt,
                       Wq, Wl, q, qr, ql, kr, c, kv, ri, inv, lpr);
    host_note_launch();
    return 0;
}
// Attention into the partials or olat, and the reduce; olat NULL: into the partials alone.  *first: the launch's first splits.  false: unsupported, nothing launched
static bool mla_attn_launch(kc_stream_t s, const MlaArgs& a, const float* ql, const float* qr, KvView kv, const RowInfo* ri, float* part, float* olat,
                            int T, int* first) {
    const int rope = rope_of(a);
    if (T < 1 || (kv.fmt != KV_BF16 && kv.fmt != KV_FP8) || (rope != 64 && rope != 128) || a.r % 8 || a.r > 64 * MLA_MAXL || a.n_splits < 1) {
        host_note_unsupported();
        return false;
    }
    if (a.n_splits > MLA_RED_MAXS) { host_note_unsupported(); return false; }
    *first = a.n_splits;
    if (a.r == 512 && rope == 64 && (((uintptr_t) ql | (uintptr_t) qr) & 15u) == 0) {   // the matrix-core kernel: 16 heads a workgroup
        constexpr int lds = mla_mfma_lds<512, 64>();
        static const hipError_t once[4] = {
            hipFuncSetAttribute((const void*) k_mla_attn_mfma<512, 64, KV_BF16, false>, hipFuncAttributeMaxDynamicSharedMemorySize, lds),
            hipFuncSetAttribute((const void*) k_mla_attn_mfma<512, 64, KV_FP8, false>, hipFuncAttributeMaxDynamicSharedMemorySize, lds),
            hipFuncSetAttribute((const void*) k_mla_attn_mfma<512, 64, KV_BF16, true>, hipFuncAttributeMaxDynamicSharedMemorySize, lds),
            hipFuncSetAttribute((const void*) k_mla_attn_mfma<512, 64, KV_FP8, true>, hipFuncAttributeMaxDynamicSharedMemorySize, lds)};
        (void) once;
        // A workgroup fills a CU: more splits of every row than fill the chip only add partials (2 KB a head and split, written and read again).  (Two or three where two
        // do not fit, by the chip's turns at them: 129 rows of 2 to 4 k positions 98 -> 84 us, 160 of 0.5 to 1 k 33 -> 43, 300 of 128 to 256 26 -> 48.)
        const int groups = (a.n_head + 15) / 16, fill = host_cu_count() / (groups * T);
        *first = a.n_splits < fill ? a.n_splits : fill < 1 ? 1 : fill;
        const bool cut = *first < a.n_splits;
        const dim3 grid((unsigned) *first, (unsigned) groups, (unsigned) T);
#define LAUNCH(FMT, CUT) hipLaunchKernelGGL((k_mla_attn_mfma<512, 64, FMT, CUT>), grid, dim3(64 * MA_NW), lds, (hipStream_t) s, a, *first, ql, qr, kv, ri, part, olat, T)
        if (kv.fmt == KV_FP8) { if (cut) LAUNCH(KV_FP8, true); else LAUNCH(KV_FP8, false); }
        else { if (cut) LAUNCH(KV_BF16, true); else LAUNCH(KV_BF16, false); }
#undef LAUNCH
    } else {
        float* o = a.n_splits > 1 ? part : olat;
        const size_t lds = sizeof(float) * (size_t) (GA_KT + GA_HW) * (size_t) (a.r + rope + 4);
        static const hipError_t once = hipFuncSetAttribute((const void*) k_mla_attn_any, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                           (int) (sizeof(float) * (GA_KT + GA_HW) * (64 * MLA_MAXL + ATT_HD + 4)));
        (void) once;
        hipLaunchKernelGGL(k_mla_attn_any, dim3((unsigned) a.n_splits, (unsigned) (a.n_head + GA_HW - 1) / GA_HW, (unsigned) T), dim3(64 * GA_HW), lds,
                           (hipStream_t) s, a, rope, ql, qr, kv, ri, o);
    }
    if (a.n_splits > 1 && olat) {
        const bool few = *first == 1;
        const int at_once = few && T < 1024 ? 1024 / T : few ? 1 : a.n_head;   // (few: as many workgroups as the chip holds, most of them to end at once)
        const dim3 grid((unsigned) (at_once < a.n_head ? at_once : a.n_head), (unsigned) T, (unsigned) (a.r + 255) / 256);
#define LAUNCH(CUT, FEW) hipLaunchKernelGGL((k_mla_reduce<CUT, FEW>), grid, dim3(256), 0, (hipStream_t) s, a, *first, ri, part, olat)
        if (few) LAUNCH(true, true);
        else if (*first < a.n_splits) LAUNCH(true, false);
        else LAUNCH(false, false);
#undef LAUNCH
    }
    host_note_launch();
    return true;
}
void kc_mla_attn(kc_stream_t s, MlaArgs a, const float* ql, const float* qr, KvView kv, const RowInfo* ri, float* part, float* olat,
                 int T) {
    int first;
    (void) mla_attn_launch(s, a, ql, qr, kv, ri, part, olat, T, &first);
}
int kc_mla_attn_vup(kc_stream_t s, MlaArgs a, const float* ql, const float* qr, KvView kv, const RowInfo* ri, float* part, HmvArgs hv, int fmt,
                    WSlice W, float* y, int T) {
    int lpr = 1, first;
    while (lpr < 64 && lpr < hv.I / 8) lpr <<= 1;
    if (a.n_splits < 2 || a.n_splits > MLA_RED_MAXS || hv.I != a.r || a.r % 8 || a.r > 64 * MLA_MAXL || hv.H != a.n_head || hv.gate ||
        (lpr != hv.I / 8 && hv.I / 8 <= 64) || hv.O < 1)
        return -1;
    if (!mla_attn_launch(s, a, ql, qr, kv, ri, part, NULL, T, &first)) return -1;
    int groups = 1024 / (a.n_head * T);   // about a thousand workgroups
    groups = groups < 1 ? 1 : groups > MLA_RV_GROUPS ? MLA_RV_GROUPS : groups;
#define LAUNCH(CUT)                                                                                                                                              \
    hipLaunchKernelGGL(k_mla_reduce_vup<CUT>, dim3((unsigned) groups, (unsigned) a.n_head, (unsigned) T), dim3(256), 0, (hipStream_t) s, a, first, ri, part, hv, \
                       fmt, W, y, lpr)
    if (first < a.n_splits) LAUNCH(true); else LAUNCH(false);
#undef LAUNCH
    host_note_launch();
    return 0;
}
void kc_kv_f32(kc_stream_t s, int fmt, const uint8_t* codes, const uint8_t* scales, int n, int rows, float* y) {
    if (rows < 1 || n < 8 || (fmt != KV_BF16 && fmt != KV_FP8)) { host_note_unsupported(); return; }
    hipLaunchKernelGGL(k_kv_f32, dim3((unsigned) ((n * rows / 8 + 127) / 128)), dim3(128), 0, (hipStream_t) s, fmt, codes, scales, n, rows, y);
    host_note_launch();
}

}   // extern "C"
