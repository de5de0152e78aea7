// Products of few rows an expert (9 .. a few hundred tokens; some decode calls of 3 .. 8): the weights are
// streamed once, straight from HBM into registers, and every token of a tile shares them.
//
// A tile is up to 32 sorted pairs of one expert (64 rows of a linear).  A block of 8 waves
// takes one tile and 8 row tiles of 16 weight rows (gate/up: 8 of gate and the same 8 of up,
// both in the same wave), and walks the whole K range or a split of it.  Lane (r, p) of a
// wave owns row r's quarter p (64 weights) of each 256-weight super-block, as in the decode
// GEMVs: 16-byte loads of whole 256-byte row runs, the quarter's own scales decoded once,
// no weight bytes through LDS.  A k step of v_mfma_f32_16x16x32_f16 takes 8 weights of each
// quarter (the order of k inside a product is free as long as both operands agree), so a
// super-block is 8 steps of 16 tokens x 16 rows.  The tokens' fp16 rows are the other
// operand: staged through two LDS buffers, one stage ahead of its use and a super-block's
// share at a time, with as many super-blocks a stage as the tile's rows leave room for.
//
// Against the 256 x 256 tiles of gemm.hip, which one expert's few rows leave nearly empty:
// no decoded scale plane is read (44 % more bytes than Q4_K's own), two blocks share a CU, so
// loads stay in flight across the barriers, and 16 tokens cost 16 rows of MFMA.
//
// What bounds it: the weight stream.  Mixtral-shaped gate/up, 24 tokens (529 MB of Q4_K): 209
// us on the 256-row tiles, 111-116 here (4.6-4.8 TB/s).  Qwen3 shape, 32
// tokens: gate/up 84 -> 42 us, down 58 -> 33; H = 4096, I = 12288 FFN of 20 rows 74 -> 44 us;
// 4096 x 6144 Q4_K linear of 33 rows 25 -> 18.6 us.  Tried and slower: two K halves in one
// block (shorter units, no better end: 43 -> 47 us), 64-pair tiles with one row tile a wave for
// gate/up (102 -> 106 us a layer; the tokens are staged twice as often), weights requested two
// super-blocks ahead (3-5 %).
// Reference: GGUFQuantMoEExperts.forward_expert (quant_kernels.py:1990-2011) ->
// exec_w4a16_matmul / exec_w8a16_matmul (:1165-1420) and model.py:916-919.
#include <algorithm>

#include "common.h"
#include "decode_kernels.h"
#include "launch.h"

namespace pgmoe {

constexpr int kThinRows = 64;  // most pairs a tile
constexpr int kThinWaves = 8;
constexpr int kThinThreads = 64 * kThinWaves;
constexpr int kThinSums = 64 * 80;  // bytes of a stage's sub-block sums
constexpr int kThinStage = kThinRows * (512 + 16);  // bytes of an LDS stage (any rows x super-blocks split)

typedef _Float16 th8 __attribute__((ext_vector_type(8)));
typedef _Float16 th2 __attribute__((ext_vector_type(2)));
typedef __bf16 tb8 __attribute__((ext_vector_type(8)));
typedef float tf4 __attribute__((ext_vector_type(4)));
typedef _Float16 th4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- weight decode
// Each lane turns its quarter's codes into fp16 MFMA operands with packed fp16 arithmetic
// (4 cycles for two weights; v_fma_mixlo / mixhi_f16 take 8 each, v_fma_mix_f32 and
// v_cvt_pk_f16_f32 4 each) that is exact, or rounds as the fp32 form would:
//   Q4_K, Q5_K: sc q (an integer below 2048, exact); the products of a super-block are summed
//               unscaled and then take d in fp32 (POST); the minima are a second product, of
//               the 6-bit m and the tokens' fp32 sums over each sub-block as three bf16 pieces
//               (their 24 bits, so exact as well), which takes dmin in fp32 (MINS);
//   Q6_K      : sc (q - 32), rounded once above 2048; d in fp32 (POST);
//   Q8_0      : d q, rounded once (the bits of the fp32 product rounded to fp16);
//   Q4_1      : d q + m in fp32, rounded once (d and m are fp16: no integer form);
//   F16       : as stored.
__device__ __forceinline__ th2 as_h2(uint32_t v) { return __builtin_bit_cast(th2, v); }
__device__ __forceinline__ th2 h2(float v) { return th2{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ th2 pk_fma(th2 a, th2 b, th2 c) { return __builtin_elementwise_fma(a, b, c); }
__device__ __forceinline__ th8 cat8(const th2 (&v)[4]) {
    return th8{v[0].x, v[0].y, v[1].x, v[1].y, v[2].x, v[2].y, v[3].x, v[3].y};
}

// Constants of the decode held in registers: v_and_or_b32 takes no literal, and one scalar.
struct ThinConst {
    uint32_t magic, mask, mask2;  // 0x6400 twice (fp16 1024); code masks of byte pairs
    uint32_t sh, sd, md, ml;      // header shifts and masks of a K-quant lane's quarter (thin_kscales)
};
template <int QT>
__device__ __forceinline__ ThinConst thin_const(int p) {
    ThinConst k{};
    k.magic = 0x64006400u;
    k.mask = QT == PGMOE_Q5_K ? 0x001f001fu : QT == PGMOE_Q6_K ? 0x003f003fu : 0x000f000fu;
    k.mask2 = 0x00f000f0u;
    asm("" : "+v"(k.magic));
    asm("" : "+s"(k.mask));
    asm("" : "+s"(k.mask2));
    if constexpr (QT == PGMOE_Q4_K || QT == PGMOE_Q5_K) {
        k.sh = 16 * (p & 1);
        k.sd = k.sh + (p < 2 ? 0 : 2);
        k.md = p < 2 ? 0x3f3fu : 0x3030u;
        k.ml = p < 2 ? 0u : 0x0f0fu;
    }
    if constexpr (QT == PGMOE_Q6_K) k.sh = 8 * (p & 1);
    return k;
}

// Codes 0 and 2, then 1 and 3, of a word's bytes under `mask` as fp16 pairs 1024 + (byte &
// mask): one v_and_or_b32 a pair.  The staged activations have the same order inside every
// four elements (thin_permute).
__device__ __forceinline__ void thin_codes(const ThinConst& k, uint32_t w, uint32_t mask, th2& m0, th2& m1) {
    m0 = as_h2((w & mask) | k.magic);
    m1 = as_h2(((w >> 8) & mask) | k.magic);
}
__device__ __forceinline__ uint32_t thin_bfi(uint32_t mask, uint32_t a, uint32_t b) { return (mask & a) | (~mask & b); }

// A lane's quarter: pair(i), i = 0..3, gives the 8-weight fragments of two k steps;
// elem(i, half) is a fragment's first element, from base(p).
template <int QT> struct ThinW;

// (scale, min) of sub-blocks 2p (low byte) and 2p + 1 from a K-quant header: for p < 2 six bits
// of D's and Mb's bytes, else the nibbles of MD's bytes with the top two bits of D's and Mb's.
__device__ __forceinline__ void thin_kscales(const ThinConst& k, const u32x4& h, uint32_t& sc, uint32_t& mn) {
    sc = ((h.y >> k.sd) & k.md) | ((h.w >> k.sh) & k.ml);
    mn = ((h.z >> k.sd) & k.md) | ((h.w >> (k.sh + 4)) & k.ml);
}
struct ThinK {  // the header of Q4_K and Q5_K
    static constexpr bool POST = true, MINS = true;
    uint32_t ddm, mn;  // d and dmin (fp16); the minima of sub-blocks 2p, 2p + 1 (bytes)
    th2 s0, s1;        // their scales, twice
    __device__ __forceinline__ ThinK(const ThinConst& kc, const u32x4& h) {
        uint32_t sc;
        thin_kscales(kc, h, sc, mn);
        ddm = h.x;
        s0 = as_h2(__builtin_amdgcn_perm(kc.magic, sc, 0x05000500u)) - h2(1024.0f);
        s1 = as_h2(__builtin_amdgcn_perm(kc.magic, sc, 0x05010501u)) - h2(1024.0f);
    }
    __device__ __forceinline__ float scale() const { return lo_half(ddm); }
    __device__ __forceinline__ float min_scale() const { return hi_half(ddm); }
    __device__ __forceinline__ tb8 mins() const {  // each minimum (6 bits, exact) against three pieces of its sum
        const uint32_t f0 = __builtin_bit_cast(uint32_t, (float)(mn & 0xff));
        const uint32_t f1 = __builtin_bit_cast(uint32_t, (float)((mn >> 8) & 0xff));
        const uint32_t a = __builtin_amdgcn_perm(f0, f0, 0x03020302u), b = __builtin_amdgcn_perm(f1, f1, 0x03020302u);
        return __builtin_bit_cast(tb8, u32x4{a, a, b, b});
    }
    __device__ static __forceinline__ constexpr int elem(int i, int half) { return 8 * i + 32 * half; }
    __device__ static __forceinline__ int base(int p) { return 64 * p; }
};
template <> struct ThinW<PGMOE_Q4_K> : ThinK {
    uint32_t w[8];
    th2 c0, c1;
    __device__ __forceinline__ ThinW(const ThinConst& kc, const Qtr<PGMOE_Q4_K>& q) : ThinK(kc, q.h) {
        w[0] = q.a.x, w[1] = q.a.y, w[2] = q.a.z, w[3] = q.a.w;
        w[4] = q.b.x, w[5] = q.b.y, w[6] = q.b.z, w[7] = q.b.w;
        s1 = s1 * h2(0.0625f);  // the high nibbles are read in place, as 1024 + 16 q
        c0 = s0 * h2(-1024.0f);
        c1 = s1 * h2(-1024.0f);
    }
    __device__ __forceinline__ void pair(const ThinConst& kc, int i, th8& lo, th8& hi) const {
        th2 m[4], n[4];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            thin_codes(kc, w[2 * i + k], kc.mask, m[2 * k], m[2 * k + 1]);
            thin_codes(kc, w[2 * i + k], kc.mask2, n[2 * k], n[2 * k + 1]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            m[k] = pk_fma(m[k], s0, c0);
            n[k] = pk_fma(n[k], s1, c1);
        }
        lo = cat8(m);
        hi = cat8(n);
    }
};
template <> struct ThinW<PGMOE_Q5_K> : ThinK {
    uint32_t w[8], hx, hy;
    th2 c0, c1;
    __device__ __forceinline__ ThinW(const ThinConst& kc, const Qtr<PGMOE_Q5_K>& q) : ThinK(kc, q.h) {
        w[0] = q.a.x, w[1] = q.a.y, w[2] = q.a.z, w[3] = q.a.w;
        w[4] = q.b.x, w[5] = q.b.y, w[6] = q.b.z, w[7] = q.b.w;
        hx = q.hb.x;
        hy = q.hb.y;
        c0 = s0 * h2(-1024.0f);
        c1 = s1 * h2(-1024.0f);
    }
    __device__ __forceinline__ void pair(const ThinConst& kc, int i, th8& lo, th8& hi) const {
        th2 m[4], n[4];
#pragma unroll
        for (int k = 0; k < 2; ++k) {  // word j: the fifth bits of its four elements are bits j + 8b of hx / hy
            const int j = 2 * i + k;
            const uint32_t bx = j < 4 ? hx << (4 - j) : hx >> (j - 4), by = j < 4 ? hy << (4 - j) : hy >> (j - 4);
            thin_codes(kc, thin_bfi(0x10101010u, bx, w[j]), kc.mask, m[2 * k], m[2 * k + 1]);
            thin_codes(kc, thin_bfi(0x10101010u, by, w[j] >> 4), kc.mask, n[2 * k], n[2 * k + 1]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            m[k] = pk_fma(m[k], s0, c0);
            n[k] = pk_fma(n[k], s1, c1);
        }
        lo = cat8(m);
        hi = cat8(n);
    }
};
template <> struct ThinW<PGMOE_Q6_K> {
    static constexpr bool POST = true, MINS = false;
    float d;
    __device__ __forceinline__ float scale() const { return d; }
    th2 s01, s23;  // scales of sub-blocks s = 0, 1 and 2, 3
    uint32_t la[4], lb[4], qh[4];
    __device__ __forceinline__ ThinW(const ThinConst& kc, const Qtr<PGMOE_Q6_K>& q) {
        d = h2f((uint16_t)q.d);
        s01 = as_h2((((q.sc.x >> kc.sh) & 0x00ff00ffu) ^ 0x00800080u) | kc.magic) - h2(1152.0f);
        s23 = as_h2((((q.sc.y >> kc.sh) & 0x00ff00ffu) ^ 0x00800080u) | kc.magic) - h2(1152.0f);
        la[0] = q.la.x, la[1] = q.la.y, la[2] = q.la.z, la[3] = q.la.w;
        lb[0] = q.lb.x, lb[1] = q.lb.y, lb[2] = q.lb.z, lb[3] = q.lb.w;
        qh[0] = q.qh.x, qh[1] = q.qh.y, qh[2] = q.qh.z, qh[3] = q.qh.w;
    }
    // step pair i: chunk la (i even) or lb, its first or second 8 bytes; sub-blocks s = i & 1
    // (low nibbles) and s + 2 (high), high bits 2s of each qh byte.  EX: what the rounding above
    // 2048 took away too (-1, 0 or 1: exact), so that lo + rlo and hi + rhi are sc (q - 32).
    __device__ __forceinline__ void pair(const ThinConst& kc, int i, th8& lo, th8& hi) const {
        th8 rlo, rhi;
        pair<false>(kc, i, lo, hi, rlo, rhi);
    }
    template <bool EX>
    __device__ __forceinline__ void pair(const ThinConst& kc, int i, th8& lo, th8& hi, th8& rlo, th8& rhi) const {
        th2 m[4], n[4], rm[4], rn[4];
        const int s = i & 1;
        const th2 a = s ? th2{s01.y, s01.y} : th2{s01.x, s01.x}, b = s ? th2{s23.y, s23.y} : th2{s23.x, s23.x};
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int j = 2 * (i >> 1) + k;
            const uint32_t l = s ? lb[j] : la[j], h = qh[j];
            thin_codes(kc, thin_bfi(0x30303030u, s ? h << 2 : h << 4, l), kc.mask, m[2 * k], m[2 * k + 1]);
            thin_codes(kc, thin_bfi(0x30303030u, s ? h >> 2 : h, l >> 4), kc.mask, n[2 * k], n[2 * k + 1]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const th2 cm = m[k] - h2(1056.0f), cn = n[k] - h2(1056.0f);
            m[k] = cm * a;
            n[k] = cn * b;
            if constexpr (EX) {
                rm[k] = pk_fma(cm, a, -m[k]);
                rn[k] = pk_fma(cn, b, -n[k]);
            }
        }
        lo = cat8(m);
        hi = cat8(n);
        if constexpr (EX) {
            rlo = cat8(rm);
            rhi = cat8(rn);
        }
    }
    __device__ static __forceinline__ constexpr int elem(int i, int half) {
        return 32 * (i & 1) + 8 * (i >> 1) + 64 * half;
    }
    __device__ static __forceinline__ int base(int p) { return 128 * (p >> 1) + 16 * (p & 1); }
};
template <> struct ThinW<PGMOE_Q8_0> {
    static constexpr bool POST = false, MINS = false;
    th2 dd;  // d of blocks 2p, 2p + 1
    u32x4 c[4];
    __device__ __forceinline__ ThinW(const ThinConst&, const Qtr<PGMOE_Q8_0>& q) {
        dd = as_h2(q.d);
        c[0] = q.c0, c[1] = q.c1, c[2] = q.c2, c[3] = q.c3;
    }
    __device__ __forceinline__ void pair(const ThinConst& kc, int i, th8& lo, th8& hi) const {
        const th2 a = i < 2 ? th2{dd.x, dd.x} : th2{dd.y, dd.y};
        const uint32_t v[4] = {c[i].x ^ 0x80808080u, c[i].y ^ 0x80808080u, c[i].z ^ 0x80808080u, c[i].w ^ 0x80808080u};
        th2 m[4], n[4];  // 1152 + q, bytes (0, 2) and (1, 3) of each word
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            m[2 * k] = as_h2(__builtin_amdgcn_perm(kc.magic, v[k], 0x05020500u));
            m[2 * k + 1] = as_h2(__builtin_amdgcn_perm(kc.magic, v[k], 0x05030501u));
            n[2 * k] = as_h2(__builtin_amdgcn_perm(kc.magic, v[2 + k], 0x05020500u));
            n[2 * k + 1] = as_h2(__builtin_amdgcn_perm(kc.magic, v[2 + k], 0x05030501u));
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            m[k] = (m[k] - h2(1152.0f)) * a;
            n[k] = (n[k] - h2(1152.0f)) * a;
        }
        lo = cat8(m);
        hi = cat8(n);
    }
    __device__ static __forceinline__ constexpr int elem(int i, int half) { return 16 * i + 8 * half; }
    __device__ static __forceinline__ int base(int p) { return 64 * p; }
};
template <> struct ThinW<PGMOE_Q4_1> {
    static constexpr bool POST = false, MINS = false;
    float a0, c0, a1, c1;
    uint32_t w[8];
    __device__ __forceinline__ ThinW(const ThinConst&, const Qtr<PGMOE_Q4_1>& q) {
        a0 = lo_half(q.dw);
        c0 = lo_half(q.mw) - 1024.0f * a0;
        const float a = hi_half(q.dw);
        c1 = hi_half(q.mw) - 64.0f * a;
        a1 = a * 0.0625f;
        w[0] = q.a.x, w[1] = q.a.y, w[2] = q.a.z, w[3] = q.a.w;
        w[4] = q.b.x, w[5] = q.b.y, w[6] = q.b.z, w[7] = q.b.w;
    }
    __device__ __forceinline__ static th2 deq(th2 v, float a, float c) {
        return th2{(_Float16)__builtin_fmaf((float)v.x, a, c), (_Float16)__builtin_fmaf((float)v.y, a, c)};
    }
    __device__ __forceinline__ void pair(const ThinConst& kc, int i, th8& lo, th8& hi) const {
        th2 m[4], n[4];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            thin_codes(kc, w[2 * i + k], kc.mask, m[2 * k], m[2 * k + 1]);
            thin_codes(kc, w[2 * i + k], kc.mask2, n[2 * k], n[2 * k + 1]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            m[k] = deq(m[k], a0, c0);
            n[k] = deq(n[k], a1, c1);
        }
        lo = cat8(m);
        hi = cat8(n);
    }
    __device__ static __forceinline__ constexpr int elem(int i, int half) { return 8 * i + 32 * half; }
    __device__ static __forceinline__ int base(int p) { return 64 * p; }
};
template <> struct ThinW<PGMOE_F16> {
    static constexpr bool POST = false, MINS = false;
    u32x4 c[8];
    __device__ __forceinline__ ThinW(const ThinConst&, const Qtr<PGMOE_F16>& q) {
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = q.c[i];
    }
    __device__ __forceinline__ void pair(const ThinConst&, int i, th8& lo, th8& hi) const {
        lo = __builtin_bit_cast(th8, c[2 * i]);
        hi = __builtin_bit_cast(th8, c[2 * i + 1]);
    }
    __device__ static __forceinline__ constexpr int elem(int i, int half) { return 16 * i + 8 * half; }
    __device__ static __forceinline__ int base(int p) { return 64 * p; }
};

// 8 activations in thin_codes' order: elements 0, 2, 1, 3 of each four.
template <int QT>
__device__ __forceinline__ u32x4 thin_permute(u32x4 v) {
    if constexpr (QT == PGMOE_F16) return v;
    u32x4 r;
    r.x = __builtin_amdgcn_perm(v.y, v.x, 0x05040100u);
    r.y = __builtin_amdgcn_perm(v.y, v.x, 0x07060302u);
    r.z = __builtin_amdgcn_perm(v.w, v.z, 0x05040100u);
    r.w = __builtin_amdgcn_perm(v.w, v.z, 0x07060302u);
    return r;
}

__device__ __forceinline__ float thin_act(int act, float g) {  // gemm.hip's hardware exp2 / reciprocal forms
    const float z = 0.7978845608028654f * (g + 0.044715f * g * g * g);
    return act ? g - g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(2.8853900817779268f * z))
               : g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * g));
}

// Quarter loads of super-block tile t (wave-uniform, at the row tile's first row): the lane
// part of every address is one of two 32-bit offsets, off0 (the row's 16 bytes) and offp (the
// quarter's first chunk of them); d: the row tile's d plane position (Q6_K).
template <int QT>
__device__ __forceinline__ void thin_offsets(int lane, int p, uint32_t& off0, uint32_t& offp) {
    off0 = (lane & 15) * 16;
    offp = off0;
    if constexpr (QT == PGMOE_Q4_K || QT == PGMOE_Q5_K) offp += (1 + 2 * p) * 1024;
    else if constexpr (QT == PGMOE_Q4_1) offp += (2 + 2 * p) * 1024;
    else if constexpr (QT == PGMOE_Q6_K) offp += (4 * (p >> 1) + (p & 1)) * 1024;
    else if constexpr (QT == PGMOE_Q8_0) offp += 4 * p * 1024;
    else offp += 8 * p * 1024;
}
template <int QT>
__device__ __forceinline__ void thin_load(Qtr<QT>& q, const uint8_t* t, const uint8_t* d, uint32_t off0, uint32_t offp,
                                          int lane, int p) {
    if constexpr (QT == PGMOE_Q4_1) {
        q.dw = *(const uint32_t*)(t + (off0 + 4 * p));
        q.mw = *(const uint32_t*)(t + (off0 + 4 * p) + 1024);
        q.a = ldq(t + offp);
        q.b = ldq(t + offp + 1024);
    } else if constexpr (QT == PGMOE_Q4_K || QT == PGMOE_Q5_K) {
        q.h = ldq(t + off0);
        q.a = ldq(t + offp);
        q.b = ldq(t + offp + 1024);
        if constexpr (QT == PGMOE_Q5_K) q.hb = *(const u32x2*)(t + (off0 + (9 + (p >> 1)) * 1024 + 8 * (p & 1)));
    } else if constexpr (QT == PGMOE_Q6_K) {
        q.la = ldq(t + offp);
        q.lb = ldq(t + offp + 2048);
        q.qh = ldq(t + (off0 + (8 + 2 * (p >> 1) + (p & 1)) * 1024));
        q.sc = *(const u32x2*)(t + (off0 + 12 * 1024 + 8 * (p >> 1)));  // bytes 2s + (p & 1) are the quarter's
        q.d = *(const uint16_t*)(d + (uint32_t)(2 * (lane & 15)));
    } else if constexpr (QT == PGMOE_F16) {
#pragma unroll
        for (int i = 0; i < 8; ++i) q.c[i] = ldq(t + (offp + (i & ~3) * 1024) + (i & 3) * 1024);
    } else {
        q.c0 = ldq(t + offp);
        q.c1 = ldq(t + offp + 1024);
        q.c2 = ldq(t + offp + 2048);
        q.c3 = ldq(t + offp + 3072);
        q.d = *(const uint32_t*)(t + (off0 + 16 * 1024 + 4 * p));
    }
}

struct ThinArgs {
    const uint8_t *w0, *w1;      // gate / up, or the one matrix
    int64_t stride0, stride1;    // between experts
    int N, K;
    const uint16_t* act;         // fp16 rows: tokens (gather through perm) or pair rows
    int gather, topk;            // gather: row of pair p is perm[p] / topk, else p
    int E, P;                    // E = 0: one matrix, pairs 0 .. P - 1 in order
    const int32_t *offsets, *perm, *tile_off;
    const float *rs, *topk_w;    // row scale and pair weight (null: 1)
    const float* bias;           // per output column (null: none)
    void* out;                   // fp32 rows [P][N] (fp16 with out_f16)
    int out_f16, act_kind;
    int kper;                    // super-blocks a split
    float* raw;                  // split K: raw sums [split][P][NC]
};

// A finite fp32 value as three bf16 pieces that add up to it, then a zero.  An infinity or NaN
// gives NaN, which thin_non_finite takes back where the call has to.
__device__ __forceinline__ u32x2 thin_split3(float v) {
    const uint32_t a = __builtin_bit_cast(uint32_t, v) & 0xffff0000u;
    const float r = v - __builtin_bit_cast(float, a);
    const uint32_t b = __builtin_bit_cast(uint32_t, r) & 0xffff0000u;
    const uint32_t c = __builtin_bit_cast(uint32_t, r - __builtin_bit_cast(float, b));
    return u32x2{(a >> 16) | b, c >> 16};
}

// Stage shape of a tile of NT token tiles: SPB super-blocks, a row 512 SPB + 16 bytes, so that
// the 16 rows of a fragment read fall on 16 bank groups.
template <int NT>
struct ThinStage {
    static constexpr int SPB = 4 / NT, ROW = 512 * SPB + 16, PIECES = 32 * SPB;  // 16-byte pieces a row
    static constexpr int SUMS = 64 * SPB + 16;  // bytes a row: 8 of each 32-element sub-block (thin_split3)
    static_assert(16 * NT * ROW <= kThinStage && 16 * NT * SUMS <= kThinSums, "a stage fits its buffers");
};

// One super-block of the wave's R row tiles over NT token tiles; load(r, b) requests row tile
// r's super-block b (R = 1: the next one before this one's products, else after them).  D of
// a product: lane l holds weight row l % 16 of tokens 4 (l / 16) + 0..3, so a row's scale is
// in the lanes that decoded it.
template <int QT, int R, int NT, bool LOAD, bool EX, class Load>
__device__ __forceinline__ void thin_block(const ThinConst& kc, const uint8_t* x, const uint8_t* xs, tf4 (&acc)[R][NT],
                                           Qtr<QT> (&q)[R], Load& load, int b) {
    constexpr int T = 16 * ThinStage<NT>::ROW;
    using W = ThinW<QT>;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const W w(kc, q[r]);
        if constexpr (LOAD && (R == 1 || NT == 1)) load(r, b + 1);
        tf4 sum[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) sum[t] = W::POST ? tf4{0.f, 0.f, 0.f, 0.f} : acc[r][t];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            th8 lo, hi, xl[NT], xh[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) xl[t] = *(const th8*)(x + T * t + 2 * W::elem(i, 0));
            if constexpr (NT * R <= 2) {
#pragma unroll
                for (int t = 0; t < NT; ++t) xh[t] = *(const th8*)(x + T * t + 2 * W::elem(i, 1));
            }
            th8 rlo, rhi;
            if constexpr (EX && QT == PGMOE_Q6_K)
                w.template pair<true>(kc, i, lo, hi, rlo, rhi);
            else
                w.pair(kc, i, lo, hi);
#pragma unroll
            for (int t = 0; t < NT; ++t) sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[t], lo, sum[t], 0, 0, 0);
            if constexpr (EX && QT == PGMOE_Q6_K)
#pragma unroll
                for (int t = 0; t < NT; ++t) sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[t], rlo, sum[t], 0, 0, 0);
            if constexpr (NT * R > 2) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < NT; ++t) xh[t] = *(const th8*)(x + T * t + 2 * W::elem(i, 1));
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[t], hi, sum[t], 0, 0, 0);
            if constexpr (EX && QT == PGMOE_Q6_K)
#pragma unroll
                for (int t = 0; t < NT; ++t) sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[t], rhi, sum[t], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (LOAD && R > 1 && NT > 1) load(r, b + 1);
        if constexpr (W::POST) {
            const float d = w.scale();
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[r][t][v] = __builtin_fmaf(d, sum[t][v], acc[r][t][v]);
        } else {
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[r][t] = sum[t];
        }
        if constexpr (W::MINS) {
            const tb8 mv = w.mins();
            const float dm = -w.min_scale();
#pragma unroll
            for (int t = 0; t < NT; ++t)
                sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const tb8*)(xs + 16 * ThinStage<NT>::SUMS * t), mv,
                                                                 tf4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[r][t][v] = __builtin_fmaf(dm, sum[t][v], acc[r][t][v]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// Element k (from super-block tile t on) of a Q4_K / Q5_K row as the 256-row tiles hold it, rounded
// to fp16 (off0: the row's 16 bytes).
template <int QT>
__device__ __forceinline__ float thin_weight(const uint8_t* t, uint32_t off0, int k) {
    t += (int64_t)(k >> 8) * (Tile<QT>::CH * 1024) + off0;
    const int s = (k >> 5) & 7, l = k & 31, j = 32 * (s >> 1) + l;  // sub-block, element of it, byte of qs
    const u32x4 h = ldq(t);
    int sc, mn, q = (t[(1 + (j >> 4)) * 1024 + (j & 15)] >> (4 * (s & 1))) & 15;
    if constexpr (QT == PGMOE_Q5_K) q |= ((t[(9 + (s >> 2)) * 1024 + 4 * (s & 3) + (l & 3)] >> (l >> 2)) & 1) << 4;
    kscale_sel(h.y, h.z, h.w, s, sc, mn);
    const float a = lo_half(h.x) * (float)sc, c = -(hi_half(h.x) * (float)mn) - 1024.0f * a;
    return (float)(_Float16)__builtin_fmaf(1024.0f + (float)q, a, c);
}

// The sums of a Q4_K / Q5_K token with an infinity or NaN are NaN here (the codes and the minima
// are products of their own: inf - inf, or inf times a zero code), where the sum of x w is +-inf
// wherever the terms that are not finite agree.  So where the K elements at x hold such terms, f
// is their sum alone, with the weights (weight(r, k): row tile r's, element k) rounded to fp16 as
// the 256-row tiles round them.  Runs only in waves that hold a NaN.
template <int R, class Weight>
__device__ __forceinline__ bool thin_non_finite(const uint16_t* x, int K, const Weight& weight, float (&f)[R]) {
    bool hit = false;
#pragma unroll
    for (int r = 0; r < R; ++r) f[r] = 0.f;
#pragma unroll 1
    for (int k = 0; k < K; k += 8) {
        const u32x4 v = ldq((const uint8_t*)(x + k));
#pragma unroll 1
        for (int c = 0; c < 8; ++c) {
            const uint32_t w = c < 4 ? (c < 2 ? v.x : v.y) : (c < 6 ? v.z : v.w);
            const uint16_t b = (uint16_t)(w >> (16 * (c & 1)));
            if ((b & 0x7c00) != 0x7c00) continue;
            hit = true;
#pragma unroll
            for (int r = 0; r < R; ++r) f[r] = __builtin_fmaf(h2f(b), weight(r, k + c), f[r]);
        }
    }
    return hit;
}

// A wave's part of a tile of n <= 16 NT pairs from m0: the K loop and the epilogue (a whole
// copy a token-tile count, so that one's registers never meet another's).  smem: two stages
// of rows, then two of sums.  weight: thin_non_finite's.
template <int QT, bool GATEUP, int R, int NT, bool EX, class Load, class Weight>
__device__ __forceinline__ void thin_tile(const ThinArgs& A, uint8_t* smem, const uint32_t* rowsrc, const float* rowscale,
                                          const ThinConst& kc, int m0, int n, int row0, int b0, int nsb,
                                          Qtr<QT> (&q)[R], Load& load, const Weight& weight) {
    using S = ThinStage<NT>;
    using W = ThinW<QT>;
    constexpr int CP = 16 * NT * S::PIECES / kThinThreads / S::SPB;  // 16-byte copies a thread and super-block step
    constexpr int RP = kThinThreads / S::PIECES;                      // rows a copy of the block covers
    const int tid = threadIdx.x, lane = tid & 63, p = lane >> 4;
    // The next stage's pieces move a few at a time, beside each super-block of this one: copy
    // c of step k is 16 bytes of row RP (CP k + c) + tid / PIECES.
    // The thread's place is formed anew at each step (opaque): held across the loop it costs
    // registers, and a spilled one a reload that waits for every weight load in flight.
    auto place = [&](int& pc, int& pr0) {
        int t = tid;
        asm volatile("" : "+v"(t));
        pc = t % S::PIECES, pr0 = t / S::PIECES;
    };
    auto fetch = [&](int s, int k, u32x4(&buf)[CP]) {
        int pc, pr0;
        place(pc, pr0);
#pragma unroll
        for (int c = 0; c < CP; ++c) {  // rows past n repeat row n - 1 (rowsrc), pieces past the split its last
            const int at = min(32 * S::SPB * s + pc, 32 * nsb - 1);
            buf[c] = *(const u32x4*)(A.act + (rowsrc[RP * (CP * k + c) + pr0] + (uint32_t)(256 * b0 + 8 * at)));
        }
    };
    auto put = [&](int s, int k, const u32x4(&buf)[CP]) {
        int pc, pr0;
        place(pc, pr0);
#pragma unroll
        for (int c = 0; c < CP; ++c) {
            const int r = RP * (CP * k + c) + pr0;
            if constexpr (W::MINS) {  // four lanes hold a sub-block's 32 elements (whole waves: xor_lane)
                const th8 h = __builtin_bit_cast(th8, buf[c]);
                float v = (((float)h[0] + (float)h[1]) + ((float)h[2] + (float)h[3])) +
                          (((float)h[4] + (float)h[5]) + ((float)h[6] + (float)h[7]));
                v += xor_lane<1>(v);
                v += xor_lane<2>(v);
                if ((tid & 3) == 0)
                    *(u32x2*)(smem + 2 * kThinStage + (s & 1) * kThinSums + r * S::SUMS + 2 * pc) = thin_split3(v);
            }
            *(u32x4*)(smem + (s & 1) * kThinStage + r * S::ROW + 16 * pc) = thin_permute<QT>(buf[c]);
        }
    };
    tf4 acc[R][NT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][t] = tf4{0.f, 0.f, 0.f, 0.f};

    // The last super-block is apart, so that every load of the loop is unconditional (with a
    // conditional one the compiler waits for every load in flight, not for the oldest).
    auto reads = [&](int s, const uint8_t*& x, const uint8_t*& xs) {  // the lane's place in stage s
        int l = lane;
        asm volatile("" : "+v"(l));
        x = smem + (s & 1) * kThinStage + (l & 15) * S::ROW + 2 * W::base(l >> 4);
        xs = smem + 2 * kThinStage + (s & 1) * kThinSums + (l & 15) * S::SUMS + 16 * (l >> 4);
    };
    const int stages = (nsb + S::SPB - 1) / S::SPB;
    {
        u32x4 first[S::SPB][CP];
#pragma unroll
        for (int k = 0; k < S::SPB; ++k) fetch(0, k, first[k]);
#pragma unroll
        for (int k = 0; k < S::SPB; ++k) put(0, k, first[k]);
    }
    __syncthreads();
    int b = 0;
    for (int s = 0; s < stages - 1; ++s) {
        const uint8_t *x, *xs;
        reads(s, x, xs);
#pragma unroll 1
        for (int k = 0; k < S::SPB; ++k, ++b, x += 512, xs += 64) {
            u32x4 buf[CP];
            fetch(s + 1, k, buf);
            thin_block<QT, R, NT, true, EX>(kc, x, xs, acc, q, load, b);
            put(s + 1, k, buf);  // buffer (s + 1) & 1: its readers passed the barrier that ended stage s - 1
        }
        __syncthreads();
    }
    if (row0 >= A.N) return;
    const uint8_t *x, *xs;
    reads(stages - 1, x, xs);
    for (; b < nsb - 1; ++b, x += 512, xs += 64) thin_block<QT, R, NT, true, EX>(kc, x, xs, acc, q, load, b);
    thin_block<QT, R, NT, false, EX>(kc, x, xs, acc, q, load, b);

    // lane l: output column row0 (+ 16 r) + l % 16 of tokens 16 t + 4 (l / 16) + 0..3
    const int col = row0 + (lane & 15);
    auto emit = [&](int tok, const float (&sum)[R]) {
        const int64_t pr = m0 + tok;
        if (A.raw) {
            const int NC = GATEUP ? 2 * A.N : A.N;
            float* rb = A.raw + ((int64_t)blockIdx.y * A.P + pr) * NC + col;
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (col + (GATEUP ? 0 : 16 * r) < A.N) rb[GATEUP ? r * A.N : 16 * r] = sum[r];
        } else if constexpr (GATEUP) {
            if (col < A.N) ((float*)A.out)[pr * A.N + col] = thin_act(A.act_kind, sum[0]) * sum[1];
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int c = col + 16 * r;
                if (c >= A.N) continue;
                float o = sum[r] * rowscale[tok];
                if (A.bias) o += A.bias[c];
                if (A.out_f16)
                    ((_Float16*)A.out)[pr * A.N + c] = (_Float16)o;
                else
                    ((float*)A.out)[pr * A.N + c] = o;
            }
        }
    };
    bool nan = false;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int tok = 16 * t + 4 * p + v;
            float sum[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                sum[r] = acc[r][t][v];
                nan |= sum[r] != sum[r];
            }
            if (tok < n) emit(tok, sum);
        }
    // (not in the decode GEMVs' place, EX: they give NaN for such tokens too)
    if constexpr (W::MINS && !EX) {
        if (!__any(nan)) return;
#pragma unroll 1
        for (int i = 0; i < 4 * NT; ++i) {
            const int tok = 16 * (i >> 2) + 4 * p + (i & 3);
            float sum[R];
            if (tok < n && thin_non_finite(A.act + rowsrc[tok] + 256 * b0, 256 * nsb, weight, sum)) emit(tok, sum);
        }
    }
}

// Tiles of up to 16 MAXNT pairs; R row tiles a wave (gate/up: gate and up rows).  EX: exact weights,
// for the decode calls.
template <int QT, bool GATEUP, int R, int MAXNT, bool EX = false>
__global__ __launch_bounds__(kThinThreads, 4) void thin_kernel(const ThinArgs A) {
    constexpr int ROWS = 16 * MAXNT;
    static_assert(!GATEUP || R == 2, "gate/up: a gate and an up row tile a wave");
    __shared__ __attribute__((aligned(16))) uint8_t smem[2 * kThinStage + 2 * kThinSums];
    __shared__ uint32_t rowsrc[ROWS];  // first element of the tile's activation rows
    __shared__ float rowscale[ROWS];  // down: rs[p] * topk_w[perm[p]]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tile = blockIdx.z;
    // the tile's expert: every wave compares the tile with 64 experts' tile ranges at a time
    int e = 0, m0, n;
    if (A.E) {
        if (tile >= A.tile_off[A.E]) return;
        int first = 0;
        for (int e0 = 0; e0 < A.E; e0 += 64) {
            const int ee = min(e0 + lane, A.E - 1);
            const int lo = A.tile_off[ee], hi = A.tile_off[ee + 1];
            const uint64_t hit = __ballot(e0 + lane < A.E && lo <= tile && tile < hi);
            if (hit) {
                const int l = __builtin_ctzll(hit);
                e = e0 + l;
                first = __builtin_amdgcn_readlane(lo, l);
                break;
            }
        }
        e = __builtin_amdgcn_readfirstlane(e);
        const int o0 = A.offsets[e], o1 = A.offsets[e + 1];
        m0 = o0 + (tile - first) * ROWS;
        n = min(ROWS, o1 - m0);
    } else {
        m0 = tile * ROWS;
        n = min(ROWS, A.P - m0);
    }
    const int nb = A.K >> 8;
    const int b0 = (int)blockIdx.y * A.kper;
    const int nsb = min(nb - b0, A.kper);

    // the wave's row tiles, and their first super-block on its way
    const int row0 = ((int)blockIdx.x * kThinWaves + wave) * (GATEUP ? 16 : 16 * R);
    const int p = lane >> 4;
    const int ngr = row_groups(A.N);
    auto row_tile = [&](int first, int r, const uint8_t*& t, const uint8_t*& d) {
        const uint8_t* mat = GATEUP && r ? A.w1 + (int64_t)e * A.stride1 : A.w0 + (int64_t)e * A.stride0;
        const int row = min(GATEUP ? first : first + 16 * r, 64 * ngr - 16);
        const int64_t g = (int64_t)(row >> 6) * nb + b0;
        t = mat + g * (Tile<QT>::CH * 1024) + (row & 63) * 16;
        d = mat + (int64_t)ngr * nb * (Tile<QT>::CH * 1024) + (g * 64 + (row & 63)) * 2;
    };
    const uint8_t *tb[R], *db[R];
#pragma unroll
    for (int r = 0; r < R; ++r) row_tile(row0, r, tb[r], db[r]);
    Qtr<QT> q[R];
    const ThinConst kc = thin_const<QT>(p);
    uint32_t off0, offp;
    thin_offsets<QT>(lane, p, off0, offp);
    auto load = [&](int r, int b) {  // super-block b < nsb of the split
        thin_load<QT>(q[r], tb[r] + (uint32_t)b * (Tile<QT>::CH * 1024), db[r] + b * 128, off0, offp, lane, p);
    };
    auto weight = [&](int r, int k) {  // (its tile found anew: kept through the K loop it costs registers)
        int first = row0;
        asm volatile("" : "+s"(first));
        const uint8_t *t, *d;
        row_tile(first, r, t, d);
        if constexpr (ThinW<QT>::MINS) return thin_weight<QT>(t, 16 * (threadIdx.x & 15), k);
        else return 0.f;
    };
#pragma unroll
    for (int r = 0; r < R; ++r) load(r, 0);
    if (tid < ROWS) {
        const int pr = m0 + min(tid, n - 1), f = A.perm ? A.perm[pr] : pr;
        rowsrc[tid] = (uint32_t)(A.gather ? f / A.topk : pr) * (uint32_t)A.K;
        if (!GATEUP) rowscale[tid] = A.rs ? (A.topk_w ? A.rs[pr] * A.topk_w[f] : A.rs[pr]) : 1.0f;
    }
    __syncthreads();

    const int nt = (n + 15) >> 4;
    if (MAXNT == 1 || nt == 1) thin_tile<QT, GATEUP, R, 1, EX>(A, smem, rowsrc, rowscale, kc, m0, n, row0, b0, nsb, q, load, weight);
    else if constexpr (MAXNT > 1) {
        if (nt == 2) thin_tile<QT, GATEUP, R, 2, EX>(A, smem, rowsrc, rowscale, kc, m0, n, row0, b0, nsb, q, load, weight);
        else if constexpr (MAXNT > 2) thin_tile<QT, GATEUP, R, 4, EX>(A, smem, rowsrc, rowscale, kc, m0, n, row0, b0, nsb, q, load, weight);
    }
}

// ---------------------------------------------------------------- when, and launches
// Tiles of thin_tile_rows() pairs.  A linear of 33 .. 128 rows takes 64, so that its weights
// are read once or twice less (2048 x 151936 Q6_K, 48 rows: 89 -> 72 us; below and above, 32 and
// 64 measured alike); the grouped products always 32: gate/up holds two row tiles a wave,
// and 64 pairs then leave one block a CU (Qwen3 skewed, 301 tokens: 142 us with 32, 154 with 64).
constexpr int kThinTile = 32;
int thin_tile_rows() { return kThinTile; }

// Whether the product of P rows with one matrix [N, K] takes thin tiles.  Each tile decodes its weights
// again (about 7 M a us), so the 256-row tiles win once the rows fill a few of them; work: the weights
// decoded in all.  Cold weights, us 256-row tiles -> thin tiles:
//   up to 256 rows, where the 256-row tiles have one M tile: gate / up (two row tiles a wave) up to
//     510 M (H = 4096, I = 12288 FFN, Q4_K: 160 rows 133 -> 112, 192 rows = 604 M 147 -> 147, 256
//     172 -> 180; Q5_K 192 150 -> 173), else up to 850 M (28672 x 4096 Q4_K, 192 rows and 704 M 107
//     -> 101) and 3.9 MB of rows, an XCD's L2 (with down products of 12288 inputs and 160 rows the
//     FFN takes 107 us, 117 without; at 192 rows they lose 2 us of 150, of 13824 inputs and 144
//     rows 5 of 160, of 20480 and 128 rows 3 of 144; 4096 x 28672 Q5_K: 16 rows 49 -> 26, 64 54 -> 51,
//     96 59 -> 71);
//   above, up to 450 M while those tiles leave most CUs idle (4096 x 6144 Q4_K linear, 512 rows: 86 ->
//     57; 512 rows and more up to 150 M: 2048 x 1024 Q8_0, 1024 rows 41 -> 20, but an I = 5632 down
//     product of 1024 rows and 369 M loses 6), Q5_K, the slowest to decode, up to 5 MB of rows (8192 x
//     2048: 300 rows 43 -> 38, 384 45.5 -> 48.6);
//   fp16 weights, which the 256-row tiles take without any decode, one tile (I = 5632 FFN: 32 rows 59 ->
//     53, 64 rows 62 -> 64).
bool thin_takes(int qtype, int64_t P, int N, int K, bool gateup) {
    if (N % 4 || P * K >= ((int64_t)1 << 31)) return false;  // split sums of four; 32-bit row offsets
    if (qtype == PGMOE_F16) return P <= kThinTile;
    const int64_t work = (int64_t)div_up(P, kThinTile) * N * K * (gateup ? 2 : 1);
    if (P <= 256) return gateup ? work <= 510000000 : work <= 850000000 && P * K <= 1970000;
    if (qtype == PGMOE_Q5_K && P * K > 2500000) return false;
    return work <= (P <= 512 ? 450000000 : 150000000) && (int64_t)div_up(P, 256) * div_up(N, gateup ? 128 : 256) <= 96;
}

// Whether an MoE layer's products take thin tiles, for every routing of M tokens to topk experts each
// (the device's alone to know).  Cold weights, us 256-row tiles -> thin tiles, a layer:
//   all tokens on the same experts, each then M rows: while the gate / up weights decoded, times the
//     K splits that keep the 256-row tiles' CUs busy on so few experts, are up to 475 M (Mixtral
//     shape 64 tokens = 470 M 135 -> 131, 72 150 -> 171, 128 168 -> 212; Qwen2 96 = 440 M 137 -> 132,
//     100 150 -> 154, 192 193 -> 207; Qwen3 448 147 -> 127; 8 experts of 6144 inputs, two splits, 64
//     = 403 M 93 -> 84, 96 103 -> 115);
//   even and Zipf-like: up to 30 pairs an expert (Qwen3 448 tokens = 28: 213 -> 167 and 149 -> 137, 512
//     = 32: 218 -> 184 and 146 -> 150), 24 where the 256-row tiles read no scale plane either (Q8_0;
//     Qwen2 96 = 12: 411 -> 367 and 256 -> 229), and 2 for F16, which they take as it is stored (H =
//     2048, I = 768, 128 experts: 32 tokens 310 -> 291, 64 326 -> 328; I = 6144, 8: 16 319 -> 329).
bool thin_takes_moe(const Mats& g, const Mats& d, int M, int topk) {
    const int64_t P = (int64_t)M * topk;
    const int E = g.n_mats;
    if (E == 1) return thin_takes(g.qtype, P, g.N, g.K, true) && thin_takes(d.qtype, P, d.N, d.K, false);
    if (g.N % 4 || d.N % 4 || P * std::max(g.K, d.K) >= ((int64_t)1 << 31)) return false;
    for (const Mats* m : {&g, &d})
        if (P > (int64_t)E * (m->qtype == PGMOE_F16 ? 2 : m->qtype == PGMOE_Q8_0 ? 24 : 30)) return false;
    return (int64_t)std::min(topk, E) * div_up(M, kThinTile) * g.N * g.K * 2 * gemm_split(P, E, g.N, g.K, true).ksplit <=
           475000000;
}

// Splits of K, cut at super-block boundaries: the count with the least estimated time, rounds
// of two blocks a CU at 3 us a super-block step of a full round (gate/up; one row tile a
// wave: 1.5) plus the raw sums' way to memory and back at 5 TB/s; no more splits than the
// 256-row tiles would take for the same product, whose scratch they use.  (H = 4096, I = 12288
// FFN of 20 rows: 96 gate/up blocks unsplit, 288 in three.)
static GemmSplit thin_split(const ThinArgs& a, bool gateup, int tile, bool scratch) {
    const int nb = a.K >> 8;
    GemmSplit best{1, nb};
    if (!scratch) return best;
    const int64_t tiles = div_up(a.P, tile) + (a.E > 0 ? std::min(a.P, a.E) / 2 : 0);
    const int64_t blocks = tiles * div_up(a.N, 16 * kThinWaves);
    const int most = gemm_split(a.P, std::max(a.E, 1), a.N, a.K, gateup).ksplit;
    double t = 1e30;
    for (int s = 1; s <= most; ++s) {
        const int kper = div_up(nb, s), n = div_up(nb, kper);
        const double raw = n > 1 ? (double)n * a.P * a.N * (gateup ? 16 : 8) / 5e6 + 2.0 : 0.0;
        const double est = (double)div_up(blocks * n, 512) * kper * (gateup ? 3.0 : 1.5) + raw;
        if (est < t) t = est, best = GemmSplit{n, kper};
    }
    return best;
}

template <int QT>
static void thin_launch_q(const ThinArgs& a, bool gateup, int tile, const dim3& grid, hipStream_t st) {
    if (gateup)
        PG_LAUNCH((thin_kernel<QT, true, 2, 2>), grid, dim3(kThinThreads), 0, st, a);
    else if (tile == 32)
        PG_LAUNCH((thin_kernel<QT, false, 1, 2>), grid, dim3(kThinThreads), 0, st, a);
    else
        PG_LAUNCH((thin_kernel<QT, false, 1, 4>), grid, dim3(kThinThreads), 0, st, a);
}

static int thin_launch(const Mats& m, ThinArgs& a, bool gateup, int tile, float* raw, GemmSplit* split,
                       hipStream_t st) {
    const GemmSplit sp = thin_split(a, gateup, tile, raw != nullptr);
    *split = sp;
    a.kper = sp.kper;
    a.raw = sp.ksplit > 1 ? raw : nullptr;
    const int tiles = a.E > 0 ? a.P / tile + std::min(a.P, a.E) : div_up(a.P, tile);
    // Tiles last: the grid holds every tile the pairs could need, and those past the last, which end at
    // once, must not lie between one split's blocks and the next's, where they put two blocks with
    // work on one CU and none on another (Mixtral shape, 24 tokens on the same experts, two splits of
    // the down product: 58 us with the splits last, 38 in this order).
    const dim3 grid(div_up(a.N, 16 * kThinWaves), sp.ksplit, tiles);
    switch (m.qtype) {
    case PGMOE_Q4_1: thin_launch_q<PGMOE_Q4_1>(a, gateup, tile, grid, st); break;
    case PGMOE_Q4_K: thin_launch_q<PGMOE_Q4_K>(a, gateup, tile, grid, st); break;
    case PGMOE_Q5_K: thin_launch_q<PGMOE_Q5_K>(a, gateup, tile, grid, st); break;
    case PGMOE_Q6_K: thin_launch_q<PGMOE_Q6_K>(a, gateup, tile, grid, st); break;
    case PGMOE_Q8_0: thin_launch_q<PGMOE_Q8_0>(a, gateup, tile, grid, st); break;
    case PGMOE_F16: thin_launch_q<PGMOE_F16>(a, gateup, tile, grid, st); break;
    default: return fail(PGMOE_E_UNSUPPORTED, "thin product: qtype %d", m.qtype);
    }
    return check_launch(gateup ? "thin gate/up" : "thin down");
}

// (The scale planes the 256-row tiles read stay required, so that whether a call is accepted
// does not depend on its size.)
static bool needs_plane(const Mats& m) { return m.qtype != PGMOE_Q8_0 && m.qtype != PGMOE_F16; }

int launch_thin_gateup(const Mats& g, const Mats& u, const uint16_t* x, int M, int topk, const int32_t* offsets,
                       const int32_t* perm, const int32_t* tile_off, float* inter, hipStream_t st, float* raw,
                       int act) {
    if (needs_plane(g) && (!g.scales || !u.scales))
        return fail(PGMOE_E_INVALID, "gemm gate/up: K-quant weights need their scale plane (pgmoe_build_scale_plane)");
    ThinArgs a{};
    a.w0 = g.base, a.w1 = u.base, a.stride0 = g.stride, a.stride1 = u.stride, a.N = g.N, a.K = g.K;
    a.act = x, a.gather = perm != nullptr, a.topk = topk;
    a.E = offsets ? g.n_mats : 0, a.P = M * topk, a.offsets = offsets, a.perm = perm, a.tile_off = tile_off;
    a.out = inter, a.act_kind = act;
    GemmSplit sp;
    int rc = thin_launch(g, a, true, kThinTile, raw, &sp, st);
    if (rc || sp.ksplit == 1) return rc;
    return launch_split_reduce(1, raw, sp.ksplit, a.P, g.N, nullptr, nullptr, nullptr, inter, st, act);
}

int launch_thin_down(const Mats& d, const uint16_t* a16, const float* rs, int M, int topk, const int32_t* offsets,
                     const int32_t* perm, const int32_t* tile_off, const float* topk_w, float* partial,
                     hipStream_t st, float* raw) {
    if (needs_plane(d) && !d.scales)
        return fail(PGMOE_E_INVALID, "gemm down: K-quant weights need their scale plane (pgmoe_build_scale_plane)");
    ThinArgs a{};
    a.w0 = d.base, a.stride0 = d.stride, a.N = d.N, a.K = d.K, a.act = a16, a.topk = topk;
    a.E = offsets ? d.n_mats : 0, a.P = M * topk, a.offsets = offsets, a.perm = perm, a.tile_off = tile_off;
    a.rs = rs, a.topk_w = topk_w, a.out = partial;
    GemmSplit sp;
    int rc = thin_launch(d, a, false, kThinTile, raw, &sp, st);
    if (rc || sp.ksplit == 1) return rc;
    return launch_split_reduce(0, raw, sp.ksplit, a.P, d.N, rs, topk_w, perm, partial, st, PGMOE_ACT_SILU);
}

// A decode linear (M <= 8) of K-quants on one thin tile, weights exact (the GEMV's precision:
// its error against float64 falls from 2e-5 .. 3.5e-6 to 2.5e-7 .. 1.3e-7).  The GEMV decodes a
// weight once but spends a dot2 and two LDS bytes on it for each token, so 8 tokens cost it twice
// the weights' time; here 16 rows of MFMA cost what one does.  2048 x 151936, us GEMV -> here:
// Q6_K 3 rows 65 -> 55, 8 rows 122 -> 56; Q4_K 56 -> 42, 106 -> 42; Q5_K 60 -> 48, 107 -> 49 (two
// rows: Q6_K 60 -> 62).  Q8_0's d q is no fp16 value, so it stays there.  K is not split: from a
// block a CU on.  The rule looks at the smallest projection of a pack, whose rows then have the
// same bits alone and packed (gate || up of 20480 rows each stays on the GEMV, as each does).
static bool thin_exact(int qtype) { return qtype == PGMOE_Q4_K || qtype == PGMOE_Q5_K || qtype == PGMOE_Q6_K; }
bool thin_takes_decode(const Mats& w, int member_rows, int M) {
    return thin_exact(w.qtype) && M > 2 && member_rows >= 32768 && (int64_t)M * w.K < ((int64_t)1 << 31);
}

int launch_thin_decode(const Mats& w, const uint16_t* x, int M, const float* bias, void* out, int out_f16,
                       hipStream_t st) {
    ThinArgs a{};
    a.w0 = w.base, a.N = w.N, a.K = w.K, a.act = x, a.topk = 1, a.P = M;
    a.bias = bias, a.out = out, a.out_f16 = out_f16, a.kper = w.K >> 8;
    const dim3 grid(div_up(a.N, 16 * kThinWaves), 1, 1);
    switch (w.qtype) {
    case PGMOE_Q4_K: PG_LAUNCH((thin_kernel<PGMOE_Q4_K, false, 1, 1, true>), grid, dim3(kThinThreads), 0, st, a); break;
    case PGMOE_Q5_K: PG_LAUNCH((thin_kernel<PGMOE_Q5_K, false, 1, 1, true>), grid, dim3(kThinThreads), 0, st, a); break;
    case PGMOE_Q6_K: PG_LAUNCH((thin_kernel<PGMOE_Q6_K, false, 1, 1, true>), grid, dim3(kThinThreads), 0, st, a); break;
    default: return fail(PGMOE_E_UNSUPPORTED, "thin decode linear: qtype %d", w.qtype);
    }
    return check_launch("thin linear");
}

// ---------------------------------------------------------------- decode FFN (M <= 8)
// A dense SwiGLU FFN of 3 .. 8 tokens with K-quant matrices on thin tiles: gate / up as the decode
// linear (exact weights, fp16 tokens), the GEMVs' activation (expf and a division; the hardware
// forms cost 2e-6 of it at -38 and save 0.3 us), and the down product on the fp32 SwiGLU rows as three
// fp16 rows each, hi + mid 2^-11 + lo 2^-22, each piece the rounded rest of the ones before.  A row
// is first brought to 2^13 .. 2^14 by a power of two, so that values within 2^-36 of its largest keep
// their 24 bits and every value 2^-60 of the largest.  (Two pieces hold 23 bits; 4 tokens 41.4 us with
// two, 42.0 with three, 8 tokens 42.6 and 44.9.)  Up to 5 tokens fill one 16-row tile, 6 .. 8 two.
// Error against float64, H = 4096, I = 12288: 3.2e-5 -> 4e-7 (Q4_K, Q6_K).
// The GEMVs' time goes with the tokens, this one's (five launches, split sums) hardly: H = 4096, I =
// 12288, us GEMV -> here 3 tokens 63 -> 42, 4 71 -> 42, 6 98 -> 44, 8 123 -> 45; 2048 x 11264 4 tokens 52
// -> 35; with two pieces 2048 x 5632 3 tokens 17 -> 27, 5 22 -> 27, 8 33.5 -> 28; 1024 x 2816 8 tokens
// 18 -> 19: from 250 M weights times tokens on.
constexpr int kThinDecRows = 8;

bool thin_takes_dense_decode(const Mats& g, const Mats& u, const Mats& d, int M) {
    return M > 2 && M <= kThinDecRows && thin_exact(g.qtype) && u.qtype == g.qtype && thin_exact(d.qtype) &&
           (int64_t)M * 3 * g.N * g.K >= 250000000;
}

// Splits of K: two blocks a CU.
static GemmSplit thin_dec_split(int N, int K) {
    const int nb = K >> 8, s = std::min(nb, std::max(1, 512 / div_up(N, 16 * kThinWaves)));
    const int kper = div_up(nb, s);
    return GemmSplit{div_up(nb, kper), kper};
}
size_t thin_dec_raw_bytes(int I, int H) {
    return 4 * std::max((size_t)thin_dec_split(I, H).ksplit * kThinDecRows * 2 * I,
                        (size_t)thin_dec_split(H, I).ksplit * 3 * kThinDecRows * H);
}

// Row m of inter (I a multiple of 256) as fp16 rows m, M + m and 2M + m of a16; rs[m] takes them back.
// One block a row, read twice (the second time from cache).
__global__ __launch_bounds__(1024) void thin_rows_kernel(const float* __restrict__ inter, int M, int I,
                                                         uint16_t* __restrict__ a16, float* __restrict__ rs) {
    __shared__ float wmx[16];
    const int tid = threadIdx.x, m = blockIdx.x, n4 = I >> 2;
    const float4* row = (const float4*)(inter + (int64_t)m * I);
    float mx = 0.f;
    for (int i = tid; i < n4; i += 1024) {
        const float4 v = row[i];
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
    mx = wave_max(mx);
    if ((tid & 63) == 0) wmx[tid >> 6] = mx;
    __syncthreads();
    mx = wmx[0];
    for (int w = 1; w < 16; ++w) mx = fmaxf(mx, wmx[w]);
    // 2^k, k = 13 - exponent(mx), -115 .. 126 (so that 2^-k is normal; a zero row: any scale)
    const int k = min(126, 140 - (int)((__builtin_bit_cast(uint32_t, mx) >> 23) & 0xff));
    const float sc = __builtin_bit_cast(float, (uint32_t)(127 + k) << 23);
    if (tid == 0) rs[m] = __builtin_bit_cast(float, (uint32_t)(127 - k) << 23);
    th4* hi = (th4*)(a16 + (int64_t)m * I);
    th4* mid = (th4*)(a16 + (int64_t)(M + m) * I);
    th4* lo = (th4*)(a16 + (int64_t)(2 * M + m) * I);
    for (int i = tid; i < n4; i += 1024) {
        const float4 v = row[i];
        const float a[4] = {v.x * sc, v.y * sc, v.z * sc, v.w * sc};
        th4 h, r, l;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            h[c] = (_Float16)a[c];
            const float rest = (a[c] - (float)h[c]) * 2048.0f;
            r[c] = (_Float16)rest;
            l[c] = (_Float16)((rest - (float)r[c]) * 2048.0f);
        }
        hi[i] = h;
        mid[i] = r;
        lo[i] = l;
    }
}

// out[m] = rs[m] (sum of row m's splits + 2^-11 of row M + m's + 2^-22 of row 2M + m's), in split order.
__global__ __launch_bounds__(256) void thin_rows_reduce_kernel(const float* __restrict__ raw, int S, int M, int N,
                                                               const float* __restrict__ rs, float* __restrict__ out) {
    const int i = blockIdx.x * 256 + threadIdx.x, N4 = N >> 2;
    if (i >= M * N4) return;
    const int m = i / N4, c = i - m * N4;
    const tf4* r = (const tf4*)raw + (int64_t)m * N4 + c;
    // eight splits' words on their way before the first is added (one split at a time, the chain of
    // loads takes three times as long: 22 splits of 8 x 2048 17.6 us)
    constexpr int G = 8;
    tf4 sum[3] = {};
    for (int s0 = 0; s0 < S; s0 += G) {
        tf4 v[G][3];
#pragma unroll
        for (int j = 0; j < G; ++j)
#pragma unroll
            for (int q = 0; q < 3; ++q) v[j][q] = r[((int64_t)min(s0 + j, S - 1) * 3 + q) * M * N4];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < G; ++j)
            if (s0 + j < S)
#pragma unroll
                for (int q = 0; q < 3; ++q) sum[q] = sum[q] + v[j][q];
    }
    ((tf4*)out)[i] = rs[m] * (sum[0] + (sum[1] + sum[2] * (1.0f / 2048.0f)) * (1.0f / 2048.0f));
}

template <bool GATEUP, int MAXNT>
static int thin_dec_launch(int qtype, ThinArgs& a, hipStream_t st) {
    const GemmSplit sp = thin_dec_split(a.N, a.K);
    a.kper = sp.kper;
    const dim3 grid(div_up(a.N, 16 * kThinWaves), sp.ksplit, 1);
    constexpr int R = GATEUP ? 2 : 1;
    switch (qtype) {
    case PGMOE_Q4_K: PG_LAUNCH((thin_kernel<PGMOE_Q4_K, GATEUP, R, MAXNT, true>), grid, dim3(kThinThreads), 0, st, a); break;
    case PGMOE_Q5_K: PG_LAUNCH((thin_kernel<PGMOE_Q5_K, GATEUP, R, MAXNT, true>), grid, dim3(kThinThreads), 0, st, a); break;
    case PGMOE_Q6_K: PG_LAUNCH((thin_kernel<PGMOE_Q6_K, GATEUP, R, MAXNT, true>), grid, dim3(kThinThreads), 0, st, a); break;
    default: return fail(PGMOE_E_UNSUPPORTED, "thin decode: qtype %d", qtype);
    }
    return check_launch("thin decode");
}

int launch_thin_dense_decode(const Mats& g, const Mats& u, const Mats& d, const uint16_t* x, int M, int act,
                             float* inter, uint16_t* a16, float* rs, float* raw, float* out, hipStream_t st) {
    ThinArgs a{};
    a.w0 = g.base, a.w1 = u.base, a.N = g.N, a.K = g.K, a.act = x, a.topk = 1, a.P = M;
    a.out = inter, a.act_kind = act, a.raw = raw;
    int rc = thin_dec_launch<true, 1>(g.qtype, a, st);
    if (rc) return rc;
    const int S = thin_dec_split(g.N, g.K).ksplit;
    if ((rc = launch_split_reduce(3, raw, S, M, g.N, nullptr, nullptr, nullptr, inter, st, act))) return rc;
    PG_LAUNCH(thin_rows_kernel, dim3(M), dim3(1024), 0, st, inter, M, g.N, a16, rs);
    ThinArgs b{};
    b.w0 = d.base, b.N = d.N, b.K = d.K, b.act = a16, b.topk = 1, b.P = 3 * M, b.raw = raw;
    if ((rc = b.P <= 16 ? thin_dec_launch<false, 1>(d.qtype, b, st) : thin_dec_launch<false, 2>(d.qtype, b, st)))
        return rc;
    PG_LAUNCH(thin_rows_reduce_kernel, dim3(div_up(M * (d.N >> 2), 256)), dim3(256), 0, st, raw,
              thin_dec_split(d.N, d.K).ksplit, M, d.N, rs, out);
    return check_launch("thin decode reduce");
}

int launch_thin_linear(const Mats& w, const uint16_t* x, int M, const float* bias, void* out, int out_f16, float* raw,
                       hipStream_t st) {
    ThinArgs a{};
    a.w0 = w.base, a.N = w.N, a.K = w.K, a.act = x, a.topk = 1, a.P = M;
    a.bias = bias, a.out = out, a.out_f16 = out_f16;
    GemmSplit sp;
    int rc = thin_launch(w, a, false, M > 32 && M <= 128 ? 64 : 32, raw, &sp, st);
    if (rc || sp.ksplit == 1) return rc;
    return launch_split_reduce(2, raw, sp.ksplit, M, w.N, bias, nullptr, nullptr, out, st, out_f16);
}

}  // namespace pgmoe
