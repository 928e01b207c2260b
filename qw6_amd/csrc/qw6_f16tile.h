// qw6_f16tile.h -- fp16 MFMA operands of the grouped contractions, decoded in
// registers from GGUF block bytes (gfx950).
//
// One 256-column block of 16 weight rows feeds eight 16x16x32 MFMA steps: step s
// multiplies columns 32 s .. 32 s + 31, one sub-block of every format, and lane (n, g) =
// (l % 16, l / 16) holds row n's columns 32 s + 8 g .. + 7.
//
// Numerics: sc * q of a Q4_K / Q5_K weight (at most 63 * 31 = 1953) and
// (2 s + 1) * lattice value of an IQ weight (at most 31 * 43 = 1333) are
// integers below 2048, exact in fp16, so the sub-block scale rides in the B
// operand and the block's factor d (block_scale) is the unit of the sums. Q6_K's
// sc * (q - 32) reaches 4096 and is not exact: its operand is q - 32 and the
// scale of a 32-column run multiplies the run's products in fp32. The K-quant
// minimum m (6 bits, exact) takes more MFMAs against the activations' sub-block
// sums.
//
// Activations are fp16 parts p0, p1 (, p2) with x = p0 + 2^-11 p1 (+ 2^-22 p2) in the
// unit of their group (group_scale: the largest is in [2^14, 2^15)), each
// with a sum of its own (join). Parts 2^11 apart keep the low ones clear of
// fp16's subnormals: two hold 22 bits of every value within 2^28 of the group's
// largest and 17 (as bf16 hi + lo) within 2^33; three hold an fp32 value exactly within
// 2^38. With the low part in the high one's unit, a value 2^20 below the largest
// kept 14 bits.
//
// Columns are stored within each quad in the order 0, 2, 1, 3 (quad_slot): two
// bytes b, b + 2 of a code word become one fp16 pair with a single v_and.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qw6_dev.h"
#include "qw6_moe.h"
#include "qw6_tile.h"

namespace qw6 {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// D[m][n]: lane l holds n = l % 16, m = 4 (l / 16) + i for i < 4.
__device__ __forceinline__ f32x4 mfma_h(const u32x4& a, const u32x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f16x2 h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ uint32_t h2b(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ f16x2 pk(float v) { return f16x2{(_Float16)v, (_Float16)v}; }

// Place of column c (of a row) in the stored order.
__host__ __device__ constexpr uint32_t quad_slot(uint32_t c) {
    return (c & ~3u) | ((c & 1u) << 1) | ((c >> 1) & 1u);
}

// Stride in 16-byte pieces of the rows of one block that a wave stages in LDS: one
// more than the block needs (raw_chunks, qw6_tile.h) where all rows would
// otherwise start in one of two banks groups (IQ3_S: 8 pieces, 128 bytes).
__host__ __device__ constexpr uint32_t stage_stride(int f) { return raw_chunks(f) + (raw_chunks(f) % 8 == 0 ? 1u : 0u); }

// A staged block in LDS that starts at an even byte offset: words are read at the
// aligned addresses around them and shifted (unaligned LDS reads work, but made
// the down kernel 1.45 times slower).
struct LdsBlock {
    const uint8_t *p, *p0, *p2;   // byte 0; the words around it and around byte 2
    uint32_t s0, s2;              // bytes from those
    __device__ __forceinline__ explicit LdsBlock(const uint8_t* smem, uint32_t R)
        : p(smem + R), p0(smem + (R & ~3u)), p2(smem + ((R + 2u) & ~3u)), s0(R & 2u), s2((R + 2u) & 2u) {}
};
template <typename T>
__device__ __forceinline__ T rd(const uint8_t* p) { return *(const T*)p; }
// The N + 1 words around the N at byte c (even; o a multiple of 4 that is not a
// constant), and the N of them.
template <int N>
__device__ __forceinline__ void rd_around(const LdsBlock& w, uint32_t c, uint32_t o, uint32_t (&v)[N + 1]) {
    const uint8_t* const q = (c & 2u ? w.p2 - 2 : w.p0) + o;
#pragma unroll
    for (int i = 0; i <= N; i++) v[i] = rd<uint32_t>(q + c + 4 * i);
}
template <int N>
__device__ __forceinline__ uint32_t word_at(const LdsBlock& w, uint32_t c, const uint32_t (&v)[N], int i) {
    return __builtin_amdgcn_alignbyte(v[i + 1], v[i], c & 2u ? w.s2 : w.s0);
}

// What the steps of one block share, of row n: the K-quants' header (d, dmin, packed
// scales), Q6_K's scales and the lane's high bits, the IQ formats' high index
// bits and scales.
template <int F> struct Head { uint32_t d; };
template <> struct Head<F_Q4K> { u32x4 hd; };
template <> struct Head<F_Q5K> { u32x4 hd; u32x2 qh; };
template <> struct Head<F_Q6K> { uint32_t sc[4], x[2][2], d; };
template <> struct Head<F_IQ2S> { uint32_t qh[2], sc[2], d; };
template <> struct Head<F_IQ3S> { uint32_t qh[2], sc, d; };

template <int F>
__device__ __forceinline__ void read_head(Head<F>& r, const LdsBlock& w, uint32_t g) {
    if constexpr (F == F_Q4K || F == F_Q5K) {
        r.hd = rd<u32x4>(w.p);
        if constexpr (F == F_Q5K) r.qh = rd<u32x2>(w.p + 16 + 8 * g);
    } else if constexpr (F == F_Q6K) {
        uint32_t v[5], x[2][3];
        rd_around<4>(w, 192, 0, v);
        rd_around<2>(w, 128, 8 * g, x[0]);
        rd_around<2>(w, 160, 8 * g, x[1]);
        r.d = rd<uint16_t>(w.p + 208);
#pragma unroll
        for (int i = 0; i < 4; i++) r.sc[i] = word_at(w, 192, v, i);
#pragma unroll
        for (int i = 0; i < 4; i++) r.x[i >> 1][i & 1] = word_at(w, 128, x[i >> 1], i & 1);
    } else {
        r.d = rd<uint16_t>(w.p);
        if constexpr (F == F_IQ2S) {
            uint32_t q[3], v[3];
            rd_around<2>(w, 66, 0, q);
            rd_around<2>(w, 74, 0, v);
#pragma unroll
            for (int i = 0; i < 2; i++) {
                r.qh[i] = word_at(w, 66, q, i);
                r.sc[i] = word_at(w, 74, v, i);
            }
        } else if constexpr (F == F_IQ3S) {
            uint32_t q[3], v[2];
            rd_around<2>(w, 66, 0, q);
            rd_around<1>(w, 106, 0, v);
            r.qh[0] = word_at(w, 66, q, 0);
            r.qh[1] = word_at(w, 66, q, 1);
            r.sc = word_at(w, 106, v, 0);
        }
    }
}

// The lane's codes of one step, as read; and the IQ formats' lattice values.
template <int F> struct Codes { u32x2 q; };
template <> struct Codes<F_Q6K> { uint32_t q[3]; };
template <> struct Codes<F_IQ2XXS> { uint32_t q, lo, hi; };
template <> struct Codes<F_IQ2S> { uint32_t q, sg; };
template <> struct Codes<F_IQ3S> { uint32_t q, sg; };
template <int F> struct Lattice {};
template <> struct Lattice<F_IQ2XXS> { u32x4 v; };
template <> struct Lattice<F_IQ2S> { u32x2 v; };
template <> struct Lattice<F_IQ3S> { u32x2 v1, v2; };

template <int F>
__device__ __forceinline__ Codes<F> read_codes(const LdsBlock& w, int s, uint32_t g) {
    Codes<F> r;
    if constexpr (F == F_Q4K || F == F_Q5K) {
        r.q = rd<u32x2>(w.p + (F == F_Q4K ? 16u : 48u) + 32 * (s >> 1) + 8 * g);
    } else if constexpr (F == F_Q6K) {
        rd_around<2>(w, 64 * (s >> 2) + 32 * (s & 1), 8 * g, r.q);
    } else if constexpr (F == F_IQ2XXS) {
        r.q = rd<uint8_t>(w.p + 2 + 8 * s + g);
        r.lo = rd<uint16_t>(w.p + 6 + 8 * s);
        r.hi = rd<uint16_t>(w.p + 8 + 8 * s);
    } else if constexpr (F == F_IQ2S) {
        r.q = rd<uint8_t>(w.p + 2 + 4 * s + g);
        r.sg = rd<uint8_t>(w.p + 34 + 4 * s + g);
    } else {
        r.q = rd<uint16_t>(w.p + 2 + 8 * s + 2 * g);
        r.sg = rd<uint8_t>(w.p + 74 + 4 * s + g);
    }
    return r;
}
// tab: the lattice in LDS (F16Grid).
template <int F>
__device__ __forceinline__ Lattice<F> look_up(const Codes<F>& q, const Head<F>& r, int s, uint32_t g, const uint8_t* tab) {
    Lattice<F> o;
    if constexpr (F == F_IQ2XXS) {
        o.v = rd<u32x4>(tab + 16 * q.q);
    } else if constexpr (F == F_IQ2S) {
        const uint32_t qh = r.qh[s >> 2] >> (8 * (s & 3));
        o.v = rd<u32x2>(tab + 8 * (q.q | ((qh << (8 - 2 * g)) & 0x300u)));
    } else if constexpr (F == F_IQ3S) {
        const uint32_t qh = r.qh[s >> 2] >> (8 * (s & 3));
        o.v1 = rd<u32x2>(tab + 8 * ((q.q & 255u) | ((qh << (8 - 2 * g)) & 256u)));
        o.v2 = rd<u32x2>(tab + 8 * ((q.q >> 8) | ((qh << (7 - 2 * g)) & 256u)));
    }
    return o;
}

// ---- decoding ---------------------------------------------------------------------

// Byte I of v as an fp16 integer in both halves: the byte pair {b, 0x64} is 1024 + b.
template <int I>
__device__ __forceinline__ f16x2 dup_byte(uint32_t v) {
    return h2(__builtin_amdgcn_perm(0x64646464u, v, I == 0 ? 0x04000400u : I == 1 ? 0x04010401u : I == 2 ? 0x04020402u : 0x04030403u)) - pk(1024.f);
}

template <int F>
__host__ __device__ constexpr bool has_min() { return F == F_Q4K || F == F_Q5K; }
// Whether the sub-block scale rides in the B operand.
template <int F>
__host__ __device__ constexpr bool folds() { return F != F_Q6K; }

// The 6-bit scales (which = 0) or minimums (1) of sub-blocks 0-3 (hi = 0) or 4-7
// of a Q4_K / Q5_K block as bytes (qw6_get_scale_min_k4, qw6.c:1480-1490).
__device__ __forceinline__ uint32_t k_bytes(const u32x4& hd, int which, int hi) {
    const uint32_t A = which ? hd.z : hd.y, C = which ? hd.w >> 4 : hd.w;
    return hi ? (C & 0x0f0f0f0fu) | ((A >> 2) & 0x30303030u) : A & 0x3f3f3f3fu;
}

// The block's minimums of sub-blocks 2 g (k-slots 0-2) and 2 g + 1 (k-slots 4-6) as
// the B operand of the minimum MFMA, against the three parts of the activation
// sums of the same sub-blocks (split_sum): 2^8, 2^-3 and 2^-14 times the minimum,
// the parts' units 2^11 apart; block_min takes the 2^8 and the sums' 2^-5 out.
template <int F>
__device__ __forceinline__ u32x4 min_operand(const Head<F>& r, uint32_t g) {
    const uint32_t m = (g & 2u ? k_bytes(r.hd, 1, 1) : k_bytes(r.hd, 1, 0)) >> (16 * (g & 1u));
    const f16x2 m0 = dup_byte<0>(m), m1 = dup_byte<1>(m);
    const f16x2 u = {(_Float16)256.f, (_Float16)0.125f}, v = {(_Float16)0x1p-14f, (_Float16)0.f};
    return u32x4{h2b(m0 * u), h2b(m0 * v), h2b(m1 * u), h2b(m1 * v)};
}

// Scale of step s's columns (Q6_K, qw6.c:1550-1578): the even one of the run's two.
__device__ __forceinline__ float run_scale(const Head<F_Q6K>& r, int s) {
    return (float)(int8_t)((r.sc[s >> 1] >> (16 * (s & 1))) & 0xffu);
}

// The signs of 8 stored values v (word k: columns 0,2 | 1,3 | 4,6 | 5,7) from
// bits 0-7 of both halves of y (bit c: column c), as apply_signs (qw6_tile.h).
__device__ __forceinline__ u32x4 flip_signs(const u32x4& v, uint32_t y) {
    const us2_t b = __builtin_bit_cast(us2_t, y);
    const us2_t s0 = {15, 13}, s1 = {14, 12}, s2 = {11, 9}, s3 = {10, 8};
    return u32x4{v.x ^ (__builtin_bit_cast(uint32_t, (us2_t)(b << s0)) & 0x80008000u),
                 v.y ^ (__builtin_bit_cast(uint32_t, (us2_t)(b << s1)) & 0x80008000u),
                 v.z ^ (__builtin_bit_cast(uint32_t, (us2_t)(b << s2)) & 0x80008000u),
                 v.w ^ (__builtin_bit_cast(uint32_t, (us2_t)(b << s3)) & 0x80008000u)};
}

// The lane's B operand of step s. A code b masked out of a word is the fp16
// subnormal b * 2^-24; times scale * 2^10 it is the normal number
// b * scale * 2^-14, exactly.
template <int F>
__device__ __forceinline__ u32x4 b_operand(const Head<F>& r, const Codes<F>& q, const Lattice<F>& t, const LdsBlock& w,
                                           int s, uint32_t g) {
    if constexpr (F == F_Q4K || F == F_Q5K) {
        const int v = s & 1;   // low or high nibbles
        const uint32_t b = k_bytes(r.hd, 0, s >> 2);
        const f16x2 sub = (s & 3) == 0 ? dup_byte<0>(b) : (s & 3) == 1 ? dup_byte<1>(b) : (s & 3) == 2 ? dup_byte<2>(b) : dup_byte<3>(b);
        const f16x2 sc = sub * pk(v ? 64.f : 1024.f);   // codes 16 q in the high nibble
        u32x4 o;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t mask = v ? 0x00f000f0u : 0x000f000fu;
            uint32_t p0 = q.q[i] & mask, p1 = (q.q[i] >> 8) & mask;
            if constexpr (F == F_Q5K) {   // fifth bit: bit s of every byte
                const uint32_t y = r.qh[i] >> s;
                p0 |= v ? (y << 8) & 0x01000100u : (y << 4) & 0x00100010u;
                p1 |= v ? y & 0x01000100u : (y >> 4) & 0x00100010u;
            }
            o[2 * i] = h2b(h2(p0) * sc);
            o[2 * i + 1] = h2b(h2(p1) * sc);
        }
        return o;
    } else if constexpr (F == F_Q6K) {
        // run k of half h (qw6.c:1550-1578): low / high nibbles of the first 32 bytes (runs 0,
        // 2) or the next (1, 3), two bits of x per run; 1024 + q - (1024 + 32)
        const int k = s & 3;
        const f16x2 z = pk(-1056.f);
        u32x4 o;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t v = word_at(w, 0, q.q, i), x = r.x[s >> 2][i];
            const uint32_t hi = k == 0 ? x << 4 : k == 1 ? x << 2 : k == 2 ? x : x >> 2;
            const uint32_t b = ((k < 2 ? v : v >> 4) & 0x0f0f0f0fu) | (hi & 0x30303030u);
            o[2 * i] = h2b(h2(__builtin_amdgcn_perm(0x64646464u, b, 0x04020400u)) + z);
            o[2 * i + 1] = h2b(h2(__builtin_amdgcn_perm(0x64646464u, b, 0x04030401u)) + z);
        }
        return o;
    } else if constexpr (F == F_IQ2XXS) {
        const uint32_t p1 = q.lo | (q.hi << 16);   // four times 7 signs, the scale
        const f16x2 sc = dup_byte<0>((p1 >> 27) | 1u);   // 2 s + 1 (bits 28-31: s; bit 27 is set either way)
        return flip_signs(u32x4{h2b(h2(t.v.x) * sc), h2b(h2(t.v.y) * sc), h2b(h2(t.v.z) * sc), h2b(h2(t.v.w) * sc)},
                          sign_pairs7((p1 >> (7 * g)) & 127u));
    } else if constexpr (F == F_IQ2S) {
        const uint32_t nib = r.sc[s >> 2] >> (8 * (s & 3) + 4 * (g >> 1));   // per 16 columns
        const f16x2 sc = dup_byte<0>(((nib << 1) & 30u) | 1u) * pk(1024.f);
        return flip_signs(u32x4{h2b(h2(t.v.x & 0x00ff00ffu) * sc), h2b(h2((t.v.x >> 8) & 0x00ff00ffu) * sc),
                                h2b(h2(t.v.y & 0x00ff00ffu) * sc), h2b(h2((t.v.y >> 8) & 0x00ff00ffu) * sc)},
                          sign_pairs(q.sg));
    } else {
        const f16x2 sc = dup_byte<0>((((r.sc >> (4 * s)) << 1) & 30u) | 1u);
        return flip_signs(u32x4{h2b(h2(t.v1.x) * sc), h2b(h2(t.v1.y) * sc), h2b(h2(t.v2.x) * sc), h2b(h2(t.v2.y) * sc)},
                          sign_pairs(q.sg));
    }
}

// The factor of a block's products: d, times 2^14 where the operands carry
// 2^-14 (b_operand), or d / 8 for the IQ2 formats, whose (0.5 + s) / 4 is
// (2 s + 1) / 8; and the K-quants' dmin in the unit of min_operand's products.
template <int F>
__device__ __forceinline__ float block_scale(const Head<F>& r) {
    if constexpr (F == F_Q4K || F == F_Q5K) return h2f(r.hd.x & 0xffffu) * 16384.f;
    else return h2f(r.d) * (F == F_IQ2XXS ? 0.125f : F == F_IQ2S ? 2048.f : 1.f);
}
template <int F>
__device__ __forceinline__ float block_min(const Head<F>& r) { return h2f(r.hd.x >> 16) * 0.125f; }

// LDS bytes of an IQ format's lattice in stored column order: fp16 values,
// except IQ2_S's 1024 entries kept as 8 bytes each.
__host__ __device__ constexpr uint32_t f16_grid_bytes(int f) {
    return f == F_IQ2XXS ? 256u * 16u : f == F_IQ2S ? 1024u * 8u : f == F_IQ3S ? 512u * 8u : 0u;
}
// Into LDS by a workgroup of NTHR threads: the loads, then (when they have landed) the
// stores.
template <int F, uint32_t NTHR>
struct F16Grid {
    static constexpr uint32_t N = F == F_IQ2XXS ? 256u : F == F_IQ2S ? 1024u : 512u, P = (N + NTHR - 1) / NTHR;
    uint64_t v[P];
    __device__ __forceinline__ void load(const IqTables& g) {
#pragma unroll
        for (uint32_t u = 0; u < P; u++) {
            const uint32_t i = min(u * NTHR + threadIdx.x, N - 1);
            v[u] = F == F_IQ2XXS ? g.iq2xxs[i] : F == F_IQ2S ? g.iq2s[i] : g.iq3s[i];
        }
    }
    __device__ __forceinline__ void store(uint8_t* tab) const {
        auto pair = [](uint32_t a, uint32_t b) {   // integers below 2048 as fp16
            return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(float)a) |
                   ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(float)b) << 16);
        };
#pragma unroll
        for (uint32_t u = 0; u < P; u++) {
            const uint32_t i = u * NTHR + threadIdx.x, a = (uint32_t)v[u], b = (uint32_t)(v[u] >> 32);
            if (i >= N) continue;
            const uint32_t lo = pair(a & 255u, (a >> 16) & 255u), hi = pair((a >> 8) & 255u, a >> 24);
            if constexpr (F == F_IQ2XXS)
                ((u32x4*)tab)[i] = u32x4{lo, hi, pair(b & 255u, (b >> 16) & 255u), pair((b >> 8) & 255u, b >> 24)};
            else ((u32x2*)tab)[i] = F == F_IQ2S ? u32x2{a, b} : u32x2{lo, hi};
        }
    }
};

// ---- activations ----------------------------------------------------------------------

constexpr float kPartUnit = 0x1p-11f;   // a part's unit in the one before's

// A power of two that brings the largest magnitude mx of a group of values
// into [2^14, 2^15); inv: its exact reciprocal. 1 for a group of zeros.
__device__ __forceinline__ float group_scale(float mx, float& inv) {
    const int ex = (int)((__float_as_uint(mx) >> 23) & 255u) - 127;   // -127: zero or subnormal
    int e = 14 - ex;
    e = e > 126 ? 126 : e;
    if (mx == 0.f) e = 0;
    inv = __uint_as_float((uint32_t)(127 - e) << 23);
    return __uint_as_float((uint32_t)(127 + e) << 23);
}
// x (scaled) as P fp16 parts; returns the represented value.
template <int P>
__device__ __forceinline__ float split_h(float x, uint16_t (&p)[P]) {
    float sum = 0.f, unit = 1.f;
#pragma unroll
    for (int i = 0; i < P; i++) {
        const _Float16 h = (_Float16)x;
        p[i] = __builtin_bit_cast(uint16_t, h);
        sum = fmaf((float)h, unit, sum);
        x = (x - (float)h) * (1.f / kPartUnit);   // exact
        unit *= kPartUnit;
    }
    return sum;
}
// The value of P parts' sums.
template <int P>
__device__ __forceinline__ float join(const float (&v)[P]) {
    float s = v[P - 1];
#pragma unroll
    for (int i = P - 2; i >= 0; i--) s = fmaf(kPartUnit, s, v[i]);
    return s;
}
// Eight scaled columns as packed parts in stored order; returns the sum of the
// represented values.
template <int P>
__device__ __forceinline__ float split8h(const float (&v)[8], float sc, uint4 (&o)[P]) {
    uint16_t h[8][P];
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) sum += split_h<P>(v[i] * sc, h[quad_slot(i)]);
#pragma unroll
    for (int p = 0; p < P; p++)
        o[p] = u4(h[0][p] | ((uint32_t)h[1][p] << 16), h[2][p] | ((uint32_t)h[3][p] << 16),
                  h[4][p] | ((uint32_t)h[5][p] << 16), h[6][p] | ((uint32_t)h[7][p] << 16));
    return sum;
}
// The sum of a sub-block's 32 values (below 2^20 in their group's unit), times 2^-5,
// as three fp16 parts 2^11 apart, a zero after: half of an A operand of the minimum
// MFMAs.
__device__ __forceinline__ uint2 split_sum(float x) {
    uint16_t p[3];
    split_h<3>(x * 0x1p-5f, p);
    return make_uint2((uint32_t)p[0] | ((uint32_t)p[1] << 16), (uint32_t)p[2]);
}

}  // namespace qw6
