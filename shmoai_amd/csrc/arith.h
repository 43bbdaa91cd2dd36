// Exact 64-bit modular arithmetic for CDNA4 (gfx950) kernels.
//
// CDNA4 has no 64x64->128 multiply instruction; __umul64hi and 64-bit
// products lower to 32-bit v_mul_hi/v_mad_u64_u32 chains. Every helper keeps
// operands below 2^62 so that lazy [0, 4q) butterflies never wrap (all primes
// are at most 61 bits).
//
// The ring degree N is a power of two (2^10 .. 2^17), so kernels split a flat
// index over [..][N] with a shift and a mask rather than a 64-bit division.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace shm {

typedef unsigned __int128 u128;

// One RNS prime with its Barrett constant floor(2^128 / q) = (mu_hi, mu_lo).
struct DevMod {
    uint64_t q;
    uint64_t mu_hi;
    uint64_t mu_lo;
};

__device__ __forceinline__ uint64_t csub(uint64_t x, uint64_t q) { return x >= q ? x - q : x; }

__device__ __forceinline__ uint64_t add_mod(uint64_t a, uint64_t b, uint64_t q) { return csub(a + b, q); }

__device__ __forceinline__ uint64_t sub_mod(uint64_t a, uint64_t b, uint64_t q) { return csub(a + q - b, q); }

__device__ __forceinline__ uint64_t neg_mod(uint64_t a, uint64_t q) { return a == 0 ? 0 : q - a; }

// Shoup product x * w mod q with ws = floor(w * 2^64 / q): result in [0, 2q)
// for any x < 2^64.
__device__ __forceinline__ uint64_t mul_shoup_lazy(uint64_t x, uint64_t w, uint64_t ws, uint64_t q) {
    return x * w - __umul64hi(x, ws) * q;
}

__device__ __forceinline__ uint64_t mul_shoup(uint64_t x, uint64_t w, uint64_t ws, uint64_t q) {
    return csub(mul_shoup_lazy(x, w, ws, q), q);
}

// Shoup companion floor(w * 2^64 / q) of w < q from the Barrett constant:
// floor(w * mu / 2^64) is at most one short, and the remainder w * 2^64 - e * q
// (exact in 64 bits, below 2q) says when.
__device__ __forceinline__ uint64_t shoup_companion(uint64_t w, const DevMod &m) {
    uint64_t e = w * m.mu_hi + __umul64hi(w, m.mu_lo);
    const uint64_t rem = 0 - e * m.q;
    return rem >= m.q ? e + 1 : e;
}

// Barrett reduction of a 128-bit value (hi, lo) with mu = floor(2^128/q).
// The quotient estimate is at most 2 short, so the remainder is in [0, 3q)
// before the final corrections.
__device__ __forceinline__ uint64_t barrett128(uint64_t hi, uint64_t lo, const DevMod &m) {
    // floor((hi*2^64 + lo) * mu / 2^128), dropping the lo*mu_lo low part.
    const uint64_t a = __umul64hi(lo, m.mu_lo);
    const uint64_t b_lo = lo * m.mu_hi, b_hi = __umul64hi(lo, m.mu_hi);
    const uint64_t c_lo = hi * m.mu_lo, c_hi = __umul64hi(hi, m.mu_lo);
    uint64_t s = a + b_lo;
    uint64_t carry = s < a;
    const uint64_t s2 = s + c_lo;
    carry += s2 < s;
    const uint64_t qest = hi * m.mu_hi + b_hi + c_hi + carry;
    uint64_t r = lo - qest * m.q;
    r = csub(r, m.q);
    return csub(r, m.q);
}

__device__ __forceinline__ uint64_t mul_mod(uint64_t a, uint64_t b, const DevMod &m) {
    return barrett128(__umul64hi(a, b), a * b, m);
}

// Reduce a single 64-bit word (any value) mod q using mu_hi = floor(2^64/q).
__device__ __forceinline__ uint64_t reduce64(uint64_t x, const DevMod &m) {
    const uint64_t qe = __umul64hi(x, m.mu_hi);
    return csub(x - qe * m.q, m.q);
}

// 128-bit accumulator helpers (explicit carries; no __int128 division).
struct Acc128 {
    uint64_t lo, hi;
};

__device__ __forceinline__ void mac128(Acc128 &acc, uint64_t a, uint64_t b) {
    const uint64_t lo = a * b, hi = __umul64hi(a, b);
    acc.lo += lo;
    acc.hi += hi + (acc.lo < lo);
}

__device__ __forceinline__ uint64_t reduce128(const Acc128 &acc, const DevMod &m) { return barrett128(acc.hi, acc.lo, m); }

// Sums of products of residues below 2^52 (every prime in (2^45, 2^52)): with
// a = a1 2^26 + a0 and b = b1 2^26 + b0, a b = a1 b1 2^52 + (a1 b0 + a0 b1) 2^26 + a0 b0,
// each partial product a 32 x 32 -> 64-bit multiply-add into one of three 64-bit
// sums (no carries: up to 64 terms stay below 2^64).
struct Acc52 {
    uint64_t s0, s1, s2;
};

struct Split26 {
    uint32_t hi, lo;
};

__device__ __forceinline__ Split26 split26(uint64_t x) { return {(uint32_t)(x >> 26), (uint32_t)x & 0x3ffffffu}; }

__device__ __forceinline__ void mac52(Acc52 &acc, Split26 a, uint64_t b) {
    const Split26 bs = split26(b);
    acc.s0 += (uint64_t)a.lo * bs.lo;
    acc.s1 += (uint64_t)a.hi * bs.lo;
    acc.s1 += (uint64_t)a.lo * bs.hi;
    acc.s2 += (uint64_t)a.hi * bs.hi;
}

// [S]_q of S = s2 2^52 + s1 2^26 + s0 < 2^109 for 2^45 < q < 2^52: T = floor(S / 2^45)
// exactly, the quotient estimate floor(T mu / 2^64) with mu = floor(2^109 / q) (from
// the Barrett constant floor(2^128 / q)) is at most 3 short, so S - qe q in [0, 4q)
// is taken in 64 bits.
__device__ __forceinline__ uint64_t reduce52(const Acc52 &a, const DevMod &m) {
    const uint64_t T = (a.s2 << 7) + (a.s1 >> 19) + ((((a.s1 & 0x7ffffull) << 26) + a.s0) >> 45);
    const uint64_t lo = a.s0 + (a.s1 << 26) + (a.s2 << 52);
    const uint64_t mu = (m.mu_hi << 45) | (m.mu_lo >> 19);
    const uint64_t r = lo - __umul64hi(T, mu) * m.q;
    return csub(csub(r, m.q << 1), m.q);
}

// a b mod q for a, b < 2^53 and 2^45 < q < 2^52: the four 26-bit split products (S < 2^106)
// and reduce52, about half the multiplies of mul_mod; the same canonical residue.
__device__ __forceinline__ uint64_t mul_mod52(uint64_t a, uint64_t b, const DevMod &m) {
    Acc52 acc{0, 0, 0};
    mac52(acc, split26(a), b);
    return reduce52(acc, m);
}

// Products by constants modulo primes just below a power of two: q = 2^b - delta,
// delta < 2^29 (every prime of a context is the largest free one of its bit size that
// is 1 mod 2N, so delta is a small multiple of 2N). A constant w < q travels as
// w = h0 2^s + l0 and 2^32 w mod q = h1 2^s + l1 with s = b - 30, so h < 2^30.
// For x = xh 2^32 + xl (signed 64-bit, any value),
//   x w = H 2^s + L (mod q),  H = xl h0 + xh h1,  L = xl l0 + xh l1,
// and 2^(s + 32) = 2^(b + 2) = 4 delta (mod q), so
//   x w = (H mod 2^32) 2^s + L + floor(H / 2^32) 4 delta (mod q):
// six 32 x 32 -> 64-bit multiply-adds, no quotient and no carry handling (a Shoup
// product with its 64-bit high part takes about twice the issue slots: every
// multiply-add, 64-bit add and shift issues in 4 cycles per wave here).
struct FoldMod {
    uint32_t pw;    // 2^s
    int32_t d4, d;  // 4 delta, delta
    uint32_t sh;    // b - 32
    uint32_t mask;  // 2^(b - 32) - 1
    uint32_t s;     // b - 30
    uint32_t twice; // one fold of a 64-bit word can leave it at 2q or more
    uint64_t off;   // the smallest multiple of q that is at least 2^63
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // (h0, l0, h1, l1)

// |result| <= 2.5 2^(b+2) + 6 2^30 delta for any signed x.
__device__ __forceinline__ uint64_t fold_mul(uint64_t x, u32x4 w, const FoldMod &f) {
    const uint32_t xl = (uint32_t)x;
    const int32_t xh = (int32_t)(x >> 32);
    const uint64_t H = (uint64_t)((int64_t)xh * (int32_t)w.z) + (uint64_t)xl * w.x;
    const uint64_t L = (uint64_t)((int64_t)xh * (int32_t)w.w) + (uint64_t)xl * w.y;
    const uint64_t r = (uint64_t)(uint32_t)H * f.pw + L;
    return (uint64_t)((int64_t)(int32_t)(H >> 32) * f.d4) + r;
}

// x mod 2^b + floor(x / 2^b) delta: congruent to a signed x and within
// (-2^(63-b) delta, 2^b + 2^(63-b) delta).
__device__ __forceinline__ uint64_t fold_tight(uint64_t x, const FoldMod &f) {
    const int32_t xh = (int32_t)(x >> 32);
    const uint64_t lo = ((uint64_t)((uint32_t)xh & f.mask) << 32) | (uint32_t)x;
    return (uint64_t)((int64_t)(xh >> f.sh) * f.d) + lo;
}

// Canonical residue of a signed x, |x| <= 2^63 - q: the offset makes it unsigned, and one
// fold (two where f.twice) leaves it below 2q.
template <bool TWICE>
__device__ __forceinline__ uint64_t fold_canon(uint64_t x, uint64_t q, const FoldMod &f) {
    auto fold = [&](uint64_t y) {
        const uint32_t yh = (uint32_t)(y >> 32);
        const uint64_t lo = ((uint64_t)(yh & f.mask) << 32) | (uint32_t)y;
        return (uint64_t)(yh >> f.sh) * (uint32_t)f.d + lo;
    };
    uint64_t y = fold(x + f.off);
    if (TWICE) y = fold(y);
    return csub(y, q);
}

// Congruent to a signed x, |x| <= 2^63 - q, in [0, 2q) (primes that fold once).
__device__ __forceinline__ uint64_t fold_positive(uint64_t x, const FoldMod &f) {
    const uint64_t y = x + f.off;
    const uint32_t yh = (uint32_t)(y >> 32);
    const uint64_t lo = ((uint64_t)(yh & f.mask) << 32) | (uint32_t)y;
    return (uint64_t)(yh >> f.sh) * (uint32_t)f.d + lo;
}

// The split form of a constant w < q given its Shoup companion.
__device__ __forceinline__ u32x4 fold_split(uint64_t w, uint64_t ws, uint64_t q, const FoldMod &f) {
    const uint64_t w1 = mul_shoup(uint64_t(1) << 32, w, ws, q);
    const uint32_t m = f.pw - 1;
    return u32x4{(uint32_t)(w >> f.s), (uint32_t)w & m, (uint32_t)(w1 >> f.s), (uint32_t)w1 & m};
}

// Base conversions sum A <= 6 products of residues y_i by constants c_i mod p, so their
// constants are split lower: c = h0 2^s + l0, 2^32 c mod p = h1 2^s + l1 with s = b - 27
// (h < 2^27), which leaves room for the sums H and L of all terms in 64 bits;
// 2^(s + 32) = 2^(b + 5) = 32 delta (mod p).
struct ConvAcc {
    uint64_t H, L;
};
__device__ __forceinline__ void conv_mac(ConvAcc &a, uint32_t yl, uint32_t yh, u32x4 c) {
    a.H += (uint64_t)yl * c.x;
    a.L += (uint64_t)yl * c.y;
    a.H += (uint64_t)yh * c.z;
    a.L += (uint64_t)yh * c.w;
}
// congruent to the sum, below conv_bound (context.hip)
__device__ __forceinline__ uint64_t conv_value(const ConvAcc &a, const FoldMod &f) {
    const uint64_t r = (uint64_t)(uint32_t)a.H * (f.pw << 3) + a.L;
    return (uint64_t)(uint32_t)(a.H >> 32) * ((uint32_t)f.d << 5) + r;
}

// [v]_q of an integral double v with |v| < 2^128; negative v maps to q - (|v| mod q),
// which is q itself when |v| is a multiple of q (callers reduce when they need [0, q)).
__device__ __forceinline__ uint64_t residue_of_rounded(double v, const DevMod &m) {
    const bool neg = signbit(v);
    const double a = fabs(v);
    uint64_t r;
    if (a < 18446744073709551616.0) {
        r = reduce64((uint64_t)a, m);
    } else {
        const uint64_t lo = (uint64_t)fmod(a, 18446744073709551616.0);
        const uint64_t hi = (uint64_t)(a / 18446744073709551616.0);
        r = barrett128(hi, lo, m);
    }
    return neg ? m.q - r : r;
}

}  // namespace shm
