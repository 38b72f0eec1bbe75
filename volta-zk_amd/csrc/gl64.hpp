// gl64.hpp -- Goldilocks field arithmetic for gfx950 (device) and the host.
//
// p = 2^64 - 2^32 + 1.  Elements are u64; "canonical" means in [0, p).
// The identities used are 2^64 = 2^32 - 1 = eps (mod p) and 2^96 = -1 (mod p),
// the same ones the reference's field uses (rust/volta-field/src/lib.rs:89-103).
//
// The device multiply forms the 128-bit product from four 32x32->64 partial
// products (v_mad_u64_u32 on gfx950) and folds the high half with the two
// identities above; no MFMA, no 64-bit hardware multiply exists on the VALU.
//
// The kernels built on this are bound by VALU issue, so every operation is
// counted in VALU instructions.  A carry or borrow out of 64 bits is corrected by
// one select and one multiply-add instead of a second carry chain: sub and
// add_lazy take 4 instructions (5 before), the general multiply 18 (20).  With
// that, lazy sums inside the DFTs and the cheap negative of the middle shifts
// (gl64_shift.hpp) a 32-point DFT takes 1,033 instead of 1,267 and a 16-point
// one 397 instead of 483; measured alternating: 2^15-point rows (C4)
// 4.47 -> 3.83 ms, the C3 step 1.674 -> 1.547 ms, C1 38.0 -> 35.9 us, the
// 2^17-point embedding commitment 2.77 -> 2.65 ms; the 2^24-point batch only
// 25.9 -> 25.4 ms, whose passes then come close to HBM as well (4.3-4.7 TB/s).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gl {

constexpr uint64_t P = 0xFFFFFFFF00000001ull;
constexpr uint64_t EPS = 0x00000000FFFFFFFFull;

// A 64-bit value from two 32-bit words, kept as one register pair on the
// device: written as (hi << 32) | lo, the compiler reads the OR as an add of
// disjoint halves and splits a later 64-bit add into two adds of zero-extended
// halves (an extra add and a register copy each time).
__host__ __device__ __forceinline__ uint64_t pack64(uint32_t lo, uint32_t hi) {
    uint64_t r = (static_cast<uint64_t>(hi) << 32) | lo;
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+v"(r));
#endif
    return r;
}

// ---- host/device scalar ops (canonical in, canonical out) ---------------

__host__ __device__ __forceinline__ uint64_t canon(uint64_t x) { return x >= P ? x - P : x; }

// m eps + t and its carry out of 2^64 (a lane mask), in one v_mad_u64_u32: the
// inline constant -1 read as an unsigned word is eps.  The compiler has no way
// to read that carry, and with eps as a literal it would expand the product.
// The mask may only be read through a SALU operation first (lane_bit's or):
// gfx950 needs two wait states between a VALU write of a mask and a VALU read
// of it, which the compiler does not see here.
// x - m' eps for m = -15 m' (m' = 0 or 1): -15 * 0x11111111 = -eps, so one
// v_mad_i64_i32 applies a borrow's correction (0x11111111 in a scalar register;
// m an inline constant of the select that made it).
#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ uint64_t mad_eps(uint32_t m, uint64_t t) {
    uint64_t r, c;
    asm("v_mad_u64_u32 %0, %1, %2, -1, %3" : "=v"(r), "=s"(c) : "v"(m), "v"(t));
    return r;
}
__device__ __forceinline__ uint64_t mad_eps(uint32_t m, uint64_t t, uint64_t* carry) {
    uint64_t r;
    asm("v_mad_u64_u32 %0, %1, %2, -1, %3" : "=v"(r), "=s"(*carry) : "v"(m), "v"(t));
    return r;
}
__device__ __forceinline__ uint64_t less_eps_word(uint64_t x, uint32_t m) {
    uint64_t r, c;
    asm("v_mad_i64_i32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(c) : "v"(m), "s"(0x11111111), "v"(x));
    return r;
}
__device__ __forceinline__ uint64_t less_eps(uint64_t x, bool borrow) {
    return less_eps_word(x, borrow ? static_cast<uint32_t>(-15) : 0u);
}
#else
__host__ __forceinline__ uint64_t mad_eps(uint32_t m, uint64_t t) { return t + m * EPS; }
__host__ __forceinline__ uint64_t less_eps(uint64_t x, bool borrow) { return x - (borrow ? EPS : 0); }
#endif

// a + b, canonical for canonical a and b.  t = a + b and s = t + eps (mod
// 2^64).  s wraps past 2^64 exactly when a + b >= p (b + eps < 2^64 for b < p),
// and then s = a + b - p < a; otherwise s >= a and the sum is t.  Two 64-bit
// adds, one compare, two selects.
__host__ __device__ __forceinline__ uint64_t add(uint64_t a, uint64_t b) {
    const uint64_t t = a + b;
    const uint64_t s = t + EPS;
    return s < a ? s : t;
}

// a + b (mod p) as some u64, for canonical b and ANY u64 a: a carry out of
// 2^64 is worth eps, and a + b - 2^64 + eps < 2^64 because
// a + b <= 2^64 - 1 + p - 1.  Four VALU instructions (64-bit add, compare,
// select, multiply-add) against add's five.
__host__ __device__ __forceinline__ uint64_t add_lazy(uint64_t a, uint64_t b) {
    const uint64_t t = a + b;
    return mad_eps(t < b ? 1u : 0u, t);
}

// a - b (mod p) for canonical b: canonical for canonical a, some u64 for ANY
// u64 a.  A borrow out of 64 bits is worth -2^64 = -eps, i.e. d - eps, which
// stays >= 0 because b <= p - 1.  Four VALU instructions: the borrow chain,
// a select and the multiply-add of less_eps (five with d - eps as a second
// borrow chain).
__host__ __device__ __forceinline__ uint64_t sub(uint64_t a, uint64_t b) {
    unsigned b0, b1;
    const uint32_t d0 = __builtin_subc(static_cast<uint32_t>(a), static_cast<uint32_t>(b), 0u, &b0);
    const uint32_t d1 = __builtin_subc(static_cast<uint32_t>(a >> 32), static_cast<uint32_t>(b >> 32), b0, &b1);
    return less_eps(pack64(d0, d1), b1 != 0);
}

__host__ __device__ __forceinline__ uint64_t neg(uint64_t a) { return a ? P - a : 0; }

// The canonical form of r + carry 2^64, where r < 2^64 - 2^33 + 1 if the carry
// is set: a carry is worth eps, and r + eps is then already canonical; without
// it r + eps is r - p exactly when r >= p.  So r + eps when either holds, else
// r: compare, select, multiply-add and one SALU or.
#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ uint64_t canon_carry(uint64_t r, uint64_t carry) {
    const uint64_t ge = __builtin_amdgcn_ballot_w64(r >= P);
    return mad_eps(__builtin_amdgcn_inverse_ballot_w64(ge | carry) ? 1u : 0u, r);
}
#endif

// Fold a 128-bit value (hi:lo) to a canonical element, any lo and hi:
// hi:lo = lo + hl 2^64 + hh 2^96 = lo + hl eps - hh (mod p).
// On the device t = lo - hh (mod p, t >= 0), then t + hl eps with its carry:
// 8 VALU instructions.
__host__ __device__ __forceinline__ uint64_t fold128(uint64_t lo, uint64_t hi) {
    const uint32_t hh = static_cast<uint32_t>(hi >> 32), hl = static_cast<uint32_t>(hi);
#if defined(__HIP_DEVICE_COMPILE__)
    // lo - hh and its borrow's correction word; written out, because a subtract
    // of zero with a borrow becomes a select and a second subtract in the
    // compiler.  The s_nop lines are the two wait states gfx950 needs between a
    // VALU write of VCC and a VALU read of it.
    uint32_t d0, d1, m;
    asm("v_sub_co_u32 %0, vcc, %3, %5\n\t"
        "s_nop 1\n\t"
        "v_subbrev_co_u32 %1, vcc, 0, %4, vcc\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32 %2, 0, -15, vcc"
        : "=&v"(d0), "=&v"(d1), "=v"(m)
        : "v"(static_cast<uint32_t>(lo)), "v"(static_cast<uint32_t>(lo >> 32)), "v"(hh)
        : "vcc");
    const uint64_t t = less_eps_word(pack64(d0, d1), m);
    uint64_t c;
    const uint64_t r = mad_eps(hl, t, &c);
    return canon_carry(r, c);
#else
    uint64_t t = lo - hh;                                   // lo - hh*2^96
    t -= (lo < hh) ? EPS : 0;                               // borrow of 2^64 = eps
    const uint64_t m = (uint64_t{hl} << 32) - hl;           // hl * eps < 2^64
    uint64_t r = t + m;
    r += (r < m) ? EPS : 0;                                 // carry of 2^64 = eps
    return r >= P ? r - P : r;
#endif
}

// hi 2^64 + lo for hi < 2^32 as some u64: the carry out of lo + hi eps is worth
// eps once more (the sum wrapped, so it is below 2^64 - 2^33 + 1).  3 VALU
// instructions on the device.
__host__ __device__ __forceinline__ uint64_t fold96_lazy(uint64_t lo, uint32_t hi) {
#if defined(__HIP_DEVICE_COMPILE__)
    uint64_t r;
    uint32_t m;
    asm("v_mad_u64_u32 %0, vcc, %2, -1, %3\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32 %1, 0, 1, vcc"
        : "=&v"(r), "=v"(m)
        : "v"(hi), "v"(lo)
        : "vcc");
    return mad_eps(m, r);
#else
    const uint64_t r = lo + hi * EPS;
    return r < lo ? r + EPS : r;
#endif
}

// Fold hi 2^64 + lo for hi < 2^32 (hi 2^64 = hi eps): fold128 without the
// hh 2^96 term, 4 VALU instructions on the device.
__host__ __device__ __forceinline__ uint64_t fold96(uint64_t lo, uint32_t hi) {
#if defined(__HIP_DEVICE_COMPILE__)
    uint64_t c;
    const uint64_t r = mad_eps(hi, lo, &c);
    return canon_carry(r, c);
#else
    return fold128(lo, hi);
#endif
}

#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ void mul_wide(uint64_t a, uint64_t b, uint64_t& lo, uint64_t& hi) {
    lo = a * b;
    hi = __umul64hi(a, b);
}
#else
inline void mul_wide(uint64_t a, uint64_t b, uint64_t& lo, uint64_t& hi) {
    const unsigned __int128 p = static_cast<unsigned __int128>(a) * b;
    lo = static_cast<uint64_t>(p);
    hi = static_cast<uint64_t>(p >> 64);
}
#endif

__host__ __device__ __forceinline__ uint64_t mul(uint64_t a, uint64_t b) {
    uint64_t lo, hi;
    mul_wide(a, b, lo, hi);
    return fold128(lo, hi);
}

// The same product from four 32x32->64 partial products, each of which maps
// onto one v_mad_u64_u32 on gfx950 (no carries can overflow: every partial
// sum stays below 2^64).
__host__ __device__ __forceinline__ uint64_t mul32x4(uint64_t a, uint64_t b) {
    const uint32_t a0 = static_cast<uint32_t>(a), a1 = static_cast<uint32_t>(a >> 32);
    const uint32_t b0 = static_cast<uint32_t>(b), b1 = static_cast<uint32_t>(b >> 32);
    const uint64_t p00 = static_cast<uint64_t>(a0) * b0;
    const uint64_t p01 = static_cast<uint64_t>(a0) * b1 + (p00 >> 32);
    const uint64_t p10 = static_cast<uint64_t>(a1) * b0 + static_cast<uint32_t>(p01);
    const uint64_t hi = static_cast<uint64_t>(a1) * b1 + (p01 >> 32) + (p10 >> 32);
    const uint64_t lo = (p10 << 32) | static_cast<uint32_t>(p00);
    return fold128(lo, hi);
}

inline uint64_t pow_host(uint64_t a, uint64_t e) {
    uint64_t acc = 1;
    while (e) {
        if (e & 1) acc = mul(acc, a);
        a = mul(a, a);
        e >>= 1;
    }
    return acc;
}

inline uint64_t inv_host(uint64_t a) { return pow_host(a, P - 2); }

// Primitive 2^bits-th root of unity 7^((p-1) >> bits): the generator and
// 2-adicity of the reference's NTT (rust/volta-pcs/src/ntt.rs:9-12).
inline uint64_t root_of_unity(unsigned bits) { return pow_host(7, (P - 1) >> bits); }

// i16 -> field: non-negative values embed as-is, negatives as p - |x|
// (rust/volta-field/src/lib.rs:32-40).
__host__ __device__ __forceinline__ uint64_t from_i16(int16_t x) {
    return x >= 0 ? static_cast<uint64_t>(x) : P - static_cast<uint64_t>(-static_cast<int32_t>(x));
}

// ---- quadratic extension Fp2 = Fp[phi]/(phi^2 - 7) -----------------------

struct alignas(8) Fp2 {
    uint64_t c0;
    uint64_t c1;
};

__host__ __device__ __forceinline__ Fp2 fp2_add(Fp2 a, Fp2 b) { return Fp2{add(a.c0, b.c0), add(a.c1, b.c1)}; }

__host__ __device__ __forceinline__ Fp2 fp2_mul(Fp2 a, Fp2 b) {
    // (a0 + a1 phi)(b0 + b1 phi) = (a0 b0 + 7 a1 b1) + (a0 b1 + a1 b0) phi
    return Fp2{add(mul(a.c0, b.c0), mul(7, mul(a.c1, b.c1))), add(mul(a.c0, b.c1), mul(a.c1, b.c0))};
}

__host__ __device__ __forceinline__ Fp2 fp2_mul_base(Fp2 a, uint64_t x) { return Fp2{mul(a.c0, x), mul(a.c1, x)}; }

}  // namespace gl
