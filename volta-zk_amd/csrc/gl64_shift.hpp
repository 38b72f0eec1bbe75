// gl64_shift.hpp -- Goldilocks multiply-by-power-of-two and the small DFTs
// built on it.
//
// 2 has multiplicative order 192 mod p (2^96 = -1), and the reference's roots
// of unity of order <= 64 are all powers of 2:
//     w_64 = 7^((p-1)/64) = 2^39,  w_32 = 2^78,  w_16 = 2^156,  w_8 = 2^120,
//     w_4 = 2^48,  w_2 = 2^96 = -1,  and  w_128 = 2^43 - 2^91.
// (checked by tests/test_fast_constants.py against 7^((p-1)/2^k)).
// So every twiddle inside a DFT of length <= 64 is a shift followed by a
// fold of the 128-bit result; no 64x64 product is needed.  All exponents are
// template parameters, so after unrolling each butterfly is straight-line
// code with immediate shift counts.
#pragma once

#include <type_traits>

#include "gl64.hpp"

namespace gl {

constexpr int E_W64 = 39;  // w_64 = 2^39
constexpr int E_W32 = 78;  // w_32 = 2^78

// x << S and x >> S as one 64-bit instruction on the device, where the compiler
// would take two 32-bit ones when it needs the halves apart.
template <int S>
__host__ __device__ __forceinline__ uint64_t shl64(uint64_t x) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (S > 0 && S < 32) {
        uint64_t r;
        asm("v_lshlrev_b64 %0, %1, %2" : "=v"(r) : "n"(S), "v"(x));
        return r;
    }
#endif
    return x << S;
}
template <int S>
__host__ __device__ __forceinline__ uint64_t shr64(uint64_t x) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (S > 0 && S < 32) {
        uint64_t r;
        asm("v_lshrrev_b64 %0, %1, %2" : "=v"(r) : "n"(S), "v"(x));
        return r;
    }
#endif
    return x >> S;
}

// The multiplications by a power of two below take any u64 and give a
// canonical result.

// x * 2^-M mod p for 1 <= M <= 32.
// With x = q 2^M + r (r < 2^M): x 2^-M = q + r 2^-M and 2^-M = -2^(96-M), so
// x 2^-M = q - r 2^(32-M) 2^64 = q - r' eps with r' = r 2^(32-M) < 2^32; both
// q < 2^(64-M) and r' eps <= (2^32-1)^2 are canonical.
template <int M>
__host__ __device__ __forceinline__ uint64_t shr_mod(uint64_t x) {
    static_assert(M >= 1 && M <= 32, "shift out of range");
    const uint64_t q = shr64<M>(x);
    const uint32_t rp = static_cast<uint32_t>(x) << (32 - M);
    return sub(q, static_cast<uint64_t>(rp) * EPS);
}

// x * 2^(32+SM) mod p for 0 <= SM < 32.
// In 32-bit words x 2^SM = W1 + W2 2^32 + W3 2^64, so x 2^(32+SM) =
// W1 2^32 + W2 2^64 + W3 2^96 = (W1 + W2) 2^32 - (W2 + W3)  (2^64 = 2^32 - 1,
// 2^96 = -1): two 32-bit sums and one borrow-corrected 64-bit difference.
template <int SM>
__host__ __device__ __forceinline__ uint64_t shl_mod_hi(uint64_t x) {
    static_assert(SM >= 0 && SM < 32, "shift out of range");
    const uint64_t xs = shl64<SM>(x);
    const uint32_t w1 = static_cast<uint32_t>(xs), w2 = static_cast<uint32_t>(xs >> 32);
    const uint32_t w3 = SM == 0 ? 0u : static_cast<uint32_t>(x >> 32) >> ((32 - SM) & 31);
    unsigned ca, cb, c2, b0, b1;
    const uint32_t a = __builtin_addc(w1, w2, 0u, &ca);  // A = a + ca 2^32
    const uint32_t b = __builtin_addc(w2, w3, 0u, &cb);  // B = b + cb 2^32 < 2^32 + 2^31
    const uint32_t h = a + ca;                           // A 2^32 = (a + ca) 2^32 - ca
    const uint32_t clo = __builtin_addc(b, 0u, ca, &c2); // C = B + ca = clo + chi 2^32
    const uint32_t chi = cb | c2;
    const uint32_t r0 = __builtin_subc(0u, clo, 0u, &b0);  // r = h 2^32 - C
    const uint32_t r1 = __builtin_subc(h, chi, b0, &b1);
    return less_eps(pack64(r0, r1), b1 != 0);  // negative: + p = - eps mod 2^64
}

// -(x * 2^(32+SM)) mod p for 0 <= SM < 32.
// With the words of x 2^SM as in shl_mod_hi, the value is (W2 + W3) - (W1 + W2) X
// (X = 2^32).  W1 + W2 = s + cs X and cs X^2 = cs (X - 1), so it is
// L - h X with h = s + cs < 2^32 (no carry: cs = 1 leaves s <= 2^32 - 2) and
// L = W2 + W3 + cs = l0 + cl X: the word l0 and the difference cl - h, formed as
// 1 - h - (1 - cl) so that one subtract-with-borrow takes both.  A borrow means
// a negative value: + p, i.e. - eps mod 2^64.  Two shifts and six VALU
// instructions, against ten for the positive value.
template <int SM>
__host__ __device__ __forceinline__ uint64_t shl_mod_hi_neg(uint64_t x) {
    static_assert(SM >= 0 && SM < 32, "shift out of range");
    const uint64_t xs = shl64<SM>(x);
    const uint32_t w1 = static_cast<uint32_t>(xs), w2 = static_cast<uint32_t>(xs >> 32);
    const uint32_t w3 = SM == 0 ? 0u : static_cast<uint32_t>(x >> 32) >> ((32 - SM) & 31);
    unsigned cs, none, cl, b;
    const uint32_t s = __builtin_addc(w1, w2, 0u, &cs);
    const uint32_t h = __builtin_addc(s, 0u, cs, &none);
    const uint32_t l0 = __builtin_addc(w2, w3, cs, &cl);
    const uint32_t hi = __builtin_subc(1u, h, cl ? 0u : 1u, &b);
    return less_eps(pack64(l0, hi), b != 0);
}

// x * 2^S mod p for 0 <= S < 96 (S = 0: x itself, canonical if x is).
template <int S>
__host__ __device__ __forceinline__ uint64_t shl_mod(uint64_t x) {
    static_assert(S >= 0 && S < 96, "shift out of range");
    if constexpr (S == 0) {
        return x;
    } else if constexpr (S < 32) {
        return fold96(x << S, static_cast<uint32_t>(x >> (64 - S)));
    } else if constexpr (S < 64) {
        return shl_mod_hi<S - 32>(x);
    } else {
        // 2^S = -2^-(96-S): one division by a power of two <= 2^32.
        return neg(shr_mod<96 - S>(x));
    }
}

// -(x * 2^S) mod p for 32 <= S < 96, whose negative is the cheaper form.
template <int S>
__host__ __device__ __forceinline__ uint64_t shl_mod_neg(uint64_t x) {
    static_assert(S >= 32 && S < 96, "no cheap negative below 2^32");
    if constexpr (S < 64) return shl_mod_hi_neg<S - 32>(x);
    else return shr_mod<96 - S>(x);
}

// x * 2^E mod p for any E >= 0: with S = (E mod 192) mod 96, 2^E = +-2^S.
template <int E>
__host__ __device__ __forceinline__ uint64_t mul_pow2(uint64_t x) {
    constexpr int S = (E % 192) % 96;
    constexpr bool minus = E % 192 >= 96;
    if constexpr (S >= 64) {
        const uint64_t t = shl_mod_neg<S>(x);
        if constexpr (minus) return t;
        else return neg(t);
    } else if constexpr (S >= 32) {
        if constexpr (minus) return shl_mod_neg<S>(x);
        else return shl_mod<S>(x);
    } else {
        const uint64_t t = shl_mod<S>(x);
        if constexpr (minus) return neg(t);
        else return t;
    }
}

// DIT butterfly (u, v) <- (u + w v, u - w v) with w = 2^E, any u64 u, and v any
// u64 unless the twiddle is trivial (E a multiple of 96), canonical then.  The
// twiddled value is canonical, so both results take the four-instruction add
// and sub; an output whose flag (CU, CV: u's, v's new value) is set is
// canonical, which needs a canonical u.
template <int E, bool CU = true, bool CV = true>
__host__ __device__ __forceinline__ void bfly_pow2(uint64_t& u, uint64_t& v) {
    // w = +-2^S with S = e mod 96; from S = 32 on the negative -(v 2^S) is the
    // cheaper form, which flips the sign once more.
    constexpr int e = E % 192, S = e % 96;
    constexpr bool neg_t = (e >= 96) != (S >= 32);
    uint64_t t;
    if constexpr (S >= 32) t = shl_mod_neg<S>(v);
    else t = shl_mod<S>(v);
    const uint64_t d = sub(u, t);
    uint64_t a;
    if constexpr (neg_t ? CV : CU) a = add(u, t);
    else a = add_lazy(u, t);
    u = neg_t ? d : a;
    v = neg_t ? a : d;
}

// Field element of a signed 64-bit integer y with |y| < 2^63: y, or y + p
// for y < 0.  In two's complement y + p = (2^64 + y) - eps, and the sign word
// y >> 63 read as an unsigned 32-bit value is eps exactly when y < 0.
__host__ __device__ __forceinline__ uint64_t from_i64(uint64_t y) {
    const uint32_t m = static_cast<uint32_t>(static_cast<int32_t>(static_cast<uint32_t>(y >> 32)) >> 31);
    return y - m;
}

// Field element of a * 2^S for |a| <= 2^15 (a signed), 0 <= S < 96.
template <int S>
__host__ __device__ __forceinline__ uint64_t small_shl_abs(uint32_t ax) {
    if constexpr (S + 16 <= 63) {
        return static_cast<uint64_t>(ax) << S;  // < 2^63 < p
    } else if constexpr (S < 64) {
        return fold96(static_cast<uint64_t>(ax) << S, static_cast<uint32_t>(static_cast<uint64_t>(ax) >> (64 - S)));
    } else {
        return shl_mod<S>(static_cast<uint64_t>(ax));
    }
}

// Field element of x * 2^E for a signed 16-bit x (any E >= 0).  Up to a
// shift of 47 the product +-x 2^s is an exact signed 64-bit integer
// (|x| <= 2^15), so one sign fix-up replaces the modular reduction.
template <int E>
__host__ __device__ __forceinline__ uint64_t i16_mul_pow2(int32_t x) {
    constexpr int e = E % 192;
    constexpr bool flip = e >= 96;
    constexpr int s = flip ? e - 96 : e;
    if constexpr (s <= 47) {
        const uint64_t v = static_cast<uint64_t>(static_cast<int64_t>(flip ? -x : x));
        return from_i64(v << s);
    } else {
        const uint32_t ax = static_cast<uint32_t>(x < 0 ? -x : x);
        const uint64_t m = small_shl_abs<s>(ax);
        const bool negate = (x < 0) != flip;
        return negate ? neg(m) : m;
    }
}

// Field element of x * w_128^k for a signed 16-bit x: w_128^k = 2^(39 k/2)
// for even k; 2^(43+c) - 2^(91+c) = 2^(43+c) (1 - 2^48) with c = 39 (k-1)/2
// for odd k.  x (1 - 2^48) is an exact signed 64-bit integer (|x| <= 2^15),
// so the odd case is one sign fix-up and one modular shift.
template <int K>
__host__ __device__ __forceinline__ uint64_t i16_mul_w128(int32_t x) {
    if constexpr (K % 2 == 0) {
        return i16_mul_pow2<E_W64 * (K / 2)>(x);
    } else {
        constexpr int c = E_W64 * ((K - 1) / 2);
        const uint64_t v = static_cast<uint64_t>(static_cast<int64_t>(x));
        return mul_pow2<43 + c>(from_i64(v - (v << 48)));
    }
}

// ---- unrolled small DFTs on register arrays -------------------------------

template <int I>
using ic = std::integral_constant<int, I>;

// Compile-time loop: f(ic<B>), f(ic<B+1>), ..., f(ic<E-1>).
template <int B, int E, class F>
__host__ __device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(ic<B>{});
        static_for<B + 1, E>(f);
    }
}

// Which positions must be canonical after the stage of span LEN of an
// N = 2^LOG point dit_pow2 with root 2^EW, so that the positions in `need` are
// canonical after its last stage: backwards through the later stages, u of a
// pair for either output, v of a pair whose twiddle is trivial.
constexpr uint64_t dit_need_after(int log, int ew, int len, uint64_t need) {
    const int n = 1 << log;
    for (int l = n; l > len; l >>= 1) {
        const int half = l / 2;
        uint64_t before = 0;
        for (int s = 0; s < n; s += l)
            for (int k = 0; k < half; ++k) {
                if (((need >> (s + k)) | (need >> (s + k + half))) & 1) before |= uint64_t{1} << (s + k);
                if ((ew * k * (n / l)) % 96 == 0) before |= uint64_t{1} << (s + k + half);
            }
        need = before;
    }
    return need;
}

constexpr uint64_t DIT_ALL = ~uint64_t{0};

// In-place radix-2 DIT DFT of length N = 2^LOG with root 2^EW on v[], which
// holds the input in bit-reversed order; output in natural order.  Inputs are
// canonical; the outputs in NEED are canonical, the others any u64 (enough for
// a value that a multiplication follows).
template <int LOG, int EW, int LEN = 2, uint64_t NEED = DIT_ALL>
__host__ __device__ __forceinline__ void dit_pow2(uint64_t* v) {
    if constexpr (LEN <= (1 << LOG)) {
        constexpr int N = 1 << LOG;
        constexpr int HALF = LEN / 2;
        constexpr uint64_t C = dit_need_after(LOG, EW, LEN, NEED);
        static_for<0, N / LEN>([&](auto g) {
            constexpr int start = decltype(g)::value * LEN;
            static_for<0, HALF>([&](auto kk) {
                constexpr int k = decltype(kk)::value;
                // w_LEN^k = w_N^(k N/LEN) = 2^(EW k N/LEN)
                bfly_pow2<EW * k * (N / LEN), ((C >> (start + k)) & 1) != 0, ((C >> (start + k + HALF)) & 1) != 0>(
                    v[start + k], v[start + k + HALF]);
            });
        });
        dit_pow2<LOG, EW, LEN * 2, NEED>(v);
    }
}

// The positions that may be nonzero after a stage of span LEN of dit_pow2
// whose input may be nonzero at the positions in m: both of a pair, if either.
constexpr uint64_t dit_mask_next(uint64_t m, int len, int n) {
    uint64_t r = 0;
    const int half = len / 2;
    for (int s = 0; s < n; s += len)
        for (int k = 0; k < half; ++k)
            if (((m >> (s + k)) | (m >> (s + k + half))) & 1) r |= (uint64_t{1} << (s + k)) | (uint64_t{1} << (s + k + half));
    return r;
}

// dit_pow2 for an input that is known to be zero outside the positions set in
// MASK (bit i: v[i] may be nonzero; the other positions must hold 0).  A
// butterfly whose second input is known zero is the copy (u, u), one whose
// inputs are both known zero is skipped, so a zero tail of the input costs no
// arithmetic in the stages it reaches.  Runs the stages of spans LEN, 2 LEN,
// ... below STOP (all of them by default); NEED as in dit_pow2, after the last
// stage of the whole DFT.
template <int LOG, int EW, uint64_t MASK, int LEN = 2, int STOP = (2 << LOG), uint64_t NEED = DIT_ALL>
__host__ __device__ __forceinline__ void dit_pow2_sparse(uint64_t* v) {
    if constexpr (LEN <= (1 << LOG) && LEN < STOP) {
        constexpr int N = 1 << LOG;
        constexpr int HALF = LEN / 2;
        constexpr uint64_t C = dit_need_after(LOG, EW, LEN, NEED);
        static_for<0, N / LEN>([&](auto g) {
            constexpr int start = decltype(g)::value * LEN;
            static_for<0, HALF>([&](auto kk) {
                constexpr int k = decltype(kk)::value;
                constexpr bool nz_u = (MASK >> (start + k)) & 1, nz_v = (MASK >> (start + k + HALF)) & 1;
                if constexpr (nz_v) {
                    bfly_pow2<EW * k * (N / LEN), ((C >> (start + k)) & 1) != 0, ((C >> (start + k + HALF)) & 1) != 0>(
                        v[start + k], v[start + k + HALF]);
                } else if constexpr (nz_u) {
                    v[start + k + HALF] = v[start + k];
                }
            });
        });
        dit_pow2_sparse<LOG, EW, dit_mask_next(MASK, LEN, N), LEN * 2, STOP, NEED>(v);
    }
}

// Bit reversal of I over LOG bits, at compile time.
constexpr int bitrev_c(int i, int log) {
    int r = 0;
    for (int b = 0; b < log; ++b) r |= ((i >> b) & 1) << (log - 1 - b);
    return r;
}

}  // namespace gl
