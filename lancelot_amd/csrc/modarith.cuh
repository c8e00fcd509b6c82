// Device-side 64-bit modular arithmetic for gfx950 (wave64, VALU integer multiplies).
//
// All routines work on residues of primes below 2^61.  "lazy" values live in [0, 4q) or [0, 8q) and
// never leave a kernel: every store to HBM that a caller can observe is the canonical residue, which
// is what makes limb-for-limb comparison with the CPU oracle meaningful.
//
// Semantics follow cahel-main/include/uintmodmath.cuh (Shoup :226-245, Barrett :112-218) and
// cahel-main/src/ntt/butterfly.cuh:10-43 (Harvey butterflies); the code is written for the CDNA4
// integer pipeline (64x64 products are assembled from v_mad_u64_u32 by the compiler).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace he {

struct Shoup {
    uint64_t w;   // operand in [0, q)
    uint64_t wq;  // floor(w * 2^64 / q)
};

__device__ __forceinline__ uint64_t mulhi64(uint64_t a, uint64_t b) { return __umul64hi(a, b); }

// x * w mod q up to one subtraction of q: result in [0, 2q).  x may be any 64-bit value.
__device__ __forceinline__ uint64_t mul_shoup_lazy(uint64_t x, Shoup s, uint64_t q) {
    uint64_t hi = mulhi64(x, s.wq);
    return x * s.w - hi * q;
}

__device__ __forceinline__ uint64_t mul_shoup(uint64_t x, Shoup s, uint64_t q) {
    uint64_t r = mul_shoup_lazy(x, s, q);
    return r >= q ? r - q : r;
}

__device__ __forceinline__ uint64_t add_mod(uint64_t a, uint64_t b, uint64_t q) {
    uint64_t s = a + b;
    return s >= q ? s - q : s;
}

__device__ __forceinline__ uint64_t sub_mod(uint64_t a, uint64_t b, uint64_t q) {
    return a >= b ? a - b : a + q - b;
}

__device__ __forceinline__ uint64_t neg_mod(uint64_t a, uint64_t q) { return a ? q - a : 0; }

// 128-bit value (hi:lo) mod q with ratio = floor(2^128 / q) = (r1:r0), q < 2^62.  r1 = floor(2^64 / q), so
// w = 2^64 mod q = 2^64 - r1 q, and r0 = floor(2^128 / q) - r1 2^64 = floor(w 2^64 / q) is the Shoup quotient of w:
// hi w - floor(hi r0 / 2^64) q lies in [0, 2q) for every hi below 2^64, and lo - floor(lo r1 / 2^64) q in [0, 2q).
// Two high and three low 64-bit products (w comes from scalar operands) where the plain Barrett reduction of the
// 128-bit value takes four and four.
__device__ __forceinline__ uint64_t barrett128(uint64_t lo, uint64_t hi, uint64_t q, uint64_t r0, uint64_t r1) {
    const uint64_t w = 0 - r1 * q;
    const uint64_t a = hi * w - mulhi64(hi, r0) * q;
    const uint64_t b = lo - mulhi64(lo, r1) * q;
    const uint64_t q2 = q << 1;
    uint64_t r = a + b;
    r = r >= q2 ? r - q2 : r;
    return r >= q ? r - q : r;
}

__device__ __forceinline__ uint64_t mul_mod(uint64_t a, uint64_t b, uint64_t q, uint64_t r0, uint64_t r1) {
    return barrett128(a * b, mulhi64(a, b), q, r0, r1);
}

// 64-bit value mod q with r1 = floor(2^64 / q).
__device__ __forceinline__ uint64_t barrett64(uint64_t x, uint64_t q, uint64_t r1) {
    uint64_t r = x - mulhi64(r1, x) * q;
    return r >= q ? r - q : r;
}

struct U128 {
    uint64_t lo, hi;
};

__device__ __forceinline__ void mac128(U128 &acc, uint64_t a, uint64_t b) {
    uint64_t lo = a * b;
    uint64_t hi = mulhi64(a, b);
    acc.lo += lo;
    acc.hi += hi + (acc.lo < lo);
}

// Lazy sum of products of residues below 2^61 with few carries.  The factors are split at bit 30
// (a = a1 2^30 + a0 with a0 < 2^30, a1 < 2^31); the four partial products of a term go, by weight, into three
// 64-bit words (ll: a0 b0 < 2^60, mid: a1 b0 + a0 b1 < 2^62, hh: a1 b1 < 2^62), each a 32 x 32 + 64 multiply-add with
// no carry out.  Four terms fit (4 * 2^62 = 2^64) before the words have to be relieved (spill3), eight when the
// residues are below 2^60 (a1 < 2^30: mid < 2^61, hh < 2^60), so a product costs 4 multiply-adds and a few
// additions instead of a 64 x 64 -> 128 product (6 multiplies) and a carry chain.  (Measured on gfx950: every
// 32-bit multiply, v_mad_u64_u32 included, issues at the rate of an FP64 fused multiply-add, half the rate of a
// 32-bit addition.)
struct Split30 {
    uint32_t lo, hi;
};

__device__ __forceinline__ Split30 split30(uint64_t a) { return Split30{(uint32_t)a & 0x3fffffffu, (uint32_t)(a >> 30)}; }

struct Lazy3 {
    uint64_t ll, mid, hh;
};

// One term for two sums that share the factor a (the two key polynomials of an inner product): eight
// v_mad_u64_u32 (32 x 32 + 64 -> 64; the carry out goes to a scalar pair that nobody reads, the sums stay below
// 2^64).  Written out because the compiler emits a multiply with a zero addend followed by a 64-bit add for
// `acc += (uint64_t)a * b`, and one statement because it separates inline-assembly statements by s_nop.
__device__ __forceinline__ void mac3x2(Lazy3 &s, Lazy3 &t, Split30 a, Split30 b, Split30 c) {
    uint64_t carry;
    asm("v_mad_u64_u32 %0, %6, %7, %9, %0\n\t"
        "v_mad_u64_u32 %1, %6, %8, %9, %1\n\t"
        "v_mad_u64_u32 %2, %6, %8, %10, %2\n\t"
        "v_mad_u64_u32 %3, %6, %7, %11, %3\n\t"
        "v_mad_u64_u32 %4, %6, %8, %11, %4\n\t"
        "v_mad_u64_u32 %5, %6, %8, %12, %5\n\t"
        "v_mad_u64_u32 %1, %6, %7, %10, %1\n\t"
        "v_mad_u64_u32 %4, %6, %7, %12, %4"
        : "+v"(s.ll), "+v"(s.mid), "+v"(s.hh), "+v"(t.ll), "+v"(t.mid), "+v"(t.hh), "=&s"(carry)
        : "v"(a.lo), "v"(a.hi), "v"(b.lo), "v"(b.hi), "v"(c.lo), "v"(c.hi));
}

// The upper halves of the three words move into three counters of weight 2^32 (two additions and a move per word:
// no carries between the words), which leaves room for the next four (eight) terms; total3 puts the six words
// together at the end.  Up to 64 terms (the counters stay below 2^37).
__device__ __forceinline__ void spill3(Lazy3 &h, Lazy3 &s) {
    h.ll += s.ll >> 32;
    s.ll &= 0xffffffffu;
    h.mid += s.mid >> 32;
    s.mid &= 0xffffffffu;
    h.hh += s.hh >> 32;
    s.hh &= 0xffffffffu;
}

__device__ __forceinline__ U128 total3(const Lazy3 &h, const Lazy3 &s) {
    typedef unsigned __int128 u128;
    const u128 t = ((u128)s.ll + ((u128)h.ll << 32)) + (((u128)s.mid + ((u128)h.mid << 32)) << 30) +
                   (((u128)s.hh + ((u128)h.hh << 32)) << 60);
    return U128{(uint64_t)t, (uint64_t)(t >> 64)};
}

// The same sum with three multiply-adds per product: a1 b0 + a0 b1 = a0 b0 + a1 b1 - (a1 - a0)(b1 - b0), the difference's product
// summed with its sign.  Residues below 2^60: |a1 - a0| < 2^30, eight terms fit into 63 bits (and sixteen into ll and hh);
// below 2^61: |a1 - a0| < 2^31, two terms.
struct Split30d {
    uint32_t lo, hi;
    int32_t d;
};

__device__ __forceinline__ Split30d split30d(uint64_t a) {
    const Split30 s = split30(a);
    return Split30d{s.lo, s.hi, (int32_t)(s.hi - s.lo)};
}

struct Sum3 {
    uint64_t ll, hh;
    int64_t mm;
};

// one term for two sums that share the factor a (see mac3x2)
__device__ __forceinline__ void mac_sum3x2(Sum3 &s, Sum3 &t, Split30d a, Split30d b, Split30d c) {
    uint64_t carry;
    asm("v_mad_u64_u32 %0, %6, %7, %10, %0\n\t"
        "v_mad_u64_u32 %3, %6, %7, %13, %3\n\t"
        "v_mad_u64_u32 %1, %6, %8, %11, %1\n\t"
        "v_mad_u64_u32 %4, %6, %8, %14, %4\n\t"
        "v_mad_i64_i32 %2, %6, %9, %12, %2\n\t"
        "v_mad_i64_i32 %5, %6, %9, %15, %5"
        : "+v"(s.ll), "+v"(s.hh), "+v"(s.mm), "+v"(t.ll), "+v"(t.hh), "+v"(t.mm), "=&s"(carry)
        : "v"(a.lo), "v"(a.hi), "v"(a.d), "v"(b.lo), "v"(b.hi), "v"(b.d), "v"(c.lo), "v"(c.hi), "v"(c.d));
}

__device__ __forceinline__ void spill_sum3(Sum3 &h, Sum3 &s) {
    h.ll += s.ll >> 32;
    s.ll &= 0xffffffffu;
    h.hh += s.hh >> 32;
    s.hh &= 0xffffffffu;
    h.mm += s.mm >> 32;
    s.mm &= 0xffffffff;
}

__device__ __forceinline__ U128 total_sum3(const Sum3 &h, const Sum3 &s) {
    typedef unsigned __int128 u128;
    const u128 ll = (u128)s.ll + ((u128)h.ll << 32), hh = (u128)s.hh + ((u128)h.hh << 32);
    const u128 mm = (u128)(__int128)s.mm + ((u128)(__int128)h.mm << 32);     // modulo 2^128; the difference below is not negative
    const u128 t = ll + ((ll + hh - mm) << 30) + (hh << 60);
    return U128{(uint64_t)t, (uint64_t)(t >> 64)};
}

// The butterflies' view of a modulus: q, and modulo 2^64 the numbers that make every sum, difference and conditional subtraction of a
// butterfly 64-bit additions (one instruction each): -q, -2q, -4q, and 4q + 1, with which x + 4q - t is (x + 4q + 1) + ~t.  Borrow chains
// through VCC need two idle issue slots between producer and consumer on this GPU, which a SIMD with one wave cannot fill (a slot costs
// such a wave 1.6 ns, any vector instruction 2.0 to 2.2; with eight waves 1.0 for the simplest and 1.75 for all others, 32-bit
// multiplications included).  The numbers pass through an empty asm statement so that the compiler does not fold them back into
// subtractions.
struct IntMod {
    uint64_t q, q4p, nq, nq2, nq4;
};

// (q is the same in every lane of a wave: a workgroup works on one limb; read from lane 0 so that the constants are
// scalars wherever the compiler cannot see that)
__device__ __forceinline__ IntMod int_mod(uint64_t q_any_lane) {
    const uint32_t q_hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(q_any_lane >> 32));
    const uint32_t q_lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)q_any_lane);   // (the builtin returns int)
    const uint64_t q = ((uint64_t)q_hi << 32) | q_lo, q2 = 2 * q, q4 = 4 * q, q4p = q4 + 1;
    // (as 32-bit scalars)
    uint32_t a0 = (uint32_t)(0 - q), a1 = (uint32_t)((0 - q) >> 32);
    uint32_t b0 = (uint32_t)(0 - q2), b1 = (uint32_t)((0 - q2) >> 32);
    uint32_t c0 = (uint32_t)(0 - q4), c1 = (uint32_t)((0 - q4) >> 32);
    uint32_t d0 = (uint32_t)q4p, d1 = (uint32_t)(q4p >> 32);
    asm volatile("" : "+s"(a0), "+s"(a1), "+s"(b0), "+s"(b1), "+s"(c0), "+s"(c1), "+s"(d0), "+s"(d1));
    return IntMod{q, ((uint64_t)d1 << 32) | d0, ((uint64_t)a1 << 32) | a0, ((uint64_t)b1 << 32) | b0, ((uint64_t)c1 << 32) | c0};
}

// floor(a b / 2^64) or up to two less: the products with one lower half enter with their upper words, that of both lower halves not at
// all (three fractions below 1 are lost)
__device__ __forceinline__ uint64_t mulhi64_low(uint64_t a, uint64_t b) {
    const uint32_t a0 = (uint32_t)a, a1 = (uint32_t)(a >> 32), b0 = (uint32_t)b, b1 = (uint32_t)(b >> 32);
    return (uint64_t)a1 * b1 + __umulhi(a0, b1) + __umulhi(a1, b0);
}

// y w mod q up to three subtractions of q, in [0, 4q), for any 64-bit y
__device__ __forceinline__ uint64_t mul_shoup_lazy(uint64_t y, Shoup s, const IntMod &m) {
    return y * s.w + mulhi64_low(y, s.wq) * m.nq;
}

// v - k q if that is not negative, else v; nkq = 2^64 - k q (v below 8q: the difference fits 63 bits)
__device__ __forceinline__ uint64_t reduce_once(uint64_t v, uint64_t nkq) {
    const uint64_t d = v + nkq;
    return (int32_t)(d >> 32) < 0 ? v : d;
}

// Cooley-Tukey butterfly, inputs in [0, 8q), outputs in [0, 8q): below 2^64 for q < 2^61.  21 vector instructions.  (With a quotient one
// less at most, in multiply-adds that wait for each other and need their addends moved, and ranges of 6q: 27, and a whole blocks pass 692
// against 502.  us: rotation on [60, 40, 40, 60], n = 2^16 27.0 -> 26.1; 2^15, 12 + 3 of 60 / 40 bits 54.9 -> 53.7; 2^16, 12 + 4 of 60 bits 90.6 ->
// 88.7; multiplication, 2^14, 4 + 1 28.6 -> 27.9 and 29.4 -> 29.0; eight limbs of 2^16 words and 60 bits 9.0 -> 8.8.)
__device__ __forceinline__ void ct_butterfly(uint64_t &x, uint64_t &y, Shoup tw, const IntMod &m) {
    const uint64_t t = mul_shoup_lazy(y, tw, m);
    const uint64_t xr = reduce_once(x, m.nq4);
    y = (xr + m.q4p) + ~t;
    x = xr + t;
}

// Gentleman-Sande butterfly with the division by two folded in (the inverse twiddles are stored
// pre-halved), inputs in [0, 4q), outputs in [0, 4q): the sum is below 8q, 4q once reduced, 2.5q once halved; the difference below
// 8q (2^64 for q < 2^61).  Both have the parity of x + y, so that the sum's halving does not wait for its reduction.
__device__ __forceinline__ void gs_butterfly(uint64_t &x, uint64_t &y, Shoup tw, const IntMod &m) {
    const uint64_t d = (x + m.q4p) + ~y;
    uint64_t s = reduce_once(x + y, m.nq4);
    s += (d & 1) ? m.q : 0;
    x = s >> 1;
    y = mul_shoup_lazy(d, tw, m);
}

// canonical from below 4q and 8q
__device__ __forceinline__ uint64_t reduce_4q(uint64_t v, const IntMod &m) { return reduce_once(reduce_once(v, m.nq2), m.nq); }
__device__ __forceinline__ uint64_t reduce_8q(uint64_t v, const IntMod &m) { return reduce_4q(reduce_once(v, m.nq4), m); }

__device__ __forceinline__ Shoup load_shoup(const uint64_t *table, size_t idx) {
    const ulonglong2 v = reinterpret_cast<const ulonglong2 *>(table)[idx];
    return Shoup{v.x, v.y};
}

// NTT-domain automorphism X -> X^elt as a gather: out[i] = in[pi(i)],
// pi(i) = bitrev(((elt * (2 bitrev(i) + 1)) >> 1) mod N)   (table of cahel-main/include/galois.cuh:45-57, on the fly)
__device__ __forceinline__ uint32_t galois_index(uint32_t i, uint32_t elt, uint32_t log_n) {
    const uint32_t r = __brev(i) >> (32 - log_n);
    const uint32_t raw = (uint32_t)(((uint64_t)elt * (2 * r + 1)) >> 1) & ((1u << log_n) - 1);
    return __brev(raw) >> (32 - log_n);
}

}  // namespace he

// ---------------------------------------------------------------------------------------------------
// FP64 modular arithmetic for primes below 2^50.
//
// v_fma_f64 / v_mul_f64 / v_add_f64 run at full rate on CDNA4, so a modular product costs six
// operations instead of the ~20 of a 64-bit Shoup product.  Every value is an integer held exactly
// in a double; residues are signed and lazy (|v| < 2^53).  All steps below are exact integer
// computations, so the canonical result equals the integer path's bit for bit.
//
//   x * w = h + l exactly (h = fl(x w), l = fma(x, w, -h)); k = rint(fl(h fl(1/q))), three roundings from
//   x w / q, differs from it by at most 1/2 + 1.5 |x w / q| 2^-52; h - k q and (h - k q) + l are integers
//   below 2^53 in magnitude, hence exact; the result is congruent to x w with
//   |r| <= (1/2 + 1.5 |x| 2^-52) q for |w| <= q, i.e. (1/2 + 0.375 b) q for |x| <= b q, q < 2^50.
//   (With the quotient from a second operand fl(w fl(1/q)) beside w the bound is the same, and a twiddle or a key word
//   costs one multiplication more.)
// ---------------------------------------------------------------------------------------------------
namespace he {

struct FpMod {
    double q, qinv;
};

// canonical residue (< 2^52) <-> exact double, through the exponent-bias trick
__device__ __forceinline__ double fp_from_u64(uint64_t x) {
    return __longlong_as_double((long long)(x | 0x4330000000000000ull)) - 4503599627370496.0;
}

__device__ __forceinline__ uint64_t fp_to_u64(double c) {  // 0 <= c < 2^52, integer
    return (uint64_t)__double_as_longlong(c + 4503599627370496.0) & 0x000FFFFFFFFFFFFFull;
}

__device__ __forceinline__ double fp_mulmod(double x, double w, FpMod m) {
    const double h = x * w;
    const double l = __builtin_fma(x, w, -h);
    const double k = __builtin_rint(h * m.qinv);
    return __builtin_fma(-k, m.q, h) + l;
}

// centred representative, |result| <= (1/2 + 2^-49) q for |v| < 2^53
__device__ __forceinline__ double fp_reduce(double v, FpMod m) {
    const double k = __builtin_rint(v * m.qinv);
    return __builtin_fma(-k, m.q, v);
}

// canonical residue in [0, q) as an exact double
__device__ __forceinline__ double fp_canonical(double v, FpMod m) {
    const double c = fp_reduce(v, m);
    return c < 0.0 ? c + m.q : c;
}

// Forward block: LOGR consecutive forward stages on 2^LOGR lazy signed doubles.  v[j] are the elements whose index differs in the
// LOGR bits that these stages pair, most significant first; idx = 2^s0 + (group number at the first stage s0); twiddle of local
// stage l, sub-block b is table[(idx << l) + b].  REDUCE_FIRST = 1 brings every input back to |v| <= q/2; from there
// (or from canonical inputs) the bound grows by 1.375 b + 0.5 per stage: 5.3 q after four stages, 7.1 q from
// canonical inputs, always below 8 q < 2^53.
// REDUCE_FIRST = 2 reduces only the inputs that the first stage adds and subtracts; those that it multiplies go into
// the modular product as they are (its result is at most (1/2 + 0.375 b) 2^50 for an input of b 2^50).  In units of
// 2^50, for every q below 2^50: the first stage ends at 1 + 0.375 b and each later one at 1.375 b' + 0.5, which
// is 5.92 after three stages from inputs of 4, 7.28 after three more, 5.63 after two more: for a chain of blocks of
// at most 3, 3 and 2 stages whose first inputs are at most 4 x 2^50, and whose consumer reduces first.
// (All of this for twiddles up to q; those of the tables are centred, so that a product grows by half of the 0.375.)
template <int LOGR, int REDUCE_FIRST>
__device__ __forceinline__ void fp_ct_block(double *v, const double *table, uint32_t idx, FpMod m) {
    constexpr int R = 1 << LOGR;
    static_assert(REDUCE_FIRST != 2 || LOGR <= 3, "bounds of the partial reduction are derived for blocks of at most 3 stages");
    if (REDUCE_FIRST) {
#pragma unroll
        for (int j = 0; j < (REDUCE_FIRST == 2 ? R / 2 : R); j++) v[j] = fp_reduce(v[j], m);
    }
#pragma unroll
    for (int l = 0; l < LOGR; l++) {
        const int half = R >> (l + 1);
#pragma unroll
        for (int b = 0; b < (1 << l); b++) {
            const double tw = table[((size_t)idx << l) + b];
#pragma unroll
            for (int j = 0; j < half; j++) {
                const double x = v[2 * b * half + j];
                const double t = fp_mulmod(v[2 * b * half + j + half], tw, m);
                v[2 * b * half + j] = x + t;
                v[2 * b * half + j + half] = x - t;
            }
        }
    }
}

// Inverse block (no halving: the factor 1/N is applied once at the end of the transform).  Sums double
// per stage, so in blocks of four or five stages the sum outputs are reduced again after every second stage (not
// after the last); outputs stay at or below 5 q (8 q from canonical inputs without REDUCE_FIRST), which is below 2^53.
template <int LOGR, bool REDUCE_FIRST>
__device__ __forceinline__ void fp_gs_block(double *v, const double *table, uint32_t idx, FpMod m) {
    constexpr int R = 1 << LOGR;
    if (REDUCE_FIRST) {
#pragma unroll
        for (int j = 0; j < R; j++) v[j] = fp_reduce(v[j], m);
    }
#pragma unroll
    for (int l = LOGR - 1; l >= 0; l--) {
        const int half = R >> (l + 1);
#pragma unroll
        for (int b = 0; b < (1 << l); b++) {
            const double tw = table[((size_t)idx << l) + b];
#pragma unroll
            for (int j = 0; j < half; j++) {
                const double x = v[2 * b * half + j], y = v[2 * b * half + j + half];
                v[2 * b * half + j] = x + y;
                v[2 * b * half + j + half] = fp_mulmod(x - y, tw, m);
            }
        }
        if (LOGR >= 4 && l > 0 && ((LOGR - l) & 1) == 0) {
#pragma unroll
            for (int b = 0; b < (1 << l); b++)
#pragma unroll
                for (int j = 0; j < half; j++) v[2 * b * half + j] = fp_reduce(v[2 * b * half + j], m);
        }
    }
}

}  // namespace he
