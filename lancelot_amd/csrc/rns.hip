// Streaming RNS kernels for gfx950: elementwise polynomial arithmetic, tensor product, NTT-domain Galois
// gather, base conversion (the modular matrix-vector product of ModUp / ModDown), the key-switch inner
// product, and the seeded samplers.  All of them are HBM-bound streams over [limb][coeff] arrays: one
// coefficient per lane, 256 consecutive coefficients per workgroup, so every access is a full-width
// coalesced row segment.
//
// What they compute follows cahel-main/src/polymath.cu (add :40, sub :108, multiply :160, mad :227/:349,
// tensor :531-612), src/galois.cu:20-30 + include/galois.cuh:45-57, src/rns_bconv.cu:587-623 and :166-198
// (base conversion, uncorrected sum, one reduction), src/eval_key_switch.cu:13-76 (inner product) and
// src/prng.cu:143-242 (distributions of the samplers).
#include <cstdlib>
#include <cstring>

#include <type_traits>

#include "chacha.cuh"
#include "kernels.h"
#include "modarith.cuh"
#include "ntt_common.cuh"

namespace he {

namespace {

constexpr int kThreads = 256;

// word `at` of a limb whose address all lanes share: a scalar address and a 32-bit distance per lane (the empty statement keeps the
// compiler from widening the distance outside a loop, which would cost a 64-bit addition per load)
__device__ __forceinline__ const uint64_t *lane_word(const uint64_t *limb, uint32_t at) {
    uint32_t bytes = at * 8u;
    asm("" : "+v"(bytes));
    return reinterpret_cast<const uint64_t *>(reinterpret_cast<const char *>(limb) + bytes);
}

__device__ __forceinline__ Words2 load_pair(const uint64_t *p) { return *reinterpret_cast<const Words2 *>(p); }

struct EwArgs {
    const uint64_t *a, *b, *c;
    uint64_t *out;
    const uint64_t *moduli, *barrett;
    LimbMap map;
    uint32_t log_n;
    int op;
};

// grid: (N / 256, limbs, polys)
__global__ __launch_bounds__(kThreads) void elementwise_kernel(EwArgs p) {
    const uint32_t limb = blockIdx.y;
    const uint32_t table = map_table(p.map, limb);
    const uint64_t q = p.moduli[table];
    const size_t idx = (((size_t)blockIdx.z * p.map.limbs + limb) << p.log_n) + blockIdx.x * kThreads + threadIdx.x;
    uint64_t r;
    switch (p.op) {
        case EW_ADD: r = add_mod(p.a[idx], p.b[idx], q); break;
        case EW_SUB: r = sub_mod(p.a[idx], p.b[idx], q); break;
        case EW_NEG: r = neg_mod(p.a[idx], q); break;
        case EW_MUL: r = mul_mod(p.a[idx], p.b[idx], q, p.barrett[2 * table], p.barrett[2 * table + 1]); break;
        default: {
            r = add_mod(mul_mod(p.a[idx], p.b[idx], q, p.barrett[2 * table], p.barrett[2 * table + 1]), p.c[idx], q);
            if (p.op == EW_MUL_ADD_NEG) r = neg_mod(r, q);
        }
    }
    p.out[idx] = r;
}

// grid: (N / 256, limbs): out = a + b * w[first + limb]
__global__ __launch_bounds__(kThreads) void scalar_mul_add_kernel(const uint64_t *a, const uint64_t *b, uint64_t *out,
                                                                  const uint64_t *moduli, const uint64_t *w,
                                                                  uint32_t first, uint32_t log_n) {
    const uint32_t table = first + blockIdx.y;
    const uint64_t q = moduli[table];
    const size_t idx = ((size_t)blockIdx.y << log_n) + blockIdx.x * kThreads + threadIdx.x;
    out[idx] = add_mod(a[idx], mul_shoup(b[idx], load_shoup(w, table), q), q);
}

// grid: (N / 256, limbs): residue of a rounded real coefficient
// blockIdx.z = item: coefficient vectors N apart, outputs out_item_stride words apart
__global__ __launch_bounds__(kThreads) void decompose_real_kernel(const double *coeffs, uint64_t *out,
                                                                  const uint64_t *moduli, const uint64_t *barrett,
                                                                  uint32_t first, uint32_t log_n, size_t out_item_stride) {
    const uint32_t table = first + blockIdx.y;
    const uint64_t q = moduli[table];
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    const double c = coeffs[((size_t)blockIdx.z << log_n) + i];
    const uint64_t r = barrett64((uint64_t)fabs(c), q, barrett[2 * table + 1]);
    out[blockIdx.z * out_item_stride + ((size_t)blockIdx.y << log_n) + i] = c < 0 ? neg_mod(r, q) : r;
}

struct TensorArgs {
    const uint64_t *ct1, *ct2;
    uint64_t *out;
    const uint64_t *moduli, *barrett;
    uint32_t L, log_n;
    uint64_t *out2;                           // d2 (out + 2 polynomials for a dense size-3 result)
    size_t in_item_stride, out_item_stride, out2_item_stride;   // blockIdx.z = item (words between items)
};

// grid: (N / 256, L).  Reads the four input limbs once, writes the three outputs: (d0, d1, d2) =
// (a0 b0, a0 b1 + a1 b0, a1 b1); out may alias ct1 (every index is read before it is written).
template <bool SQUARE>
__global__ __launch_bounds__(kThreads) void tensor_kernel(TensorArgs p) {
    const uint32_t limb = blockIdx.y;
    const uint64_t q = p.moduli[limb], r0 = p.barrett[2 * limb], r1 = p.barrett[2 * limb + 1];
    const size_t poly = (size_t)p.L << p.log_n;
    const size_t idx = ((size_t)limb << p.log_n) + blockIdx.x * kThreads + threadIdx.x;
    const uint64_t *ct1 = p.ct1 + blockIdx.z * p.in_item_stride, *ct2 = p.ct2 + blockIdx.z * p.in_item_stride;
    uint64_t *out = p.out + blockIdx.z * p.out_item_stride, *out2 = p.out2 + blockIdx.z * p.out2_item_stride;
    const uint64_t a0 = ct1[idx], a1 = ct1[idx + poly];
    uint64_t d0, d1, d2;
    if (SQUARE) {
        d0 = mul_mod(a0, a0, q, r0, r1);
        d2 = mul_mod(a1, a1, q, r0, r1);
        uint64_t m = mul_mod(a0, a1, q, r0, r1);
        d1 = add_mod(m, m, q);
    } else {
        const uint64_t b0 = ct2[idx], b1 = ct2[idx + poly];
        d0 = mul_mod(a0, b0, q, r0, r1);
        d2 = mul_mod(a1, b1, q, r0, r1);
        // Karatsuba: (a0 + a1)(b0 + b1) - d0 - d2; the sums stay below 2^62
        uint64_t m = mul_mod(a0 + a1, b0 + b1, q, r0, r1);
        d1 = sub_mod(sub_mod(m, d0, q), d2, q);
    }
    out[idx] = d0;
    out[idx + poly] = d1;
    out2[idx] = d2;
}

// The same in exact FP64 arithmetic (every prime below 2^50): about 60 instructions per coefficient instead of
// about 260, the same canonical residues.
template <bool SQUARE>
__global__ __launch_bounds__(kThreads) void tensor_fp_kernel(TensorArgs p, const double *fp_consts) {
    const uint32_t limb = blockIdx.y;
    const FpMod m{fp_consts[4 * limb], fp_consts[4 * limb + 1]};
    const size_t poly = (size_t)p.L << p.log_n;
    const size_t idx = ((size_t)limb << p.log_n) + blockIdx.x * kThreads + threadIdx.x;
    const uint64_t *ct1 = p.ct1 + blockIdx.z * p.in_item_stride, *ct2 = p.ct2 + blockIdx.z * p.in_item_stride;
    uint64_t *out = p.out + blockIdx.z * p.out_item_stride, *out2 = p.out2 + blockIdx.z * p.out2_item_stride;
    const double a0 = fp_from_u64(ct1[idx]), a1 = fp_from_u64(ct1[idx + poly]);
    double d0, d1, d2;
    if (SQUARE) {
        d0 = fp_canonical(fp_mulmod(a0, a0, m), m);
        d2 = fp_canonical(fp_mulmod(a1, a1, m), m);
        const double mm = fp_mulmod(a0, a1, m);
        d1 = fp_canonical(mm + mm, m);
    } else {
        const double b0 = fp_from_u64(ct2[idx]), b1 = fp_from_u64(ct2[idx + poly]);
        d0 = fp_canonical(fp_mulmod(a0, b0, m), m);
        d2 = fp_canonical(fp_mulmod(a1, b1, m), m);
        const double sb = b0 + b1;
        const double mm = fp_mulmod(a0 + a1, sb, m);
        d1 = fp_canonical(mm - d0 - d2, m);
    }
    out[idx] = fp_to_u64(d0);
    out[idx + poly] = fp_to_u64(d1);
    out2[idx] = fp_to_u64(d2);
}

// General tensor product: grid (N / 256, L); ct1 [S1][L][N], ct2 [S2][L][N] -> out [S1 + S2 - 1][L][N],
// out_j = sum over a + b = j of ct1_a * ct2_b with the products summed in 128 bits and reduced once (at most three
// products of 61-bit factors).  Sizes are template parameters: the operands stay in registers, nothing is allocated
// on the device.  out may be ct1's buffer: every coefficient is read before it is written.
template <int S1, int S2>
__global__ __launch_bounds__(kThreads) void tensor_mxn_kernel(TensorArgs p) {
    const uint32_t limb = blockIdx.y;
    const uint64_t q = p.moduli[limb], r0 = p.barrett[2 * limb], r1 = p.barrett[2 * limb + 1];
    const size_t poly = (size_t)p.L << p.log_n;
    const size_t idx = ((size_t)limb << p.log_n) + blockIdx.x * kThreads + threadIdx.x;
    uint64_t c1[S1], c2[S2], o[S1 + S2 - 1];
#pragma unroll
    for (int a = 0; a < S1; a++) c1[a] = p.ct1[idx + poly * a];
#pragma unroll
    for (int b = 0; b < S2; b++) c2[b] = p.ct2[idx + poly * b];
#pragma unroll
    for (int j = 0; j < S1 + S2 - 1; j++) {
        U128 acc{0, 0};
#pragma unroll
        for (int a = 0; a < S1; a++)
            if (j - a >= 0 && j - a < S2) mac128(acc, c1[a], c2[j - a]);
        o[j] = barrett128(acc.lo, acc.hi, q, r0, r1);
    }
#pragma unroll
    for (int j = 0; j < S1 + S2 - 1; j++) p.out[idx + poly * j] = o[j];
}

// The same product for operands of any size (run-time sizes, up to 16 polynomials each): nothing is kept in registers,
// the operands are read where they are needed (a coefficient's S1 + S2 words stay in the first-level cache), at most
// 16 products of 61-bit factors are summed in 128 bits per output.  Outputs are formed from the last to the first, so
// that out may be ct1's buffer: output j overwrites word j of ct1, which only the outputs from j on read.
__global__ __launch_bounds__(kThreads) void tensor_any_kernel(TensorArgs p, uint32_t s1, uint32_t s2) {
    const uint32_t limb = blockIdx.y;
    const uint64_t q = p.moduli[limb], r0 = p.barrett[2 * limb], r1 = p.barrett[2 * limb + 1];
    const size_t poly = (size_t)p.L << p.log_n;
    const size_t idx = ((size_t)limb << p.log_n) + blockIdx.x * kThreads + threadIdx.x;
    for (uint32_t j = s1 + s2 - 1; j-- > 0;) {
        const uint32_t a_first = j >= s2 ? j - (s2 - 1) : 0, a_last = j < s1 ? j : s1 - 1;
        U128 acc{0, 0};
        for (uint32_t a = a_first; a <= a_last; a++) mac128(acc, p.ct1[idx + poly * a], p.ct2[idx + poly * (j - a)]);
        p.out[idx + poly * j] = barrett128(acc.lo, acc.hi, q, r0, r1);
    }
}

// grid: (N / 256, limbs, items).  out[item][limb] = c0 + c1 * s (+ noise[item][limb]) for the ciphertext cts[item]
__global__ __launch_bounds__(kThreads) void decrypt_gather_kernel(const uint64_t *const *cts, const uint64_t *sk,
                                                                  const uint64_t *noise, uint64_t *out,
                                                                  const uint64_t *moduli, const uint64_t *barrett,
                                                                  uint32_t limbs, uint32_t log_n) {
    const uint32_t limb = blockIdx.y;
    const uint64_t q = moduli[limb], r0 = barrett[2 * limb], r1 = barrett[2 * limb + 1];
    const size_t idx = ((size_t)limb << log_n) + blockIdx.x * kThreads + threadIdx.x;
    const size_t poly = (size_t)limbs << log_n;
    const uint64_t *ct = cts[blockIdx.z];
    uint64_t v = add_mod(ct[idx], mul_mod(ct[idx + poly], sk[idx], q, r0, r1), q);
    const size_t o = (size_t)blockIdx.z * poly + idx;
    if (noise) v = add_mod(v, noise[o], q);
    out[o] = v;
}

// Sums of ciphertexts and of products of ciphertexts, each of `count` terms: what a row of a distance matrix or a masked sum of
// updates is.  A call per term read and wrote the running sum each time (3 us of launch and latency a term at N = 2^16, two or
// three limbs: 90 terms of ten row sums 290 us, 20 of two masked sums 110 us); here every term is read once, by all sums together.
struct SumArgs {
    const uint64_t *const *cts;   // device array [items][count], or [items][count][2] for products
    uint64_t *out;
    const uint64_t *moduli, *barrett;
    uint32_t limbs, log_n, polys, count;
};

typedef const uint64_t *const __attribute__((address_space(4))) *ScalarPtr;
__device__ __forceinline__ ScalarPtr scalar(const uint64_t *const *p) { return (ScalarPtr)(uintptr_t)p; }

// grid: (N / 512, limbs, items * polys), two words per thread
__global__ __launch_bounds__(kThreads) void sum_kernel(SumArgs p) {
    const uint32_t limb = blockIdx.y, item = blockIdx.z / p.polys, poly = blockIdx.z - item * p.polys;
    const size_t at = ((size_t)(poly * p.limbs + limb) << p.log_n) + 2 * (blockIdx.x * kThreads + threadIdx.x);
    const uint64_t q = scalar(p.moduli)[limb];
    const ScalarPtr ct = scalar(p.cts) + (size_t)item * p.count;
    Words2 acc = load_pair(ct[0] + at);
#pragma unroll 4
    for (uint32_t k = 1; k < p.count; k++) {
        const Words2 w = load_pair(ct[k] + at);
        acc.x = add_mod(acc.x, w.x, q);
        acc.y = add_mod(acc.y, w.y, q);
    }
    *reinterpret_cast<Words2 *>(p.out + (((size_t)item * p.polys * p.limbs) << p.log_n) + at) = acc;
}

// grid: (N / 512, limbs, items): (d0, d1, d2) = sum of (a0 b0, a0 b1 + a1 b0, a1 b1), residues below 2^61: the 128-bit sums
// take 16 terms (32 products below 2^122 in d1) before they are reduced
__global__ __launch_bounds__(kThreads) void multiply_sum_kernel(SumArgs p) {
    const uint32_t limb = blockIdx.y;
    const uint64_t q = scalar(p.moduli)[limb], r0 = scalar(p.barrett)[2 * limb], r1 = scalar(p.barrett)[2 * limb + 1];
    const size_t poly = (size_t)p.limbs << p.log_n, at = ((size_t)limb << p.log_n) + 2 * (blockIdx.x * kThreads + threadIdx.x);
    const ScalarPtr pair = scalar(p.cts) + (size_t)blockIdx.z * p.count * 2;
    U128 s[3][2];
#pragma unroll
    for (int i = 0; i < 3; i++) s[i][0] = s[i][1] = U128{0, 0};
    for (uint32_t k = 0; k < p.count; k++) {
        const uint64_t *a = pair[2 * k] + at, *b = pair[2 * k + 1] + at;
        const Words2 a0 = load_pair(a), a1 = load_pair(a + poly), b0 = load_pair(b), b1 = load_pair(b + poly);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            mac128(s[0][j], a0[j], b0[j]);
            mac128(s[1][j], a0[j], b1[j]);
            mac128(s[1][j], a1[j], b0[j]);
            mac128(s[2][j], a1[j], b1[j]);
        }
        if (k % 16 == 15) {
#pragma unroll
            for (int i = 0; i < 3; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) s[i][j] = U128{barrett128(s[i][j].lo, s[i][j].hi, q, r0, r1), 0};
        }
    }
    uint64_t *out = p.out + (size_t)blockIdx.z * 3 * poly + at;
#pragma unroll
    for (int i = 0; i < 3; i++)
        *reinterpret_cast<Words2 *>(out + i * poly) = Words2{barrett128(s[i][0].lo, s[i][0].hi, q, r0, r1),
                                                             barrett128(s[i][1].lo, s[i][1].hi, q, r0, r1)};
}

// Squared distances for Krum, as size-3 ciphertexts (lazy relinearisation) whose third polynomial, the key switch's input, has a
// buffer of its own, so that (d0, d1) is a dense batch of size-2 ciphertexts.
// Two distances can share a ciphertext: the squared differences of real messages have real slots, and X^(N/2) multiplies every slot by
// i, so that out = first + X^(N/2) second carries one sum in the real and one in the imaginary parts through relinearisation,
// rescale and slot sum (all of them linear and compatible with i), at half the work per distance.
struct SquareSumArgs {
    const uint64_t *const *table;   // device table of ciphertexts [2][L][N]
    uint64_t *sums;                 // row_square_kernel: what client_sums_kernel has left
    uint64_t *out01, *out2;         // [items][2][L][N] (d0, d1) and [items][L][N] (d2)
    const uint64_t *moduli, *barrett, *psi;
    uint32_t L, log_n, count, parts;
};

// W neighbouring words of a thread
template <int W>
__device__ __forceinline__ void load_words(uint64_t (&v)[W], const uint64_t *p) {
    static_assert(W == 1 || W == 2, "8 or 16 bytes");
    if constexpr (W == 1) {
        v[0] = *p;
    } else {
        const Words2 w = load_pair(p);
        v[0] = w.x;
        v[1] = w.y;
    }
}

template <int W>
__device__ __forceinline__ void store_words(uint64_t *p, const uint64_t (&v)[W]) {
    if constexpr (W == 1)
        *p = v[0];
    else
        *reinterpret_cast<Words2 *>(p) = Words2{v[0], v[1]};
}

// sums of products below 2^122, W words a thread: 64 of them fit into 128 bits
template <int W>
struct SquareSums {
    U128 s[3][W];
    uint64_t q, r0, r1;
    __device__ __forceinline__ SquareSums(const SquareSumArgs &p, uint32_t limb)
        : q(scalar(p.moduli)[limb]), r0(scalar(p.barrett)[2 * limb]), r1(scalar(p.barrett)[2 * limb + 1]) {
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < W; j++) s[i][j] = U128{0, 0};
    }
    __device__ __forceinline__ uint64_t reduced(int i, int j) const { return barrett128(s[i][j].lo, s[i][j].hi, q, r0, r1); }
    // after term k, the number of products a term adds to one sum being at most two
    __device__ __forceinline__ void relieve(uint32_t k) {
        if (k % 16 != 15) return;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < W; j++) s[i][j] = U128{reduced(i, j), 0};
    }
    // the first part's sums
    __device__ __forceinline__ void real_part(uint64_t (&d)[3][W]) const {
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < W; j++) d[i][j] = reduced(i, j);
    }
    // d gains the second part's times X^(N/2): w = psi^(N/2) at the words of the NTT order's first half, its negative at those of the
    // second
    __device__ __forceinline__ void add_imaginary_part(uint64_t (&d)[3][W], Shoup w, bool upper) const {
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < W; j++) {
                const uint64_t v = mul_shoup(reduced(i, j), w, q);
                d[i][j] = add_mod(d[i][j], upper ? neg_mod(v, q) : v, q);
            }
    }
};

// psi^(N/2), which X^(N/2) is at half of the words
__device__ __forceinline__ Shoup half_root(const SquareSumArgs &p, uint32_t limb) { return scalar_shoup(p.psi, ((size_t)limb << p.log_n) + 1); }

template <int W>
__device__ __forceinline__ void store_squares(const SquareSumArgs &p, uint32_t item, size_t at, const uint64_t (&d)[3][W]) {
    const size_t poly = (size_t)p.L << p.log_n;
    uint64_t *out = p.out01 + (size_t)item * 2 * poly + at;
    store_words(out, d[0]);
    store_words(out + poly, d[1]);
    store_words(p.out2 + (size_t)item * poly + at, d[2]);
}

// grid: (N / (256 W), L, items).  Item = sum of (a - b)^2 over the `count` pairs of its row of the table [items][PARTS][count][2], plus
// X^(N/2) times that over its second part's (null: no second part): the subtraction, the tensor square and the accumulation in one
// pass over the inputs.
// What bounds it: integer multiplies, about 1000 instructions a thread, and close behind them its traffic (45 pairs of two chunks, three
// limbs of 2^16 words, two pairs an item: 81 us for 407 MB, 5.0 TB/s; one reduction per sum and half the outputs buy what the reductions
// of X^(N/2) cost: 90 us with a reduction per term and a pair an item.  An order of workgroups in which the items that share a ciphertext
// meet on one XCD: the same).
template <int PARTS, int W>
__global__ __launch_bounds__(kThreads) void pair_square_sum_kernel(SquareSumArgs p) {
    const uint32_t limb = blockIdx.y, word = W * (blockIdx.x * kThreads + threadIdx.x), item = blockIdx.z;
    const size_t poly = (size_t)p.L << p.log_n, at = ((size_t)limb << p.log_n) + word;
    uint64_t d[3][W];
    for (int part = 0; part < PARTS; part++) {
        const ScalarPtr pair = scalar(p.table) + ((size_t)item * PARTS + part) * p.count * 2;
        if (part && !pair[0]) break;
        SquareSums<W> sums(p, limb);
        const uint64_t q = sums.q;
#pragma unroll 2
        for (uint32_t k = 0; k < p.count; k++) {
            const uint64_t *a = pair[2 * k] + at, *b = pair[2 * k + 1] + at;
            uint64_t a0[W], a1[W], b0[W], b1[W];
            load_words(a0, a);
            load_words(a1, a + poly);
            load_words(b0, b);
            load_words(b1, b + poly);
#pragma unroll
            for (int j = 0; j < W; j++) {
                const uint64_t x0 = sub_mod(a0[j], b0[j], q), x1 = sub_mod(a1[j], b1[j], q);
                mac128(sums.s[0][j], x0, x0);
                mac128(sums.s[1][j], x0, add_mod(x1, x1, q));
                mac128(sums.s[2][j], x1, x1);
            }
            sums.relieve(k);
        }
        if (part == 0)
            sums.real_part(d);
        else
            sums.add_imaginary_part(d, half_root(p, limb), word >> (p.log_n - 1));
    }
    store_squares(p, item, at, d);
}

// The sum of a client's squared distances to all others, sum_j (x_i - x_j)^2 = x_i (n x_i - 2 S) + T with S = sum x_j and
// T = sum x_j^2, word for word the same modulo q and n products instead of n (n - 1): client_sums_kernel leaves S of every chunk
// [chunks][2][L][N] and T [3][L][N] (over all chunks), row_square_kernel forms two clients' sums per item.
// 10 clients of two chunks: 22 + 37 us.
// table [clients][chunks], count = clients, parts = chunks.  grid: (N / 512, L)
__global__ __launch_bounds__(kThreads) void client_sums_kernel(SquareSumArgs p) {
    const uint32_t limb = blockIdx.y;
    const size_t poly = (size_t)p.L << p.log_n, at = ((size_t)limb << p.log_n) + 2 * (blockIdx.x * kThreads + threadIdx.x);
    SquareSums<2> squares(p, limb);
    const uint64_t q = squares.q;
    for (uint32_t c = 0, term = 0; c < p.parts; c++) {
        Words2 s0{0, 0}, s1{0, 0};
#pragma unroll 4
        for (uint32_t k = 0; k < p.count; k++, term++) {
            const uint64_t *ct = scalar(p.table)[(size_t)k * p.parts + c] + at;
            const Words2 x0 = load_pair(ct), x1 = load_pair(ct + poly);
            s0 = Words2{add_mod(s0.x, x0.x, q), add_mod(s0.y, x0.y, q)};
            s1 = Words2{add_mod(s1.x, x1.x, q), add_mod(s1.y, x1.y, q)};
#pragma unroll
            for (int j = 0; j < 2; j++) {
                mac128(squares.s[0][j], x0[j], x0[j]);
                mac128(squares.s[1][j], x0[j], add_mod(x1[j], x1[j], q));
                mac128(squares.s[2][j], x1[j], x1[j]);
            }
            squares.relieve(term);
        }
        uint64_t *out = p.sums + (size_t)c * 2 * poly + at;
        *reinterpret_cast<Words2 *>(out) = s0;
        *reinterpret_cast<Words2 *>(out + poly) = s1;
    }
#pragma unroll
    for (int i = 0; i < 3; i++)
        *reinterpret_cast<Words2 *>(p.sums + ((size_t)2 * p.parts + i) * poly + at) = Words2{squares.reduced(i, 0), squares.reduced(i, 1)};
}

// grid: (N / 512, L, items): item k holds client 2 k, and client 2 k + 1 (if there is one) times X^(N/2)
__global__ __launch_bounds__(kThreads) void row_square_kernel(SquareSumArgs p) {
    const uint32_t limb = blockIdx.y, j2 = 2 * (blockIdx.x * kThreads + threadIdx.x), item = blockIdx.z;
    const size_t poly = (size_t)p.L << p.log_n, at = ((size_t)limb << p.log_n) + j2;
    uint64_t d[3][2];
    for (uint32_t part = 0; part < 2; part++) {
        const uint32_t client = 2 * item + part;
        if (client >= p.count) break;
        SquareSums<2> sums(p, limb);
        const uint64_t q = sums.q;
        for (int i = 0; i < 3; i++) {
            const Words2 t = load_pair(p.sums + ((size_t)2 * p.parts + i) * poly + at);
            sums.s[i][0] = U128{t.x, 0};
            sums.s[i][1] = U128{t.y, 0};
        }
#pragma unroll 2
        for (uint32_t c = 0; c < p.parts; c++) {
            const uint64_t *ct = scalar(p.table)[(size_t)client * p.parts + c] + at, *s = p.sums + (size_t)c * 2 * poly + at;
            const Words2 x0 = load_pair(ct), x1 = load_pair(ct + poly), s0 = load_pair(s), s1 = load_pair(s + poly);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                // n x - 2 S
                auto spread = [&](uint64_t x, uint64_t sum) {
                    const uint64_t nx = mul_mod(x, p.count, q, sums.r0, sums.r1);
                    return sub_mod(sub_mod(nx, sum, q), sum, q);
                };
                const uint64_t y0 = spread(x0[j], s0[j]), y1 = spread(x1[j], s1[j]);
                mac128(sums.s[0][j], x0[j], y0);
                mac128(sums.s[1][j], x0[j], y1);
                mac128(sums.s[1][j], x1[j], y0);
                mac128(sums.s[2][j], x1[j], y1);
            }
            sums.relieve(c);
        }
        if (part == 0)
            sums.real_part(d);
        else
            sums.add_imaginary_part(d, half_root(p, limb), j2 >> (p.log_n - 1));
    }
    store_squares(p, item, at, d);
}

// grid: (N / 256, total limbs)
__global__ __launch_bounds__(kThreads) void galois_kernel(const uint64_t *in, uint64_t *out, uint32_t elt,
                                                          uint32_t log_n) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    const size_t base = (size_t)blockIdx.y << log_n;
    out[base + i] = in[base + galois_index(i, elt, log_n)];
}

// Base conversion of one digit: thread = one coefficient x kRows output limbs.
constexpr int kRows = 4;

struct BconvKArgs {
    BconvArgs a;
    const uint64_t *moduli, *barrett;
    uint32_t log_n;
};

template <int NIN>
__global__ __launch_bounds__(kThreads) void bconv_kernel(BconvKArgs p) {
    const size_t j = (size_t)blockIdx.x * kThreads + threadIdx.x;
    const uint32_t n_in = NIN > 0 ? NIN : p.a.n_in;
    uint64_t x[NIN > 0 ? NIN : 1];
    if (NIN > 0) {
#pragma unroll
        for (int i = 0; i < NIN; i++) x[i] = p.a.x[((size_t)i << p.log_n) + j];
    }
    for (uint32_t rr = 0; rr < kRows; rr++) {
        const uint32_t row = blockIdx.y * kRows + rr;
        if (row >= p.a.n_out) return;
        const uint64_t *m = p.a.mat + (size_t)row * n_in;
        U128 acc{0, 0};
        if (NIN > 0) {
#pragma unroll
            for (int i = 0; i < NIN; i++) mac128(acc, x[i], m[i]);
        } else {
            for (uint32_t i = 0; i < n_in; i++) mac128(acc, p.a.x[((size_t)i << p.log_n) + j], m[i]);
        }
        const uint32_t t = p.a.out_table[row];
        p.a.out[((size_t)p.a.out_limb[row] << p.log_n) + j] =
            barrett128(acc.lo, acc.hi, p.moduli[t], p.barrett[2 * t], p.barrett[2 * t + 1]);
    }
}

// output limbs per thread in the batched base conversion: the inputs are re-read once per row group

constexpr int kBatchIn = 8;

struct BconvBatchK {
    BconvBatch b;
    const uint64_t *moduli, *barrett;
    uint32_t log_n, compute_groups, rows_per;
};

// grid: (N / 256, compute groups + copy groups, units); thread = one coefficient x kBatchRows output limbs
__global__ __launch_bounds__(kThreads) void bconv_batched_kernel(BconvBatchK p) {
    const uint32_t item = blockIdx.z / p.b.n_units;
    const BconvDesc d = p.b.descs[blockIdx.z - item * p.b.n_units];
    const size_t j = (size_t)blockIdx.x * kThreads + threadIdx.x;
    uint64_t *out = p.b.out_base + item * p.b.out_item_stride + d.out_off;
    if (blockIdx.y >= p.compute_groups) {
        // limbs that pass through unchanged
        const uint64_t *from = p.b.copy_base + item * p.b.copy_item_stride;
        const uint32_t first = (blockIdx.y - p.compute_groups) * p.rows_per;
        for (uint32_t r = first; r < first + p.rows_per && r < d.copy_count; r++) {
            const size_t idx = ((size_t)(d.copy_first + r) << p.log_n) + j;
            out[idx] = from[idx];
        }
        return;
    }
    const uint32_t row0 = blockIdx.y * p.rows_per;
    if (row0 >= d.n_out) return;
    const uint64_t *x = p.b.x_base + item * p.b.x_item_stride + d.x_off;
    uint64_t xv[kBatchIn];
#pragma unroll
    for (int i = 0; i < kBatchIn; i++) xv[i] = (uint32_t)i < d.n_in ? x[((size_t)i << p.log_n) + j] : 0;
    const uint64_t *mat = p.b.mat_base + d.mat_off;
    for (uint32_t row = row0; row < row0 + p.rows_per && row < d.n_out; row++) {
        const uint64_t *m = mat + (size_t)row * d.n_in;
        const uint32_t t = p.b.out_table[d.map_off + row];
        uint64_t r;
        if (d.n_in == 1 && m[0] == 1) {
            // a digit of one limb (one special prime): Q_d / q_i = 1, the conversion is a plain reduction
            r = barrett64(xv[0], p.moduli[t], p.barrett[2 * t + 1]);
        } else {
            U128 acc{0, 0};
#pragma unroll
            for (int i = 0; i < kBatchIn; i++)
                if ((uint32_t)i < d.n_in) mac128(acc, xv[i], m[i]);
            r = barrett128(acc.lo, acc.hi, p.moduli[t], p.barrett[2 * t], p.barrett[2 * t + 1]);
        }
        out[((size_t)p.b.out_limb[d.map_off + row] << p.log_n) + j] = r;
    }
}

// FP64 variant: every product is reduced on the fly to |r| <= 0.875 m (fp_mulmod, words below 2^50), so the sum of up to 8 terms stays
// an exact integer of at most 7 m < 2^53; one canonicalisation per output.
__global__ __launch_bounds__(kThreads) void bconv_batched_fp_kernel(BconvBatchK p) {
    const uint32_t item = blockIdx.z / p.b.n_units;
    const BconvDesc d = p.b.descs[blockIdx.z - item * p.b.n_units];
    const size_t j = (size_t)blockIdx.x * kThreads + threadIdx.x;
    uint64_t *out = p.b.out_base + item * p.b.out_item_stride + d.out_off;
    if (blockIdx.y >= p.compute_groups) {
        const uint64_t *from = p.b.copy_base + item * p.b.copy_item_stride;
        const uint32_t first = (blockIdx.y - p.compute_groups) * p.rows_per;
        for (uint32_t r = first; r < first + p.rows_per && r < d.copy_count; r++) {
            const size_t idx = ((size_t)(d.copy_first + r) << p.log_n) + j;
            out[idx] = from[idx];
        }
        return;
    }
    const uint32_t row0 = blockIdx.y * p.rows_per;
    if (row0 >= d.n_out) return;
    const uint64_t *x = p.b.x_base + item * p.b.x_item_stride + d.x_off;
    double xv[kBatchIn];
#pragma unroll
    for (int i = 0; i < kBatchIn; i++) xv[i] = (uint32_t)i < d.n_in ? fp_from_u64(x[((size_t)i << p.log_n) + j]) : 0.0;
    const double *mat = p.b.mat_fp + d.mat_off;
    for (uint32_t row = row0; row < row0 + p.rows_per && row < d.n_out; row++) {
        const double *m = mat + (size_t)row * d.n_in;
        const uint32_t t = p.b.out_table[d.map_off + row];
        const FpMod mod{p.b.fp_consts[4 * t], p.b.fp_consts[4 * t + 1]};
        double acc = 0.0;
#pragma unroll
        for (int i = 0; i < kBatchIn; i++)
            if ((uint32_t)i < d.n_in) acc += fp_mulmod(xv[i], m[i], mod);
        out[((size_t)p.b.out_limb[d.map_off + row] << p.log_n) + j] = fp_to_u64(fp_canonical(acc, mod));
    }
}

struct InnerArgs {
    const uint64_t *y;
    uint64_t *out;
    const uint64_t *moduli, *barrett;
    EvkPtrs evk;
    uint32_t L, K, size_q, beta, log_n, galois_elt;
    int accumulate;
    const uint64_t *fold_ct, *fold_w;
    size_t y_item_stride, out_item_stride, fold_item_stride;   // blockIdx.z = item (words between items)
    const uint64_t *add_c0, *p_mod_q;
    uint32_t add_elt;
    const uint64_t *own;            // optional: the key-switch input [L][N]; a digit's own limbs are read from it (their
    size_t own_item_stride;         // slots in y were left unwritten), items own_item_stride words apart
    uint32_t own_elt;               // != 0: the key-switch input is sigma(own), gathered here (X -> X^own_elt)
};

// grid: (N / 256, L + K, items).  Streams beta digit limbs of y and 2 beta key limbs, writes (or accumulates) the
// two output limbs.  The products are summed in 128 bits and reduced once (beta <= 64 products of
// 61-bit factors cannot overflow).
__global__ __launch_bounds__(kThreads) void inner_product_kernel(InnerArgs p) {
    const uint32_t t = blockIdx.y;
    const uint32_t LK = p.L + p.K;
    const uint32_t table = t < p.L ? t : p.size_q + (t - p.L);
    const uint32_t j = blockIdx.x * kThreads + threadIdx.x;
    const uint32_t src = p.galois_elt ? galois_index(j, p.galois_elt, p.log_n) : j;
    const size_t key_off = ((size_t)table << p.log_n) + j;
    const size_t key_poly = (size_t)(p.size_q + p.K) << p.log_n;
    // (the argument struct stays untouched: a modified copy would move its pointer table to scratch memory)
    const uint64_t *y = p.y + blockIdx.z * p.y_item_stride;
    uint64_t *out = p.out + blockIdx.z * p.out_item_stride;
    const uint64_t *own = p.own ? p.own + blockIdx.z * p.own_item_stride + ((size_t)t << p.log_n) : nullptr;
    const uint32_t own_d = (own && t < p.L) ? t / p.K : 0xffffffffu;
    const uint32_t own_src = p.own_elt ? galois_index(j, p.own_elt, p.log_n) : src;
    U128 a0{0, 0}, a1{0, 0};
    for (uint32_t d = 0; d < p.beta; d++) {
        const uint64_t v = d == own_d ? own[own_src] : y[(((size_t)d * LK + t) << p.log_n) + src];
        const uint64_t *k = p.evk.p[d];
        mac128(a0, v, k[key_off]);
        mac128(a1, v, k[key_off + key_poly]);
    }
    const uint64_t q = p.moduli[table], r0 = p.barrett[2 * table], r1 = p.barrett[2 * table + 1];
    uint64_t o0 = barrett128(a0.lo, a0.hi, q, r0, r1);
    uint64_t o1 = barrett128(a1.lo, a1.hi, q, r0, r1);
    const size_t o = ((size_t)t << p.log_n) + j;
    const size_t opoly = (size_t)LK << p.log_n;
    if (p.accumulate) {
        o0 = add_mod(o0, out[o], q);
        o1 = add_mod(o1, out[o + opoly], q);
    }
    if (p.add_c0 && t < p.L) {
        // a rotation: polynomial 0 gains P sigma(c0), which ModDown's division by P turns into sigma(c0)
        const uint32_t g = p.add_elt ? galois_index(j, p.add_elt, p.log_n) : j;
        o0 = add_mod(o0, mul_shoup(p.add_c0[((size_t)t << p.log_n) + g], load_shoup(p.p_mod_q, t), q), q);
    }
    if (p.fold_ct && t == p.L - 1) {
        const Shoup w = load_shoup(p.fold_w, 0);
        const size_t cpoly = (size_t)p.L << p.log_n;
        const uint64_t *fold = p.fold_ct + blockIdx.z * p.fold_item_stride;
        o0 = add_mod(mul_shoup(o0, w, q), fold[o], q);
        o1 = add_mod(mul_shoup(o1, w, q), fold[o + cpoly], q);
    }
    out[o] = o0;
    out[o + opoly] = o1;
}

struct HoistArgs {
    const uint64_t *y, *c0;
    uint64_t *out, *c0_out;
    const uint64_t *moduli, *barrett;
    EvkPtrs evk;                    // [step * beta + digit]
    uint32_t elts[kMaxDigits];      // Galois element of every step
    uint32_t n_steps, L, K, size_q, beta, log_n;
    int accumulate, with_self;
    uint32_t items;
    size_t ct_item_stride;          // words between the ciphertexts of consecutive items (blockIdx.z), in and out
    const double *fp_consts;        // [tables][4] of the FP64 back end
    uint64_t fp_mask;               // bit t: the products of table t (a prime below 2^50) are formed in FP64
    int own_from_ct;                // a digit's own limbs are read from c1 of the input (c0 + L limbs), not from y
    uint32_t rows, groups;          // grid: N / 256 blocks x rows x groups of items, as one dimension
    int xcd_map;                    // workgroup order that keeps the sharers of a key block on one XCD
};

// The two words that an automorphism brings to coefficients j and j + 1 (j even), src its gather index of j: odd elements
// keep aligned pairs of the NTT order together, so they are one 16-byte access, in their order or turned round.
__device__ __forceinline__ void turned(uint64_t *v, Words2 w, uint32_t src) {
    v[0] = src & 1 ? w.y : w.x;
    v[1] = src & 1 ? w.x : w.y;
}

// Hoisted rotations in one launch: grid (N / 256, (L + K) + L [+ L], ceil(items / I)); a thread serves the same
// coefficient of I consecutive items, so that a key word is loaded once for all of them.
// rows t < L + K:  out[p][t] = sum_s sum_d sigma_s(y_d)[t] * evk_{s,d}[p][t]  (n_steps * beta <= 64 products, summed
//                  lazily as partial products of factors split at bit 30, see Sum3, and reduced once); the automorphism is the
//                  gather index of the load of y.  The kernel is bound by instruction issue (its multiply-adds).
// rows L + K + t:  c0_out[t] = sum_s sigma_s(c0)[t]  (+ c0[t] with_self)
// rows L + K + L + t (with_self only): c1 is copied to the output, so that the ModDown that follows adds onto
//                  the input ciphertext: ct_out = ct_in + sum_s rot_s(ct_in)
// LOCAL: every step's Galois element is 1 modulo 2^(log_n - 7) (steps that are multiples of N / 512), so the
// automorphism permutes inside each aligned block of 256 NTT-order words: a workgroup stages its block of every item
// and digit in LDS once (I * beta <= kHoistLocalTiles) and gathers from there, instead of one global gather per step.
// 45 ciphertexts of [60, 40 | 60] bits at N = 2^16, 15 steps: 331 -> 255 us block-local (three multiply-adds per
// product instead of four, no register moves between terms, c0 from LDS, four waves per SIMD), 7 and 15 steps with gathers from memory 334 -> 320 us on average (four ciphertexts per thread there too).
constexpr int kHoistLocalTiles = 16;
template <int I, bool LOCAL>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void hoist_inner_kernel(HoistArgs p) {
    __shared__ uint64_t ybuf[LOCAL ? kHoistLocalTiles * kThreads : 1];
    const uint32_t LK = p.L + p.K;
    // Workgroup -> (block of 256 coefficients bx, row by, group of items bz).  The workgroups that share key words
    // (same block and row, every group) get linear ids 8 apart and consecutive in that sequence: the hardware deals
    // consecutive ids round-robin to the 8 XCDs, so they run on one XCD at about the same time and all but the first
    // find the keys in that XCD's L2 (p.xcd_map; otherwise the plain order).
    uint32_t bx, by, bz;
    {
        const uint32_t nb = (1u << p.log_n) / kThreads, id = blockIdx.x;
        if (p.xcd_map) {
            // xcd_map 2 (gathers from memory, N >= 2^15): an XCD also takes the 16 blocks of an aligned 4,096-word
            // stretch of one row one after the other, so that the words which the steps' gathers bring into its L2 (a
            // step of 8 k permutes inside such stretches) are found there by the neighbouring workgroups; the stretches
            // of every row are dealt to the XCDs in turn, heavy rows first everywhere
            const uint32_t s = id >> 3;
            uint32_t pair = (s / p.groups) * 8 + (id & 7);
            if (p.xcd_map == 2) {
                const uint32_t q = s / p.groups, u = (q >> 4) * 8 + (id & 7), stretches = nb >> 4;
                pair = (u / stretches) * nb + (u % stretches) * 16 + (q & 15);
            }
            bz = s % p.groups;
            bx = pair % nb;
            by = pair / nb;
        } else {
            bx = id % nb;
            by = (id / nb) % p.rows;
            bz = id / (nb * p.rows);
        }
    }
    const uint32_t j = bx * kThreads + threadIdx.x;
    const uint32_t item0 = bz * I;
    const uint32_t count = p.items - item0 < (uint32_t)I ? p.items - item0 : (uint32_t)I;
    // (the argument struct stays untouched: a modified copy would move its tables to scratch memory)
    if (by >= LK) {
        const size_t o = ((size_t)(by - LK) << p.log_n) + j;
        if (by >= LK + p.L) {
            if (!p.accumulate)
                for (uint32_t it = 0; it < count; it++)
                    p.c0_out[(item0 + it) * p.ct_item_stride + o] = p.c0[(item0 + it) * p.ct_item_stride + o];
            return;
        }
        const uint32_t t = by - LK;
        const uint64_t q = p.moduli[t];
        const uint64_t *in = p.c0 + item0 * p.ct_item_stride + ((size_t)t << p.log_n);
        uint64_t *c0_out = p.c0_out + item0 * p.ct_item_stride + ((size_t)t << p.log_n);
        if constexpr (LOCAL) {
            // every step permutes the block's words: they come from LDS, one index per step for all items
            uint64_t acc[I];
#pragma unroll
            for (int it = 0; it < I; it++) {
                const uint64_t w = in[((uint32_t)it < count ? it : count - 1) * p.ct_item_stride + j];
                ybuf[it * kThreads + threadIdx.x] = w;
                acc[it] = p.accumulate ? c0_out[((uint32_t)it < count ? it : count - 1) * p.ct_item_stride + j] : p.with_self ? w : 0;
            }
            __syncthreads();
#pragma unroll 4
            for (uint32_t s = 0; s < p.n_steps; s++) {
                const uint32_t g = galois_index(j, p.elts[s], p.log_n) & (kThreads - 1);
#pragma unroll
                for (int it = 0; it < I; it++) acc[it] = add_mod(acc[it], ybuf[it * kThreads + g], q);
            }
#pragma unroll
            for (int it = 0; it < I; it++)
                if ((uint32_t)it < count) c0_out[it * p.ct_item_stride + j] = acc[it];
        } else {
            // two neighbouring words per thread (see turned) of half the items; the gathers of a step are independent of the running
            // sums, several steps' are in flight
            constexpr int H = (I + 1) / 2;
            const uint32_t half = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / (kThreads / 2)) * H;
            const uint32_t j2 = bx * kThreads + 2 * (threadIdx.x % (kThreads / 2));
            const uint64_t *src[H];
            Words2 acc[H];
#pragma unroll
            for (int it = 0; it < H; it++) {
                const size_t at = (half + it < count ? half + it : count - 1) * p.ct_item_stride;
                src[it] = in + at;
                acc[it] = p.accumulate ? load_pair(c0_out + at + j2) : p.with_self ? load_pair(in + at + j2) : Words2{0, 0};
            }
#pragma unroll 4
            for (uint32_t s = 0; s < p.n_steps; s++) {
                const uint32_t g = galois_index(j2, p.elts[s], p.log_n);
#pragma unroll
                for (int it = 0; it < H; it++) {
                    uint64_t v[2];
                    turned(v, load_pair(lane_word(src[it], g & ~1u)), g);
                    acc[it].x = add_mod(acc[it].x, v[0], q);
                    acc[it].y = add_mod(acc[it].y, v[1], q);
                }
            }
#pragma unroll
            for (int it = 0; it < H; it++)
                if (half + it < count) *reinterpret_cast<Words2 *>(c0_out + (half + it) * p.ct_item_stride + j2) = acc[it];
        }
        return;
    }
    const uint32_t t = by;
    const size_t y_item = (size_t)p.beta * LK << p.log_n;
    const uint64_t *y = p.y + item0 * y_item + ((size_t)t << p.log_n);
    const uint32_t table = t < p.L ? t : p.size_q + (t - p.L);
    const size_t key_row = (size_t)table << p.log_n;
    const size_t key_poly = (size_t)(p.size_q + p.K) << p.log_n;
    const size_t digit = (size_t)LK << p.log_n;
    // the digit that owns limb t: its "lifted" limb is the input's c1 itself
    const uint32_t own = (p.own_from_ct && t < p.L) ? t / p.K : 0xffffffffu;
    const uint64_t *c1 = p.c0 + item0 * p.ct_item_stride + ((size_t)(p.L + t) << p.log_n);
    const uint32_t n_terms = p.n_steps * p.beta;
    if (LOCAL) {
        for (uint32_t d = 0; d < p.beta; d++)
#pragma unroll
            for (int it = 0; it < I; it++) {
                const uint32_t i = (uint32_t)it < count ? it : count - 1;
                ybuf[(d * I + it) * kThreads + threadIdx.x] = *lane_word(d == own ? c1 + i * p.ct_item_stride : y + i * y_item + d * digit, j);
            }
        __syncthreads();
    }
    // The operands of one term are requested while another is multiplied, in two sets by turns, so that a wave neither waits for
    // memory once per term nor moves a set; the gather index belongs to the step.  Every request is made on every path, past the end
    // for the last term again: behind a branch that may skip loads the compiler waits for all of them.  (A thread's items past
    // the last one read that one again.)
    struct Term {
        uint64_t k0, k1, v[I];
    };
    uint32_t st = 0, d = 0, next = 0, src = galois_index(j, p.elts[0], p.log_n);
    const uint64_t *yd = y;
    auto fetch = [&](Term &x) {
        const uint64_t *k = p.evk.p[next] + key_row;
        x.k0 = *lane_word(k, j);
        x.k1 = *lane_word(k + key_poly, j);
        const bool mine = d == own;
        const uint64_t *w = mine ? c1 : yd;
        const size_t stride = mine ? p.ct_item_stride : y_item;
#pragma unroll
        for (int it = 0; it < I; it++) {
            x.v[it] = LOCAL ? ybuf[(d * I + it) * kThreads + (src & (kThreads - 1))] : *lane_word(w, src);
            w += (uint32_t)it + 1 < count ? stride : 0;
        }
        const bool more = next + 1 < n_terms, wrap = more && d + 1 == p.beta;
        next += more ? 1 : 0;
        d = wrap ? 0 : d + (more ? 1 : 0);
        yd = wrap ? y : yd + (more ? digit : 0);
        if (wrap) src = galois_index(j, p.elts[++st], p.log_n);
    };
    auto terms = [&](auto &&take) {
        Term x, z;
        fetch(x);
        uint32_t e = 0;
        if (n_terms > 1) {
            do {
                fetch(z);
                asm volatile("" ::: "memory");       // (a compiler barrier: without it the loads, whose values are first used in the
                __builtin_amdgcn_sched_barrier(0);   //  next half, sink to the end of this one and every term waits for its operands)
                take(e, x);
                fetch(x);
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                take(e + 1, z);
                e += 2;
            } while (e + 1 < n_terms);
        }
        if (e < n_terms) take(e, x);
    };
    const size_t o = ((size_t)t << p.log_n) + j;
    const size_t opoly = (size_t)LK << p.log_n;
    if (table < 64 && ((p.fp_mask >> table) & 1)) {
        // a prime below 2^50: the sum of the products as an exact pair (hi, lo) before any reduction, four FP64
        // operations per product.  hi runs in [2^B, 2^(B+1)), where doubles are the multiples of 2^(B-52): the fused
        // multiply-add t = fl(x w + hi) rounds the exact sum to such a multiple, t - hi is exact, x w - (t - hi) is the
        // rounding error, an integer of at most 2^(B-53) in magnitude that the second fused multiply-add returns
        // exactly.  B = 103 takes 8 products below 2^100 between two folds (8 errors sum exactly, <= 2^53); when
        // n_terms q^2 <= 2^100 a smaller B takes all of them (at most 64) in one go.
        const FpMod m{p.fp_consts[4 * table], p.fp_consts[4 * table + 1]};
        const uint32_t qbits = 64 - __builtin_clzll(p.moduli[table]);              // q < 2^qbits
        const uint32_t tbits = 32 - __builtin_clz(n_terms);                        // n_terms < 2^tbits
        const bool one_go = 2 * qbits + tbits <= 100;
        const uint32_t B = !one_go ? 103 : 2 * qbits + tbits < 60 ? 60 : 2 * qbits + tbits;   // (any B up to 100 serves small primes)
        const uint32_t fold_mask = one_go ? 0xffffffffu : 7u;
        const double base = __hiloint2double((int)((1023 + B) << 20), 0);
        const double down = __hiloint2double((int)((1023 + 52 - B) << 20), 0);     // 2^-(B-52)
        const double cB = fp_reduce(__hiloint2double((int)((1023 + B - 52) << 20), 0), m);
        double hi0[I], lo0[I], hi1[I], lo1[I], f0[I], f1[I];
#pragma unroll
        for (int it = 0; it < I; it++) {
            hi0[it] = hi1[it] = base;
            lo0[it] = lo1[it] = f0[it] = f1[it] = 0.0;
        }
        // (hi - 2^B) / 2^(B-52) is an integer below 2^52; times 2^(B-52) mod q it is congruent to the high part, and the
        // modular product takes it as it is (result at most 2.5 q in magnitude)
        auto fold = [&]() {
#pragma unroll
            for (int it = 0; it < I; it++) {
                f0[it] = fp_reduce(f0[it] + fp_mulmod((hi0[it] - base) * down, cB, m) + fp_reduce(lo0[it], m), m);
                f1[it] = fp_reduce(f1[it] + fp_mulmod((hi1[it] - base) * down, cB, m) + fp_reduce(lo1[it], m), m);
                hi0[it] = hi1[it] = base;
                lo0[it] = lo1[it] = 0.0;
            }
        };
        terms([&](uint32_t e, const Term &x) {
            const double w0 = fp_from_u64(x.k0), w1 = fp_from_u64(x.k1);
#pragma unroll
            for (int it = 0; it < I; it++) {
                const double v = fp_from_u64(x.v[it]);
                const double t0 = __builtin_fma(v, w0, hi0[it]), t1 = __builtin_fma(v, w1, hi1[it]);
                lo0[it] += __builtin_fma(v, w0, -(t0 - hi0[it]));
                lo1[it] += __builtin_fma(v, w1, -(t1 - hi1[it]));
                hi0[it] = t0;
                hi1[it] = t1;
            }
            if ((e & fold_mask) == fold_mask) fold();
        });
        fold();   // (what the last full eight terms left, possibly nothing)
#pragma unroll
        for (int it = 0; it < I; it++) {
            if ((uint32_t)it >= count) break;
            uint64_t *out = p.out + (item0 + it) * ((size_t)2 * LK << p.log_n);
            double o0 = f0[it], o1 = f1[it];
            if (p.accumulate) {
                o0 += fp_from_u64(out[o]);
                o1 += fp_from_u64(out[o + opoly]);
            }
            out[o] = fp_to_u64(fp_canonical(o0, m));
            out[o + opoly] = fp_to_u64(fp_canonical(o1, m));
        }
        return;
    }
    Sum3 s0[I], s1[I], h0[I], h1[I];
    // the words are relieved every 8 terms for a prime below 2^60, every 2 otherwise (see Sum3)
    const uint32_t spill_mask = (p.moduli[table] >> 60) ? 1u : 7u;
#pragma unroll
    for (int it = 0; it < I; it++) s0[it] = s1[it] = h0[it] = h1[it] = Sum3{0, 0, 0};
    terms([&](uint32_t e, const Term &x) {
        const Split30d ks0 = split30d(x.k0), ks1 = split30d(x.k1);
#pragma unroll
        for (int it = 0; it < I; it++) mac_sum3x2(s0[it], s1[it], split30d(x.v[it]), ks0, ks1);
        if ((e & spill_mask) == spill_mask) {
#pragma unroll
            for (int it = 0; it < I; it++) {
                spill_sum3(h0[it], s0[it]);
                spill_sum3(h1[it], s1[it]);
            }
        }
    });
    const uint64_t q = p.moduli[table], r0 = p.barrett[2 * table], r1 = p.barrett[2 * table + 1];
#pragma unroll
    for (int it = 0; it < I; it++) {
        if ((uint32_t)it >= count) break;
        uint64_t *out = p.out + (item0 + it) * ((size_t)2 * LK << p.log_n);
        const U128 a0 = total_sum3(h0[it], s0[it]), a1 = total_sum3(h1[it], s1[it]);
        uint64_t o0 = barrett128(a0.lo, a0.hi, q, r0, r1);
        uint64_t o1 = barrett128(a1.lo, a1.hi, q, r0, r1);
        if (p.accumulate) {
            o0 = add_mod(o0, out[o], q);
            o1 = add_mod(o1, out[o + opoly], q);
        }
        out[o] = o0;
        out[o + opoly] = o1;
    }
}

// Sums of one wave's terms of a hoisted inner product: both key polynomials, two coefficients per lane.
// A prime below 2^50: exact (hi, lo) pairs of doubles, see hoist_inner_kernel.
struct HoistSumsFp {
    FpMod m;
    double base, down, hi[4], lo[4], f[4];
    double cB;
    uint32_t period, pending;
    __device__ __forceinline__ HoistSumsFp(const double *consts, uint64_t q, uint32_t n_terms) : m{scalar(consts)[0], scalar(consts)[1]} {
        const uint32_t qbits = 64 - __builtin_clzll(q), tbits = 32 - __builtin_clz(n_terms);
        const bool one_go = 2 * qbits + tbits <= 100;
        const uint32_t B = !one_go ? 103 : 2 * qbits + tbits < 60 ? 60 : 2 * qbits + tbits;
        period = one_go ? n_terms : 8;
        pending = 0;
        base = __hiloint2double((int)((1023 + B) << 20), 0);
        down = __hiloint2double((int)((1023 + 52 - B) << 20), 0);
        cB = fp_reduce(__hiloint2double((int)((1023 + B - 52) << 20), 0), m);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            hi[i] = base;
            lo[i] = f[i] = 0.0;
        }
    }
    __device__ __forceinline__ void fold() {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            f[i] = fp_reduce(f[i] + fp_mulmod((hi[i] - base) * down, cB, m) + fp_reduce(lo[i], m), m);
            hi[i] = base;
            lo[i] = 0.0;
        }
        pending = 0;
    }
    // v: words of the two coefficients; k: the key polynomials' words, [polynomial][coefficient]
    __device__ __forceinline__ void add(const uint64_t *v, const uint64_t (*k)[2]) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const double x = fp_from_u64(v[c]);
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const double w = fp_from_u64(k[r][c]), t = __builtin_fma(x, w, hi[2 * r + c]);
                lo[2 * r + c] += __builtin_fma(x, w, -(t - hi[2 * r + c]));
                hi[2 * r + c] = t;
            }
        }
        if (++pending == period) fold();
    }
    __device__ __forceinline__ void finish(uint64_t (*o)[2]) {
        if (pending) fold();
#pragma unroll
        for (int i = 0; i < 4; i++) o[i >> 1][i & 1] = fp_to_u64(fp_canonical(f[i], m));
    }
};

// Any prime: sums of partial products (Lazy3)
struct HoistSumsInt {
    Lazy3 s[4], h[4];
    uint64_t q, r0, r1;
    uint32_t period, pending;
    __device__ __forceinline__ HoistSumsInt(uint64_t q_, uint64_t r0_, uint64_t r1_) : q(q_), r0(r0_), r1(r1_) {
        period = (q >> 60) ? 4 : 8;
        pending = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) s[i] = h[i] = Lazy3{0, 0, 0};
    }
    __device__ __forceinline__ void add(const uint64_t *v, const uint64_t (*k)[2]) {
#pragma unroll
        for (int c = 0; c < 2; c++) mac3x2(s[c], s[2 + c], split30(v[c]), split30(k[0][c]), split30(k[1][c]));
        if (++pending == period) {
#pragma unroll
            for (int i = 0; i < 4; i++) spill3(h[i], s[i]);
            pending = 0;
        }
    }
    __device__ __forceinline__ void finish(uint64_t (*o)[2]) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const U128 a = total3(h[i], s[i]);
            o[i >> 1][i & 1] = barrett128(a.lo, a.hi, q, r0, r1);
        }
    }
};

__device__ __forceinline__ Words2 stream_pair(const uint64_t *p) { return __builtin_nontemporal_load(reinterpret_cast<const Words2 *>(p)); }

// Terms [first, last) of limb t for the coefficients j, j + 1 of every lane; two terms are multiplied while the next two are
// on their way.
template <class Sums>
__device__ __forceinline__ void hoist_terms(const HoistArgs &p, uint32_t t, uint32_t table, uint32_t j, uint32_t first, uint32_t last,
                                            Sums &sums) {
    constexpr uint32_t U = 2;
    const uint32_t LK = p.L + p.K;
    const uint64_t *y = p.y + ((size_t)t << p.log_n), *c1 = p.c0 + ((size_t)(p.L + t) << p.log_n);
    const size_t key_off = ((size_t)table << p.log_n) + j, key_poly = (size_t)(p.size_q + p.K) << p.log_n;
    const size_t digit = (size_t)LK << p.log_n;
    const uint32_t own = (p.own_from_ct && t < p.L) ? t / p.K : 0xffffffffu;
    uint32_t st = first / p.beta, d = first - st * p.beta, src = galois_index(j, p.elts[st], p.log_n);
    Words2 k[2][U][2], w[2][U];
    uint32_t turn[2][U];
    uint32_t at = first;
    auto fetch = [&](int b) {
#pragma unroll
        for (int u = 0; u < (int)U; u++) {
            if (at >= last) break;
            const uint64_t *key = p.evk.p[at] + key_off;
            k[b][u][0] = stream_pair(key);
            k[b][u][1] = stream_pair(key + key_poly);
            w[b][u] = load_pair((d == own ? c1 : y + d * digit) + (src & ~1u));
            turn[b][u] = src;
            if (++d == p.beta) {
                d = 0;
                st++;
                if (at + 1 < last) src = galois_index(j, p.elts[st], p.log_n);
            }
            at++;
        }
    };
    auto take = [&](int b, uint32_t e) {
#pragma unroll
        for (int u = 0; u < (int)U; u++) {
            if (e + u >= last) break;
            uint64_t v[2], kk[2][2];
            turned(v, w[b][u], turn[b][u]);
#pragma unroll
            for (int r = 0; r < 2; r++) {
                kk[r][0] = k[b][u][r].x;
                kk[r][1] = k[b][u][r].y;
            }
            sums.add(v, kk);
        }
    };
    if (first >= last) return;
    fetch(0);
    for (uint32_t e = first;; e += 2 * U) {
        if (e + U < last) fetch(1);
        __builtin_amdgcn_sched_barrier(0);   // (the loads stay ahead of the products)
        take(0, e);
        if (e + U >= last) return;
        if (e + 2 * U < last) fetch(0);
        __builtin_amdgcn_sched_barrier(0);
        take(1, e + U);
        if (e + 2 * U >= last) return;
    }
}

// Hoisted rotations of one ciphertext (hoist_inner_kernel's rows, same results).  Every key word is read once, so the kernel is
// bound by that stream when there are many limbs and by the chain of a wave's terms when there are few.  A lane serves two
// neighbouring coefficients with 16-byte accesses; an XCD takes a contiguous eighth of the (limb, block) sequence, so that
// the words which the steps gather from a limb come from its own L2 after the first step, and the keys pass by without
// staying there.  SPLIT = 4: the four waves of a workgroup deal the terms of one block out and add their sums in LDS.
// Against one coefficient per lane, one term ahead, blocks dealt to the XCDs in turn: hoisting of 7 steps at N = 2^16,
// L = 24, K = 8 303 -> 248 us (704 MB of keys, 5.5 TB/s in this kernel), of 15 steps at L = 2, K = 1 60 -> 52 us.
template <int SPLIT>
__global__ __launch_bounds__(kThreads) void hoist_one_kernel(HoistArgs p) {
    constexpr uint32_t PER = 2 * kThreads / SPLIT;   // coefficients of a workgroup
    __shared__ uint64_t part_lds[SPLIT > 1 ? SPLIT : 1][2][SPLIT > 1 ? PER : 1];
    touch_arguments<sizeof(HoistArgs)>();
    const uint32_t LK = p.L + p.K, log_b = p.log_n - (SPLIT == 1 ? 9 : 7), heavy = LK << log_b;
    const uint32_t lane = threadIdx.x & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t id = blockIdx.x;
    auto contiguous = [](uint32_t i, uint32_t n) { return n % 8 == 0 ? (i & 7) * (n >> 3) + (i >> 3) : i; };
    if (id >= heavy) {
        // sums of the permuted c0, and the copy of c1
        id = contiguous(id - heavy, gridDim.x - heavy);
        const uint32_t t = id >> (p.log_n - 9), j = ((id & ((1u << (p.log_n - 9)) - 1)) << 9) + 2 * threadIdx.x;
        const size_t o = ((size_t)t << p.log_n) + j;
        Words2 *out = reinterpret_cast<Words2 *>(p.c0_out + o);
        if (t >= p.L) {
            if (!p.accumulate) *out = load_pair(p.c0 + o);
            return;
        }
        const uint64_t q = scalar(p.moduli)[t];
        const uint64_t *in = p.c0 + ((size_t)t << p.log_n);
        Words2 acc = p.accumulate ? *out : p.with_self ? load_pair(in + j) : Words2{0, 0};
#pragma unroll 4
        for (uint32_t s = 0; s < p.n_steps; s++) {
            const uint32_t g = galois_index(j, p.elts[s], p.log_n);
            uint64_t v[2];
            turned(v, load_pair(in + (g & ~1u)), g);
            acc.x = add_mod(acc.x, v[0], q);
            acc.y = add_mod(acc.y, v[1], q);
        }
        *out = acc;
        return;
    }
    id = contiguous(id, heavy);
    const uint32_t t = id >> log_b, base = (id & ((1u << log_b) - 1)) * PER, table = t < p.L ? t : p.size_q + (t - p.L);
    const uint32_t j = base + (SPLIT == 1 ? 128 * wave : 0) + 2 * lane;
    const uint32_t n_terms = p.n_steps * p.beta, share = (n_terms + SPLIT - 1) / SPLIT;
    const uint32_t first = SPLIT == 1 ? 0 : wave * share, last = SPLIT == 1 || first + share > n_terms ? n_terms : first + share;
    const uint64_t q = scalar(p.moduli)[table];
    uint64_t o[2][2];
    if (table < 64 && ((p.fp_mask >> table) & 1)) {
        HoistSumsFp sums(p.fp_consts + 4 * (size_t)table, q, n_terms);
        hoist_terms(p, t, table, j, first, last, sums);
        sums.finish(o);
    } else {
        HoistSumsInt sums(q, scalar(p.barrett)[2 * table], scalar(p.barrett)[2 * table + 1]);
        hoist_terms(p, t, table, j, first, last, sums);
        sums.finish(o);
    }
    if constexpr (SPLIT > 1) {
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int c = 0; c < 2; c++) part_lds[wave][r][2 * lane + c] = o[r][c];
        __syncthreads();
        if (wave > 1) return;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            uint64_t v = part_lds[0][wave][2 * lane + c];
#pragma unroll
            for (int i = 1; i < SPLIT; i++) v = add_mod(v, part_lds[i][wave][2 * lane + c], q);
            o[0][c] = v;
        }
    }
#pragma unroll
    for (int r = 0; r < (SPLIT > 1 ? 1 : 2); r++) {
        Words2 *out = reinterpret_cast<Words2 *>(p.out + ((size_t)((SPLIT > 1 ? wave : (uint32_t)r) * LK + t) << p.log_n) + j);
        Words2 v{o[r][0], o[r][1]};
        if (p.accumulate) {
            const Words2 old = *out;
            v.x = add_mod(v.x, old.x, q);
            v.y = add_mod(v.y, old.y, q);
        }
        *out = v;
    }
}

struct SampleArgs {
    uint64_t *out;
    const uint64_t *moduli, *barrett;
    const uint64_t *cdt;
    ChaChaKey key;
    uint64_t stream;
    LimbMap map;
    uint32_t log_n, cdt_len;
    int kind;
    uint32_t stream_stride;
    size_t out_item_stride;
};

// the first entry of the cumulative table above u (the table ascends)
__device__ __forceinline__ uint32_t cdt_magnitude(const uint64_t *cdt, uint32_t len, uint64_t u) {
    uint32_t lo = 0, hi = len;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (u >= cdt[mid])
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// ternary / error / gauss: one thread = one ChaCha block = 16 (ternary) or 8 coefficients, the same
// signed value written to every limb.  uniform: one thread = one block = 4 residues of one limb.
// KIND is a template parameter so that the loops over the block's words unroll and the words stay in registers (with
// a run-time count the array lived in scratch memory); a thread's 16 or 8 consecutive output words leave as 16-byte
// stores.
template <int KIND>
__device__ __forceinline__ void sample_signed(const SampleArgs &p, uint32_t b, uint64_t stream, uint64_t *out);

template <int KIND>
__global__ __launch_bounds__(kThreads) void sample_kernel(SampleArgs p) {
    const uint32_t n = 1u << p.log_n;
    const uint32_t b = blockIdx.x * kThreads + threadIdx.x;
    // blockIdx.y = item: its own stream id, its own polynomial
    const uint64_t stream = p.stream + (uint64_t)blockIdx.y * p.stream_stride;
    uint64_t *out = p.out + blockIdx.y * p.out_item_stride;
    uint32_t w[16];
    if (KIND == SAMPLE_UNIFORM) {
        const uint32_t per_limb = n / 4;
        if (b >= per_limb * p.map.limbs) return;
        const uint32_t limb = b / per_limb, blk = b % per_limb;
        const uint32_t table = map_table(p.map, limb);
        const uint64_t q = p.moduli[table], r0 = p.barrett[2 * table], r1 = p.barrett[2 * table + 1];
        chacha20_block(p.key, b, stream, w);
        uint64_t r[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            uint64_t lo = ((uint64_t)w[4 * e + 1] << 32) | w[4 * e];
            uint64_t hi = ((uint64_t)w[4 * e + 3] << 32) | w[4 * e + 2];
            r[e] = barrett128(lo, hi, q, r0, r1);
        }
        ulonglong2 *dst = reinterpret_cast<ulonglong2 *>(out + ((size_t)limb << p.log_n) + 4 * blk);
        dst[0] = ulonglong2{r[0], r[1]};
        dst[1] = ulonglong2{r[2], r[3]};
        return;
    }
    sample_signed<KIND>(p, b, stream, out);
}

// the signed coefficients of one ChaCha block (16 words w)
template <int KIND>
__device__ __forceinline__ void signed_values(int *v, const uint32_t *w, const uint64_t *cdt, uint32_t cdt_len) {
    constexpr int per_block = KIND == SAMPLE_TERNARY ? 16 : 8;
#pragma unroll
    for (int e = 0; e < per_block; e++) {
        if (KIND == SAMPLE_TERNARY) {
            v[e] = ternary_value(w[e]);
        } else if (KIND == SAMPLE_ERROR) {
            v[e] = error_value(w[2 * e], w[2 * e + 1]);
        } else {
            uint64_t u = ((uint64_t)w[2 * e + 1] << 32) | w[2 * e];
            const bool neg = u >> 63;
            u &= 0x7FFFFFFFFFFFFFFFull;
            const uint32_t mag = cdt_magnitude(cdt, cdt_len, u);
            v[e] = neg ? -(int)mag : (int)mag;
        }
    }
}

// ternary / error / gauss coefficients of ChaCha block b of `stream`, the same signed value to every limb of `out`
template <int KIND>
__device__ __forceinline__ void sample_signed(const SampleArgs &p, uint32_t b, uint64_t stream, uint64_t *out) {
    const uint32_t n = 1u << p.log_n;
    uint32_t w[16];
    constexpr int per_block = KIND == SAMPLE_TERNARY ? 16 : 8;
    if (b >= n / per_block) return;
    chacha20_block(p.key, b, stream, w);
    int v[per_block];
    signed_values<KIND>(v, w, p.cdt, p.cdt_len);
    for (uint32_t limb = 0; limb < p.map.limbs; limb++) {
        const uint64_t q = p.moduli[map_table(p.map, limb)];
        ulonglong2 *dst = reinterpret_cast<ulonglong2 *>(out + ((size_t)limb << p.log_n) + (size_t)per_block * b);
#pragma unroll
        for (int e = 0; e < per_block; e += 2)
            dst[e / 2] = ulonglong2{v[e] < 0 ? q - (uint64_t)(-v[e]) : (uint64_t)v[e],
                                    v[e + 1] < 0 ? q - (uint64_t)(-v[e + 1]) : (uint64_t)v[e + 1]};
    }
}

// Sampled polynomials as one signed byte per coefficient (the residues are made where the transform reads them: a launch
// that wrote them for every limb took 12 us for u, e0, e1 of one encryption and 16 us for one noise polynomial; its threads, one per
// ChaCha block, had 8 to 16 words to store per limb and the table of the Gaussian to walk in memory, which is in LDS here).
// One wave per workgroup: a polynomial has at most 8,192 blocks.
struct SmallArgs {
    int8_t *out;
    const uint64_t *cdt;
    ChaChaKey key;
    uint64_t stream;
    uint32_t log_n, cdt_len, items;
};
constexpr int kSmallThreads = 64;

template <int KIND>
__device__ __forceinline__ void sample_bytes(const SmallArgs &p, uint64_t stream, int8_t *out) {
    static_assert(KIND != SAMPLE_GAUSS, "has a kernel of its own");
    constexpr int per_block = KIND == SAMPLE_TERNARY ? 16 : 8;
    const uint32_t b = blockIdx.x * kSmallThreads + threadIdx.x;
    if (b >= (1u << p.log_n) / per_block) return;
    uint32_t w[16];
    chacha20_block(p.key, b, stream, w);
    int v[per_block];
    signed_values<KIND>(v, w, nullptr, 0);
    uint32_t *dst = reinterpret_cast<uint32_t *>(out + (size_t)per_block * b);
#pragma unroll
    for (int e = 0; e < per_block; e += 4) dst[e / 4] = four_bytes(v[e], v[e + 1], v[e + 2], v[e + 3]);
}

// u of every item, then e0, e1 of every item; blockIdx.y = polynomial
__global__ __launch_bounds__(kSmallThreads) void sample_encrypt_kernel(SmallArgs p) {
    const uint32_t y = blockIdx.y;
    int8_t *out = p.out + ((size_t)y << p.log_n);
    if (y < p.items) {
        sample_bytes<SAMPLE_TERNARY>(p, p.stream + 3 * (uint64_t)y, out);
    } else {
        const uint32_t e = y - p.items;
        sample_bytes<SAMPLE_ERROR>(p, p.stream + 3 * (uint64_t)(e >> 1) + 1 + (e & 1), out);
    }
}

// blockIdx.y = item.  Bound by the chain of a search: see gauss_bytes.
__global__ __launch_bounds__(kSmallThreads) void sample_gauss_small_kernel(SmallArgs p) {
    __shared__ uint64_t cdt[kSmallCdt];
    for (uint32_t i = threadIdx.x; i < kSmallCdt; i += kSmallThreads) cdt[i] = padded_cdt(p.cdt, p.cdt_len, i);
    const uint32_t b = blockIdx.x * kSmallThreads + threadIdx.x;
    uint32_t w[16];
    chacha20_block(p.key, b, p.stream + blockIdx.y, w);
    __syncthreads();
    if (b >= (1u << p.log_n) / 8) return;
    uint32_t o[2];
    gauss_bytes<8>(o, w, cdt);
    uint32_t *dst = reinterpret_cast<uint32_t *>(p.out + ((size_t)blockIdx.y << p.log_n) + 8 * (size_t)b);
    dst[0] = o[0];
    dst[1] = o[1];
}

}  // namespace

hipError_t launch_elementwise(const Tables &t, int op, const uint64_t *a, const uint64_t *b, const uint64_t *c,
                              uint64_t *out, uint32_t n_polys, LimbMap map, hipStream_t s) {
    if (n_polys == 0 || map.limbs == 0) return hipSuccess;
    EwArgs p{a, b, c, out, t.moduli, t.barrett, map, t.log_n, op};
    hipLaunchKernelGGL(elementwise_kernel, dim3((1u << t.log_n) / kThreads, map.limbs, n_polys), dim3(kThreads), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_scalar_mul_add(const Tables &t, const uint64_t *a, const uint64_t *b, uint64_t *out,
                                 const uint64_t *w, uint32_t first, uint32_t limbs, hipStream_t s) {
    if (limbs == 0) return hipSuccess;
    hipLaunchKernelGGL(scalar_mul_add_kernel, dim3((1u << t.log_n) / kThreads, limbs), dim3(kThreads), 0, s, a, b, out,
                       t.moduli, w, first, t.log_n);
    return hipGetLastError();
}

hipError_t launch_decompose_real(const Tables &t, const double *coeffs, uint64_t *out, uint32_t limbs, uint32_t first,
                                 uint32_t items, size_t out_item_stride, hipStream_t s) {
    if (limbs == 0 || items == 0) return hipSuccess;
    if (items > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(decompose_real_kernel, dim3((1u << t.log_n) / kThreads, limbs, items), dim3(kThreads), 0, s, coeffs,
                       out, t.moduli, t.barrett, first, t.log_n, out_item_stride);
    return hipGetLastError();
}

hipError_t launch_tensor(const Tables &t, const uint64_t *ct1, const uint64_t *ct2, uint64_t *out, uint32_t L,
                         bool square, hipStream_t s, const double *fp_consts, uint32_t items, uint64_t *out2) {
    if (items == 0 || items > 65535 || (items > 1 && !out2)) return hipErrorInvalidValue;
    const size_t poly = (size_t)L << t.log_n;
    TensorArgs p{ct1, ct2, out, t.moduli, t.barrett, L, t.log_n, out2 ? out2 : out + 2 * poly, 2 * poly, 2 * poly, poly};
    dim3 grid((1u << t.log_n) / kThreads, L, items);
    if (fp_consts && square)
        hipLaunchKernelGGL(tensor_fp_kernel<true>, grid, dim3(kThreads), 0, s, p, fp_consts);
    else if (fp_consts)
        hipLaunchKernelGGL(tensor_fp_kernel<false>, grid, dim3(kThreads), 0, s, p, fp_consts);
    else if (square)
        hipLaunchKernelGGL(tensor_kernel<true>, grid, dim3(kThreads), 0, s, p);
    else
        hipLaunchKernelGGL(tensor_kernel<false>, grid, dim3(kThreads), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_tensor_mxn(const Tables &t, const uint64_t *ct1, uint32_t s1, const uint64_t *ct2, uint32_t s2,
                             uint64_t *out, uint32_t L, hipStream_t s) {
    const size_t poly = (size_t)L << t.log_n;
    TensorArgs p{ct1, ct2, out, t.moduli, t.barrett, L, t.log_n, out, 0, 0, poly};
    dim3 grid((1u << t.log_n) / kThreads, L);
#define HE_CASE(A, B) \
    if (s1 == A && s2 == B) hipLaunchKernelGGL((tensor_mxn_kernel<A, B>), grid, dim3(kThreads), 0, s, p); else
    HE_CASE(1, 1) HE_CASE(1, 2) HE_CASE(1, 3) HE_CASE(2, 1) HE_CASE(2, 2) HE_CASE(2, 3) HE_CASE(3, 1) HE_CASE(3, 2)
    HE_CASE(3, 3) {
        if (s1 == 0 || s2 == 0 || s1 > 16 || s2 > 16) return hipErrorInvalidValue;
        hipLaunchKernelGGL(tensor_any_kernel, grid, dim3(kThreads), 0, s, p, s1, s2);
    }
#undef HE_CASE
    return hipGetLastError();
}

hipError_t launch_pair_square_sum(const Tables &t, const uint64_t *psi, const uint64_t *const *pairs, uint64_t *out01, uint64_t *out2,
                                  uint32_t L, uint32_t items, uint32_t parts, uint32_t count, hipStream_t s) {
    if (items == 0 || items > 65535 || count == 0 || L == 0 || parts == 0 || parts > 2) return hipErrorInvalidValue;
    SquareSumArgs p{pairs, nullptr, out01, out2, t.moduli, t.barrett, psi, L, t.log_n, count, parts};
    // One part: while the launch is small its time is the chain of a thread, with one word half as long as with two; once the operands
    // fill the caches 16-byte accesses win.  us of one word a thread / two, two terms an item: 3 limbs of 2^12 words 2.62 / 3.28, 6 of 2^16
    // 5.66 / 5.91, 16 of 2^16 10.38 / 10.97, 24 of 2^16 15.8 / 16.2, 32 of 2^16 26.0 / 25.0, 160 of 2^16 152 / 132; ten terms, 10 of 2^15
    // 23.2 / 19.7.
    const uint32_t blocks = (1u << t.log_n) / kThreads;
    const bool one_word = (uint64_t)count * items * L << t.log_n <= (uint64_t)48 << 16;
    if (parts == 2)
        hipLaunchKernelGGL((pair_square_sum_kernel<2, 2>), dim3(blocks / 2, L, items), dim3(kThreads), 0, s, p);
    else if (one_word)
        hipLaunchKernelGGL((pair_square_sum_kernel<1, 1>), dim3(blocks, L, items), dim3(kThreads), 0, s, p);
    else
        hipLaunchKernelGGL((pair_square_sum_kernel<1, 2>), dim3(blocks / 2, L, items), dim3(kThreads), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_row_square_sums(const Tables &t, const uint64_t *psi, const uint64_t *const *cts, uint64_t *out01, uint64_t *out2,
                                  uint64_t *sums, uint32_t L, uint32_t clients, uint32_t chunks, hipStream_t s) {
    if (clients == 0 || clients > 2 * 65535 || chunks == 0 || L == 0) return hipErrorInvalidValue;
    SquareSumArgs p{cts, sums, out01, out2, t.moduli, t.barrett, psi, L, t.log_n, clients, chunks};
    const uint32_t wgs = (1u << t.log_n) / (2 * kThreads);
    hipLaunchKernelGGL(client_sums_kernel, dim3(wgs, L), dim3(kThreads), 0, s, p);
    if (hipError_t e = hipGetLastError()) return e;
    hipLaunchKernelGGL(row_square_kernel, dim3(wgs, L, (clients + 1) / 2), dim3(kThreads), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_sum(const Tables &t, const uint64_t *const *cts, uint64_t *out, uint32_t limbs, uint32_t polys, uint32_t items,
                      uint32_t count, hipStream_t s) {
    // (one launch holds 65535 polynomials: more rows take several)
    const uint32_t per_launch = 65535u / polys;
    for (uint32_t first = 0; first < items; first += per_launch) {
        const uint32_t rows = items - first < per_launch ? items - first : per_launch;
        SumArgs p{cts + (size_t)first * count, out + ((size_t)first * polys * limbs << t.log_n), t.moduli, t.barrett, limbs, t.log_n, polys, count};
        hipLaunchKernelGGL(sum_kernel, dim3((1u << t.log_n) / (2 * kThreads), limbs, rows * polys), dim3(kThreads), 0, s, p);
        if (hipError_t e = hipGetLastError()) return e;
    }
    return hipSuccess;
}

hipError_t launch_multiply_sum(const Tables &t, const uint64_t *const *pairs, uint64_t *out, uint32_t limbs, uint32_t items,
                               uint32_t count, hipStream_t s) {
    SumArgs p{pairs, out, t.moduli, t.barrett, limbs, t.log_n, 2, count};
    hipLaunchKernelGGL(multiply_sum_kernel, dim3((1u << t.log_n) / (2 * kThreads), limbs, items), dim3(kThreads), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_decrypt_gather(const Tables &t, const uint64_t *const *cts, const uint64_t *sk, const uint64_t *noise,
                                 uint64_t *out, uint32_t limbs, uint32_t items, hipStream_t s) {
    if (items == 0 || items > 65535 || limbs == 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(decrypt_gather_kernel, dim3((1u << t.log_n) / kThreads, limbs, items), dim3(kThreads), 0, s, cts, sk,
                       noise, out, t.moduli, t.barrett, limbs, t.log_n);
    return hipGetLastError();
}

hipError_t launch_galois(const Tables &t, const uint64_t *in, uint64_t *out, uint32_t total_limbs, uint32_t elt,
                         hipStream_t s) {
    if (total_limbs == 0) return hipSuccess;
    hipLaunchKernelGGL(galois_kernel, dim3((1u << t.log_n) / kThreads, total_limbs), dim3(kThreads), 0, s, in, out, elt,
                       t.log_n);
    return hipGetLastError();
}

hipError_t launch_bconv(const Tables &t, const BconvArgs &a, hipStream_t s) {
    if (a.n_out == 0) return hipSuccess;
    BconvKArgs p{a, t.moduli, t.barrett, t.log_n};
    dim3 grid((1u << t.log_n) / kThreads, (a.n_out + kRows - 1) / kRows);
    switch (a.n_in) {
#define HE_CASE(NIN) \
    case NIN: hipLaunchKernelGGL(bconv_kernel<NIN>, grid, dim3(kThreads), 0, s, p); break;
        HE_CASE(1) HE_CASE(2) HE_CASE(3) HE_CASE(4) HE_CASE(5) HE_CASE(6) HE_CASE(7) HE_CASE(8)
#undef HE_CASE
        default: hipLaunchKernelGGL(bconv_kernel<0>, grid, dim3(kThreads), 0, s, p);
    }
    return hipGetLastError();
}

hipError_t launch_bconv_batched(const Tables &t, const BconvBatch &b, const Tuning &tune, hipStream_t s) {
    if (b.n_units == 0) return hipSuccess;
    const uint32_t target = tune.bconv_rows >= 1 && tune.bconv_rows <= 64 ? tune.bconv_rows : 6;
    const uint32_t cg = (b.max_rows + target - 1) / target;
    const uint32_t rows_per = (b.max_rows + cg - 1) / cg;
    const uint32_t kg = (b.max_copy + rows_per - 1) / rows_per;
    BconvBatchK p{b, t.moduli, t.barrett, t.log_n, cg, rows_per};
    const uint32_t items = b.items ? b.items : 1;
    if ((uint64_t)b.n_units * items > 65535) return hipErrorInvalidValue;
    const dim3 grid((1u << t.log_n) / kThreads, cg + kg, b.n_units * items);
    if (b.mat_fp)
        hipLaunchKernelGGL(bconv_batched_fp_kernel, grid, dim3(kThreads), 0, s, p);
    else
        hipLaunchKernelGGL(bconv_batched_kernel, grid, dim3(kThreads), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_inner_product(const Tables &t, const uint64_t *y, const EvkPtrs &evk, uint64_t *out, uint32_t L,
                                uint32_t K, uint32_t size_q, uint32_t beta, uint32_t galois_elt, bool accumulate,
                                const uint64_t *fold_ct, const uint64_t *fold_w, uint32_t items, size_t fold_item_stride,
                                hipStream_t s, const uint64_t *add_c0, uint32_t add_elt, const uint64_t *p_mod_q,
                                const uint64_t *own, size_t own_item_stride, uint32_t own_elt) {
    const size_t n = (size_t)1 << t.log_n;
    InnerArgs p{y, out, t.moduli, t.barrett, evk, L, K, size_q, beta, t.log_n, galois_elt, accumulate ? 1 : 0,
                fold_ct, fold_w, (size_t)beta * (L + K) * n, 2 * (size_t)(L + K) * n, fold_item_stride,
                add_c0, p_mod_q, add_elt, own, own_item_stride, own_elt};
    if (items == 0 || items > 65535 || (add_c0 && (items != 1 || !p_mod_q))) return hipErrorInvalidValue;
    hipLaunchKernelGGL(inner_product_kernel, dim3((1u << t.log_n) / kThreads, L + K, items), dim3(kThreads), 0, s, p);
    return hipGetLastError();
}

struct InnerFpArgs {
    const uint64_t *y, *own;
    uint64_t *out;
    const double *fp_consts;
    EvkPtrs evk;
    uint32_t L, K, size_q, beta, log_n, items;
    const uint64_t *fold_ct, *fold_w;
    size_t y_item_stride, own_item_stride, out_item_stride, fold_item_stride;
};

// The inner product of a batch on the FP64 back end (every prime below 2^50).  grid: (N / 512, L + K, groups of I
// items); a thread holds two coefficients of I items.  A key word is loaded and converted once and multiplies all I
// items, so the 2 beta key limbs are read once per group instead of once per item; a digit's own limbs are read from
// the key switch's input (own, NTT form) rather than from a copy inside y.  Terms stay below 0.875 q, eight of them
// fit between two reductions; the stores are canonical, hence equal to the integer kernel's.
template <int I>
__global__ __launch_bounds__(kThreads) void inner_product_fp_kernel(InnerFpArgs p) {
    const uint32_t t = blockIdx.y;
    const uint32_t LK = p.L + p.K;
    const uint32_t table = t < p.L ? t : p.size_q + (t - p.L);
    const FpMod m{p.fp_consts[4 * table], p.fp_consts[4 * table + 1]};
    const size_t j = 2 * ((size_t)blockIdx.x * kThreads + threadIdx.x);
    const size_t key_off = ((size_t)table << p.log_n) + j;
    const size_t key_poly = (size_t)(p.size_q + p.K) << p.log_n;
    const uint32_t item0 = blockIdx.z * I;
    const uint32_t own_digit = t < p.L ? t / p.K : 0xffffffffu;
    double acc[I][4];
#pragma unroll
    for (int i = 0; i < I; i++) acc[i][0] = acc[i][1] = acc[i][2] = acc[i][3] = 0.0;
    for (uint32_t d = 0; d < p.beta; d++) {
        const uint64_t *k = p.evk.p[d];
        const ulonglong2 k0 = *reinterpret_cast<const ulonglong2 *>(k + key_off);
        const ulonglong2 k1 = *reinterpret_cast<const ulonglong2 *>(k + key_off + key_poly);
        const double w00 = fp_from_u64(k0.x), w01 = fp_from_u64(k0.y), w10 = fp_from_u64(k1.x), w11 = fp_from_u64(k1.y);
        const bool is_own = d == own_digit;
        const uint64_t *src = is_own ? p.own + ((size_t)t << p.log_n) + j : p.y + (((size_t)d * LK + t) << p.log_n) + j;
        const size_t stride = is_own ? p.own_item_stride : p.y_item_stride;
#pragma unroll
        for (int i = 0; i < I; i++) {
            const uint32_t item = item0 + i < p.items ? item0 + i : p.items - 1;
            const ulonglong2 v = *reinterpret_cast<const ulonglong2 *>(src + item * stride);
            const double y0 = fp_from_u64(v.x), y1 = fp_from_u64(v.y);
            acc[i][0] += fp_mulmod(y0, w00, m);
            acc[i][1] += fp_mulmod(y1, w01, m);
            acc[i][2] += fp_mulmod(y0, w10, m);
            acc[i][3] += fp_mulmod(y1, w11, m);
        }
        if ((d & 7) == 7) {
#pragma unroll
            for (int i = 0; i < I; i++)
                for (int c = 0; c < 4; c++) acc[i][c] = fp_reduce(acc[i][c], m);
        }
    }
    const size_t o = ((size_t)t << p.log_n) + j;
    const size_t opoly = (size_t)LK << p.log_n;
    const bool fold = p.fold_ct && t == p.L - 1;
    const double fw = fold ? fp_from_u64(p.fold_w[0]) : 0.0;
#pragma unroll
    for (int i = 0; i < I; i++) {
        if (item0 + i >= p.items) break;
        double r[4];
        for (int c = 0; c < 4; c++) r[c] = fp_canonical(acc[i][c], m);
        if (fold) {
            const uint64_t *f = p.fold_ct + (item0 + i) * p.fold_item_stride + o;
            const ulonglong2 f0 = *reinterpret_cast<const ulonglong2 *>(f);
            const ulonglong2 f1 = *reinterpret_cast<const ulonglong2 *>(f + ((size_t)p.L << p.log_n));
            r[0] = fp_canonical(fp_mulmod(r[0], fw, m) + fp_from_u64(f0.x), m);
            r[1] = fp_canonical(fp_mulmod(r[1], fw, m) + fp_from_u64(f0.y), m);
            r[2] = fp_canonical(fp_mulmod(r[2], fw, m) + fp_from_u64(f1.x), m);
            r[3] = fp_canonical(fp_mulmod(r[3], fw, m) + fp_from_u64(f1.y), m);
        }
        uint64_t *out = p.out + (item0 + i) * p.out_item_stride + o;
        *reinterpret_cast<ulonglong2 *>(out) = ulonglong2{fp_to_u64(r[0]), fp_to_u64(r[1])};
        *reinterpret_cast<ulonglong2 *>(out + opoly) = ulonglong2{fp_to_u64(r[2]), fp_to_u64(r[3])};
    }
}

hipError_t launch_inner_product_fp(const Tables &t, const double *fp_consts, const uint64_t *y, const uint64_t *own,
                                   size_t own_item_stride, const EvkPtrs &evk, uint64_t *out, uint32_t L, uint32_t K,
                                   uint32_t size_q, uint32_t beta, const uint64_t *fold_ct, const uint64_t *fold_w,
                                   uint32_t items, size_t fold_item_stride, hipStream_t s) {
    const size_t n = (size_t)1 << t.log_n;
    if (items == 0 || n < 2 * kThreads || !fp_consts || !own) return hipErrorInvalidValue;
    InnerFpArgs p{y, own, out, fp_consts, evk, L, K, size_q, beta, t.log_n, items, fold_ct, fold_w,
                  (size_t)beta * (L + K) * n, own_item_stride, 2 * (size_t)(L + K) * n, fold_item_stride};
    auto grid = [&](uint32_t per) { return dim3((uint32_t)(n / (2 * kThreads)), L + K, (items + per - 1) / per); };
    if ((items + 7) / 8 > 65535) return hipErrorInvalidValue;
    if (items >= 7)
        hipLaunchKernelGGL(inner_product_fp_kernel<8>, grid(8), dim3(kThreads), 0, s, p);
    else if (items >= 3)
        hipLaunchKernelGGL(inner_product_fp_kernel<4>, grid(4), dim3(kThreads), 0, s, p);
    else
        hipLaunchKernelGGL(inner_product_fp_kernel<2>, grid(2), dim3(kThreads), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_hoist_inner(const Tables &t, const Tuning &tune, const uint64_t *y, const uint64_t *c0, const uint64_t *const *evk,
                              const uint32_t *elts, uint32_t n_steps, uint64_t *out, uint64_t *c0_out, uint32_t L,
                              uint32_t K, uint32_t size_q, uint32_t beta, bool accumulate, bool with_self, uint32_t items,
                              size_t ct_item_stride, hipStream_t s, const double *fp_consts, uint64_t fp_mask,
                              bool own_from_ct) {
    if (n_steps == 0 || n_steps * beta > (uint32_t)kMaxDigits || items == 0 || items > 65535) return hipErrorInvalidValue;
    HoistArgs p;
    memset(&p, 0, sizeof(p));
    p.y = y;
    p.c0 = c0;
    p.out = out;
    p.c0_out = c0_out;
    p.moduli = t.moduli;
    p.barrett = t.barrett;
    for (uint32_t i = 0; i < n_steps * beta; i++) p.evk.p[i] = evk[i];
    for (uint32_t i = 0; i < n_steps; i++) p.elts[i] = elts[i];
    p.n_steps = n_steps;
    p.L = L;
    p.K = K;
    p.size_q = size_q;
    p.beta = beta;
    p.log_n = t.log_n;
    p.accumulate = accumulate ? 1 : 0;
    p.with_self = with_self ? 1 : 0;
    p.ct_item_stride = ct_item_stride;
    p.items = items;
    p.fp_consts = fp_consts;
    p.fp_mask = fp_consts ? fp_mask : 0;
    p.own_from_ct = own_from_ct ? 1 : 0;
    const uint32_t rows = (L + K) + (with_self ? 2 : 1) * L;
    const uint32_t nb = (1u << t.log_n) / kThreads;
    p.rows = rows;
    // every automorphism of the launch stays inside the aligned 256-word blocks of the NTT order
    bool local = t.log_n >= 8 && beta * 4 <= (uint32_t)kHoistLocalTiles;
    for (uint32_t i = 0; i < n_steps && local; i++) local = t.log_n < 9 || ((elts[i] - 1) & ((1u << (t.log_n - 7)) - 1)) == 0;
    const bool no_local = tune.hoist_no_local, no_xcd = tune.hoist_no_xcd, no_contig = tune.hoist_no_contig;
    if (no_local) local = false;
    // ... or inside the aligned stretches of 4,096 words (steps that are multiples of N / 8192)
    bool stretch_local = t.log_n >= 12;
    for (uint32_t i = 0; i < n_steps && stretch_local; i++) stretch_local = ((elts[i] - 1) & ((1u << (t.log_n - 11)) - 1)) == 0;
    // One ciphertext: four waves share a block as long as that leaves at most four waves on a SIMD (hoisting split / unsplit:
    // n = 2^12, 3 + 1 limbs, 7 steps of 2 digits 28.2 / 31.4 us; n = 2^15, 10 + 3 limbs, 5 steps of 4 digits 100.0 / 101.7 us;
    // from 2^16 x 12 limbs on the unsplit form wins, 99.7 against 102.5 us, and 247.9 against 255.9 us at L = 24, K = 8)
    const bool hoist_split = n_steps * beta >= 4 && ((uint64_t)(L + K) << (t.log_n - 7)) <= 4096;
    if (items == 1 && t.log_n >= 9) {
        const uint32_t light = (rows - (L + K)) << (t.log_n - 9);
        if (hoist_split)
            hipLaunchKernelGGL(hoist_one_kernel<4>, dim3(((L + K) << (t.log_n - 7)) + light), dim3(kThreads), 0, s, p);
        else
            hipLaunchKernelGGL(hoist_one_kernel<1>, dim3(((L + K) << (t.log_n - 9)) + light), dim3(kThreads), 0, s, p);
        return hipGetLastError();
    }
    const bool p_xcd_ok = !no_xcd && (nb * rows) % 8 == 0;
    const bool stretches = !local && !no_contig && stretch_local && nb >= 128 && (nb >> 4) % 8 == 0;
    auto launch = [&](auto kernel, uint32_t per) {
        p.groups = (items + per - 1) / per;
        // (one group shares its keys with nobody, but its gathers still want a stretch's words in one L2: 4 items of 2^16 words, steps
        // that are multiples of 8, the whole call 99.9 -> 76.3 us)
        p.xcd_map = !p_xcd_ok ? 0 : stretches ? 2 : p.groups > 1 ? 1 : 0;
        const uint64_t wgs = (uint64_t)nb * rows * p.groups;
        if (wgs > most_workgroups(kThreads)) return hipErrorInvalidValue;
        hipLaunchKernelGGL(kernel, dim3((uint32_t)wgs), dim3(kThreads), 0, s, p);
        return hipGetLastError();
    };
    // Items of a thread.  More of them read the keys less often but need more registers (5, 6 and 8 at 3, 2 and 2 waves per SIMD: 6 %,
    // 5 to 20 % and 20 % slower than 4 at 4 waves), and a thread multiplies for all of its places, also those past the last item: 5 as 4
    // and 1 cost what 8 do, as 3 and 2 what 6 do.  A group's own cost is about an item's.  Calls on [60, 40 | 60] bits, 15 steps, as 4 / as
    // 3: 2^16 words, 5 items block-local 98.2 / 94.1 us, from memory 109.6 / 104.2, 9 items 138.7 / 133.1 and 156.8 / 148.1, but 7 items
    // 111.0 / 116.1 and 8 items 126.9 / 136.9; 3 items as 2 and 1 / as 3, block-local 71.5 / 64.8.
    // Below five workgroups for every two CUs two items, block-local below two a CU: more waves hide more than fewer key words save.  As 4 /
    // 3 / 2: 9 items of 2^14 words from memory 67.4 / 65.4 / 62.9, 23 of 2^13 71.8 / 67.6 / 68.1; block-local 11 of 2^14 (576 workgroups)
    // 61.2 / 59.2 / 63.8, 7 of 2^14 (384) 47.9 / 48.4 / 46.6.
    auto cost = [&](uint32_t per) { return (items + per - 1) / per * (per + 1); };
    uint32_t per = 4;
    for (uint32_t i = 3; i >= 2; i--)
        if (cost(i) < cost(per)) per = i;
    const uint64_t heavy = (uint64_t)nb * (L + K) * ((items + per - 1) / per);
    if (2 * heavy < (local ? 4 : 5) * (uint64_t)tune.cus) per = 2;
#define HE_HOIST(I) return local ? launch(hoist_inner_kernel<I, true>, I) : launch(hoist_inner_kernel<I, false>, I)
    if (per == 4) HE_HOIST(4);
    if (per == 3) HE_HOIST(3);
    HE_HOIST(2);
#undef HE_HOIST
}

hipError_t launch_sample(const Tables &t, int kind, ChaChaKey key, uint64_t stream_id, uint64_t *out, LimbMap map,
                         const uint64_t *cdt, uint32_t cdt_len, uint32_t items, uint32_t stream_stride,
                         size_t out_item_stride, hipStream_t s) {
    if (items == 0 || items > 65535) return hipErrorInvalidValue;
    const uint32_t n = 1u << t.log_n;
    uint32_t blocks = kind == SAMPLE_UNIFORM ? (n / 4) * map.limbs : (kind == SAMPLE_TERNARY ? n / 16 : n / 8);
    // (a thread's words leave as 16-byte stores)
    if ((reinterpret_cast<uintptr_t>(out) & 15) || (out_item_stride & 1)) return hipErrorInvalidValue;
    SampleArgs p{out, t.moduli, t.barrett, cdt, key, stream_id, map, t.log_n, cdt_len, kind, stream_stride, out_item_stride};
    const dim3 grid((blocks + kThreads - 1) / kThreads, items);
    switch (kind) {
        case SAMPLE_UNIFORM: hipLaunchKernelGGL(sample_kernel<SAMPLE_UNIFORM>, grid, dim3(kThreads), 0, s, p); break;
        case SAMPLE_TERNARY: hipLaunchKernelGGL(sample_kernel<SAMPLE_TERNARY>, grid, dim3(kThreads), 0, s, p); break;
        case SAMPLE_ERROR: hipLaunchKernelGGL(sample_kernel<SAMPLE_ERROR>, grid, dim3(kThreads), 0, s, p); break;
        case SAMPLE_GAUSS: hipLaunchKernelGGL(sample_kernel<SAMPLE_GAUSS>, grid, dim3(kThreads), 0, s, p); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_sample_encrypt(uint32_t log_n, ChaChaKey key, uint64_t stream_id, int8_t *out, uint32_t items, hipStream_t s) {
    if (items == 0 || 3 * (uint64_t)items > 65535 || log_n < 7) return hipErrorInvalidValue;
    const SmallArgs p{out, nullptr, key, stream_id, log_n, 0, items};
    // (the grid covers the error polynomials' blocks; the surplus threads of the ternary ones leave at once)
    const dim3 grid(((1u << log_n) / 8 + kSmallThreads - 1) / kSmallThreads, 3 * items);
    hipLaunchKernelGGL(sample_encrypt_kernel, grid, dim3(kSmallThreads), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_sample_gauss_small(uint32_t log_n, ChaChaKey key, uint64_t stream_id, int8_t *out, const uint64_t *cdt,
                                     uint32_t cdt_len, uint32_t items, hipStream_t s) {
    if (items == 0 || items > 65535 || log_n < 7 || cdt_len == 0 || cdt_len >= kSmallCdt) return hipErrorInvalidValue;
    const SmallArgs p{out, cdt, key, stream_id, log_n, cdt_len, items};
    const dim3 grid(((1u << log_n) / 8 + kSmallThreads - 1) / kSmallThreads, items);
    hipLaunchKernelGGL(sample_gauss_small_kernel, grid, dim3(kSmallThreads), 0, s, p);
    return hipGetLastError();
}

}  // namespace he
