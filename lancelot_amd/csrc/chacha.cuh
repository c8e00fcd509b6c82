// The random words of the samplers, and the discrete Gaussian made of them.
#pragma once
#include "kernels.h"

namespace he {

namespace {

// ---------------------------------------------------------------------------------------------------
// samplers: ChaCha20 block function (RFC 8439 section 2.3), 64-bit block counter in words 12-13,
// 64-bit stream id in words 14-15
// ---------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t rotl32(uint32_t v, int c) { return (v << c) | (v >> (32 - c)); }

#define HE_QR(a, b, c, d) \
    a += b; d ^= a; d = rotl32(d, 16); \
    c += d; b ^= c; b = rotl32(b, 12); \
    a += b; d ^= a; d = rotl32(d, 8);  \
    c += d; b ^= c; b = rotl32(b, 7);

__device__ void chacha20_block(const ChaChaKey &key, uint64_t counter, uint64_t stream, uint32_t *out) {
    uint32_t s[16] = {0x61707865u, 0x3320646eu, 0x79622d32u, 0x6b206574u,
                      key.k[0], key.k[1], key.k[2], key.k[3], key.k[4], key.k[5], key.k[6], key.k[7],
                      (uint32_t)counter, (uint32_t)(counter >> 32), (uint32_t)stream, (uint32_t)(stream >> 32)};
    uint32_t x[16];
#pragma unroll
    for (int i = 0; i < 16; i++) x[i] = s[i];
    for (int i = 0; i < 10; i++) {
        HE_QR(x[0], x[4], x[8], x[12]) HE_QR(x[1], x[5], x[9], x[13]) HE_QR(x[2], x[6], x[10], x[14]) HE_QR(x[3], x[7], x[11], x[15])
        HE_QR(x[0], x[5], x[10], x[15]) HE_QR(x[1], x[6], x[11], x[12]) HE_QR(x[2], x[7], x[8], x[13]) HE_QR(x[3], x[4], x[9], x[14])
    }
#pragma unroll
    for (int i = 0; i < 16; i++) out[i] = x[i] + s[i];
}

// A ternary coefficient of one word, and an error (centred binomial, 21 bits a side) of two
__device__ __forceinline__ int ternary_value(uint32_t w) { return (int)(((uint64_t)w * 3) >> 32) - 1; }
__device__ __forceinline__ int error_value(uint32_t w0, uint32_t w1) { return __popc(w0 & 0x1FFFFFu) - __popc(w1 & 0x1FFFFFu); }
__device__ __forceinline__ uint32_t four_bytes(int a, int b, int c, int d) {
    return (uint32_t)(a & 255) | ((uint32_t)(b & 255) << 8) | ((uint32_t)(c & 255) << 16) | ((uint32_t)(d & 255) << 24);
}

// The cumulative table of the discrete Gaussian, padded to 128 entries that nothing reaches, so that all searches take the same seven
// steps and those of a thread go together, their LDS reads behind one another instead of each search after the one before
// (one polynomial of 2^16 coefficients 7.9 -> 5.1 us).
constexpr uint32_t kSmallCdt = 128;
__device__ __forceinline__ uint64_t padded_cdt(const uint64_t *cdt, uint32_t len, uint32_t i) { return i < len ? cdt[i] : ~(uint64_t)0; }

// COUNT coefficients from as many pairs of words, a signed byte each, four to an element of o
template <int COUNT>
__device__ __forceinline__ void gauss_bytes(uint32_t *o, const uint32_t *w, const uint64_t *cdt) {
    uint64_t u[COUNT];
    uint32_t mag[COUNT];
#pragma unroll
    for (int e = 0; e < COUNT; e++) {
        u[e] = (((uint64_t)w[2 * e + 1] << 32) | w[2 * e]) & 0x7FFFFFFFFFFFFFFFull;
        mag[e] = 0;
    }
    // the number of entries that are not above u (the table ascends)
#pragma unroll
    for (uint32_t step = kSmallCdt / 2; step; step >>= 1) {
#pragma unroll
        for (int e = 0; e < COUNT; e++) mag[e] += u[e] >= cdt[mag[e] + step - 1] ? step : 0;
    }
#pragma unroll
    for (int e = 0; e < COUNT; e += 4) o[e / 4] = 0;
#pragma unroll
    for (int e = 0; e < COUNT; e++) {
        const uint32_t v = w[2 * e + 1] >> 31 ? 0u - mag[e] : mag[e];
        o[e / 4] |= (v & 255) << (8 * (e % 4));
    }
}

}  // namespace

}  // namespace he
