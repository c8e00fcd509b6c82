// Base conversion fused with the rows pass of the forward transform that follows it, 4 words per thread, every back end.
//
// Both operate on the same set of coefficients: a tile of all N / 256 rows x C columns of a limb's (N / 256) x 256 view.  A workgroup
// of 512 threads owns a tile of 2048 words of one unit (a ModUp digit or a ModDown polynomial) and a group of the unit's output limbs;
// a thread keeps its 4 words of each of the (at most 8) input limbs in registers, and for every output limb of the group it
// forms sum_i x_i M[r][i] and goes straight on with the rows pass (Tile4 of ntt_common.cuh): the converted limbs never
// exist in coefficient form in memory.  The groups of one tile re-read the same inputs (from L2: they run on one XCD).
//
// mdr (merged ModDown + rescale): the last matrix row belongs to the limb that the rescale drops; with
// r = t - P^-1 sum_i x_i M[last][i] mod q_last (t: the limb right before the unit's inputs), output limb j receives
// P^-1 sum_i x_i M[j][i] + (r mod q_j).  (FP64: the matrix carries the factor P^-1.)
//
// What bounds it: instruction issue, about 390 instructions for a thread's 4 words of an output limb with 8 input limbs (their loads and
// set-up included), and the wait for the inputs that every workgroup starts with; 4 words a thread leave room for four waves per SIMD with 8
// input limbs in registers (on integers two or three), where 8 words left two.  One product against a kernel with 8 words per thread (FP64 only):
// n = 2^15, 10 of 12 limbs, K = 3 64.7 -> 55.8 us; n = 2^14, 8 limbs, K = 2 42.6 -> 38.4; a batch of 8, n = 2^15, 12 limbs, K = 4
// 233 -> 219; L = 24, K = 8 the same 150 us.  Levels with a prime from 2^50 on against conversion kernel + rows pass: n = 2^15, 10 of
// 12 limbs of 60 / 40 bits 77.5 -> 71.6 us; n = 2^13, 6 limbs, K = 2 45.4 -> 38.3; n = 2^16, 24 + 8 limbs 217 -> 204; a batch of 8,
// n = 2^15, 12 limbs, K = 3 323 -> 277.
// The unit, its rows and their primes are worked out from a few scalars (BconvUnit): looked up in the arguments, a description and two
// lists, one behind the other, they cost 1.2 us a product (n = 2^15, 10 of 12 limbs of 60 / 40 bits 67.4 -> 66.1 us; n = 2^13, 6
// limbs, K = 2 36.2 -> 35.1; n = 2^16, 24 + 8 limbs 141.8 -> 139.8).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.h"
#include "modarith.cuh"
#include "ntt_common.cuh"

namespace he {

namespace {

constexpr int kTileLog = 11;

// Conversion in FP64 (every prime of the level below 2^50).  The inputs are held as x' = x - 2^49 and the matrix entries centred, so that
// a product is below 2^98 in magnitude; what the shift takes away comes back with the row's constant (BconvRows::rows_fp).
template <int NIN, bool MDR, bool TILED>
struct ConvFp {
    double x[NIN][4], rr[MDR ? 4 : 1];
    // (tiled words are doubles, and shifted already)
    static __device__ __forceinline__ double value(uint64_t w) {
        return TILED ? FpArith::from_word(w) : __longlong_as_double((long long)(w | 0x4330000000000000ull)) - 0x1.2p52;
    }
    __device__ __forceinline__ void take(int k, int j, uint64_t w) { x[k][j] = value(w); }
    static __device__ __forceinline__ ScalarF64 row_of(const BconvExtra &b, const BconvUnit &d, uint32_t r) {
        return scalar(static_cast<const double *>(b.mat)) + (size_t)(d.row_off + r) * kConversionRow;
    }
    // v = sum of x M mod q, at most 1.01 q in magnitude, the sums' low part starting from lo.
    // The sum as an exact pair (hi, lo) before any reduction, four operations per term.  hi runs in [2^102, 2^103], where doubles are the
    // multiples of 2^50: t = fl(x w + hi) rounds the exact sum to such a multiple (eight products below 2^98 stay within 2^101 of
    // 1.5 2^102), t - hi is exact, x w - (t - hi) is the rounding error, an integer of at most 2^49 that the second fused multiply-add
    // returns exactly; eight of those, the row's constant below 2^49 and a residue below 2^50 sum exactly, to less than 2^52.5.
    // With H = hi - 1.5 2^102, a multiple of 2^50 up to 2^101, and c = 2^50 mod q the sum is H 2^-50 c + lo = h + l + lo, h = fl(H 2^-50 c),
    // up to 2^100, and one quotient serves all three: k = rint(lo / q + h / q), of which h's part is off by at most 3/8 (three roundings of a
    // number up to 2^50) and their sum by 1/8; h - k q is within q + 2^47 of -lo, below 2^53 as is every sum after it, and exact.
    static __device__ __forceinline__ void sum(double *v, const double (*x)[4], ScalarF64 row, uint32_t n_in, FpMod m, const double *lo0) {
        double hi[4], lo[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            hi[j] = 0x1.8p102;
            lo[j] = lo0[j];
        }
        double w[NIN];
#pragma unroll
        for (int k = 0; k < NIN; k++) w[k] = row[k];
        const double c = row[9];
#pragma unroll
        for (int k = 0; k < NIN; k++) {
            if ((uint32_t)k >= n_in) break;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const double t = __builtin_fma(x[k][j], w[k], hi[j]);
                lo[j] += __builtin_fma(x[k][j], w[k], -(t - hi[j]));
                hi[j] = t;
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const double big = hi[j] - 0x1.8p102, h = big * c, l = __builtin_fma(big, c, -h);
            const double k = __builtin_rint(__builtin_fma(lo[j], m.qinv, h * m.qinv));
            v[j] = (__builtin_fma(-k, m.q, h) + l) + lo[j];
        }
    }
    __device__ __forceinline__ void dropped(const NttArgs &a, const BconvExtra &b, const BconvUnit &d, const uint64_t *t) {
        const uint32_t last = d.n_out - 1;
        const FpMod m = fp_ctx(a, map_table(a.map, last)).m;
        const ScalarF64 row = row_of(b, d, last);
        double v[4], lo[4];
#pragma unroll
        for (int j = 0; j < 4; j++) lo[j] = row[8];
        sum(v, x, row, d.n_in, m, lo);
#pragma unroll
        for (int j = 0; j < 4; j++) rr[j] = fp_canonical((value(t[j]) + 0x1p49) - v[j], m);
    }
    __device__ __forceinline__ void convert(double *v, const NttArgs &, const BconvExtra &b, const BconvUnit &d, uint32_t r, uint32_t,
                                            const FpArith &ar) const {
        const ScalarF64 row = row_of(b, d, r);
        double lo[4];
#pragma unroll
        for (int j = 0; j < 4; j++) lo[j] = MDR ? rr[j] + row[8] : row[8];
        sum(v, x, row, d.n_in, ar.m, lo);
    }
};

// Conversion of integer inputs (any primes) in the arithmetic of the output limb.
template <int NIN, bool MDR>
struct ConvInt {
    Split30 x[NIN][4];
    uint64_t rr[MDR ? 4 : 1];
    __device__ __forceinline__ void take(int k, int j, uint64_t w) { x[k][j] = split30(w); }
    // sums of words j, j + 1 (the partial products are relieved every four terms: see Lazy3)
    __device__ __forceinline__ void sum(uint64_t *o, int j, const uint64_t *row, uint32_t n_in, uint64_t q, uint64_t r0, uint64_t r1) const {
        Lazy3 s0{0, 0, 0}, s1{0, 0, 0}, h0{0, 0, 0}, h1{0, 0, 0};
#pragma unroll
        for (int k = 0; k < NIN; k++) {
            if ((uint32_t)k >= n_in) break;
            mac3x2(s0, s1, split30(scalar(row)[k]), x[k][j], x[k][j + 1]);
            if (k % 4 == 3 && k + 1 < NIN) {
                spill3(h0, s0);
                spill3(h1, s1);
            }
        }
        const U128 a0 = total3(h0, s0), a1 = total3(h1, s1);
        o[0] = barrett128(a0.lo, a0.hi, q, r0, r1);
        o[1] = barrett128(a1.lo, a1.hi, q, r0, r1);
    }
    __device__ __forceinline__ void sums(uint64_t *o, const NttArgs &a, const BconvExtra &b, const BconvUnit &d, uint32_t r, uint32_t table) const {
        const uint64_t q = scalar(a.moduli)[table], r0 = scalar(a.barrett)[2 * table], r1 = scalar(a.barrett)[2 * table + 1];
        const uint64_t *row = static_cast<const uint64_t *>(b.mat) + d.mat_off + (size_t)r * d.n_in;
        sum(o, 0, row, d.n_in, q, r0, r1);
        sum(o + 2, 2, row, d.n_in, q, r0, r1);
    }
    __device__ __forceinline__ void dropped(const NttArgs &a, const BconvExtra &b, const BconvUnit &d, const uint64_t *t) {
        const uint32_t last = d.n_out - 1, table = map_table(a.map, last);
        const uint64_t q = scalar(a.moduli)[table];
        const Shoup w = scalar_shoup(static_cast<const uint64_t *>(b.w), last);
        uint64_t s[4];
        sums(s, a, b, d, last, table);
#pragma unroll
        for (int j = 0; j < 4; j++) rr[j] = sub_mod(t[j], mul_shoup(s[j], w, q), q);
    }
    __device__ __forceinline__ void convert(uint64_t *v, const NttArgs &a, const BconvExtra &b, const BconvUnit &d, uint32_t r, uint32_t table,
                                            const IntArith &) const {
        sums(v, a, b, d, r, table);
        if constexpr (MDR) {
            const uint64_t q = scalar(a.moduli)[table], r1 = scalar(a.barrett)[2 * table + 1];
            const Shoup w = scalar_shoup(static_cast<const uint64_t *>(b.w), r);
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = add_mod(mul_shoup(v[j], w, q), barrett64(rr[j], q, r1), q);
        }
    }
    // An output limb below 2^50: x = xh 2^30 + xl in FP64, sum of xh (M 2^30 mod q) + xl M (mod q), at most 1.01 q in magnitude.  As
    // ConvFp::sum: a product is below 2^80, hi runs around 1.5 2^86, where doubles are the multiples of 2^34, with sums below 2^85, and
    // what is left of a product is an integer of at most 2^33.  Four operations and a conversion a product, where integers take four
    // multiply-adds a term and sixty instructions to put a word together and reduce it.  Chains of 60 / 40 bits, integers -> FP64, one
    // product: n = 2^15, 10 of 12 limbs, K = 3 62.1 -> 60.7 us; n = 2^16, 12 + 4 limbs 91.6 -> 90.3, a batch of four 244 -> 239; a batch of
    // 8, n = 2^14, 8 limbs, K = 2 98.4 -> 94.6.
    __device__ __forceinline__ void convert(double *v, const NttArgs &, const BconvExtra &b, const BconvUnit &d, uint32_t r, uint32_t,
                                            const FpArith &ar) {
        // (the halves stay integers between the rows: as doubles of all inputs they would not fit in the registers)
#pragma unroll
        for (int k = 0; k < NIN; k++)
#pragma unroll
            for (int j = 0; j < 4; j++) asm volatile("" : "+v"(x[k][j].lo), "+v"(x[k][j].hi));
        if constexpr (MDR) {
#pragma unroll
            for (int j = 0; j < 4; j++) asm volatile("" : "+v"(rr[j]));
        }
        const ScalarF64 row = scalar(b.rows_mixed) + (size_t)(d.row_off + r) * kMixedRow;
        const FpMod m = ar.m;
        double hi[4], lo[4];
        auto add = [&](int j, double x, double w) {
            const double t = __builtin_fma(x, w, hi[j]);
            lo[j] += __builtin_fma(x, w, -(t - hi[j]));
            hi[j] = t;
        };
#pragma unroll
        for (int j = 0; j < 4; j++) {
            hi[j] = 0x1.8p86;
            lo[j] = 0.0;
            if constexpr (MDR) {
                const Split30 s = split30(rr[j]);
                lo[j] = (double)s.lo;
                add(j, (double)s.hi, row[17]);
            }
        }
#pragma unroll
        for (int k = 0; k < NIN; k++) {
            if ((uint32_t)k >= d.n_in) break;
            const double wh = row[k], wl = row[8 + k];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                add(j, (double)x[k][j].hi, wh);
                add(j, (double)x[k][j].lo, wl);
            }
        }
        const double c = row[16];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const double big = hi[j] - 0x1.8p86, h = big * c, l = __builtin_fma(big, c, -h);
            const double k = __builtin_rint(__builtin_fma(lo[j], m.qinv, h * m.qinv));
            v[j] = (__builtin_fma(-k, m.q, h) + l) + lo[j];
        }
    }
};

// BE: NTT_BACKEND_FP: the whole level is below 2^50; otherwise the inputs are integers, and MIXED: bit `table` of a.fp_mask says in which
// arithmetic the limb is converted and transformed
// TILED: the input limbs are in the order of conversion_word (BconvRows::tiled)
template <int LD, int BE, int NIN, bool MDR, bool TILED>
__global__ __launch_bounds__(1 << (kTileLog - 2)) __attribute__((amdgpu_waves_per_eu(BE == NTT_BACKEND_FP || NIN <= 4 ? 4 : 2)))
void bconv_rows4_kernel(HE_HEAD_PARAMS, BconvExtra b) {
    using T4 = Tile4<kTileLog, LD>;
    constexpr int LOGC = kTileLog - LD, NB = T4::kBlocks;
    constexpr uint32_t C = 1u << LOGC, tiles_per_limb = 256u >> LOGC;
    // (two tiles in turn: the barriers of one output limb say that the tile of the limb before is free again)
    __shared__ uint64_t lds[2][(1 << kTileLog) + (1 << (kTileLog - 4))];
    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    const size_t n = (size_t)1 << a.log_n;
    uint32_t lb = logical_block(h4);
    const uint32_t compute_groups = h2 & 0xffff, groups = compute_groups + (h2 >> 16), grp = lb % groups, rows_per = h5;
    lb /= groups;
    const uint32_t col0 = (lb % tiles_per_limb) << LOGC;
    const uint32_t K = h1 >> 16;
    const BconvUnit d = bconv_unit(a, h1 & 0xffff, K, lb / tiles_per_limb, TILED ? K + (MDR ? 1 : 0) : 0);
    const uint32_t t = ((uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) << 6) | (threadIdx.x & 63);
    // word j of layout k: a scalar distance from the lane's first one
    auto first = [&](int k) {
        const uint32_t e = T4::word(k, t, 0);
        return (e >> LOGC) * 256 + col0 + (e & (C - 1));
    };
    auto step = [](int k, int j) {
        const uint32_t e = (uint32_t)j << (kTileLog - 2 * k - 2);
        return (e >> LOGC) * 256 + (e & (C - 1));
    };
    const uint32_t in0 = first(0), out0 = first(NB - 1);
    if (grp >= compute_groups) {
        // limbs that pass through unchanged (a digit's own limbs keep their NTT form)
        const uint64_t *from = b.copy_base + d.item * b.copy_item_stride;
        const uint32_t c0 = (grp - compute_groups) * rows_per;
        for (uint32_t r = c0; r < c0 + rows_per && r < d.n_in; r++) {
            const size_t limb = (size_t)(d.copy_first + r) << a.log_n;
            uint64_t w[4];
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = (from + limb + step(0, j))[in0];
#pragma unroll
            for (int j = 0; j < 4; j++) (d.out + limb + step(0, j))[in0] = w[j];
        }
        return;
    }
    const uint32_t n_rows = MDR ? d.n_out - 1 : d.n_out, r_begin = grp * rows_per;
    const uint32_t r_end = r_begin + rows_per < n_rows ? r_begin + rows_per : n_rows;
    if (r_begin >= n_rows) return;
    typename std::conditional<BE == NTT_BACKEND_FP, ConvFp<NIN, MDR, TILED>, ConvInt<NIN, MDR>>::type conv;
    const uint64_t *x = d.in;
    {
        uint64_t w[NIN][4], tw[4];
        if constexpr (TILED) {
            const uint32_t at = conversion_word<kTileLog, LD>(col0 >> LOGC, t);
#pragma unroll
            for (int k = 0; k < NIN; k++) load_tiled(w[k], x + ((size_t)((uint32_t)k < d.n_in ? (uint32_t)k : d.n_in - 1) << a.log_n) + at);
            if constexpr (MDR) load_tiled(tw, x - n + at);
        } else {
#pragma unroll
            for (int k = 0; k < NIN; k++) {
                const uint32_t kk = (uint32_t)k < d.n_in ? (uint32_t)k : d.n_in - 1;
#pragma unroll
                for (int j = 0; j < 4; j++) w[k][j] = (x + ((size_t)kk << a.log_n) + step(0, j))[in0];
            }
            if constexpr (MDR) {
#pragma unroll
                for (int j = 0; j < 4; j++) tw[j] = (x - n + step(0, j))[in0];
            }
        }
#pragma unroll
        for (int k = 0; k < NIN; k++)
#pragma unroll
            for (int j = 0; j < 4; j++) conv.take(k, j, w[k][j]);
        if constexpr (MDR) conv.dropped(a, b, d, tw);
    }
    for (uint32_t r = r_begin; r < r_end; r++) {
        const uint32_t limb = d.limb(r), table = map_table(a.map, limb);
        uint64_t *dst = d.out + ((size_t)limb << a.log_n), *tile = lds[(r - r_begin) & 1];
        auto row = [&](const auto &ar) {
            using A = typename std::remove_cv<typename std::remove_reference<decltype(ar)>::type>::type;
            typename A::V v[4];
            typename A::Tw tw[NB];
            T4::template load_tw<A, 0>(tw, ar, 1, t);
            conv.convert(v, a, b, d, r, table, ar);
            T4::template forward<A>(v, tw, ar, tile, t);
#pragma unroll
            for (int j = 0; j < 4; j++) (dst + step(NB - 1, j))[out0] = A::to_word(v[j]);
        };
        if constexpr (BE == NTT_BACKEND_FP) {
            row(fp_arith(a, table));
        } else if constexpr (BE == NTT_BACKEND_INT) {
            row(int_arith(a, table));
        } else {
            if ((a.fp_mask >> table) & 1)
                row(fp_arith(a, table));
            else
                row(int_arith(a, table));
        }
    }
}

template <int BE, int NIN, bool MDR, bool TILED>
hipError_t launch_nin(const NttHead &h, uint32_t log_n, const BconvExtra &b, hipStream_t s) {
#define HE_CASE(LD)                                                                                                              \
    case LD:                                                                                                                     \
        hipLaunchKernelGGL((bconv_rows4_kernel<LD, BE, NIN, MDR, TILED>), dim3(h.h4), dim3(1 << (kTileLog - 2)), 0, s, HE_HEAD_ARGS(h), b); \
        break;
    if constexpr (TILED) {
        switch (log_n - 8) {
            HE_CASE(8)
            default: return hipErrorInvalidValue;
        }
    } else {
        switch (log_n - 8) {
            HE_CASE(4) HE_CASE(5) HE_CASE(6) HE_CASE(7) HE_CASE(8)
            default: return hipErrorInvalidValue;
        }
    }
#undef HE_CASE
    return hipGetLastError();
}

}  // namespace

hipError_t launch_bconv_rows4(const NttHead &head, const BconvRows &b, hipStream_t s) {
    NttHead h = head;
    const uint32_t log_n = h.h0 & 31, groups = (h.h2 & 0xffff) + (h.h2 >> 16);
    const uint64_t wgs = (uint64_t)b.units * (b.items ? b.items : 1) * (1u << (log_n - kTileLog)) * groups;
    if (log_n < 12 || log_n > 16 || b.K == 0 || b.K > 8 || (!b.rows_fp && (!b.mat || (h.fp_mask && !b.rows_mixed))) || wgs == 0 || wgs > most_workgroups(1 << (kTileLog - 2)))
        return hipErrorInvalidValue;
    h.h4 = (uint32_t)wgs;
    const BconvExtra x{b.rows_fp ? static_cast<const void *>(b.rows_fp) : b.mat, b.w, b.copy_base, b.copy_item_stride, b.rows_mixed};
#define HE_TILED(BE, NIN, MDR) (b.tiled ? launch_nin<BE, NIN, MDR, true>(h, log_n, x, s) : launch_nin<BE, NIN, MDR, false>(h, log_n, x, s))
#define HE_NIN(BE, MDR) (b.K <= 4 ? HE_TILED(BE, 4, MDR) : HE_TILED(BE, 8, MDR))
#define HE_MDR(BE) (b.mdr ? HE_NIN(BE, true) : HE_NIN(BE, false))
    if (b.rows_fp) return HE_MDR(NTT_BACKEND_FP);
    // (no limb on FP64: without that branch the kernel needs fewer registers)
    return h.fp_mask ? HE_MDR(NTT_BACKEND_MIXED) : HE_MDR(NTT_BACKEND_INT);
#undef HE_MDR
#undef HE_NIN
#undef HE_TILED
}

}  // namespace he
