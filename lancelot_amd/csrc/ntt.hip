// Batched negacyclic NTT / inverse NTT over RNS limbs for gfx950.
//
// Mathematics (what the CPU oracle and the reference compute; cahel-main/src/ntt/fntt_2d.cu:8-246,
// src/ntt/intt_2d.cu:8-198, src/ntt/butterfly.cuh): forward = log2(N) Cooley-Tukey stages m = 1, 2, ..., N/2
// with twiddle psi^bitrev(m+k) for group k, output in bit-reversed order, canonical residues; inverse =
// the Gentleman-Sande stages in the opposite order including the factor 1/N.
//
// Decomposition for the GPU: N = R x 256.  A limb is an R x 256 row-major matrix.
//   rows pass   : the first log2(R) stages pair elements that are whole rows apart.  A workgroup owns a
//                 tile of R rows x C columns in LDS; global accesses run along the columns (C consecutive words
//                 per row).
//   blocks pass : the last 8 stages stay inside one row (256 consecutive words), which a wave owns.
// The forward transform runs rows pass then blocks pass, the inverse
// the other way round.  The passes, and the inner product, the tensor product, encryption and decryption fused with the blocks pass,
// are in ntt_passes.hip, base conversions fused with the rows pass in ntt_bconv.hip.  This file holds the whole-limb kernel of the
// small degrees and the conversion on the matrix cores, and chooses between them.
//
// Two arithmetic back ends share this skeleton:
//   integer : 64-bit Shoup/Harvey butterflies, any prime below 2^61 (25 VALU instructions per butterfly, 31 back);
//             inverse twiddles are pre-halved so that 1/N comes for free
//   FP64    : exact integer arithmetic in doubles for primes below 2^50 (8 full-rate operations per
//             butterfly, see modarith.cuh); values between the two passes are lazy signed doubles stored
//             in the same 8-byte words; the factor 1/N is folded into the last multiplication
// A launch uses the FP64 back end when every limb it touches has a prime below 2^50, the integer one when none
// has, and otherwise the mixed instantiations, in which every workgroup follows its own limb's prime.
#include <cstdlib>
#include <type_traits>

#include "kernels.h"
#include "modarith.cuh"
#include "ntt_common.cuh"

namespace he {

namespace {

// ---------------------------------------------------------------------------------------------------
// Whole-limb transform for N <= 2^14 (FP64 back end, plain forward / inverse with the optional inverse scaling):
// one workgroup of N / 16 threads per limb keeps the limb in LDS (at most 136 KiB of the CU's 160) between its
// register blocks, so the limb crosses memory once in each direction instead of twice, in one launch instead of two.
// Forward: the first block (stages 0..3, words t + j N/16) comes straight from the coalesced load; the blocks after
// it exchange through LDS (skewed by a word per 16); the last block's results return to LDS for a coalesced store of
// canonical residues.  Inverse: the mirror image, the last block (words t + j N/16) is scaled and stored from
// registers.  LOGN = 4 NB4 + REM: NB4 blocks of four stages and one of REM stages at the fine end.
// ---------------------------------------------------------------------------------------------------
template <int LOGN, bool FWD>
__global__ __launch_bounds__((1 << LOGN) / 16) void ntt_limb_fp_kernel(NttArgs a) {
    constexpr uint32_t N = 1u << LOGN, T = N / 16;
    constexpr int NB4 = LOGN / 4, REM = LOGN % 4, PER = 16 >> REM;
    static_assert(LOGN >= 9 && LOGN <= 14, "a limb of at most 2^14 words");
    __shared__ double ld[N + N / 16];
    const Job job = decode_job(a, blockIdx.x);
    const FpCtx c = fp_ctx(a, job.table);
    const FpMod m = c.m;
    const uint32_t t = threadIdx.x;
    double v[16];
    // block k (stages 4k .. 4k+3) of thread t: words base + (j << low), twiddle index (1 << 4k) + upper
    auto geom = [&](int k, uint32_t &base, uint32_t &low, uint32_t &idx) {
        low = (uint32_t)(LOGN - 4 * (k + 1));
        const uint32_t upper = t >> low;
        base = (upper << (low + 4)) | (t & ((1u << low) - 1));
        idx = (1u << (4 * k)) + upper;
    };
    if (FWD) {
#pragma unroll
        for (int j = 0; j < 16; j++) v[j] = fp_from_u64(job.in[t + T * j]);
        fp_ct_block<4, false>(v, c.tw, 1u, m);
#pragma unroll
        for (int j = 0; j < 16; j++) ld[skew(t + T * j)] = v[j];
        lds_barrier();
#pragma unroll
        for (int k = 1; k < NB4; k++) {
            uint32_t base, low, idx;
            geom(k, base, low, idx);
#pragma unroll
            for (int j = 0; j < 16; j++) v[j] = ld[skew(base + ((uint32_t)j << low))];
            fp_ct_block<4, true>(v, c.tw, idx, m);
#pragma unroll
            for (int j = 0; j < 16; j++) ld[skew(base + ((uint32_t)j << low))] = v[j];
            lds_barrier();
        }
        if constexpr (REM > 0) {
#pragma unroll
            for (int gi = 0; gi < PER; gi++) {
                const uint32_t g = t * PER + gi, base = g << REM;
                double w[1 << REM];
#pragma unroll
                for (int j = 0; j < (1 << REM); j++) w[j] = ld[skew(base + j)];
                fp_ct_block<(REM > 0 ? REM : 1), true>(w, c.tw, (1u << (4 * NB4)) + g, m);
#pragma unroll
                for (int j = 0; j < (1 << REM); j++) ld[skew(base + j)] = w[j];
            }
            lds_barrier();
        }
#pragma unroll
        for (int j = 0; j < 16; j++) job.out[t + T * j] = fp_to_u64(fp_canonical(ld[skew(t + T * j)], m));
    } else {
#pragma unroll
        for (int j = 0; j < 16; j++) ld[skew(t + T * j)] = fp_from_u64(job.in[t + T * j]);
        lds_barrier();
        if constexpr (REM > 0) {
#pragma unroll
            for (int gi = 0; gi < PER; gi++) {
                const uint32_t g = t * PER + gi, base = g << REM;
                double w[1 << REM];
#pragma unroll
                for (int j = 0; j < (1 << REM); j++) w[j] = ld[skew(base + j)];
                fp_gs_block<(REM > 0 ? REM : 1), false>(w, c.tw, (1u << (4 * NB4)) + g, m);
#pragma unroll
                for (int j = 0; j < (1 << REM); j++) ld[skew(base + j)] = w[j];
            }
            lds_barrier();
        }
#pragma unroll
        for (int k = NB4 - 1; k >= 0; k--) {
            uint32_t base, low, idx;
            geom(k, base, low, idx);
#pragma unroll
            for (int j = 0; j < 16; j++) v[j] = ld[skew(base + ((uint32_t)j << low))];
            if (REM == 0 && k == NB4 - 1)
                fp_gs_block<4, false>(v, c.tw, idx, m);   // canonical inputs
            else
                fp_gs_block<4, true>(v, c.tw, idx, m);
            if (k > 0) {
#pragma unroll
                for (int j = 0; j < 16; j++) ld[skew(base + ((uint32_t)j << low))] = v[j];
                lds_barrier();
            }
        }
        // block 0: base = t, low = log2(T): the coalesced store pattern
        const double scale = inverse_scale(a, job, m);
#pragma unroll
        for (int j = 0; j < 16; j++) job.out[t + T * j] = fp_to_u64(fp_canonical(fp_mulmod(v[j], scale, m), m));
    }
}

// The same for N = 2^10 and 2^12 with 4 words a thread (N / 4 threads), on every back end.  What bounds a transform of this size is the
// chain of one workgroup: with 16 words a thread N / 1024 waves a SIMD go through blocks of four stages, each behind a fetch of its 15
// twiddles and a trip of all its words through LDS; here all twiddles are requested together with the words, and only the
// exchanges of more than 256 words (two at 2^12) go through LDS, the others stay in a wave's registers (Tile4).
// Six limbs of 50 bits, forward and inverse, the GPU's time of calls in a row: 2^10 4.39 -> 2.32 and 4.91 -> 2.48 us, 2^12 5.37 -> 4.67 and
// 5.95 -> 4.76; of 60 bits at 2^10, against rows pass and blocks pass, 5.66 -> 3.14 and 5.76 -> 3.46.
template <int LOGN, bool FWD, int BE>
__global__ __launch_bounds__(1 << (LOGN - 2)) void ntt_limb4_kernel(HE_HEAD_PARAMS, const uint64_t *w) {
    using T4 = Tile4<LOGN, LOGN>;
    constexpr int NB = T4::kBlocks;
    __shared__ uint64_t lds[(1 << LOGN) + (1 << (LOGN - 4))];
    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    a.w = w;
    a.epi_mode = h5;
    const Job job = decode_job(a, blockIdx.x);
    const uint32_t t = ((uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) << 6) | (threadIdx.x & 63);
    const bool fp = BE == NTT_BACKEND_FP || (BE == NTT_BACKEND_MIXED && ((a.fp_mask >> job.table) & 1));
    uint64_t x[4];
    // (the forward direction starts from the layout of block 0, words N / 4 apart, and ends with four neighbouring words a thread; the
    // inverse the other way round)
    if (FWD) {
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = job.in[T4::word(0, t, j)];
    } else {
        load4(x, job.in + 4 * t);
    }
    if (BE != NTT_BACKEND_INT && fp) {
        const FpArith ar = fp_arith(a, job.table);
        FpArith::Tw tw[NB];
        T4::template load_tw<FpArith, 0>(tw, ar, 1, t);
        double v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = fp_from_u64(x[j]);
        if (FWD) {
            T4::template forward<FpArith>(v, tw, ar, lds, t);
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = fp_to_u64(fp_canonical(v[j], ar.m));
        } else {
            const double scale = inverse_scale(a, job, ar.m);
            T4::template inverse<FpArith>(v, tw, ar, lds, t);
            ar.template scale<T4::stages(0)>(x, v, scale);
        }
    }
    if constexpr (BE != NTT_BACKEND_FP) {
        if (!fp) {
            const IntArith ar = int_arith(a, job.table);
            const uint64_t q = scalar(a.moduli)[job.table];
            IntArith::Tw tw[NB];
            T4::template load_tw<IntArith, 0>(tw, ar, 1, t);
            if (FWD) {
                T4::template forward<IntArith>(x, tw, ar, lds, t);
#pragma unroll
                for (int j = 0; j < 4; j++) x[j] = reduce_8q(x[j], ar.m);
            } else {
                Shoup w{0, 0};
                if (a.epi_mode == NTT_EPI_MUL) w = scalar_shoup(a.w, job.limb);
                T4::template inverse<IntArith>(x, tw, ar, lds, t);
#pragma unroll
                for (int j = 0; j < 4; j++) x[j] = a.epi_mode == NTT_EPI_MUL ? mul_shoup(x[j], w, q) : reduce_4q(x[j], ar.m);
            }
        }
    }
    if (FWD) {
        store4(job.out + 4 * t, x);
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++) job.out[T4::word(0, t, j)] = x[j];
    }
}

// 4 words a thread or 16 (FP64) at 2^12: 16 waves a limb shorten its chain, 4 issue fewer instructions, which counts once every CU has
// a limb of its own (forward / inverse, us: 6 limbs 4.67 / 4.76 against 5.37 / 5.95, 192 5.64 / 5.67 against 6.18 / 6.72, 576 12.8 / 12.9 against
// 11.9 / 13.4, 960 16.1 / 16.7 against 14.9 / 16.8).
inline bool limb4(const NttArgs &a, int backend, uint32_t n_jobs) {
    return a.log_n == 10 || (a.log_n == 12 && (backend != NTT_BACKEND_FP || n_jobs <= a.cus));
}

template <bool FWD>
hipError_t launch_limbs(const NttArgs &a, uint32_t n_jobs, bool four, int backend, hipStream_t s) {
    if (four) {
        const NttHead head = ntt_head(a, n_jobs, (uint32_t)a.epi_mode);
#define HE_LIMB4(LOGN)                                                                                                                  \
    do {                                                                                                                                \
        const dim3 block((1u << LOGN) / 4);                                                                                             \
        if (backend == NTT_BACKEND_MIXED)                                                                                               \
            hipLaunchKernelGGL((ntt_limb4_kernel<LOGN, FWD, NTT_BACKEND_MIXED>), dim3(n_jobs), block, 0, s, HE_HEAD_ARGS(head), a.w);                         \
        else if (backend)                                                                                                               \
            hipLaunchKernelGGL((ntt_limb4_kernel<LOGN, FWD, NTT_BACKEND_FP>), dim3(n_jobs), block, 0, s, HE_HEAD_ARGS(head), a.w);                            \
        else                                                                                                                            \
            hipLaunchKernelGGL((ntt_limb4_kernel<LOGN, FWD, NTT_BACKEND_INT>), dim3(n_jobs), block, 0, s, HE_HEAD_ARGS(head), a.w);                           \
    } while (0)
        if (a.log_n == 10)
            HE_LIMB4(10);
        else
            HE_LIMB4(12);
#undef HE_LIMB4
        return hipGetLastError();
    }
    switch (a.log_n) {
#define HE_CASE(LOGN) \
    case LOGN: hipLaunchKernelGGL((ntt_limb_fp_kernel<LOGN, FWD>), dim3(n_jobs), dim3((1u << LOGN) / 16), 0, s, a); break;
        HE_CASE(9) HE_CASE(11) HE_CASE(12) HE_CASE(13) HE_CASE(14)
#undef HE_CASE
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// With 4 words a thread one launch does not hold the threads from 2^34 words (137 GB) on: whole polynomials, as many as it holds, go
// into each of several.
template <bool FWD>
hipError_t launch_limb(NttArgs a, uint32_t n_polys, int backend, hipStream_t s) {
    const bool four = limb4(a, backend, n_polys * a.map.limbs);
    const uint32_t per_launch = most_workgroups((1u << a.log_n) / (four ? 4 : 16)) / a.map.limbs;
    for (;;) {
        const uint32_t polys = n_polys < per_launch ? n_polys : per_launch;
        if (hipError_t e = launch_limbs<FWD>(a, polys * a.map.limbs, four, backend, s)) return e;
        n_polys -= polys;
        if (n_polys == 0) return hipSuccess;
        a.in += (size_t)polys * a.in_poly_stride << a.log_n;
        a.out += (size_t)polys * a.out_poly_stride << a.log_n;
    }
}

// The launches that a whole-limb kernel covers and wins; us of one launch against rows pass and blocks pass, forward / inverse.  A limb
// is one workgroup on one CU.  Up to N = 2^12 that is faster on FP64 whatever the number of limbs, or as fast and one launch for the
// host instead of two (2^12, 6 limbs 4.67 / 4.76 against 5.46 / 5.14, 960 14.9 / 16.8 against 21.2 / 22.3; 2^9, 96 limbs 5.0 / 5.6 against 4.6 /
// 4.7, 960 5.2 / 5.8 against 6.2 / 6.0).  A limb of 2^13 or 2^14 words takes one CU longer than two launches of a few limbs take: at 2^13 the
// kernel pays from a limb for every second CU on (96 limbs 9.2 / 10.8 against 8.1 / 8.3, 129 9.5 / 11.1 against 10.2 / 10.6, 192 9.9 / 11.4 against
// 12.1 / 12.3, 960 32.5 / 38.1 against 50.2 / 49.7), at 2^14 from three limbs for every four CUs on in the forward direction (129 limbs 16.0
// against 15.9, 192 17.1 against 19.0, 960 71.4 against 84.4; its inverse, whose first blocks wait for the whole limb, takes 18.7 against 16.7
// with 129 and 63.3 against 54.1 with 576).  Integers take 2.5 times the instructions: one launch at 2^10 always, at 2^12 from five limbs for every
// eight CUs on (6 limbs 7.0 / 7.3 against 6.2 / 6.3, 128 7.6 / 7.9 against 7.5 / 7.6, 192 8.0 / 8.2 against 9.9 / 10.3, 960 24.4 / 25.6 against 29.1 /
// 31.5; 60 and 40 bits, 128 limbs 7.4 / 7.7 against 6.9 / 7.1, 160 7.6 / 7.9 against 7.8 / 7.8).  a.one_pass = 2 forces it (tests).
inline bool one_pass_ok(const NttArgs &a, int backend, bool forward, uint32_t n_jobs) {
    if (!a.one_pass || a.log_n > 14 || a.jobs || a.pro_mode != NTT_PLAIN || a.in_galois ||
        !(a.epi_mode == NTT_PLAIN || (!forward && a.epi_mode == NTT_EPI_MUL)))
        return false;
    if (backend != NTT_BACKEND_FP) return a.log_n == 10 || (a.log_n == 12 && (a.one_pass == 2 || 8 * (uint64_t)n_jobs >= 5 * (uint64_t)a.cus));
    return a.one_pass == 2 || a.log_n <= 12 || (a.log_n == 13 && 2 * (uint64_t)n_jobs >= a.cus) || (a.log_n == 14 && forward && 4 * (uint64_t)n_jobs >= 3 * (uint64_t)a.cus);
}

constexpr int kFuseLog = 11;
constexpr uint32_t kFuseWords = 1u << kFuseLog;


// see the matrix-core kernel below
__device__ __forceinline__ uint32_t swz8(uint32_t e) { return e ^ ((((e >> 5) ^ (e >> 8)) & 3u) << 3); }

// the last two stages of a tile that lives in LDS, 8 words per thread; twl: entries 0..255 of the limb's twiddle table, in LDS;
// the results go to global memory as lazy signed doubles for the blocks pass
__device__ __forceinline__ void fuse_last(const double *ld, const double *twl, FpMod m, uint64_t *dst, uint32_t col0) {
#pragma unroll
    for (int gi = 0; gi < 2; gi++) {
        const uint32_t g = threadIdx.x + 256 * gi, upper = g >> 3, base = (upper << 5) | (g & 7);
        double v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = ld[swz8(base + ((uint32_t)j << 3))];
        fp_ct_block<2, 1>(v, twl, 64u + upper, m);   // (at most 1.8 q: see FpArith)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t e = base + ((uint32_t)j << 3);
            dst[(size_t)(e >> 3) * 256 + col0 + (e & 7)] = (uint64_t)__double_as_longlong(v[j]);
        }
    }
}

// a value that every lane of the wave holds (read from LDS with one address) as a scalar
__device__ __forceinline__ double uniform_f64(double v) {
    const long long b = __double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b), hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// output limbs per workgroup, at most (the LDS arrays of the rows' constants have this many entries; their loader
// strides over the workgroup, whatever its size)
constexpr uint32_t kFuseMaxRows = 24;

// ---------------------------------------------------------------------------------------------------
// Base conversion fused with the rows pass of the transform that follows it (ntt_bconv.hip) at N = 2^16, with the matrix product of
// the conversion on the int8 matrix cores.
//
// sum_i x_i M[r][i] mod q_r is a 64-term integer product per 7-bit digit of the constants M_ij = M[r][i] 2^(8 j) mod q_r,
// over the bytes x_ij of the inputs as they lie in memory (BconvRows::mx_tab).  One v_mfma_i32_16x16x64_i8 forms it for 16
// coefficients, four output rows and four digits; two of them (digits 0..3, 4..7) leave the 8 digit sums S_e < 2^21 of
// (row rr, coefficient c) in lane 16 rr + c, and
//     sum_e S_e 2^(7 e) = lo + 2^28 hi,   lo = S_0 + 2^7 S_1 + 2^14 S_2 + 2^21 S_3 < 2^43,  hi likewise,
// becomes the lazy residue (hi x (2^28 mod q)) mod q + lo with one modular product: 13 FP64-rate operations and two
// matrix instructions per word against 44 operations for the eight exact multiply-adds on the vector units.  (When it runs: see
// launch_bconv_rows.)
//
// Wave w of the workgroup owns the coefficients of rows w + 4 j + 32 i (j, i < 8) of the 256 x 8 tile; lane (kg, c) keeps the words of input limbs 2 kg, 2 kg + 1 for coefficient c of each of 32 sets of 16
// coefficients (set (g, i): (j, column) = (2 g + c / 8, c % 8), row w + 4 j + 32 i), which is at once the B operand of the
// set.  Output rows go four at a time: lane (rr, c) receives row rr's words of every set, i.e. for each g the 8 words
// i = 0..7 of one first register block, runs the block on them and stores them to row rr's tile in LDS.  The second block
// (stages 3..5) stays inside the wave tile by tile, the third follows a workgroup barrier.
//
// LDS index of tile word e = (row << 3) | column: bits 4..3 are XORed with bits 6..5 and bits 9..8.  The accesses of
// a half-wave vary the column and either bit 5 (first block), bits 9..8 (second) or bits 6..5 (third) with bits 4..3
// fixed, so they fall into distinct 8-byte banks; consecutive tiles start 16 words apart modulo 32, which separates the
// two output rows that the lanes of a half-wave store in the first block.
// ---------------------------------------------------------------------------------------------------
typedef int v4i __attribute__((ext_vector_type(4)));
constexpr uint32_t kMxStride = kFuseWords + 16;

template <bool MDR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void bconv_rows_mx_kernel(HE_HEAD_PARAMS, BconvExtra b) {
    __shared__ double tiles[4 * kMxStride];
    __shared__ double twl[4][256];
    __shared__ double rconst[2][4][4];         // per group parity and row: q, 1/q, the constant that the digit sums lack
    __shared__ uint32_t rlimb[2][4];
    __shared__ uint32_t rtable[kFuseMaxRows + 4];
    constexpr int LOGC = 3;
    constexpr uint32_t tiles_per_limb = 32;

    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    uint32_t lb = logical_block(h4);
    const uint32_t compute_groups = h2 & 0xffff, groups = compute_groups + (h2 >> 16), rows_per = h5;
    const uint32_t grp = lb % groups;
    lb /= groups;
    const BconvUnit d = bconv_unit(a, h1 & 0xffff, h1 >> 16, lb / tiles_per_limb);
    const uint32_t col0 = (lb % tiles_per_limb) << LOGC;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, kg = lane >> 4, cn = lane & 15;
    uint64_t *out = d.out;

    if (grp >= compute_groups) {
        // limbs that pass through unchanged (a digit's own limbs keep their NTT form)
        const uint64_t *from = b.copy_base + d.item * b.copy_item_stride;
        const uint32_t first = (grp - compute_groups) * rows_per;
        const size_t g0 = (size_t)(threadIdx.x >> LOGC) * 256 + col0 + (threadIdx.x & 7);
        for (uint32_t r = first; r < first + rows_per && r < d.n_in; r++) {
            const size_t limb = (size_t)(d.copy_first + r) << 16;
            uint64_t w[8];
#pragma unroll
            for (int i = 0; i < 8; i++) w[i] = from[limb + g0 + (size_t)i * 32 * 256];
#pragma unroll
            for (int i = 0; i < 8; i++) out[limb + g0 + (size_t)i * 32 * 256] = w[i];
        }
        return;
    }
    const uint32_t n_rows = MDR ? d.n_out - 1 : d.n_out;
    const uint32_t r_begin = grp * rows_per;
    const uint32_t r_end = r_begin + rows_per < n_rows ? r_begin + rows_per : n_rows;
    if (r_begin >= n_rows) return;

    // the tables of this workgroup's rows (rows past the end repeat the last one; they are computed and not stored)
    if (threadIdx.x < kFuseMaxRows + 4) {
        const uint32_t r = r_begin + threadIdx.x < r_end ? r_begin + threadIdx.x : r_end - 1;
        rtable[threadIdx.x] = map_table(a.map, d.limb(r));
    }
    // the inputs: bytes 0..6 as signed numbers (x - 128), byte 7 (zero: the residues are below 2^50) stays zero
    const uint64_t *x = d.in;
    const uint32_t l0 = 2 * kg < d.n_in ? 2 * kg : d.n_in - 1, l1 = 2 * kg + 1 < d.n_in ? 2 * kg + 1 : d.n_in - 1;
    // (a uniform base and 32-bit byte offsets: one address register per load in flight instead of two)
    const char *xbytes = reinterpret_cast<const char *>(x);
    int xb[32][4];   // (scalars: the merged mode rewrites single bytes of them in place)
    auto operand = [&](int s) { return v4i{xb[s][0], xb[s][1], xb[s][2], xb[s][3]}; };
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const uint32_t G = cn + 16 * g;
        const uint32_t o = ((wave + 4 * (G >> 3)) * 256 + (G & 7) + col0) * 8;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t oi = o + (uint32_t)i * (32 * 256 * 8);
            const uint64_t u0 = *reinterpret_cast<const uint64_t *>(xbytes + ((l0 << 19) + oi)) ^ 0x0080808080808080ull;
            const uint64_t u1 = *reinterpret_cast<const uint64_t *>(xbytes + ((l1 << 19) + oi)) ^ 0x0080808080808080ull;
            xb[8 * g + i][0] = (int)(uint32_t)u0;
            xb[8 * g + i][1] = (int)(uint32_t)(u0 >> 32);
            xb[8 * g + i][2] = (int)(uint32_t)u1;
            xb[8 * g + i][3] = (int)(uint32_t)(u1 >> 32);
        }
    }
    if (MDR) {
        // merged ModDown + rescale: r = (t - sum_i x_i M[last][i]) mod q_last, canonical, is added to every output row;
        // its bytes 0..6 go into byte 7 of the words of limbs 0..6, where the rows' records hold the digits of 2^(8 i).
        // The record of the dropped row repeats it in all four row slots, so that every lane holds r of its coefficient.
        // t, the limb before the unit's inputs, crosses LDS (the tiles are not in use yet): fetched per lane where it is
        // needed, its 32 words would wait in registers beside the inputs.
        {
            const uint64_t *tsrc = x - ((size_t)1 << 16) + col0 + (size_t)(threadIdx.x >> LOGC) * 256 + (threadIdx.x & 7);
            uint64_t *tl = reinterpret_cast<uint64_t *>(tiles);
            uint64_t tw[8];
#pragma unroll
            for (int i = 0; i < 8; i++) tw[i] = tsrc[(size_t)i * 32 * 256];
#pragma unroll
            for (int i = 0; i < 8; i++) tl[threadIdx.x + 256 * i] = tw[i];   // tile word (row << 3) | column
        }
        lds_barrier();
        const uint32_t ltable = map_table(a.map, d.n_out - 1);
        const FpMod ml{a.fp_consts[4 * (size_t)ltable], a.fp_consts[4 * (size_t)ltable + 1]};
        const v4i *lrec = static_cast<const v4i *>(b.w);
        const v4i la = lrec[lane], lh = lrec[64 + lane];
        const double *loff = reinterpret_cast<const double *>(lrec + 128);
        const double off = loff[0];
        const double c28 = fp_reduce(0x1p28, ml);
        const uint64_t *tl = reinterpret_cast<const uint64_t *>(tiles);
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const uint32_t G = cn + 16 * g;
            const uint32_t e = ((wave + 4 * (G >> 3)) << LOGC) | (G & 7);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const v4i zero = {0, 0, 0, 0};
                const v4i lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(la, operand(8 * g + i), zero, 0, 0, 0);
                const v4i hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(lh, operand(8 * g + i), zero, 0, 0, 0);
                const int l01 = lo.x + lo.y * 128, l23 = lo.z + lo.w * 128;
                const int h01 = hi.x + hi.y * 128, h23 = hi.z + hi.w * 128;
                const double ld = __builtin_fma((double)l23, 16384.0, (double)l01) + off;
                const double hd = __builtin_fma((double)h23, 16384.0, (double)h01);
                const double t = fp_from_u64(tl[e + ((uint32_t)(32 * i) << LOGC)]);
                const uint64_t r = fp_to_u64(fp_canonical(t - (fp_mulmod(hd, c28, ml) + ld), ml));
                const uint32_t b0 = (uint32_t)(r >> (16 * kg)) & 0xffu, b1 = (uint32_t)(r >> (16 * kg + 8)) & 0xffu;
                // (in place: as a new value in the source, the compiler keeps the old and the new operand beside each other,
                // 32 times four registers)
                asm volatile("v_or_b32 %0, %0, %1" : "+v"(xb[8 * g + i][1]) : "v"((b0 ^ 0x80u) << 24));
                asm volatile("v_or_b32 %0, %0, %1" : "+v"(xb[8 * g + i][3]) : "v"((b1 ^ 0x80u) << 24));
            }
        }
        lds_barrier();   // the tiles are free again
    }
    const v4i *rec = static_cast<const v4i *>(b.mat) + ((size_t)d.mx_off + (r_begin >> 2)) * kMxRecord;
    lds_barrier();   // rtable

    // Twiddles: entries 1..63 of a row's table serve the first two blocks, 64..255 the third.  Thread t fetches entry
    // t % 64 of row t / 64 for the first part and entries 64 + t % 64 + 64 c (c < 3) of that row for the second.
    const uint32_t trow = threadIdx.x >> 6, tcol = threadIdx.x & 63;
    auto low_part = [&](uint32_t k) {   // group k of this workgroup: (entry tcol of row trow, that row's constants)
        return a.tw_fp[((size_t)rtable[4 * k + trow] << 16) + tcol];
    };
    auto stage_consts = [&](uint32_t k, const v4i *rc) {
        if (threadIdx.x < 16) {
            const uint32_t rr = threadIdx.x >> 2, c = threadIdx.x & 3;
            const double *off = reinterpret_cast<const double *>(rc + 128);
            rconst[k & 1][rr][c] = c < 2 ? a.fp_consts[4 * (size_t)rtable[4 * k + rr] + c] : off[2 * rr + (c - 2)];
        }
        if (threadIdx.x >= 16 && threadIdx.x < 20) {
            const uint32_t rr = threadIdx.x - 16;
            const uint32_t r = r_begin + 4 * k + rr < r_end ? r_begin + 4 * k + rr : r_end - 1;
            rlimb[k & 1][rr] = d.limb(r);
        }
    };
    twl[trow][tcol] = low_part(0);
    stage_consts(0, rec);
    lds_barrier();

    // a group's matrix digits (from L2: every workgroup of the unit reads the same ones); the next group's are requested
    // as soon as the first block has issued its last product
    v4i alo = rec[lane], ahi = rec[64 + lane];
    uint32_t k = 0;
    for (uint32_t r0 = r_begin; r0 < r_end; r0 += 4, rec += kMxRecord, k++) {
        const uint32_t nr = r_end - r0 < 4 ? r_end - r0 : 4;
        const bool more = r0 + 4 < r_end;
        {
            // first block, lane (rr, c) on row rr = kg
            const FpMod mod{rconst[k & 1][kg][0], rconst[k & 1][kg][1]};
            const double off = rconst[k & 1][kg][2];
            const double c28 = fp_reduce(0x1p28, mod);
            const double *tws = twl[kg];
            double *tile_ld = tiles + kg * kMxStride;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                // (opaque: computed once for the whole loop, the 32 store addresses would occupy registers through all of it)
                uint32_t cn_ = cn;
                asm volatile("" : "+v"(cn_));
                const uint32_t G = cn_ + 16 * g;
                const uint32_t z = swz8(((wave + 4 * (G >> 3)) << LOGC) | (G & 7));
                double v[8];
                // (the products of set i + 1 are issued before set i's are taken up: the matrix cores need 16 cycles each)
                const v4i zero = {0, 0, 0, 0};
                v4i lo_next = __builtin_amdgcn_mfma_i32_16x16x64_i8(alo, operand(8 * g), zero, 0, 0, 0);
                v4i hi_next = __builtin_amdgcn_mfma_i32_16x16x64_i8(ahi, operand(8 * g), zero, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const v4i lo = lo_next, hi = hi_next;
                    if (i < 7) {
                        lo_next = __builtin_amdgcn_mfma_i32_16x16x64_i8(alo, operand(8 * g + i + 1), zero, 0, 0, 0);
                        hi_next = __builtin_amdgcn_mfma_i32_16x16x64_i8(ahi, operand(8 * g + i + 1), zero, 0, 0, 0);
                    }
                    // signed digit sums (the bytes entered as x - 128): |S| < 2^21, the pairs below 2^29, lo and hi exact
                    const int l01 = lo.x + lo.y * 128, l23 = lo.z + lo.w * 128;
                    const int h01 = hi.x + hi.y * 128, h23 = hi.z + hi.w * 128;
                    const double ld = __builtin_fma((double)l23, 16384.0, (double)l01) + off;
                    const double hd = __builtin_fma((double)h23, 16384.0, (double)h01);
                    // |v| <= (1/2 + 2^-8) q + 2^44 + q: within the 4 x 2^50 that the register blocks of this pass start from
                    v[i] = fp_mulmod(hd, c28, mod) + ld;
                }
                fp_ct_block<3, 2>(v, tws, 1u, mod);
                // word i is 32 i rows further: bits 10..8 of the tile index, of which the slot takes bits 9..8 into bits 4..3
#pragma unroll
                for (int i = 0; i < 8; i++) tile_ld[z ^ (uint32_t)(((i & 3) << 3) | (i << 8))] = v[i];
            }
        }
        if (more) {
            alo = rec[kMxRecord + lane];
            ahi = rec[kMxRecord + 64 + lane];
        }
        // the twiddles of the third block travel during the second
        double tw_hi[3];
#pragma unroll
        for (int c = 0; c < 3; c++) tw_hi[c] = a.tw_fp[((size_t)rtable[4 * k + trow] << 16) + 64 + tcol + 64 * c];
        // stages 3..5 inside the wave, tile by tile: lane (u, col) takes rows 32 u + 4 j + wave, which lanes of this wave wrote
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        {
            // (all four tiles, also those of rows past the end: the words of the next tile are read before the block of
            // the current one runs)
            const uint32_t u = lane >> 3;
            const uint32_t base = ((32 * u + wave) << LOGC) + (lane & 7);
            double vn[8];
#pragma unroll
            for (int j = 0; j < 8; j++) vn[j] = tiles[swz8(base + ((uint32_t)(4 * j) << LOGC))];
#pragma unroll
            for (int rr = 0; rr < 4; rr++) {
                const FpMod mod{uniform_f64(rconst[k & 1][rr][0]), uniform_f64(rconst[k & 1][rr][1])};
                double *tile_ld = tiles + rr * kMxStride;
                double v[8];
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = vn[j];
                if (rr < 3) {
#pragma unroll
                    for (int j = 0; j < 8; j++) vn[j] = tile_ld[kMxStride + swz8(base + ((uint32_t)(4 * j) << LOGC))];
                }
                fp_ct_block<3, 2>(v, twl[rr], 8u + u, mod);
#pragma unroll
                for (int j = 0; j < 8; j++) tile_ld[swz8(base + ((uint32_t)(4 * j) << LOGC))] = v[j];
            }
        }
        // (the third block of the previous group, the last reader of these entries, ended before that group's last barrier)
#pragma unroll
        for (int c = 0; c < 3; c++) twl[trow][64 + tcol + 64 * c] = tw_hi[c];
        lds_barrier();
        // the next group's first twiddles and constants travel during the third block
        double tw_lo = 0.0;
        if (more) tw_lo = low_part(k + 1);
        for (uint32_t rr = 0; rr < nr; rr++) {
            const FpMod mod{uniform_f64(rconst[k & 1][rr][0]), uniform_f64(rconst[k & 1][rr][1])};
            const uint32_t limb = __builtin_amdgcn_readfirstlane(rlimb[k & 1][rr]);
            fuse_last(tiles + rr * kMxStride, twl[rr], mod, out + ((size_t)limb << 16), col0);
        }
        if (more) {
            // entries 0..63 were last read by the second block, before the barrier above
            twl[trow][tcol] = tw_lo;
            stage_consts(k + 1, rec + kMxRecord);
        }
        lds_barrier();  // every read of the tiles is done before the next four rows overwrite them
    }
}

}  // namespace

// The matrix-core kernel (N = 2^16) multiplies 8 input limbs deep whatever there are, takes the output rows four at a time and two
// workgroups to a CU: it pays from five limbs on, and once the tiles alone give every CU a workgroup.  us with it / without, all of
// a multiplication: K = 8, L = 24: one 140.0 / 139.0, two 241.5 / 241.4, three 338.8 / 340.6, four 422 / 436, eight 805 / 840;
// K = 6, L = 30: one 203.0 / 201.2; K = 4, L = 12: one 80.8 / 74.4, two 129.7 / 124.4, eight 410 / 403.  (Merged ModDown +
// rescale, K = 8: eight 106 / 122 us.)
static bool bconv_on_matrix_cores(uint32_t log_n, const BconvRows &b, const Tuning &tune) {
    return log_n == 16 && b.rows_fp && b.mx_tab && !b.tiled && !tune.no_matrix_bconv && b.K > 4 && (!b.mdr || b.mx_last) &&
           ((uint64_t)b.units * (b.items ? b.items : 1) << (log_n - kFuseLog)) >= (tune.cus ? tune.cus : 256);
}

// Tiled inputs (conversion_word): what a workgroup of the vector kernel fetches first, 64 KB to 144 KB, lay in segments of 64 bytes at N = 2^16,
// which took 10 us of a launch's 28 with all workgroups at it.  The rows pass before it needs a buffer to leave them in, whose lines no cache
// holds yet; that costs rotations what they gain while there are few limbs, and batches past 64 limbs, whose words go past the caches.  us
// natural / tiled, n = 2^16, L + K limbs.  Rotation 24 + 8 113.1 / 108.8, 16 + 8 78.4 / 75.1, 8 + 8 50.9 / 49.1, 10 + 3 65.7 / 64.7, 16 + 2 105.0 /
// 103.5, 8 + 2 52.9 / 53.2, 6 + 4 43.6 / 44.4; hoisting 24 + 8 238.6 / 235.6; 60 / 40 bits: rotation 24 + 8 157.3 / 153.2, 8 + 2 65.4 / 64.2, 8 + 3
// 63.7 / 62.1, 6 + 4 55.1 / 54.0, 3 + 8 52.1 / 53.5.  Products, limbs x items: 24 + 8 136.9 / 132.1, 16 + 8 94.6 / 90.5, 9 + 3 55.9 / 53.8, 12 + 4 x 2
// 111.8 / 108.8, x 3 151.3 / 148.7, x 4 182.1 / 180.5, x 5 240 / 242, 16 + 4 x 3 201 / 197, x 4 252 / 254, 9 + 3 x 4 141.8 / 141.3; 60 / 40 bits 12 + 4
// x 4 244.4 / 245.9, x 6 366 / 367; 60 bits x 4 292.7 / 292.7.  Products that would gain below the lower line, which is the rotations': 8 + 2 55.3 /
// 53.2, x 4 139.9 / 137.1, x 6 201 / 195, 6 + 2 x 4 105.4 / 100.0, but 6 + 3 x 4 98.5 / 98.3; 60 / 40 bits 6 + 2 63.6 / 62.0, x 4 138.8 / 137.3, but 6 +
// 3 x 4 129.6 / 131.9.  At 2^15 the segments are whole lines already: rotation 24 + 8 68.0 / 67.3, 10 + 3 43.7 / 44.6.
bool bconv_wants_tiles(const NttArgs &inv, int inv_backend, const BconvRows &b, const Tuning &tune) {
    const uint32_t limbs = b.map.limbs, items = b.items ? b.items : 1;
    if (inv.log_n != 16 || b.map.split < 6 || limbs < (b.rows_fp ? 12 : 10) || (uint64_t)limbs * items > 64) return false;
    return !bconv_on_matrix_cores(inv.log_n, b, tune) && (b.rows_fp != nullptr) == (inv_backend == NTT_BACKEND_FP);
}

hipError_t launch_bconv_rows(const NttArgs &a, const BconvRows &b, int backend, const Tuning &tune, hipStream_t s) {
    if (a.log_n < 12 || a.log_n > 16 || b.units == 0 || b.K == 0 || b.K > 8) return hipErrorInvalidValue;
    const uint32_t forced = tune.fuse_rows_forced <= kFuseMaxRows ? tune.fuse_rows_forced : 0;
    const uint32_t items = b.items ? b.items : 1;
    const int ld = (int)a.log_n - 8;
    const uint32_t tiles = 256u >> (kFuseLog - ld);
    // (the most of a unit: ModUp, the last digit's)
    const uint32_t L = b.map.split, last = L % b.K ? L % b.K : b.K;
    const uint32_t rows = b.up ? b.map.limbs - last : b.mdr ? L - 1 : L;
    if (rows == 0) return hipErrorInvalidValue;
    const uint32_t cus = tune.cus ? tune.cus : 256;
    const bool mx = bconv_on_matrix_cores(a.log_n, b, tune);
    // Output limbs per workgroup.  The kernel is bound by instruction issue, so a CU's time is the number of workgroups it is dealt
    // times a workgroup's work: r rows plus the fetching of the inputs and setting up, one row's worth and a half with 4 waves and a
    // tile of 8 words per thread; with 8 waves and 4 words half a row's with eight inputs and K / 16 of one with up to four (K / 20 on
    // integers, whose rows take longer).  Few rows per workgroup pay that often, many leave CUs with one workgroup more than others.  A CU
    // with a single workgroup has fewer waves to cover its waits with: as much as two take (4 waves), 15 % (8 waves, 10 % on
    // integers), and some of it where an odd number leaves one for the end.  Measured at n = 2^16 (8 waves, inputs in their own order), us
    // with 1, 2, 3, 4, 5, 6, 8 rows a workgroup: K = 8, 24 rows for 96 tiles 32.0, 25.0, 24.0, 31.3, 25.5, 28.7, 34.2; 23 rows for 64 tiles 26.0,
    // 23.6, 21.0, 25.3, 27.6, 22.5, 27.0; 16 rows for 64 15.5, 14.6, 16.4, 15.0, 16.5, 17.4, 21.4; K = 4, 12 rows for 96 tiles 13.4, 14.2, 14.4, 16.2,
    // 18.1, 16.0, 18.8; 12 for 64 9.6, 11.0, 10.5, 11.6, -, 14.2; 24 for 192 39.0, 35.4, 33.0, 34.1, 35.2, 35.3, 39.0; integers, K = 4, 12 rows for 96
    // 19.3, 20.4, 21.6, 24.8, 26.3, 23.2, 25.2; n = 2^15, K = 3, 12 for 64 14.0, 14.4, 13.7, 15.0, 18.1, 18.8, 22.3.  Against half a row's set-up for every
    // K: rotations, n = 2^16, 12 + 4 limbs 63.4 / 62.8 us, 9 of 12 + 4 59.8 / 58.6, of 60 / 40 bits 79.2 / 77.0, 73.4 / 71.0, 16 + 8 102.3 / 100.1.
    const uint32_t step = mx ? 4 : 1;
    uint32_t target = mx ? (forced + 3) / 4 * 4 : forced;
    if (!target) {
        uint64_t best = ~0ull;
        const uint32_t set_up = b.K > 4 ? 40 : b.rows_fp ? 5 * b.K : 4 * b.K, alone = b.rows_fp ? 23 : 22, odd = b.rows_fp ? 3 : 1;
        for (uint32_t r = step; r <= kFuseMaxRows && r < rows + step; r += step) {
            const uint64_t wgs = (uint64_t)b.units * items * tiles * ((rows + r - 1) / r);
            const uint64_t per_cu = (wgs + cus - 1) / cus;
            const uint64_t cost = mx ? (per_cu < 2 ? 2 : per_cu) * (2 * r + 3)
                                     : (per_cu < 2 ? alone : 20 * per_cu + (per_cu & 1 ? odd : 0)) * (80 * r + set_up);
            if (cost < best) {
                best = cost;
                target = r;
            }
        }
    }
    const uint32_t compute_groups = (rows + target - 1) / target, copy_groups = b.copy_base ? ((L < b.K ? L : b.K) + target - 1) / target : 0;
    const uint64_t wgs = (uint64_t)b.units * items * tiles * (compute_groups + copy_groups);
    if (wgs > most_workgroups(256)) return hipErrorInvalidValue;
    NttArgs m = a;
    m.in = b.in;
    m.out = b.out;
    m.map = b.map;
    m.pro_mode = b.up;
    if (!b.rows_fp) m.fp_mask = backend == NTT_BACKEND_INT ? 0 : backend == NTT_BACKEND_FP ? ~(uint64_t)0 : a.fp_mask;
    NttHead h = ntt_head(m, (uint32_t)wgs, target);
    h.h1 = b.units | b.K << 16;
    h.h2 = compute_groups | copy_groups << 16;
    if (mx) {
        const BconvExtra x{b.mx_tab, b.mx_last, b.copy_base, b.copy_item_stride, nullptr};
        if (b.mdr)
            hipLaunchKernelGGL(bconv_rows_mx_kernel<true>, dim3(h.h4), dim3(256), 0, s, HE_HEAD_ARGS(h), x);
        else
            hipLaunchKernelGGL(bconv_rows_mx_kernel<false>, dim3(h.h4), dim3(256), 0, s, HE_HEAD_ARGS(h), x);
        return hipGetLastError();
    }
    return launch_bconv_rows4(h, b, s);
}

hipError_t launch_ntt_forward(const NttArgs &a, uint32_t n_polys, int backend, hipStream_t s, bool rows_done) {
    if (a.log_n < 9 || a.log_n > 17 || backend < NTT_BACKEND_INT || backend > NTT_BACKEND_MIXED) return hipErrorInvalidValue;
    const uint32_t n_jobs = a.jobs ? a.n_jobs * (a.items ? a.items : 1) : n_polys * a.map.limbs;
    if (n_jobs == 0) return hipSuccess;
    if (!rows_done && one_pass_ok(a, backend, true, n_jobs)) return launch_limb<true>(a, n_polys, backend, s);
    const hipError_t e = rows_done ? hipSuccess : launch_ntt_rows(a, n_jobs, true, backend, s);
    return e != hipSuccess ? e : launch_ntt_blocks(a, n_polys, true, backend, s);
}

hipError_t launch_ntt_inverse(const NttArgs &a, uint32_t n_polys, int backend, hipStream_t s, bool blocks_done,
                              bool rows_skipped) {
    if (a.log_n < 9 || a.log_n > 17 || backend < NTT_BACKEND_INT || backend > NTT_BACKEND_MIXED) return hipErrorInvalidValue;
    const uint32_t n_jobs = a.jobs ? a.n_jobs * (a.items ? a.items : 1) : n_polys * a.map.limbs;
    if (n_jobs == 0) return hipSuccess;
    if (!blocks_done && !rows_skipped && one_pass_ok(a, backend, false, n_jobs)) return launch_limb<false>(a, n_polys, backend, s);
    const hipError_t e = blocks_done ? hipSuccess : launch_ntt_blocks(a, n_polys, false, backend, s);
    if (e != hipSuccess || rows_skipped) return e;
    NttArgs rows = a;
    rows.in = a.out;  // the rows pass continues in place on the output buffer
    rows.in_poly_stride = a.out_poly_stride;
    if (a.tiles) {
        rows.out = a.tiles;
        rows.out_poly_stride = a.tiles_poly_stride;
    }
    return launch_ntt_rows(rows, n_jobs, false, backend, s);
}

}  // namespace he
