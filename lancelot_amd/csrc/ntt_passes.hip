// The two passes of the transform (ntt.hip's header says how a limb splits into them), 4 words per thread.
//
// What bounds a pass is how many waves a SIMD has to switch between while loads, twiddle look-ups and LDS exchanges are on
// their way, so a thread holds little: 4 words, its twiddles (at most 12, requested together with the words) and no more, 52
// to 110 registers, 4 to 8 waves per SIMD.  The stages run as register blocks of two; the exchanges between them, all of
// a blocks pass's and all but the first (two for 2048-word tiles) of a rows pass's, stay inside one wave and move words between its
// lanes in registers; the others go through LDS.  Passes with 16 words per thread (radix-16 blocks, half the LDS exchanges, at most 2 waves per SIMD on
// FP64 and 3 on integers), which this layout replaced, measured against it: 2 x 24 limbs at N = 2^16 30.0 against 27.3 us
// (50 bits) and 43.5 against 37.5 us (60 bits), 8 x 24 limbs of 60 bits 139 against 112 us, 12 x 24 of 50 bits the same
// 112 us (5.3 TB/s: the two trips through memory), 2 limbs at N = 2^13 9.8 against 8.1 us (50 bits) and 13 against 8.5 us
// (60 bits).
#include <hip/hip_runtime.h>

#include <cstring>
#include <type_traits>

#include "chacha.cuh"
#include "kernels.h"
#include "modarith.cuh"
#include "ntt_common.cuh"

namespace he {

namespace {

// What a rows pass's mode needs behind NttHead.
struct RowsExtra {
    const uint64_t *p0, *p1, *p2;   // inverse: w; NTT_PRO_SOURCE_[INTT_|SMALL_]REDUCE: pro_itw or pro_values, pro_small; NTT_PRO_MODDOWN_RESCALE: pro_src, pro_src2 (or pro_itw), pro_w
    uint64_t u0, u1, mask;          // list: item_stride, pro_item_stride; NTT_PRO_ROUND, NTT_PRO_SOURCE_SMALL_REDUCE: pro_fix (, pro_log_slots); NTT_PRO_MODDOWN_RESCALE: strides, pro_last and pro_k1
    uint32_t w0;                    // inverse: epi_mode; NTT_PRO_SOURCE_[INTT_|SMALL_]REDUCE in map mode: pro_src_table
};

RowsExtra rows_extra(const NttArgs &a, bool fwd) {
    RowsExtra e{nullptr, nullptr, nullptr, a.item_stride, a.pro_item_stride, a.pro_src_fp_mask, 0};
    if (!fwd) {
        e.p0 = a.w;
        e.w0 = (uint32_t)a.epi_mode;
    } else if (a.pro_mode == NTT_PRO_SOURCE_SMALL_REDUCE) {
        e.p0 = reinterpret_cast<const uint64_t *>(a.pro_values);
        e.p1 = reinterpret_cast<const uint64_t *>(a.pro_small);
        memcpy(&e.u0, &a.pro_fix, sizeof(e.u0));
        e.u1 = a.pro_log_slots;
        e.w0 = a.pro_src_table;
    } else if (a.pro_mode == NTT_PRO_SOURCE_INTT_REDUCE) {
        e.p0 = a.pro_itw;
        e.p1 = reinterpret_cast<const uint64_t *>(a.pro_small);
        e.w0 = a.pro_src_table;
    } else if (a.pro_mode == NTT_PRO_MODDOWN_RESCALE && a.pro_itw) {
        e.p0 = a.pro_src;
        e.p1 = a.pro_itw;
        e.p2 = a.pro_w;
        e.u0 = a.pro_poly_stride;
        e.u1 = a.pro_last;
        e.w0 = a.pro_src_table;
    } else if (a.pro_mode == NTT_PRO_MODDOWN_RESCALE) {
        e.p0 = a.pro_src;
        e.p1 = a.pro_src2;
        e.p2 = a.pro_w;
        e.u0 = a.pro_poly_stride | (uint64_t)a.pro2_poly_stride << 32;
        e.u1 = a.pro_last | (uint64_t)a.pro_k1 << 32;
    } else if (a.pro_mode == NTT_PRO_ROUND) {
        memcpy(&e.u0, &a.pro_fix, sizeof(e.u0));
    }
    return e;
}

template <bool FWD, bool SRC_INTT, bool MDR>
__device__ __forceinline__ void set_extra(NttArgs &a, const RowsExtra &e) {
    a.epi_mode = FWD ? NTT_PLAIN : (int)e.w0;
    a.w = FWD ? nullptr : e.p0;
    a.item_stride = e.u0;
    a.pro_item_stride = e.u1;
    a.pro_fix = __longlong_as_double((long long)e.u0);
    a.pro_small = reinterpret_cast<const int8_t *>(e.p1);
    a.pro_values = reinterpret_cast<const double *>(e.p0);
    a.pro_log_slots = (uint32_t)e.u1;
    if constexpr (FWD && !MDR) a.pro_src_table = e.w0;
    if constexpr (SRC_INTT) {
        set_inverse_block(a, MDR ? e.p1 : e.p0);
        a.pro_src_fp_mask = e.mask;
        a.pro_src_table = e.w0;
    }
    if constexpr (MDR && SRC_INTT) {
        // (the special limb lies behind the dropped one)
        a.pro_src = e.p0;
        a.pro_src2 = e.p0 + ((size_t)1 << a.log_n);
        a.pro_w = e.p2;
        a.pro_poly_stride = a.pro2_poly_stride = (uint32_t)e.u0;
        a.pro_last = (uint32_t)e.u1;
        a.pro_k1 = 1;
    } else if constexpr (MDR) {
        a.pro_src = e.p0;
        a.pro_src2 = e.p1;
        a.pro_w = e.p2;
        a.pro_poly_stride = (uint32_t)e.u0;
        a.pro2_poly_stride = (uint32_t)(e.u0 >> 32);
        a.pro_last = (uint32_t)e.u1;
        a.pro_k1 = (int)(e.u1 >> 32);
    }
}

// The inverse rows pass of a source limb's tile: lazy words of the last block's layout become canonical coefficients in the first
// block's.  (Behind the request of the forward twiddles: the exchanges' compiler barriers would hold that back until the inverse
// pass has ended.)
// behind: requests what is needed after the pass (loads return in order: in front of the twiddles, the pass would wait for them)
template <class T4, class Behind>
__device__ __forceinline__ void source_words(uint64_t (&s)[4], const NttArgs &a, uint32_t st, uint64_t *lds, uint32_t t, Behind &&behind) {
    constexpr int NB = T4::kBlocks;
    if ((a.pro_src_fp_mask >> st) & 1) {
        const FpArith ar{fp_ctx(a, st).m, a.pro_itw_fp + ((size_t)st << a.log_n)};
        double v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = FpArith::from_word(s[j]);
        FpArith::Tw tw[NB];
        T4::template load_tw<FpArith, 0>(tw, ar, 1, t);
        behind();
        T4::template inverse<FpArith>(v, tw, ar, lds, t);
        const ScalarF64 cc = scalar(a.fp_consts) + 4 * (size_t)st;
        const double ninv = cc[2];
        ar.template scale<T4::stages(0)>(s, v, ninv);
    } else {
        const uint64_t q = scalar(a.moduli)[st];
        const IntArith ar{int_mod(q), a.pro_itw + ((size_t)st << (a.log_n + 1))};
        IntArith::Tw tw[NB];
        T4::template load_tw<IntArith, 0>(tw, ar, 1, t);
        behind();
        T4::template inverse<IntArith>(s, tw, ar, lds, t);
#pragma unroll
        for (int j = 0; j < 4; j++) s[j] = reduce_4q(s[j], ar.m);
    }
}

// Rows pass.  The thread index is (wave, lane), the wave the same scalar in all its lanes, so that the twiddles of the
// first two blocks come through scalar loads.
// SRC_INTT (forward, NTT_PRO_SOURCE_INTT_REDUCE): the inverse rows pass of the source limb's tile runs first; it leaves the
// coefficients where the forward pass takes them from.  With MDR (one special prime) those of the dropped limb and of the special
// one behind it, which every output limb's workgroup transforms anew: a launch less, and CUs that were idle (see ntt_two_sources_ok).
// B = log2(words of a tile): 2^LD rows x 2^(B - LD) columns
// TILES (inverse): the coefficients leave where a fused conversion looks for them (conversion_word), on the FP64 back end as doubles.
// SMALL: NTT_PRO_SOURCE_SMALL_REDUCE, or SRC_INTT with pro_small.
template <int LD, bool FWD, int BE, bool SRC_INTT, bool MDR, int B, bool TILES, bool SMALL>
__global__ __launch_bounds__(1 << (B - 2)) void ntt_rows_kernel(HE_HEAD_PARAMS, RowsExtra x) {
    NttArgs a;
    using T4 = Tile4<B, LD>;
    constexpr int LOGC = B - LD, NB = T4::kBlocks;
    constexpr uint32_t C = 1u << LOGC, tiles_per_limb = 256u >> LOGC;
    __shared__ uint64_t lds[(1 << B) + (1 << (B - 4))], lds2[SRC_INTT && MDR ? (1 << B) + (1 << (B - 4)) : 1];
    set_head(a, HE_HEAD_NAMES);
    set_extra<FWD, SRC_INTT, MDR>(a, x);
    const uint32_t lb = logical_block(h4);
    const Job job = decode_job<SRC_INTT && !MDR>(a, a.first_job + lb / tiles_per_limb);
    const uint32_t col0 = (lb % tiles_per_limb) << LOGC;
    const uint32_t t = ((uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) << 6) | (threadIdx.x & 63);
    auto glob = [&](int k, int j) {
        const uint32_t e = T4::word(k, t, j);
        return (size_t)(e >> LOGC) * 256 + col0 + (e & (C - 1));
    };
    uint64_t s[4], s2[4];   // canonical coefficients of the source limbs
    if constexpr (SRC_INTT) {
        const uint64_t *src = MDR ? a.pro_src + ((size_t)job.poly * a.pro_poly_stride << a.log_n) : job.src;
#pragma unroll
        for (int j = 0; j < 4; j++) s[j] = src[glob(NB - 1, j)];
        if constexpr (MDR) {
#pragma unroll
            for (int j = 0; j < 4; j++) s2[j] = (src + ((size_t)1 << a.log_n))[glob(NB - 1, j)];
        }
    }
    int small[4] = {0, 0, 0, 0};   // an encryption's errors (pro_small)
    uint64_t src_q = 0, dst_q = 0, dst_r1 = 0;
    auto sources = [&]() {
        if constexpr (!MDR) {
            src_q = scalar(a.moduli)[job.src_table];
            dst_q = scalar(a.moduli)[job.table];
            dst_r1 = scalar(a.barrett)[2 * job.table + 1];
        }
        source_words<T4>(s, a, MDR ? a.pro_last : job.src_table, lds, t, [&]() {
            // (the moduli too: behind the pass they would be another trip to memory)
            if constexpr (!MDR) asm volatile("" ::"s"(src_q), "s"(dst_q), "s"(dst_r1));
            if constexpr (SMALL) {
#pragma unroll
                for (int j = 0; j < 4; j++) small[j] = (a.pro_small + ((size_t)job.poly << a.log_n))[glob(0, j)];
            }
        });
        if constexpr (SMALL) {
#pragma unroll
            for (int j = 0; j < 4; j++) s[j] = add_small(s[j], small[j], src_q);
        }
        if constexpr (MDR) source_words<T4>(s2, a, a.pro_src_table, lds2, t, []() {});
    };
    // the last words of an inverse pass: to their places in the limb, or where a conversion looks for them
    auto leave = [&](const uint64_t *w) {
        if constexpr (TILES) {
            store_tiled(job.out + conversion_word<B, LD>(lb % tiles_per_limb, t), w);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) job.out[glob(0, j)] = w[j];
        }
    };
    const bool fp = BE == NTT_BACKEND_FP || (BE == NTT_BACKEND_MIXED && ((a.fp_mask >> job.table) & 1));
    if (BE != NTT_BACKEND_INT && fp) {
        const FpCtx c = fp_ctx(a, job.table);
        const FpArith ar{c.m, c.tw};
        double v[4];
        FpArith::Tw tw[NB];
        if (FWD) {
            T4::template load_tw<FpArith, 0>(tw, ar, 1, t);
            if constexpr (SRC_INTT) sources();
            if constexpr (SRC_INTT && !MDR) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint64_t w = barrett64(s[j], dst_q, dst_r1);
                    v[j] = fp_from_u64(SMALL ? add_small(w, -small[j], dst_q) : w);
                }
            } else if constexpr (SMALL) {
                const bool values = a.pro_values && !(job.poly & 1);
                double r[4];
                small_source(s, r, a, job, values, [&](int j) { return glob(0, j); });
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = fp_from_u64(s[j]);
                if (values) {
                    const double p = fp_from_u64(scalar_shoup(a.barrett + p_constants_from_barrett(a.size_qp), job.limb).w);
#pragma unroll
                    for (int j = 0; j < 4; j++) v[j] -= fp_mulmod(fp_reduce(r[j], c.m), p, c.m);
                    ar.reduce(v);
                }
            } else if (rows_input_fp<MDR, SRC_INTT>(v, a, job, c, [&](int j) { return glob(0, j); }, s, s2)) {
                ar.reduce(v);
            }
            T4::template forward<FpArith>(v, tw, ar, lds, t);
            // lazy signed doubles go to the blocks pass
#pragma unroll
            for (int j = 0; j < 4; j++) job.out[glob(NB - 1, j)] = FpArith::to_word(v[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = FpArith::from_word(job.in[glob(NB - 1, j)]);
            T4::template load_tw<FpArith, 0>(tw, ar, 1, t);
            const double scale = inverse_scale(a, job, c.m);
            T4::template inverse<FpArith>(v, tw, ar, lds, t);
            ar.template scale<T4::stages(0)>(v, scale);
            uint64_t w[4];
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = TILES && BE == NTT_BACKEND_FP ? FpArith::to_word(v[j] - 0x1p49) : fp_to_u64(v[j]);
            leave(w);
        }
        return;
    }
    if constexpr (BE != NTT_BACKEND_FP) {
        const IntArith ar = int_arith(a, job.table);
        const uint64_t q = scalar(a.moduli)[job.table];
        uint64_t v[4];
        IntArith::Tw tw[NB];
        if (FWD) {
            T4::template load_tw<IntArith, 0>(tw, ar, 1, t);
            if constexpr (SRC_INTT) sources();
            if constexpr (SRC_INTT && !MDR) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint64_t w = barrett64(s[j], dst_q, dst_r1);
                    v[j] = SMALL ? add_small(w, -small[j], dst_q) : w;
                }
            } else if constexpr (SMALL) {
                const bool values = a.pro_values && !(job.poly & 1);
                const uint64_t r1 = scalar(a.barrett)[2 * job.table + 1];
                double r[4];
                small_source(v, r, a, job, values, [&](int j) { return glob(0, j); });
                if (values) {
                    const Shoup p = scalar_shoup(a.barrett + p_constants_from_barrett(a.size_qp), job.limb);
#pragma unroll
                    for (int j = 0; j < 4; j++) v[j] = sub_mod(v[j], mul_shoup(rounded_residue(r[j], q, r1), p, q), q);
                }
            } else {
                rows_input_int<MDR, SRC_INTT>(v, a, job, q, [&](int j) { return glob(0, j); }, s, s2);
            }
            T4::template forward<IntArith>(v, tw, ar, lds, t);
            // lazy values in [0, 8q) go to the blocks pass
#pragma unroll
            for (int j = 0; j < 4; j++) job.out[glob(NB - 1, j)] = v[j];
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = job.in[glob(NB - 1, j)];
            T4::template load_tw<IntArith, 0>(tw, ar, 1, t);
            Shoup w{0, 0};
            if (a.epi_mode == NTT_EPI_MUL) w = scalar_shoup(a.w, job.limb);
            T4::template inverse<IntArith>(v, tw, ar, lds, t);
            if (a.epi_mode == NTT_EPI_MUL) {
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = mul_shoup(v[j], w, q);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = reduce_4q(v[j], ar.m);
            }
            leave(v);
        }
    }
}

constexpr int kBlockWaves = 2;   // 256-word blocks of a workgroup, one per wave

// What a blocks pass's mode needs behind NttHead: the operands of an epilogue, or the list.
struct BlocksExtra {
    const void *p0, *p1, *p2, *p3, *p4;   // epi_a, epi_b, epi_dst, w, pro_w; or jobs, groups, item_stride
    uint32_t u0, u1, u2, n_polys;         // strides of epi_a and epi_b, of epi_dst and epi_mode, epi_b_mask; or n_groups, items; in_galois
};

BlocksExtra blocks_extra(const NttArgs &a, bool fwd) {
    if (a.jobs) return BlocksExtra{a.jobs, a.groups, reinterpret_cast<const void *>(a.item_stride), nullptr, nullptr, a.n_groups, a.items, 0, a.n_polys};
    return BlocksExtra{a.epi_a, a.epi_b, a.epi_dst, a.w, a.pro_w, a.epi_a_poly_stride | a.epi_b_poly_stride << 16,
                       a.epi_dst_poly_stride | (uint32_t)a.epi_mode << 16, fwd ? a.epi_b_mask : a.in_galois, a.n_polys};
}

__device__ __forceinline__ void set_extra(NttArgs &a, const BlocksExtra &e, bool fwd) {
    a.n_polys = e.n_polys;
    a.in_galois = fwd ? 0 : e.u2;
    a.jobs = static_cast<const LimbJob *>(e.p0);
    a.groups = static_cast<const LimbGroup *>(e.p1);
    a.item_stride = reinterpret_cast<size_t>(e.p2);
    a.n_groups = e.u0;
    a.items = e.u1;
    a.epi_a = static_cast<const uint64_t *>(e.p0);
    a.epi_b = static_cast<const uint64_t *>(e.p1);
    a.epi_dst = static_cast<uint64_t *>(const_cast<void *>(e.p2));
    a.w = static_cast<const uint64_t *>(e.p3);
    a.pro_w = static_cast<const uint64_t *>(e.p4);
    a.epi_a_poly_stride = e.u0 & 0xffff;
    a.epi_b_poly_stride = e.u0 >> 16;
    a.epi_dst_poly_stride = e.u1 & 0xffff;
    a.epi_mode = e.u1 >> 16;
    a.epi_b_mask = e.u2;
}

// Operands of a fused forward epilogue at the lane's two pairs of words, and its constants
struct EpiOperands {
    bool fma, add;
    uint64_t a[4], b[4];
    uint64_t *dst;
    Shoup w, pro_w;
};

__device__ __forceinline__ EpiOperands load_epilogue(const NttArgs &a, const Job &job, size_t off) {
    EpiOperands o;
    o.fma = a.epi_mode == NTT_EPI_FMA_SUB_MUL;
    o.add = o.fma || (a.epi_mode == NTT_EPI_SUB_MUL_ADD && ((a.epi_b_mask >> (job.poly & 31)) & 1));
    const size_t n = (size_t)1 << a.log_n, at = off + (size_t)job.limb * n;
    o.dst = a.epi_dst + (size_t)job.poly * a.epi_dst_poly_stride * n + at;
    load_pairs(o.a, a.epi_a + (size_t)job.poly * a.epi_a_poly_stride * n + at);
    if (o.add) load_pairs(o.b, a.epi_b + (size_t)job.poly * a.epi_b_poly_stride * n + at);
    o.w = scalar_shoup(a.w, job.limb);
    o.pro_w = Shoup{0, 0};
    if (o.fma) o.pro_w = scalar_shoup(a.pro_w, job.limb);
    return o;
}

// The limbs that a wave takes in turn at its block: they share a prime, so its twiddles are loaded once.
// Map mode: limb `limb` of the polynomials p0 .. p0 + count - 1.  List mode: the jobs of one group, for the items i0 ...
struct BlockUnit {
    uint32_t first, per, stride, count;   // job b of the unit: first + (b / per) * stride + b % per
    __device__ __forceinline__ uint32_t job(uint32_t b) const { return per == 1 ? first + b * stride : first + (b / per) * stride + b % per; }
};

__device__ __forceinline__ BlockUnit block_unit(const NttArgs &a, uint32_t u) {
    if (a.listed) {
        const uint32_t items = a.items ? a.items : 1;
        uint32_t first, per, chunk;
        if (a.groups) {
            chunk = u / a.n_groups;
            const LimbGroup g = a.groups[u - chunk * a.n_groups];
            first = g.first;
            per = g.count;
        } else {
            chunk = u / a.n_jobs;
            first = u - chunk * a.n_jobs;
            per = 1;
        }
        const uint32_t i0 = chunk * a.batch, n = items - i0 < a.batch ? items - i0 : a.batch;
        return BlockUnit{i0 * a.n_jobs + first, per, a.n_jobs, n * per};
    }
    const uint32_t limb = u % a.map.limbs, p0 = (u / a.map.limbs) * a.batch;
    return BlockUnit{p0 * a.map.limbs + limb, 1, a.map.limbs, a.n_polys - p0 < a.batch ? a.n_polys - p0 : a.batch};
}

// Blocks pass: a wave owns one block of 256 consecutive words of every limb of its unit, every exchange stays inside the
// wave.  The next limb's words are requested before the current one's butterflies.
template <bool FWD, bool EPI, bool LOOP, class A>
__device__ __forceinline__ void blocks_pass(const NttArgs &a, const BlockUnit &unit, Job job, const A &ar, uint64_t q, uint32_t blk,
                                              uint32_t lane) {
    using T4 = Tile4<8, 8>;
    constexpr bool FP = std::is_base_of<FpArith, A>::value;
    const size_t off = (size_t)blk * 256;
    auto fetch = [&](uint64_t *x, const Job &j) {
        if (FWD) {
            // the rows pass left its words in out
#pragma unroll
            for (int i = 0; i < 4; i++) x[i] = j.out[off + T4::word(0, lane, i)];
        } else if (a.in_galois) {
#pragma unroll
            for (int i = 0; i < 4; i++) x[i] = j.in[galois_index((uint32_t)off + pair_lane(lane) + pair_word(i), a.in_galois, a.log_n)];
        } else {
            load_pairs(x, j.in + off + pair_lane(lane));
        }
    };
    uint64_t x[4], nx[4];
    fetch(nx, job);
    typename A::Tw tw[4];
    T4::template load_tw<A, 0>(tw, ar, (1u << (a.log_n - 8)) + blk, lane);
    for (uint32_t b = 0;; b++) {
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = nx[j];
        const bool more = LOOP && b + 1 < unit.count;
        EpiOperands e;
        if (FWD && EPI) e = load_epilogue(a, job, off + pair_lane(lane));
        Job next = job;
        if (more) {
            next = decode_job<false, true>(a, unit.job(b + 1));
            fetch(nx, next);
        }
        typename A::V v[4];
        if constexpr (FP) {
            const FpMod m = ar.m;
            if (FWD) {
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = A::from_word(x[j]);
                T4::template forward<A>(v, tw, ar, nullptr, lane);
                turn_pairs(v);
                if (EPI) {
                    // (the word enters the difference as the last stage leaves it: at most 3.8 q, minuend below 1.9 q)
                    const double ew = fp_from_u64(e.w.w);
                    if (e.fma) {
                        const double pw = fp_from_u64(e.pro_w.w);
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const double lhs = fp_mulmod(fp_from_u64(e.a[j]), pw, m) + fp_from_u64(e.b[j]);
                            v[j] = fp_mulmod(lhs - v[j], ew, m);
                        }
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            v[j] = fp_mulmod(fp_from_u64(e.a[j]) - v[j], ew, m);
                            if (e.add) v[j] += fp_from_u64(e.b[j]);
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < 4; j++) x[j] = fp_to_u64(fp_canonical(v[j], m));
                store_pairs(EPI ? e.dst : job.out + off + pair_lane(lane), x);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = fp_from_u64(x[j]);
                turn_pairs(v);
                T4::template inverse<A>(v, tw, ar, nullptr, lane);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = x[j];
            if (FWD) {
                T4::template forward<A>(v, tw, ar, nullptr, lane);
                turn_pairs(v);
#pragma unroll
                for (int j = 0; j < 4; j++) x[j] = reduce_8q(v[j], ar.m);
                if (EPI) {
                    const Shoup ew = e.w;
                    if (e.fma) {
                        const Shoup pw = e.pro_w;
#pragma unroll
                        for (int j = 0; j < 4; j++)
                            x[j] = mul_shoup(sub_mod(add_mod(mul_shoup(e.a[j], pw, q), e.b[j], q), x[j], q), ew, q);
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            x[j] = mul_shoup(sub_mod(e.a[j], x[j], q), ew, q);
                            if (e.add) x[j] = add_mod(x[j], e.b[j], q);
                        }
                    }
                }
                store_pairs(EPI ? e.dst : job.out + off + pair_lane(lane), x);
            } else {
                turn_pairs(v);
                T4::template inverse<A>(v, tw, ar, nullptr, lane);
            }
        }
        if (!FWD) {
            // lazy words (signed doubles, or integers in [0, 4q)) go to the rows pass
#pragma unroll
            for (int j = 0; j < 4; j++) job.out[off + T4::word(0, lane, j)] = A::to_word(v[j]);
        }
        if (!more) break;
        job = next;
    }
}

// PRODUCTS: see FpProducts (launch_ntt_blocks says when)
template <bool FWD, bool EPI, bool LOOP, int BE, bool PRODUCTS>
__global__ __launch_bounds__(64 * kBlockWaves) void ntt_blocks_kernel(HE_HEAD_PARAMS, BlocksExtra x) {
    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    set_extra(a, x, FWD);
    const uint32_t lr = a.log_n - 8, lane = threadIdx.x & 63;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t id = (EPI ? limb_block(h4, lr - 1, h0) : logical_block(h4)) * kBlockWaves + w;   // (a limb has an even number of blocks)
    const BlockUnit unit = block_unit(a, id >> lr);
    const uint32_t blk = id & ((1u << lr) - 1);
    const Job job = decode_job<false, true>(a, unit.job(0));
    const bool fp = BE == NTT_BACKEND_FP || (BE == NTT_BACKEND_MIXED && ((a.fp_mask >> job.table) & 1));
    if (BE != NTT_BACKEND_INT && fp) {
        const typename std::conditional<PRODUCTS, FpProducts<false>, FpArith>::type ar{fp_arith(a, job.table)};
        blocks_pass<FWD, EPI, LOOP>(a, unit, job, ar, 0, blk, lane);
    }
    if constexpr (BE != NTT_BACKEND_FP) {
        if (!fp) blocks_pass<FWD, EPI, LOOP>(a, unit, job, int_arith(a, job.table), scalar(a.moduli)[job.table], blk, lane);
    }
}

// Sum over the digits of (word x key word) for four words of both key polynomials.
// FP64: a transformed word enters as the last stage leaves it (at most 3.63 q: a term below 1.9 q), the sums are reduced after
// every fourth digit and stay below 8 q.  Integers: 128-bit sums of at most 64 products below 2^122 of canonical words, or, with primes
// below 2^60, of at most 32 products of words as the last stage leaves them (below 8 q):
// a wave's share of kMaxDigits, since only waves that share a block leave them so.
struct FpSums {
    double s[2][4];
    uint32_t pending = 0;
    __device__ __forceinline__ FpSums() {
#pragma unroll
        for (int j = 0; j < 4; j++) s[0][j] = s[1][j] = 0.0;
    }
    __device__ __forceinline__ void add(const double *v, const uint64_t (*k)[4], const FpArith &ar) {
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const double w = fp_from_u64(k[r][j]);
                s[r][j] += fp_mulmod(v[j], w, ar.m);
            }
        if (++pending == 4) {
            pending = 0;
            ar.reduce(s[0]);
            ar.reduce(s[1]);
        }
    }
};

struct IntSums {
    U128 s[2][4];
    __device__ __forceinline__ IntSums() {
#pragma unroll
        for (int j = 0; j < 4; j++) s[0][j] = s[1][j] = U128{0, 0};
    }
    __device__ __forceinline__ void add(const uint64_t *v, const uint64_t (*k)[4], const IntArith &ar) {
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int j = 0; j < 4; j++) mac128(s[r][j], v[j], k[r][j]);
    }
};

// What the inner product needs behind NttHead: up to three digits of one item, or any number of both.
struct InnerFew {
    static constexpr uint32_t kDigits = 3;
    const uint64_t *itw, *addend;   // the inverse direction's block; add_c0 or fold_ct
    uint64_t *out;
    uint32_t own_galois, inv_first;  // inv_first: bit 16: addend is add_c0, bit 17: it is fold_ct
    const uint64_t *evk[kDigits];
    __device__ __forceinline__ size_t item_stride() const { return 0; }
    __device__ __forceinline__ size_t own_item_stride() const { return 0; }
    __device__ __forceinline__ size_t fold_item_stride() const { return 0; }
};
struct InnerMany {
    static constexpr uint32_t kDigits = kMaxDigits;
    const uint64_t *itw, *addend;
    uint64_t *out;
    uint32_t own_galois, inv_first;
    size_t strides[3];
    const uint64_t *evk[kDigits];
    __device__ __forceinline__ size_t item_stride() const { return strides[0]; }
    __device__ __forceinline__ size_t own_item_stride() const { return strides[1]; }
    __device__ __forceinline__ size_t fold_item_stride() const { return strides[2]; }
};

// Blocks pass of ModUp's forward transform fused with the key-switch inner product: a wave owns one block of 256 words of limb t of
// Ql u P, takes it through the last 8 stages for every digit in turn and multiplies it by both key polynomials; the digit
// that owns limb t contributes the input itself.  The transformed limbs never reach memory, and the limbs of the sum that
// ModDown needs in coefficient form leave through the inverse blocks pass (a launch and two trips of those limbs less: one
// product at L = 24, K = 8 157 -> 153 us, n = 2^14, 4 + 1 limbs 38 -> 34 us, although the second set of twiddles takes the
// FP64 kernel from 96 registers to 120).
// SPLIT waves share a block when there are few: wave `part` takes every SPLIT-th digit, the partial sums meet in LDS (`sums_lds`),
// and waves 0 and 1 finish one polynomial each.
// STREAM: 1: the key words pass by the caches; 2: the digits' words do, which nothing reads again; 3: both (launch_ntt_inner says when).
template <int SPLIT, int STREAM, class A, class X>
__device__ __forceinline__ void inner_block(const NttArgs &a, const X &x, uint32_t L, uint32_t LK, uint32_t beta, uint32_t t,
                                            uint32_t table, uint32_t blk, uint32_t item, uint32_t lane, const A &ar, uint32_t part,
                                            uint64_t *sums_lds) {
    using T4 = Tile4<8, 8>;
    constexpr bool FP = std::is_base_of<FpArith, A>::value;
    const size_t n = (size_t)1 << a.log_n, off = (size_t)blk * 256, at = off + pair_lane(lane);
    const uint32_t own = t < L ? t / (LK - L) : 0xffffffffu;
    const uint64_t *lazy = a.out + (size_t)t * n + off;   // words left by the rows pass, digit 0
    if (item) lazy += item * x.item_stride();
    const size_t digit_stride = (size_t)LK * n, key_off = (size_t)table * n + at, key_poly = (size_t)a.size_qp * n;
    // the digits to transform: all but the own one, the own one counting as the first for the deal
    auto skip_own = [&](uint32_t d) { return d == own ? d + 1 : d; };
    auto next_digit = [&](uint32_t d) {
#pragma unroll
        for (int i = 0; i < SPLIT; i++) d = skip_own(d + 1);
        return d;
    };
    auto fetch = [&](uint64_t *w, uint32_t d) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint64_t *p = lazy + d * digit_stride + T4::word(0, lane, j);
            w[j] = STREAM & 2 ? __builtin_nontemporal_load(p) : *p;
        }
    };
    auto keys = [&](uint64_t (*k)[4], uint32_t d) {
        load_pairs_or_stream<(STREAM & 1) != 0>(k[0], x.evk[d] + key_off);
        load_pairs_or_stream<(STREAM & 1) != 0>(k[1], x.evk[d] + key_poly + key_off);
    };
    typename A::Tw tw[4];
    uint64_t nx[4];
    uint32_t d = skip_own(0);
    if constexpr (SPLIT > 1) {
        const uint32_t skip = own == 0xffffffffu ? part : (part + SPLIT - 1) % SPLIT;
        for (uint32_t i = 0; i < skip; i++) d = skip_own(d + 1);
    }
    if (d < beta) fetch(nx, d);
    T4::template load_tw<A, 0>(tw, ar, (1u << (a.log_n - 8)) + blk, lane);
    const bool add = (x.inv_first >> 16 & 1) && t < L;                 // polynomial 0 gains P sigma(c0) (a rotation)
    const bool fold = (x.inv_first >> 17 & 1) && t == L - 1;
    Shoup add_w{0, 0}, fold_w{0, 0};
    const uint64_t *p_mod_q = a.barrett + p_constants_from_barrett(a.size_qp);   // and P^-1 behind it (NttArgs::tw)
    if (add) add_w = scalar_shoup(p_mod_q, t);
    if (fold) fold_w = scalar_shoup(p_mod_q, a.map.tail_first + t);
    const uint64_t r0 = scalar(a.barrett)[2 * table], r1 = scalar(a.barrett)[2 * table + 1];
    // (the words of a limb that ModDown transforms back go through the inverse blocks pass before they leave the wave)
    const bool invert = t >= (x.inv_first & 0xffff);
    A iar = ar;
    if constexpr (FP)
        iar.table = a.pro_itw_fp + ((size_t)table << a.log_n);
    else
        iar.table = a.pro_itw + ((size_t)table << (a.log_n + 1));
    typename A::Tw itw[SPLIT > 1 ? 4 : 1];
    uint64_t c0[4], cl[4];
    auto fetch_addends = [&](uint32_t r) {
        if (add && r == 0) {
            const uint64_t *src = x.addend + (size_t)t * n;
            if (x.own_galois) {
#pragma unroll
                for (int j = 0; j < 4; j++) c0[j] = src[galois_index((uint32_t)at + pair_word(j), x.own_galois, a.log_n)];
            } else {
                load_pairs(c0, src + at);
            }
        }
        if (fold) load_pairs(cl, x.addend + item * x.fold_item_stride() + ((size_t)r * L + t) * n + at);
    };
    if constexpr (SPLIT > 1) {
        // (what the two waves that finish need after the sums have met is requested before the digits)
        if (part < 2) {
            if (invert) T4::template load_tw<A, 0>(itw, iar, (1u << (a.log_n - 8)) + blk, lane);
            fetch_addends(part);
        }
    }
    bool canonical = false;
    if constexpr (!FP) canonical = ar.m.q >> 60;
    typename std::conditional<FP, FpSums, IntSums>::type sums;
    if (own != 0xffffffffu && part == 0) {
        const uint64_t *src = a.in + (size_t)t * n;
        if (item) src += item * x.own_item_stride();
        uint64_t c[4], k[2][4];
        keys(k, own);
        if (x.own_galois) {
#pragma unroll
            for (int j = 0; j < 4; j++) c[j] = src[galois_index((uint32_t)at + pair_word(j), x.own_galois, a.log_n)];
        } else {
            load_pairs_or_stream<(STREAM & 2) != 0>(c, src + at);
        }
        typename A::V v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if constexpr (FP)
                v[j] = fp_from_u64(c[j]);
            else
                v[j] = c[j];
        }
        sums.add(v, k, ar);
    }
    while (d < beta) {
        uint64_t k[2][4];
        keys(k, d);
        typename A::V v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = A::from_word(nx[j]);
        const uint32_t now = d;
        d = next_digit(d);
        // (behind a branch that may skip these loads the compiler waits for them with the keys; short chains fetch their last digit
        // again instead: n = 2^15, 10 of 12 limbs 71.5 -> 69.8 us.  One wave a block loses by it: L = 24, K = 8 153 against 156 us)
        if (SPLIT > 1 || d < beta) fetch(nx, d < beta ? d : now);
        T4::template forward<A>(v, tw, ar, nullptr, lane);
        turn_pairs(v);
        if constexpr (!FP) {
            if (SPLIT == 1 || canonical) {   // (one wave a block: the branch costs what it saves)
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = reduce_8q(v[j], ar.m);
            }
        }
        sums.add(v, k, ar);
    }
    if constexpr (SPLIT > 1) {
        // (integers: the 128-bit sums as they are, so that each is reduced once, by the wave that finishes it, and not by all that share it;
        // with the words' reductions left out where they can be, rotations: n = 2^15, 10 + 3 limbs of 60 / 40 bits 51.9 -> 50.8 us; 2^14, 4 + 1
        // of 60 bits 23.6 -> 22.7; 2^16, 2 + 1 29.5 -> 28.8.  A wave's sum of lazy words is below 2^128 q^2 / 2^120 (two waves) or half of that
        // (four); from 33 digits on all of them could pass 2^128, so one that has reached 2^127 (2^126) gives q 2^67 (q 2^66) away and is below it
        // again.  A reduction of every word instead took 2 to 3.5 % of a whole product: 36 digits of 2^13 and 60 bits 141.5 / 137.0 us.)
        static_assert(kMaxDigits <= 64, "a wave's sum fits 128 bits");
        if constexpr (!FP) {
            constexpr int top = SPLIT == 2 ? 63 : 62;
            if (beta > 32 && !canonical) {
#pragma unroll
                for (int r = 0; r < 2; r++)
#pragma unroll
                    for (int j = 0; j < 4; j++) sums.s[r][j].hi -= sums.s[r][j].hi >> top ? ar.m.q << (top - 60) : 0;
            }
        }
#pragma unroll
        for (int r = 0; r < 2; r++) {
            uint64_t w[4];
            if constexpr (FP) {
                ar.reduce(sums.s[r]);
#pragma unroll
                for (int j = 0; j < 4; j++) w[j] = A::to_word(sums.s[r][j]);
                store_pairs(sums_lds + (2 * part + r) * 256 + pair_lane(lane), w);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) w[j] = sums.s[r][j].lo;
                store_pairs(sums_lds + (4 * part + 2 * r) * 256 + pair_lane(lane), w);
#pragma unroll
                for (int j = 0; j < 4; j++) w[j] = sums.s[r][j].hi;
                store_pairs(sums_lds + (4 * part + 2 * r + 1) * 256 + pair_lane(lane), w);
            }
        }
        lds_barrier();
        if (part > 1) return;
    }
    if (SPLIT == 1 && invert) T4::template load_tw<A, 0>(tw, iar, (1u << (a.log_n - 8)) + blk, lane);
    // one wave finishes both polynomials, or waves 0 and 1 one each
#pragma unroll
    for (int both = 0; both < (SPLIT > 1 ? 1 : 2); both++) {
        const uint32_t r = SPLIT > 1 ? part : (uint32_t)both;
        typename A::V v[4];
        if (SPLIT == 1) fetch_addends(r);
        if constexpr (FP) {
            const FpMod m = ar.m;
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = SPLIT > 1 ? 0.0 : sums.s[both][j];
            if constexpr (SPLIT > 1) {
#pragma unroll
                for (int i = 0; i < SPLIT; i++) {
                    uint64_t w[4];
                    load_pairs(w, sums_lds + (2 * i + r) * 256 + pair_lane(lane));
#pragma unroll
                    for (int j = 0; j < 4; j++) v[j] += A::from_word(w[j]);
                }
            }
            if (add && r == 0) {
                const double pd = fp_from_u64(add_w.w);
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] += fp_mulmod(fp_from_u64(c0[j]), pd, m);
            }
            if (fold) {
                const double wd = fp_from_u64(fold_w.w);
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = fp_mulmod(v[j], wd, m) + fp_from_u64(cl[j]);
            }
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = fp_canonical(v[j], m);
        } else {
            const uint64_t q = ar.m.q;
            U128 total[4];
#pragma unroll
            for (int j = 0; j < 4; j++) total[j] = SPLIT > 1 ? U128{0, 0} : sums.s[both][j];
            if constexpr (SPLIT > 1) {
#pragma unroll
                for (int i = 0; i < SPLIT; i++) {
                    uint64_t lo[4], hi[4];
                    load_pairs(lo, sums_lds + (4 * i + 2 * r) * 256 + pair_lane(lane));
                    load_pairs(hi, sums_lds + (4 * i + 2 * r + 1) * 256 + pair_lane(lane));
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        total[j].lo += lo[j];
                        total[j].hi += hi[j] + (total[j].lo < lo[j]);
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = barrett128(total[j].lo, total[j].hi, q, r0, r1);
            if (add && r == 0) {
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = add_mod(v[j], mul_shoup(c0[j], add_w, q), q);
            }
            if (fold) {
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] = add_mod(mul_shoup(v[j], fold_w, q), cl[j], q);
            }
        }
        uint64_t *o = x.out + item * (2 * (size_t)LK * n) + (size_t)r * LK * n + (size_t)t * n;
        if (invert) {
            turn_pairs(v);
            T4::template inverse<A>(v, SPLIT > 1 ? itw : tw, iar, nullptr, lane);
#pragma unroll
            for (int j = 0; j < 4; j++) o[off + T4::word(0, lane, j)] = A::to_word(v[j]);
        } else {
            uint64_t res[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (FP)
                    res[j] = fp_to_u64(v[j]);
                else
                    res[j] = v[j];
            }
            store_pairs(o + at, res);
        }
    }
}

// Waves of a workgroup: of one item, neighbouring blocks; of a batch, the same block of neighbouring items, which find the
// key words of the first in the CU's cache.  Across workgroups the items of a block run next to each other on one XCD.
constexpr int kInnerWaves = 4;

// PRODUCTS: see FpProducts (launch_ntt_inner says when)
template <int BE, int SPLIT, int STREAM, bool PRODUCTS, class X>
__global__ __launch_bounds__(64 * kInnerWaves) void ntt_inner_kernel(HE_HEAD_PARAMS, X x) {
    __shared__ uint64_t sums_all[SPLIT > 1 ? kInnerWaves / SPLIT : 1][SPLIT > 1 ? (BE == NTT_BACKEND_FP ? 2 : 4) * SPLIT * 256 : 1];
    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    set_inverse_block(a, x.itw);
    const uint32_t LK = a.map.limbs, L = a.map.split, items = h5 >> 8;
    const uint32_t lr = a.log_n - 8, lane = threadIdx.x & 63, pairs = LK << lr;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6), part = w % SPLIT;
    uint32_t pair, item = 0;
    if (SPLIT == 1 && items > 1) {
        const uint32_t groups = (items + kInnerWaves - 1) / kInnerWaves, id = blockIdx.x;
        uint32_t g;
        if (pairs % 8 == 0) {
            // hardware id -> XCD id & 7; inside an XCD the groups of one pair are consecutive
            const uint32_t s = id >> 3;
            g = s % groups;
            pair = (s / groups) * 8 + (id & 7);
        } else {
            g = id / pairs;
            pair = id - g * pairs;
        }
        item = g * kInnerWaves + w;
        if (item >= items) return;
    } else {
        // last limb first: the special limbs have one digit more to transform than the others
        // (a limb has an even number of blocks: with SPLIT > 1 no wave is left over, and a workgroup's blocks share their limb)
        pair = blockIdx.x * (kInnerWaves / SPLIT) + w / SPLIT;
        if (SPLIT == 1 && pair >= pairs) return;
        pair = pairs - 1 - pair;
    }
    uint32_t t = pair >> lr;
    if (BE == NTT_BACKEND_MIXED && LK <= 16) t = (uint32_t)((((uint64_t)h2 << 32) | h1) >> (4 * t)) & 15;
    const uint32_t blk = pair & ((1u << lr) - 1), table = map_table(a.map, t);
    const bool fp = BE == NTT_BACKEND_FP || (BE == NTT_BACKEND_MIXED && ((a.fp_mask >> table) & 1));
    uint64_t *sums = sums_all[SPLIT > 1 ? w / SPLIT : 0];
    if (BE != NTT_BACKEND_INT && fp) {
        const typename std::conditional<PRODUCTS, FpProducts<true>, FpArith>::type ar{fp_arith(a, table)};
        inner_block<SPLIT, STREAM>(a, x, L, LK, h5 & 255, t, table, blk, item, lane, ar, part, sums);
    }
    if constexpr (BE != NTT_BACKEND_FP) {
        if (!fp) inner_block<SPLIT, STREAM>(a, x, L, LK, h5 & 255, t, table, blk, item, lane, int_arith(a, table), part, sums);
    }
}

// (d0, d1, d2) = (a0 b0, a0 b1 + a1 b0, a1 b1) mod q, canonical, of four words each
__device__ __forceinline__ void tensor4(const FpArith &ar, const NttArgs &, uint32_t, const uint64_t *a0, const uint64_t *a1,
                                        const uint64_t *b0, const uint64_t *b1, double *d0, double *d1, double *d2) {
    const FpMod m = ar.m;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const double x0 = fp_from_u64(a0[j]), x1 = fp_from_u64(a1[j]), y0 = fp_from_u64(b0[j]), y1 = fp_from_u64(b1[j]);
        d0[j] = fp_canonical(fp_mulmod(x0, y0, m), m);
        d2[j] = fp_canonical(fp_mulmod(x1, y1, m), m);
        // Karatsuba: both factors are below 2 q, the product is reduced to |r| <= 2 q, the difference stays below 4 q
        const double sy = y0 + y1, mm = fp_mulmod(x0 + x1, sy, m);
        d1[j] = fp_canonical(mm - d0[j] - d2[j], m);
    }
}

__device__ __forceinline__ void tensor4(const IntArith &ar, const NttArgs &a, uint32_t table, const uint64_t *a0, const uint64_t *a1,
                                        const uint64_t *b0, const uint64_t *b1, uint64_t *d0, uint64_t *d1, uint64_t *d2) {
    const uint64_t q = ar.m.q, r0 = scalar(a.barrett)[2 * table], r1 = scalar(a.barrett)[2 * table + 1];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        d0[j] = mul_mod(a0[j], b0[j], q, r0, r1);
        d2[j] = mul_mod(a1[j], b1[j], q, r0, r1);
        // Karatsuba; the sums stay below 2^62
        d1[j] = sub_mod(sub_mod(mul_mod(a0[j] + a1[j], b0[j] + b1[j], q, r0, r1), d0[j], q), d2[j], q);
    }
}

// x y mod q of four canonical words: as the arithmetic's values and as words, canonical
__device__ __forceinline__ void product4(const FpArith &ar, const NttArgs &, uint32_t, const uint64_t *x, const uint64_t *y, double *d, uint64_t *w) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
        d[j] = fp_canonical(fp_mulmod(fp_from_u64(x[j]), fp_from_u64(y[j]), ar.m), ar.m);
        w[j] = fp_to_u64(d[j]);
    }
}

__device__ __forceinline__ void product4(const IntArith &ar, const NttArgs &a, uint32_t table, const uint64_t *x, const uint64_t *y, uint64_t *d,
                                         uint64_t *w) {
    const uint64_t r0 = scalar(a.barrett)[2 * table], r1 = scalar(a.barrett)[2 * table + 1];
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = d[j] = mul_mod(x[j], y[j], ar.m.q, r0, r1);
}

// Tensor product fused with the blocks pass of the inverse transform of its third polynomial: a wave forms the three products
// of one block of 256 words, stores them (d2 in NTT form is what the key switch multiplies by its own digit's key) and takes d2
// through the 8 inverse stages; the lazy words are left in a.out for the rows pass.  One read of d2 and one launch less
// than tensor kernel + inverse transform.
template <class A>
__device__ __forceinline__ void tensor_block(const NttArgs &a, const TensorFuse &x, const Job &job, const A &ar, uint32_t blk,
                                             uint32_t lane) {
    using T4 = Tile4<8, 8>;
    constexpr bool FP = std::is_base_of<FpArith, A>::value;
    const size_t n = (size_t)1 << a.log_n, poly = (size_t)x.L * n, off = (size_t)blk * 256, at = off + pair_lane(lane);
    const size_t ct = 2 * job.poly * poly + job.limb * n + at;
    uint64_t a0[4], a1[4], b0[4], b1[4];
    load_pairs(a0, x.ct1 + ct);
    load_pairs(a1, x.ct1 + ct + poly);
    if (!x.square) {
        load_pairs(b0, x.ct2 + ct);
        load_pairs(b1, x.ct2 + ct + poly);
    }
    typename A::Tw tw[4];
    T4::template load_tw<A, 0>(tw, ar, (1u << (a.log_n - 8)) + blk, lane);
    if (x.square) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            b0[j] = a0[j];
            b1[j] = a1[j];
        }
    }
    typename A::V d0[4], d1[4], d2[4];
    tensor4(ar, a, job.table, a0, a1, b0, b1, d0, d1, d2);
    uint64_t o0[4], o1[4], o2[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if constexpr (FP) {
            o0[j] = fp_to_u64(d0[j]);
            o1[j] = fp_to_u64(d1[j]);
            o2[j] = fp_to_u64(d2[j]);
        } else {
            o0[j] = d0[j];
            o1[j] = d1[j];
            o2[j] = d2[j];
        }
    }
    store_pairs(x.d01 + ct, o0);
    store_pairs(x.d01 + ct + poly, o1);
    store_pairs(x.d2 + job.poly * poly + job.limb * n + at, o2);
    turn_pairs(d2);
    T4::template inverse<A>(d2, tw, ar, nullptr, lane);
#pragma unroll
    for (int j = 0; j < 4; j++) job.out[off + T4::word(0, lane, j)] = A::to_word(d2[j]);
}

// the third polynomial alone (TensorFuse::last_only)
template <class A>
__device__ __forceinline__ void third_block(const NttArgs &a, const TensorFuse &x, const Job &job, const A &ar, uint32_t blk, uint32_t lane) {
    using T4 = Tile4<8, 8>;
    const size_t n = (size_t)1 << a.log_n, poly = (size_t)x.L * n, off = (size_t)blk * 256, at = off + pair_lane(lane);
    const size_t ct = (2 * job.poly + 1) * poly + job.limb * n + at;
    uint64_t a1[4], b1[4];
    load_pairs(a1, x.ct1 + ct);
    load_pairs(b1, (x.square ? x.ct1 : x.ct2) + ct);
    typename A::Tw tw[4];
    T4::template load_tw<A, 0>(tw, ar, (1u << (a.log_n - 8)) + blk, lane);
    typename A::V d2[4];
    uint64_t w[4];
    product4(ar, a, job.table, a1, b1, d2, w);
    store_pairs(x.d2 + job.poly * poly + job.limb * n + at, w);
    turn_pairs(d2);
    T4::template inverse<A>(d2, tw, ar, nullptr, lane);
#pragma unroll
    for (int j = 0; j < 4; j++) job.out[off + T4::word(0, lane, j)] = A::to_word(d2[j]);
}

template <int BE, bool LAST_ONLY>
__global__ __launch_bounds__(64 * kBlockWaves) void tensor_intt_blocks_kernel(HE_HEAD_PARAMS, const uint64_t *ct2, uint64_t *d01, uint64_t *d2) {
    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    const TensorFuse x{h_in, ct2, d01, d2, a.map.limbs, (int)h5, LAST_ONLY};
    const uint32_t lr = a.log_n - 8, lane = threadIdx.x & 63;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t id = limb_block(h4, lr - 1, h0) * kBlockWaves + w, blk = id & ((1u << lr) - 1);
    const Job job = decode_job(a, id >> lr);
    const bool fp = BE == NTT_BACKEND_FP || (BE == NTT_BACKEND_MIXED && ((a.fp_mask >> job.table) & 1));
    auto block = [&](const auto &ar) {
        if (LAST_ONLY && job.limb + 1 != a.map.limbs)
            third_block(a, x, job, ar, blk, lane);
        else
            tensor_block(a, x, job, ar, blk, lane);
    };
    if (BE != NTT_BACKEND_INT && fp) block(fp_arith(a, job.table));
    if constexpr (BE != NTT_BACKEND_FP) {
        if (!fp) block(int_arith(a, job.table));
    }
}

// out = (c P^-1 + d - v) q_last^-1 of four words: v as the forward stages have left it, d = x y or x y + z w of canonical words
__device__ __forceinline__ void end4(const FpArith &ar, const NttArgs &, uint32_t, const double *v, const uint64_t *c, const uint64_t *x, const uint64_t *y,
                                     const uint64_t *z, const uint64_t *w, Shoup p_inv, Shoup q_inv, uint64_t *out) {
    const FpMod m = ar.m;
    const double pw = fp_from_u64(p_inv.w), ew = fp_from_u64(q_inv.w);
    // (three products below q, less a word of at most 3.8 q: below 8 q)
#pragma unroll
    for (int j = 0; j < 4; j++) {
        double d = fp_mulmod(fp_from_u64(c[j]), pw, m) + fp_mulmod(fp_from_u64(x[j]), fp_from_u64(y[j]), m);
        if (z) d += fp_mulmod(fp_from_u64(z[j]), fp_from_u64(w[j]), m);
        out[j] = fp_to_u64(fp_canonical(fp_mulmod(d - v[j], ew, m), m));
    }
}

__device__ __forceinline__ void end4(const IntArith &ar, const NttArgs &a, uint32_t table, const uint64_t *v, const uint64_t *c, const uint64_t *x,
                                     const uint64_t *y, const uint64_t *z, const uint64_t *w, Shoup p_inv, Shoup q_inv, uint64_t *out) {
    const uint64_t q = ar.m.q, r0 = scalar(a.barrett)[2 * table], r1 = scalar(a.barrett)[2 * table + 1];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        U128 d{0, 0};
        mac128(d, x[j], y[j]);
        if (z) mac128(d, z[j], w[j]);
        const uint64_t lhs = add_mod(mul_shoup(c[j], p_inv, q), barrett128(d.lo, d.hi, q, r0, r1), q);
        out[j] = mul_shoup(sub_mod(lhs, reduce_8q(v[j], ar.m), q), q_inv, q);
    }
}

// what ProductEnd has behind the head, whose input is the first factor
struct EndExtra {
    const uint64_t *cx, *ct2;
    uint64_t *out;
    const uint64_t *p_inv, *q_last_inv;
    uint32_t cx_stride;
};

// A product's last pass (ProductEnd): a wave takes one block of both polynomials, so that it reads the four factors once.  Bound by memory:
// the factors are read again (four polynomials) in place of d0 and d1 (two), which the first pass then neither forms nor stores, and for which
// it does not read two of the factors.  Eight products of 24 + 8 limbs of 2^16 words, the first and the last pass: 140 + 163 us -> 77
// + 190, and 90 + 147 with words that pass by the caches.
// STREAM: 1: the rows pass's words and the sums pass by the caches; 2: the factors do as well.
template <int STREAM, class A>
__device__ __forceinline__ void product_end_block(const NttArgs &a, const EndExtra &x, const Job &job, const A &ar, uint32_t blk,
                                                  uint32_t lane) {
    using T4 = Tile4<8, 8>;
    const uint32_t L = a.map.limbs + 1;
    const size_t n = (size_t)1 << a.log_n, off = (size_t)blk * 256, at = off + pair_lane(lane), item = job.poly;
    const size_t ct = (2 * item * L + job.limb) * n + at, poly = (size_t)L * n;
    const uint64_t *cx = x.cx + (2 * item * x.cx_stride + job.limb) * n + at;
    uint64_t lazy[2][4], c[2][4], f[2][4], g[2][4];
#pragma unroll
    for (int r = 0; r < 2; r++) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint64_t *p = job.out + r * poly + off + T4::word(0, lane, j);
            lazy[r][j] = STREAM ? __builtin_nontemporal_load(p) : *p;
        }
    }
    typename A::Tw tw[4];
    T4::template load_tw<A, 0>(tw, ar, (1u << (a.log_n - 8)) + blk, lane);
#pragma unroll
    for (int r = 0; r < 2; r++) {
        load_pairs_or_stream<STREAM != 0>(c[r], cx + r * (size_t)x.cx_stride * n);
        load_pairs_or_stream<STREAM == 2>(f[r], a.in + ct + r * poly);
        load_pairs_or_stream<STREAM == 2>(g[r], x.ct2 + ct + r * poly);
    }
    const Shoup p_inv = scalar_shoup(x.p_inv, job.limb), q_inv = scalar_shoup(x.q_last_inv, job.limb);
    uint64_t *out = x.out + (2 * item * (L - 1) + job.limb) * n + at;
#pragma unroll
    for (int r = 0; r < 2; r++) {
        typename A::V v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = A::from_word(lazy[r][j]);
        T4::template forward<A>(v, tw, ar, nullptr, lane);
        turn_pairs(v);
        uint64_t o[4];
        if (r == 0)
            end4(ar, a, job.table, v, c[0], f[0], g[0], nullptr, nullptr, p_inv, q_inv, o);
        else
            end4(ar, a, job.table, v, c[1], f[0], g[1], f[1], g[0], p_inv, q_inv, o);
        store_pairs(out + r * (size_t)(L - 1) * n, o);
    }
}

// PRODUCTS: see FpProducts (launch_product_end says when)
template <int BE, int STREAM, bool PRODUCTS>
__global__ __launch_bounds__(64 * kBlockWaves) void product_end_kernel(HE_HEAD_PARAMS, EndExtra x) {
    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    const uint32_t lr = a.log_n - 8, lane = threadIdx.x & 63;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t id = limb_block(h4, lr - 1, h0) * kBlockWaves + w, blk = id & ((1u << lr) - 1);
    const Job job = decode_job(a, id >> lr);
    const bool fp = BE == NTT_BACKEND_FP || (BE == NTT_BACKEND_MIXED && ((a.fp_mask >> job.table) & 1));
    if (BE != NTT_BACKEND_INT && fp) {
        const typename std::conditional<PRODUCTS, FpProducts<false>, FpArith>::type ar{fp_arith(a, job.table)};
        product_end_block<STREAM>(a, x, job, ar, blk, lane);
    }
    if constexpr (BE != NTT_BACKEND_FP) {
        if (!fp) product_end_block<STREAM>(a, x, job, int_arith(a, job.table), blk, lane);
    }
}

// a word that the forward stages have left (lazy) as a canonical residue, and a canonical word as the arithmetic's value
__device__ __forceinline__ uint64_t canonical_word(double v, const FpArith &ar) { return fp_to_u64(fp_canonical(v, ar.m)); }
__device__ __forceinline__ uint64_t canonical_word(uint64_t v, const IntArith &ar) { return reduce_8q(v, ar.m); }

// v + x * y mod q for canonical words x, y and v as the forward stages have left it; canonical
__device__ __forceinline__ uint64_t add_product(double v, uint64_t x, uint64_t y, const FpArith &ar, uint64_t, uint64_t) {
    const double w = fp_from_u64(y);
    return fp_to_u64(fp_canonical(v + fp_mulmod(fp_from_u64(x), w, ar.m), ar.m));
}
__device__ __forceinline__ uint64_t add_product(uint64_t v, uint64_t x, uint64_t y, const IntArith &ar, uint64_t r0, uint64_t r1) {
    return add_mod(reduce_8q(v, ar.m), mul_mod(x, y, ar.m.q, r0, r1), ar.m.q);
}

// Encryption with several special primes: three waves take their block of u, e0 and e1 of one limb through the last 8 stages; the transformed u stays in
// LDS, from where the other two add u pk_i to their e_i and store the sums, a special limb's through the inverse blocks pass
// (ModDown follows).  (One wave for all three: 14.8 against 11.4 us for 4 limbs of 2^16 words.)
template <class A>
__device__ __forceinline__ void encrypt_block(const NttArgs &a, const uint64_t *pk, uint32_t L, uint32_t LK, uint32_t size_qp, uint32_t t,
                                              uint32_t table, uint32_t blk, uint32_t item, uint32_t items, uint32_t w, uint32_t lane,
                                              const A &ar, uint64_t *u_lds) {
    using T4 = Tile4<8, 8>;
    constexpr bool FP = std::is_base_of<FpArith, A>::value;
    const size_t n = (size_t)1 << a.log_n, off = (size_t)blk * 256, at = off + pair_lane(lane);
    uint64_t *poly = a.out + ((size_t)(w == 0 ? item : items + 2 * item + w - 1) * LK + t) * n;
    const uint64_t r0 = scalar(a.barrett)[2 * table], r1 = scalar(a.barrett)[2 * table + 1];
    uint64_t x[4], k[4], u[4];
#pragma unroll
    for (int j = 0; j < 4; j++) x[j] = poly[off + T4::word(0, lane, j)];
    typename A::Tw tw[4];
    T4::template load_tw<A, 0>(tw, ar, (1u << (a.log_n - 8)) + blk, lane);
    if (w) load_pairs(k, pk + ((size_t)(w - 1) * size_qp + table) * n + at);
    typename A::V v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = A::from_word(x[j]);
    T4::template forward<A>(v, tw, ar, nullptr, lane);
    turn_pairs(v);
    if (w == 0) {
#pragma unroll
        for (int j = 0; j < 4; j++) u[j] = canonical_word(v[j], ar);
        store_pairs(u_lds + pair_lane(lane), u);
    }
    A iar = ar;
    if (w && t >= L) {
        if constexpr (FP)
            iar.table = a.pro_itw_fp + ((size_t)table << a.log_n);
        else
            iar.table = a.pro_itw + ((size_t)table << (a.log_n + 1));
        T4::template load_tw<A, 0>(tw, iar, (1u << (a.log_n - 8)) + blk, lane);
    }
    lds_barrier();
    if (w == 0) return;
    load_pairs(u, u_lds + pair_lane(lane));
    uint64_t o[4];
#pragma unroll
    for (int j = 0; j < 4; j++) o[j] = add_product(v[j], u[j], k[j], ar, r0, r1);
    if (t >= L) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if constexpr (FP)
                v[j] = fp_from_u64(o[j]);
            else
                v[j] = o[j];
        }
        turn_pairs(v);
        T4::template inverse<A>(v, tw, iar, nullptr, lane);
#pragma unroll
        for (int j = 0; j < 4; j++) poly[off + T4::word(0, lane, j)] = A::to_word(v[j]);
    } else {
        store_pairs(poly + at, o);
    }
}

template <int BE>
__global__ __launch_bounds__(192) void encrypt_blocks_kernel(HE_HEAD_PARAMS, const uint64_t *itw) {
    __shared__ uint64_t u_lds[256];
    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    set_inverse_block(a, itw);
    const uint64_t *pk = a.in;
    const uint32_t lr = a.log_n - 8, lane = threadIdx.x & 63, LK = a.map.limbs, L = a.map.split, items = h1, first_item = h5;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t id = limb_block(h4, lr, h0), blk = id & ((1u << lr) - 1), it = id >> lr;
    const uint32_t of_launch = it / LK, item = first_item + of_launch, t = it - of_launch * LK, table = map_table(a.map, t);
    const bool fp = BE == NTT_BACKEND_FP || (BE == NTT_BACKEND_MIXED && ((a.fp_mask >> table) & 1));
    if (BE != NTT_BACKEND_INT && fp)
        encrypt_block(a, pk, L, LK, a.size_qp, t, table, blk, item, items, w, lane, fp_arith(a, table), u_lds);
    if constexpr (BE != NTT_BACKEND_FP) {
        if (!fp) encrypt_block(a, pk, L, LK, a.size_qp, t, table, blk, item, items, w, lane, int_arith(a, table), u_lds);
    }
}

// x times v as the forward stages have left it, mod q, canonical
__device__ __forceinline__ uint64_t lazy_product(double v, uint64_t x, const FpArith &ar, uint64_t, uint64_t) {
    return fp_to_u64(fp_canonical(fp_mulmod(fp_canonical(v, ar.m), fp_from_u64(x), ar.m), ar.m));
}
__device__ __forceinline__ uint64_t lazy_product(uint64_t v, uint64_t x, const IntArith &ar, uint64_t r0, uint64_t r1) {
    return mul_mod(reduce_8q(v, ar.m), x, ar.m.q, r0, r1);
}

// Encryption with one special prime P: the errors e_i never come here.  With d = (u pk_i + e_i) mod P,
// (u pk_i + e_i - d) / P = (u pk_i - NTT(d - e_i)) / P modulo q, so ModDown's transform of d takes e_i along, and the
// special limb gains it as the coefficients that it is: L + 1 transforms of u, 2 L of d - e_i, where those of e_0 and e_1 were
// 2 (L + 1) more.  A wave transforms its block of u and multiplies by both pk_i; a special limb's two products go through the inverse
// blocks pass on a wave each, with the block of u on both (one after the other they would be the launch's longest chain).
// Encryption against three transforms each, us: [60, 40, 40 | 60], 2^16 words, 1, 4, 20 items 29.5 -> 26.7, 66.0 -> 52.5, 212 -> 168,
// primes of 60 bits 33.7 -> 29.0, 71.5 -> 57.8, 249 -> 186, of 50 bits 26.1 -> 23.9, 51.8 -> 46.3, 175 -> 141; 2^12 and 2^13 words, 1 or 2
// items the same within 1 %.
template <bool SPECIAL, class A>
__device__ __forceinline__ void encrypt_products(const NttArgs &a, const uint64_t *pk, uint64_t *wide, uint32_t LK, uint32_t t, uint32_t table,
                                                 uint32_t r, uint32_t blk, uint32_t item, uint32_t lane, const A &ar) {
    using T4 = Tile4<8, 8>;
    constexpr bool FP = std::is_base_of<FpArith, A>::value;
    const size_t n = (size_t)1 << a.log_n, off = (size_t)blk * 256, at = off + pair_lane(lane), key_poly = (size_t)a.size_qp * n;
    const uint64_t *u = a.out + ((size_t)item * LK + t) * n;
    const uint64_t *key = pk + (size_t)table * n + r * key_poly + at;
    uint64_t *out = wide + ((size_t)(2 * item + r) * LK + t) * n;
    const uint64_t r0 = scalar(a.barrett)[2 * table], r1 = scalar(a.barrett)[2 * table + 1];
    uint64_t x[4], k[4], k1[4], o[4];
#pragma unroll
    for (int j = 0; j < 4; j++) x[j] = u[off + T4::word(0, lane, j)];
    typename A::Tw tw[T4::kBlocks];
    T4::template load_tw<A, 0>(tw, ar, (1u << (a.log_n - 8)) + blk, lane);
    load_pairs(k, key);
    if constexpr (!SPECIAL) load_pairs(k1, key + key_poly);
    typename A::V v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = A::from_word(x[j]);
    T4::template forward<A>(v, tw, ar, nullptr, lane);
    A iar = ar;
    if constexpr (SPECIAL) {
        if constexpr (FP)
            iar.table = a.pro_itw_fp + ((size_t)table << a.log_n);
        else
            iar.table = a.pro_itw + ((size_t)table << (a.log_n + 1));
        T4::template load_tw<A, 0>(tw, iar, (1u << (a.log_n - 8)) + blk, lane);
    }
    turn_pairs(v);
#pragma unroll
    for (int j = 0; j < 4; j++) o[j] = lazy_product(v[j], k[j], ar, r0, r1);
    if constexpr (SPECIAL) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if constexpr (FP)
                v[j] = fp_from_u64(o[j]);
            else
                v[j] = o[j];
        }
        turn_pairs(v);
        T4::template inverse<A>(v, tw, iar, nullptr, lane);
#pragma unroll
        for (int j = 0; j < 4; j++) out[off + T4::word(0, lane, j)] = A::to_word(v[j]);
    } else {
        store_pairs(out + at, o);
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = lazy_product(v[j], k1[j], ar, r0, r1);
        store_pairs(out + LK * n + at, o);
    }
}

// (units of an item: its L data limbs, then both polynomials of the special ones)
template <int BE>
__global__ __launch_bounds__(64 * kBlockWaves) void encrypt_products_kernel(HE_HEAD_PARAMS, const uint64_t *itw, uint64_t *wide) {
    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    set_inverse_block(a, itw);
    const uint64_t *pk = a.in;
    const uint32_t lr = a.log_n - 8, lane = threadIdx.x & 63, LK = a.map.limbs, L = a.map.split, units = 2 * LK - L;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t id = limb_block(h4, lr - 1, h0) * kBlockWaves + w, blk = id & ((1u << lr) - 1), it = id >> lr;
    const uint32_t of_launch = it / units, unit = it - of_launch * units, item = h5 + of_launch;
    const bool special = unit >= L;
    const uint32_t t = special ? L + ((unit - L) >> 1) : unit, r = (unit - L) & 1, table = map_table(a.map, t);
    const bool fp = BE == NTT_BACKEND_FP || (BE == NTT_BACKEND_MIXED && ((a.fp_mask >> table) & 1));
    auto block = [&](const auto &ar) {
        if (special)
            encrypt_products<true>(a, pk, wide, LK, t, table, r, blk, item, lane, ar);
        else
            encrypt_products<false>(a, pk, wide, LK, t, table, 0, blk, item, lane, ar);
    };
    if (BE != NTT_BACKEND_INT && fp) block(fp_arith(a, table));
    if constexpr (BE != NTT_BACKEND_FP) {
        if (!fp) block(int_arith(a, table));
    }
}

// Decryption: the flooding noise's block through the last 8 stages, plus c0 + c1 s [+ c2 s^2].
template <class A>
__device__ __forceinline__ void decrypt_block(const NttArgs &a, const DecryptArgs &d, const Job &job, uint32_t blk, uint32_t lane,
                                              const A &ar) {
    using T4 = Tile4<8, 8>;
    const size_t n = (size_t)1 << a.log_n, off = (size_t)blk * 256, at = off + pair_lane(lane), poly = (size_t)a.map.limbs * n;
    const uint64_t q = scalar(a.moduli)[job.table], r0 = scalar(a.barrett)[2 * job.table], r1 = scalar(a.barrett)[2 * job.table + 1];
    const uint64_t *ct = (a.in ? a.in : d.cts[job.poly]) + job.limb * n + at;
    const uint64_t *sk = d.sk + job.limb * n + at;
    uint64_t x[4], c0[4], c1[4], s1[4], c2[4], s2[4];
#pragma unroll
    for (int j = 0; j < 4; j++) x[j] = job.out[off + T4::word(0, lane, j)];
    typename A::Tw tw[4];
    T4::template load_tw<A, 0>(tw, ar, (1u << (a.log_n - 8)) + blk, lane);
    load_pairs(c0, ct);
    load_pairs(c1, ct + poly);
    load_pairs(s1, sk);
    if (d.size > 2) {
        load_pairs(c2, ct + 2 * poly);
        load_pairs(s2, sk + d.sk_stride);
    }
    typename A::V v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = A::from_word(x[j]);
    T4::template forward<A>(v, tw, ar, nullptr, lane);
    turn_pairs(v);
    uint64_t o[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        o[j] = add_mod(add_product(v[j], c1[j], s1[j], ar, r0, r1), c0[j], q);
        if (d.size > 2) o[j] = add_mod(o[j], mul_mod(c2[j], s2[j], q, r0, r1), q);
    }
    store_pairs(job.out + at, o);
}

template <int BE>
__global__ __launch_bounds__(64 * kBlockWaves) void decrypt_blocks_kernel(HE_HEAD_PARAMS, DecryptArgs d) {
    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    const uint32_t lr = a.log_n - 8, lane = threadIdx.x & 63;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t id = logical_block(h4) * kBlockWaves + w, blk = id & ((1u << lr) - 1);
    const Job job = decode_job(a, id >> lr);
    const bool fp = BE == NTT_BACKEND_FP || (BE == NTT_BACKEND_MIXED && ((a.fp_mask >> job.table) & 1));
    if (BE != NTT_BACKEND_INT && fp) decrypt_block(a, d, job, blk, lane, fp_arith(a, job.table));
    if constexpr (BE != NTT_BACKEND_FP) {
        if (!fp) decrypt_block(a, d, job, blk, lane, int_arith(a, job.table));
    }
}

// What the noise's rows pass needs behind NttHead.
struct FloodExtra {
    ChaChaKey key;
    uint64_t stream;
    const uint64_t *cdt;
    uint32_t cdt_len;
    int8_t *errors;
};

// The rows pass of a small Gaussian polynomial that is sampled on the spot: a thread makes four neighbouring coefficients of its tile
// (half of its ChaCha block), a byte each in LDS.  Every limb's workgroups sample anew, on CUs that a launch of a few limbs leaves
// idle, which costs less than a sampler's launch and the bytes' way through memory: decryption of two limbs of
// 2^16 coefficients 10.7 -> 8.9 us.
// ENCRYPT: u instead (a quarter of a ChaCha block a thread); the workgroups behind the tiles make a block's errors a
// thread.  he_encrypt_batch on three limbs and a special one of 2^15, 2^14, 2^12 words 23.2 -> 22.4, 19.1 -> 18.2, 18.0 -> 17.1 us.
template <int LD, bool ENCRYPT>
__global__ __launch_bounds__(256) void flood_rows_kernel(HE_HEAD_PARAMS, FloodExtra f) {
    using T4 = Tile4<10, LD>;
    constexpr int LOGC = 10 - LD, NB = T4::kBlocks;
    constexpr uint32_t C = 1u << LOGC, tiles_per_limb = 256u >> LOGC;
    __shared__ uint64_t lds[(1 << 10) + (1 << 6)], cdt[ENCRYPT ? 1 : kSmallCdt];
    __shared__ uint32_t noise[256];
    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    if constexpr (ENCRYPT) {
        if (blockIdx.x >= h4) {
            const uint32_t i = blockIdx.x - h4, poly = i >> (LD - 3), b = (i & ((1u << (LD - 3)) - 1)) * 256 + threadIdx.x;
            uint32_t w[16];
            chacha20_block(f.key, b, f.stream + 3 * (uint64_t)(poly >> 1) + 1 + (poly & 1), w);
            uint32_t *dst = reinterpret_cast<uint32_t *>(f.errors + ((size_t)poly << a.log_n) + 8 * (size_t)b);
#pragma unroll
            for (int e = 0; e < 2; e++)
                dst[e] = four_bytes(error_value(w[8 * e], w[8 * e + 1]), error_value(w[8 * e + 2], w[8 * e + 3]),
                                    error_value(w[8 * e + 4], w[8 * e + 5]), error_value(w[8 * e + 6], w[8 * e + 7]));
            return;
        }
    }
    const uint32_t lb = logical_block(h4);
    const Job job = decode_job(a, lb / tiles_per_limb);
    const uint32_t col0 = (lb % tiles_per_limb) << LOGC;
    const uint32_t t = ((uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) << 6) | (threadIdx.x & 63);
    if (!ENCRYPT && t < kSmallCdt) cdt[t] = padded_cdt(f.cdt, f.cdt_len, t);
    auto glob = [&](int k, int j) {
        const uint32_t e = T4::word(k, t, j);
        return (size_t)(e >> LOGC) * 256 + col0 + (e & (C - 1));
    };
    auto sample = [&]() {
        const uint32_t at = ((4 * t) >> LOGC) * 256 + col0 + ((4 * t) & (C - 1));
        uint32_t w[16];
        if constexpr (ENCRYPT) {
            chacha20_block(f.key, at >> 4, f.stream + 3 * (uint64_t)job.poly, w);
#pragma unroll
            for (int e = 0; e < 8; e++) w[e] = at & 8 ? w[8 + e] : w[e];
#pragma unroll
            for (int e = 0; e < 4; e++) w[e] = at & 4 ? w[4 + e] : w[e];
            noise[t] = four_bytes(ternary_value(w[0]), ternary_value(w[1]), ternary_value(w[2]), ternary_value(w[3]));
            lds_barrier();
            return;
        }
        chacha20_block(f.key, at >> 3, f.stream + job.poly, w);
        const bool upper = at & 4;
#pragma unroll
        for (int e = 0; e < 8; e++) w[e] = upper ? w[8 + e] : w[e];
        lds_barrier();   // cdt
        gauss_bytes<4>(noise + t, w, cdt);
        lds_barrier();
    };
    auto value = [&](int j) { return (int)reinterpret_cast<const int8_t *>(noise)[T4::word(0, t, j)]; };
    if ((a.fp_mask >> job.table) & 1) {
        const FpArith ar = fp_arith(a, job.table);
        FpArith::Tw tw[NB];
        T4::template load_tw<FpArith, 0>(tw, ar, 1, t);
        sample();
        double v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = (double)value(j);
        T4::template forward<FpArith>(v, tw, ar, lds, t);
#pragma unroll
        for (int j = 0; j < 4; j++) job.out[glob(NB - 1, j)] = FpArith::to_word(v[j]);
    } else {
        const IntArith ar = int_arith(a, job.table);
        IntArith::Tw tw[NB];
        T4::template load_tw<IntArith, 0>(tw, ar, 1, t);
        sample();
        uint64_t v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t x = value(j);
            v[j] = (uint64_t)x + (x < 0 ? ar.m.q : 0);
        }
        T4::template forward<IntArith>(v, tw, ar, lds, t);
#pragma unroll
        for (int j = 0; j < 4; j++) job.out[glob(NB - 1, j)] = v[j];
    }
}

// Which launches deal every limb's workgroups to all XCDs (limb_block).  Otherwise an XCD has a contiguous range of the launch, which
// the passes need that go over the same words one after the other: they meet them in the XCD's L2 (2 x 6 limbs of 2^16 words 10.8 us, dealt
// out 13.1).  But with few limbs of both arithmetics, two XCDs have all the work of a 60-bit limb and two that of a 40-bit one.
//
// Encryption's blocks pass with several special primes (the lines were measured with one as well): up to four items, of which an XCD's range is half of one or less; a range over more evens itself out.
// Together / dealt, us of an encryption on 60 + 40 .. + 60 bits, L + K limbs x items: 2^16, 3 + 1 x 1 32.4 / 29.2, x 2 48.1 / 44.0, x 4
// 64.4 / 63.5, x 6 81.3 / 83.0, x 20 210 / 211, 20 + 4 x 1 96.9 / 84.2, x 4 254 / 240; 2^15, 10 + 2 x 1 43.3 / 38.2, x 4 82.5 / 80.9.  Short
// limbs need more workgroups: 2^14, 12 + 4 x 1 35.0 / 31.1, 3 + 1 x 2 23.4 / 24.1, x 3 27.1 / 29.1, x 6 33.6 / 38.5, 12 + 4 x 2 47.3 / 45.4, x 4
// 62.2 / 61.6; 2^13, 8 + 1 x 1 (288 workgroups) 20.1 / 21.0, 10 + 2 x 1 (384) 27.1 / 26.0, 3 + 1 x 8 26.0 / 29.8.
bool spread_encryption(const NttArgs &a, int backend, uint32_t items, uint64_t wgs) {
    if (backend != NTT_BACKEND_MIXED || items > 4) return false;
    const uint64_t halves = a.log_n >= 15 || items == 1 ? 3 : items == 2 ? 6 : 24;   // workgroups for every two CUs
    return 2 * wgs >= halves * a.cus;
}

// Encryption with one special prime (encrypt_products_kernel), which is shorter: limbs of 2^16 words, of 2^15 up to 16 of them, of fewer a
// single encryption's; not four items of up to eight limbs: half an item an XCD, together or dealt out.  Together / dealt, us, limbs x items: 2^16, 4 x 1
// 27.0 / 25.8, 4 x 3 46.9 / 46.1, 4 x 4 51.9 / 54.1, 4 x 5 64.0 / 61.7, 4 x 10 96.3 / 93.4, 4 x 20 169 / 163, 3 x 4 44.9 / 44.9, 7 x 1 32.9 / 32.4, 7 x 2 47.8 / 48.3,
// 7 x 4 69.6 / 70.5, 7 x 8 120 / 114, 13 x 1 44.9 / 43.0, 13 x 4 106.6 / 102.2; 2^15, 10 x 1 28.4 / 27.3, 4 x 2 26.9 / 26.5, 4 x 4 34.9 / 35.4, 4 x 5 39.7 / 40.5, 10 x 2
// 37.8 / 38.3, 4 x 8 50.5 / 53.1; 2^14, 13 x 1 23.8 / 22.9, 21 x 1 27.9 / 26.6, 4 x 2 22.0 / 22.1; 2^13, 10 x 1 18.5 / 18.6, 10 x 4 26.5 / 28.0.
bool spread_encrypt_products(const NttArgs &a, int backend, uint32_t items, uint32_t limbs) {
    if (backend != NTT_BACKEND_MIXED || 2 * ((uint64_t)items * limbs << (a.log_n - 8)) < 3 * (uint64_t)a.cus) return false;
    if (items == 4 && limbs <= 8) return false;
    return a.log_n >= 16 || (a.log_n == 15 ? (uint64_t)items * limbs <= 16 : items == 1);
}

// A blocks pass with an epilogue, where its caller asks for it (NttArgs::deal) and from three workgroups per CU on.  Behind an inner
// product, which leaves an operand that no order of this launch finds in its XCD's L2: multiplication with 10 + 2 limbs of 2^15 words
// 61.1 / 60.6, 20 + 4 of 2^14 61.9 / 61.2, eight of 10 + 2 of 2^16 446 / 438, rotation with 5 + 1 limbs of 2^16 49.2 / 47.8, 12 + 4 of 2^14
// 41.2 / 40.1; with 2 + 1 of 2^16 (512 workgroups) 27.6 / 27.9.  Behind other passes only long limbs gain, and a single ciphertext's
// encryption: encryption with 3 + 1 limbs of 2^16 words -4.7 %, 10 + 2 of 2^15 -6.2 %, hoisting of four ciphertexts, 4 + 2 limbs of 2^15
// -1.5 %, but encryption of four, 8 + 1 limbs of 2^14 + 7.4 %, hoisting of eight, 5 + 1 of 2^13 + 3.2 %.  ModDown and rescale alone find their
// operands where the passes before them have left them, rescale of 12 + 4 limbs of 2^16 22.3 / 24.2, ModDown of 8 + 1 20.9 / 22.4, and gain
// while a ciphertext has no more limbs than there are XCDs: rescale of 4 + 2 16.0 / 15.5, ModDown of 3 + 1 15.9 / 15.5.
bool spread_epilogue(const NttArgs &a, int backend, uint32_t limbs, uint32_t polys, uint64_t wgs) {
    if (backend != NTT_BACKEND_MIXED || wgs < 3 * (uint64_t)a.cus) return false;
    return a.deal == NTT_DEAL_ALWAYS || (a.deal == NTT_DEAL_LONG && a.log_n >= 15) || (polys <= 2 && limbs * polys <= 8);
}

// Words of a tile, log2: 1024 (4 columns at N = 2^16) for launches that would otherwise leave CUs without a workgroup, 2048
// (twice the columns of a memory access) from 32 limbs of 2^16 words on (2 x 24 limbs 28.0 against 27.3 us); N < 2^12 takes
// tiles of one wave, N = 2^17 needs 2048.
template <bool FWD, int BE, bool SRC_INTT = false, bool MDR = false, bool TILES = false, bool SMALL = false>
hipError_t launch_rows(NttArgs a, uint32_t n_jobs, hipStream_t s) {
    const uint32_t ld = a.log_n - 8;
    const bool large = ((uint64_t)n_jobs << a.log_n) >= ((uint64_t)32 << 16);
    const uint32_t b = ld < 4 ? 8 : (large || ld > 8) ? 11 : 10;
    // (from 2^34 words on, 137 GB, one launch does not hold the threads)
    const uint32_t per_launch = most_workgroups(1u << (b - 2)) >> (a.log_n - b);
    while (n_jobs > per_launch) {
        if (hipError_t e = launch_rows<FWD, BE, SRC_INTT, MDR, TILES, SMALL>(a, per_launch, s)) return e;
        a.first_job += per_launch;
        n_jobs -= per_launch;
    }
    const dim3 grid(n_jobs << (a.log_n - b)), block(1u << (b - 2));
    const NttHead head = ntt_head(a, grid.x, a.first_job);
    const RowsExtra extra = rows_extra(a, FWD);
#define HE_ROWS(LD, B) hipLaunchKernelGGL((ntt_rows_kernel<LD, FWD, BE, SRC_INTT, MDR, B, TILES, SMALL>), grid, block, 0, s, HE_HEAD_ARGS(head), extra)
#define HE_CASE(LD)         \
    case LD:                \
        if (large)          \
            HE_ROWS(LD, 11); \
        else                \
            HE_ROWS(LD, 10); \
        break;
    if constexpr (!SRC_INTT && !TILES) {
        switch (ld) {
            case 1: HE_ROWS(1, 8); return hipGetLastError();
            case 2: HE_ROWS(2, 8); return hipGetLastError();
            case 3: HE_ROWS(3, 8); return hipGetLastError();
            case 9: HE_ROWS(9, 11); return hipGetLastError();
            default: break;
        }
    }
    if constexpr (TILES) {
        switch (ld) {
            HE_CASE(8)
            default: return hipErrorInvalidValue;
        }
    } else {
        switch (ld) {
            HE_CASE(4) HE_CASE(5) HE_CASE(6) HE_CASE(7) HE_CASE(8)
            default: return hipErrorInvalidValue;
        }
    }
#undef HE_CASE
#undef HE_ROWS
    return hipGetLastError();
}

}  // namespace

bool ntt_source_intt_ok(uint32_t log_n, uint32_t n_jobs, uint32_t n_tables) {
    return log_n >= 12 && log_n <= 16 && n_tables <= 64 && ((uint64_t)n_jobs << log_n) <= ((uint64_t)16 << 16);
}

// ModDown + rescale with one special prime: two inverse rows passes in front of every output limb's, which pay as long as the launch is
// small: every limb repeats them, on CUs that are idle otherwise.  The line is where integers, with 2.5 times the instructions, cease to
// gain.  Multiplication with a launch for them -> without, by n_jobs limbs of 2^16 words.  60 bits, the GPU's time, us: 0.1 (n = 2^12, L =
// 2) 27.9 -> 25.7, 1.5 (2^14, 4) 32.8 -> 30.6, 3.5 (2^14, 8) 46.9 -> 44.5, 4 (2^15, 5) 46.7 -> 45.6; back to back: 6 (2^15, 7) 56.5 -> 55.5, 6 (2^16,
// 4) 54.2 -> 54.0, 7 (2^15, 8) 61.7 -> 61.9, 8 (2^16, 5) 62.5 -> 63.5, 10 (2^16, 6) 72.0 -> 75.1.  50 bits: 0.1 22.6 -> 20.1, 1.5 26.2 -> 24.0,
// 4 (2^15, 5) 35.6 -> 33.6, 7 48.6 -> 47.5, 8 48.9 -> 47.5, 10 56.4 -> 55.7, 14 71.0 -> 72.0; 60 and 40 bits: 7 54.1 -> 53.0, 8 57.7 -> 56.2, 10
// 63.3 -> 64.3.  (With primes below 2^50 it would pay to 10.)
bool ntt_two_sources_ok(uint32_t log_n, uint32_t n_jobs, uint32_t n_tables) {
    return ntt_source_intt_ok(log_n, n_jobs, n_tables) && ((uint64_t)n_jobs << log_n) <= ((uint64_t)7 << 16);
}

hipError_t launch_ntt_rows(const NttArgs &args, uint32_t n_jobs, bool forward, int backend, hipStream_t s) {
    if (args.log_n < 9 || args.log_n > 17) return hipErrorInvalidValue;
    NttArgs a = args;
    if (forward && a.pro_mode != NTT_PLAIN && a.pro_mode != NTT_PRO_MODDOWN_RESCALE) {
        // the source in place of the input, which these prologues do not read (see Job::src and rows_input_fp)
        a.in = a.pro_src;
        a.in_poly_stride = a.pro_mode == NTT_PRO_ROUND ? a.pro_log_slots : a.pro_poly_stride;
    }
    if (a.pro_mode == NTT_PRO_SOURCE_INTT_REDUCE) {
        // one instantiation per degree, which follows fp_mask limb by limb: the mask stands for the launch's back end here
        if (!forward || !a.pro_itw || (a.pro_src_fp_mask && !a.pro_itw_fp)) return hipErrorInvalidValue;
        a.fp_mask = backend == NTT_BACKEND_INT ? 0 : (backend == NTT_BACKEND_FP ? ~(uint64_t)0 : a.fp_mask);
        if (a.pro_small) return launch_rows<true, NTT_BACKEND_MIXED, true, false, false, true>(a, n_jobs, s);
        return launch_rows<true, NTT_BACKEND_MIXED, true>(a, n_jobs, s);
    }
    if (forward && a.pro_mode == NTT_PRO_SOURCE_SMALL_REDUCE)
        return backend == NTT_BACKEND_MIXED ? launch_rows<true, NTT_BACKEND_MIXED, false, false, false, true>(a, n_jobs, s)
               : backend                    ? launch_rows<true, NTT_BACKEND_FP, false, false, false, true>(a, n_jobs, s)
                                            : launch_rows<true, NTT_BACKEND_INT, false, false, false, true>(a, n_jobs, s);
    if (forward && a.pro_mode == NTT_PRO_MODDOWN_RESCALE && a.pro_itw) {
        if (!a.pro_k1 || a.pro_poly_stride != a.pro2_poly_stride || a.pro_src2 != a.pro_src + ((size_t)1 << a.log_n)) return hipErrorInvalidValue;
        a.fp_mask = backend == NTT_BACKEND_INT ? 0 : (backend == NTT_BACKEND_FP ? ~(uint64_t)0 : a.fp_mask);
        return launch_rows<true, NTT_BACKEND_MIXED, true, true>(a, n_jobs, s);
    }
    if (forward && a.pro_mode == NTT_PRO_MODDOWN_RESCALE)
        return backend == NTT_BACKEND_MIXED ? launch_rows<true, NTT_BACKEND_MIXED, false, true>(a, n_jobs, s)
               : backend                    ? launch_rows<true, NTT_BACKEND_FP, false, true>(a, n_jobs, s)
                                            : launch_rows<true, NTT_BACKEND_INT, false, true>(a, n_jobs, s);
    if (forward)
        return backend == NTT_BACKEND_MIXED ? launch_rows<true, NTT_BACKEND_MIXED>(a, n_jobs, s)
               : backend                    ? launch_rows<true, NTT_BACKEND_FP>(a, n_jobs, s)
                                            : launch_rows<true, NTT_BACKEND_INT>(a, n_jobs, s);
    if (a.tiles)
        return backend == NTT_BACKEND_MIXED ? launch_rows<false, NTT_BACKEND_MIXED, false, false, true>(a, n_jobs, s)
               : backend                    ? launch_rows<false, NTT_BACKEND_FP, false, false, true>(a, n_jobs, s)
                                            : launch_rows<false, NTT_BACKEND_INT, false, false, true>(a, n_jobs, s);
    return backend == NTT_BACKEND_MIXED ? launch_rows<false, NTT_BACKEND_MIXED>(a, n_jobs, s)
           : backend                    ? launch_rows<false, NTT_BACKEND_FP>(a, n_jobs, s)
                                        : launch_rows<false, NTT_BACKEND_INT>(a, n_jobs, s);
}

// one workgroup for every CU: 4 limbs of 2^16 coefficients 11.5 -> 9.9 us with the blocks pass behind them, 16 of 2^14 10.6 -> 9.4; half as
// many workgroups more and the sampling is no longer hidden (6 of 2^16: 12.4 -> 12.5 us, 24 of 2^14: 11.5 -> 12.0)
bool flood_rows_ok(uint32_t log_n, uint32_t limbs, uint32_t items, uint32_t cus) {
    return log_n >= 12 && log_n <= 16 && limbs <= 64 && ((uint64_t)items * limbs << (log_n - 10)) <= cus;
}

hipError_t launch_flood_rows(const NttArgs &args, ChaChaKey key, uint64_t stream_id, const uint64_t *cdt, uint32_t cdt_len, uint32_t items,
                             int backend, hipStream_t s) {
    const uint32_t n_jobs = items * args.map.limbs;
    if (items == 0 || items > 65535 || args.jobs || cdt_len == 0 || cdt_len >= kSmallCdt || !flood_rows_ok(args.log_n, args.map.limbs, items, args.cus)) return hipErrorInvalidValue;
    NttArgs a = args;
    a.fp_mask = backend == NTT_BACKEND_INT ? 0 : (backend == NTT_BACKEND_FP ? ~(uint64_t)0 : a.fp_mask);
    const dim3 grid(n_jobs << (a.log_n - 10));
    const NttHead head = ntt_head(a, grid.x, 0);
    const FloodExtra f{key, stream_id, cdt, cdt_len, nullptr};
    switch (a.log_n - 8) {
#define HE_CASE(LD) case LD: hipLaunchKernelGGL((flood_rows_kernel<LD, false>), grid, dim3(256), 0, s, HE_HEAD_ARGS(head), f); break;
        HE_CASE(4) HE_CASE(5) HE_CASE(6) HE_CASE(7) HE_CASE(8)
#undef HE_CASE
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// One workgroup for every CU, those with the errors counted: 4 limbs of 2^16 words, 256 of tiles and 64 of errors, take as long as the two
// launches (8.0 us)
bool encrypt_rows_ok(uint32_t log_n, uint32_t limbs, uint32_t items, uint32_t cus) {
    return flood_rows_ok(log_n, limbs, items, cus) && ((uint64_t)items * (limbs + 1) << (log_n - 10)) <= cus;
}

hipError_t launch_encrypt_rows(const NttArgs &args, ChaChaKey key, uint64_t stream_id, int8_t *small, uint32_t items, int backend, hipStream_t s) {
    const uint32_t n_jobs = items * args.map.limbs;
    if (items == 0 || args.jobs || !encrypt_rows_ok(args.log_n, args.map.limbs, items, args.cus)) return hipErrorInvalidValue;
    NttArgs a = args;
    a.fp_mask = backend == NTT_BACKEND_INT ? 0 : (backend == NTT_BACKEND_FP ? ~(uint64_t)0 : a.fp_mask);
    const uint32_t tiles = n_jobs << (a.log_n - 10);
    const dim3 grid(tiles + (2 * items << (a.log_n - 11)));
    const NttHead head = ntt_head(a, tiles, 0);
    const FloodExtra f{key, stream_id, nullptr, 0, small + ((size_t)items << a.log_n)};
    switch (a.log_n - 8) {
#define HE_CASE(LD) case LD: hipLaunchKernelGGL((flood_rows_kernel<LD, true>), grid, dim3(256), 0, s, HE_HEAD_ARGS(head), f); break;
        HE_CASE(4) HE_CASE(5) HE_CASE(6) HE_CASE(7) HE_CASE(8)
#undef HE_CASE
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Limbs of one prime in turn on one wave, which reads its twiddles once: saves up to a third of the traffic (FP64; half of it
// on the integer back end), but each wave then works longer and there are fewer.  It pays from four limbs in turn on
// (two: 29.9 against 27.1 us for 2 x 24 limbs) as long as the launch keeps six waves per SIMD: 12 x 24 limbs 130 -> 112 us,
// 8 x 24 of 60 bits 126 -> 112 us.
constexpr uint32_t kLoopWaves = 6144;

hipError_t launch_ntt_blocks(NttArgs a, uint32_t n_polys, bool forward, int backend, hipStream_t s) {
    if (a.log_n < 9 || a.log_n > 17) return hipErrorInvalidValue;
    const uint32_t blocks = 1u << (a.log_n - 8), repeats = a.jobs ? (a.items ? a.items : 1) : n_polys;
    // (job lists: the groups of one table come into play when even four-limb units leave that many waves)
    if (a.jobs && (uint64_t)a.n_groups * repeats * blocks < 4 * kLoopWaves) a.groups = nullptr;
    const uint32_t kinds = !a.jobs ? a.map.limbs : a.groups ? a.n_groups : a.n_jobs;
    const uint64_t waves = (uint64_t)kinds * blocks;
    const uint32_t split = waves >= kLoopWaves ? 1 : (uint32_t)((kLoopWaves + waves - 1) / waves);
    a.batch = (repeats + split - 1) / split;
    if (a.batch < 4 && !a.groups) a.batch = 1;
    a.n_polys = n_polys;
    const uint64_t wgs = (uint64_t)kinds * ((repeats + a.batch - 1) / a.batch) * (blocks / kBlockWaves);
    if (wgs > most_workgroups(64 * kBlockWaves)) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)wgs), block(64 * kBlockWaves);
    const bool epi = forward && (a.epi_mode == NTT_EPI_SUB_MUL || a.epi_mode == NTT_EPI_SUB_MUL_ADD || a.epi_mode == NTT_EPI_FMA_SUB_MUL);
    a.spread = epi && spread_epilogue(a, backend, kinds, repeats, wgs);
    const NttHead head = ntt_head(a, grid.x, a.batch);
    const BlocksExtra extra = blocks_extra(a, forward);
#define HE_LAUNCH(FWD, EPI, LOOP, PRODUCTS)                                                                                       \
    do {                                                                                                                          \
        if (backend == NTT_BACKEND_MIXED)                                                                                         \
            hipLaunchKernelGGL((ntt_blocks_kernel<FWD, EPI, LOOP, NTT_BACKEND_MIXED, PRODUCTS>), grid, block, 0, s, HE_HEAD_ARGS(head), extra); \
        else if (backend)                                                                                                         \
            hipLaunchKernelGGL((ntt_blocks_kernel<FWD, EPI, LOOP, NTT_BACKEND_FP, PRODUCTS>), grid, block, 0, s, HE_HEAD_ARGS(head), extra); \
        else                                                                                                                      \
            hipLaunchKernelGGL((ntt_blocks_kernel<FWD, EPI, LOOP, NTT_BACKEND_INT, false>), grid, block, 0, s, HE_HEAD_ARGS(head), extra); \
    } while (0)
    const bool loop = a.batch > 1 || a.groups;
    // Twiddles worked out (FpProducts).  In front of an epilogue, on FP64 from one wave for every SIMD on: fewer wait for their two products
    // more than for what they move.  us in this pass, waves, read / worked out: 64 3.40 / 3.50, 256 3.24 / 3.42, 448 3.68 / 3.78, 512 3.36 / 3.52, 1024 4.16 / 4.16,
    // 1280 4.68 / 4.56, 2048 5.60 / 5.10, 4096 8.24 / 7.42; a whole product of 4 + 1 limbs of 2^14 (384 waves) 22.95 / 23.04, of 8 + 2 of 2^12 26.60 / 26.69, of 3 + 1
    // of 2^13 19.96 / 20.06.  With limbs of both arithmetics the integers' waves are the longer ones: 4 + 1 of 2^13 24.53 / 24.39, rotation, 2 + 1 of 2^14 20.55 /
    // 20.48, 24 + 8 of 2^12 42.58 / 42.54.  By itself a pass over 32 * 2^16 words finds them in the L2s in a repeated
    // transform, one over 36 does not.  Transforms, us read / worked out: 2 x 16 limbs of 2^16 words 15.1 / 15.6, 2 x 20 19.1 / 18.0, 2 x 24 back 22.8 /
    // 21.0, of 60 / 40 bits 23.7 / 22.0, 3 x 24 of 2^15 17.3 / 16.8, 4 x 24 of 2^14 12.1 / 12.7.  A job list's words (hoisting's ModUp) come from one
    // buffer and go to another: FP64 from 64 on, 36 limbs 10.46 / 10.50, 49 12.40 / 12.56, 64 15.26 / 15.24, 72 17.38 / 17.20, 100 20.80 / 20.38; 60 / 40 bits 36 limbs
    // 13.32 / 13.28, 49 16.12 / 16.02, 72 22.02 / 21.68.
    const uint64_t line = a.jobs && backend == NTT_BACKEND_FP ? 64 : 36;
    const bool products = ((uint64_t)kinds * repeats << a.log_n) >= line << 16 && !a.in_galois;
    const bool epi_products = backend == NTT_BACKEND_MIXED || (uint64_t)kinds * repeats * blocks >= 4 * (uint64_t)a.cus;
    if (epi && loop)
        HE_LAUNCH(true, true, true, false);
    else if (epi && epi_products)
        HE_LAUNCH(true, true, false, true);
    else if (epi)
        HE_LAUNCH(true, true, false, false);
    else if (forward && loop)
        HE_LAUNCH(true, false, true, false);
    else if (forward && products)
        HE_LAUNCH(true, false, false, true);
    else if (forward)
        HE_LAUNCH(true, false, false, false);
    else if (loop)
        HE_LAUNCH(false, false, true, false);
    else if (products)
        HE_LAUNCH(false, false, false, true);
    else
        HE_LAUNCH(false, false, false, false);
#undef HE_LAUNCH
    return hipGetLastError();
}

// Words that are read for the last time pass by the caches (the digits' words and the sums of a product), from 2^20 words a polynomial of the
// whole batch on: they leave the last-level cache to what the kernels behind them read.  Products, us with such words kept / passing by:
// FP64: 8 x 24 + 8 limbs of 2^16 words 742 / 694, 4 x 389 / 364, 1 x 124.0 / 122.7, 16 x 12 + 4 695 / 648, 2 x 111.4 / 107.2, 2 x 8 + 2 85.5 / 83.3, 8 x
// 12 + 4 of 2^15 186 / 175, 32 x 6 + 2 of 2^13 96.4 / 92.0; 60 / 40 bits: 8 x 12 + 4 of 2^16 456 / 435, 16 x 3 + 1 221 / 215; 60 bits: 8 x 12 + 4
// 533 / 520, 2 x 8 + 2 136.1 / 134.5; below the line 8 x 8 + 1 of 2^13 57.5 / 58.0, 1 x 8 + 2 of 2^16 55.4 / 55.9, 2 x 12 + 4 of 2^15 67.3 / 67.6, but 4 x 3 +
// 1 of 60 bits 86.4 / 84.4.  (The result stored past the caches would be 1 % more, and the caller's next call would read it from memory.)
bool stream_products(uint32_t items, uint32_t L, uint32_t log_n) { return ((uint64_t)items * L << log_n) >= (uint64_t)16 << 16; }

hipError_t launch_ntt_inner(const NttArgs &args, const KsFuseArgs &x, int backend, hipStream_t s) {
    NttArgs a = args;
    if (a.log_n < 9 || a.log_n > 17 || x.items > 0xffffff || x.beta > 255) return hipErrorInvalidValue;
    const uint32_t items = x.items ? x.items : 1;
    if (items > 1 && (x.own_galois || x.add_c0)) return hipErrorInvalidValue;
    const uint64_t pairs = (uint64_t)(x.L + x.K) << (a.log_n - 8);
    // Few blocks: what a wave does in turn (a transform per digit, for a special limb two inverse ones) is the kernel's time, so
    // two or four waves share a block as long as the chip has room for them (two, four waves per SIMD).  One product, one
    // wave against two against four a block: n = 2^12, 3 limbs 35.6 / 30.6 / 23.8 us; n = 2^14, 4 limbs 37.9 / 33.8 / 27.0;
    // n = 2^16, 2 limbs of two digits 44.5 / 38.3; n = 2^15, 10 limbs in 5 digits 78.5 / 74.5 / 76.1; n = 2^16, 6 limbs (2048
    // blocks) 64.4 / 64.3 / 64.5; from 3072 blocks on nothing is gained, at 8192 four waves lose 5 %.
    const int split = items > 1 || x.beta < 2 ? 1 : x.beta > 2 && pairs <= 512 ? 4 : pairs <= 2048 ? 2 : 1;
    const uint64_t wgs = items > 1 ? pairs * ((items + kInnerWaves - 1) / kInnerWaves) : (pairs * split + kInnerWaves - 1) / kInnerWaves;
    if (wgs > most_workgroups(64 * kInnerWaves)) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)wgs), block(64 * kInnerWaves);
    a.in = x.own;
    a.map = LimbMap{x.L + x.K, 0, x.L, x.size_q};
    if (x.add_c0 && x.fold_ct) return hipErrorInvalidValue;
    NttHead head = ntt_head(a, (uint32_t)wgs, x.beta | items << 8);
    if (backend == NTT_BACKEND_MIXED && x.L + x.K <= 16) {
        // The launch walks its limbs from the last to the first.  With more than one workgroup for every CU the integer
        // limbs, whose waves issue three times the instructions, take the last places, so that a CU's second workgroup is one of the short
        // ones (a rotation on [60, 40, 40, 60], two limbs of 2^16 words: 30.4 -> 29.1 us, in this kernel 9.8 -> 8.5)
        const bool reorder = items == 1 && wgs > a.cus;
        uint64_t order = 0;
        uint32_t at = x.L + x.K;
        for (int fp = 0; fp < 2; fp++)
            for (uint32_t t = x.L + x.K; t-- > 0;)
                if (reorder ? (int)((a.fp_mask >> map_table(a.map, t)) & 1) == fp : fp == 0) order |= (uint64_t)t << (4 * --at);
        head.h1 = (uint32_t)order;
        head.h2 = (uint32_t)(order >> 32);
    }
    const uint64_t *addend = x.add_c0 ? x.add_c0 : x.fold_ct;
    const uint32_t inv_first = x.inv_first | (x.add_c0 ? 1u << 16 : 0) | (x.fold_ct ? 1u << 17 : 0);
    InnerFew few{a.pro_itw, addend, x.out, x.own_galois, inv_first, {x.evk.p[0], x.evk.p[1], x.evk.p[2]}};
    InnerMany many{a.pro_itw, addend, x.out, x.own_galois, inv_first, {a.item_stride, x.own_item_stride, x.fold_item_stride}, {}};
    memcpy(many.evk, x.evk.p, sizeof(many.evk));
    // Key words that pass by the caches leave them to the other operands, which the kernels around this one wrote or will read; but a
    // key that would have stayed there for the next call comes from memory then.  So the line is where a key switch's words (key, digits,
    // their sum, input and result) come near the 256 MiB of the last-level cache: 400 limbs of 2^16 words.  Rotations, us with keys kept /
    // passing by (n = 2^16, L + K limbs, so many limbs in all): 16 + 4 (344) 82.6 / 83.7, 10 + 1 (392) 80.0 / 81.7, 20 + 8 (388) 104.8 /
    // 104.9, 22 + 8 (414) 110.6 / 109.1, 18 + 4 (446) 104.7 / 103.7, 24 + 8 (448) 115.0 / 112.8, 12 + 1 (542) 105.6 / 104.9, 24 + 4 (656)
    // 140.5 / 131.8, 14 + 1 (720) 132.7 / 125.4; 60 / 40 bits 10 + 1 87.7 / 89.7, 22 + 8 154.4 / 152.1, 24 + 4 167.8 / 161.4.  A batch's
    // waves share their keys in a CU's cache: eight products 791 / 856.
    const bool stream_keys = items == 1 && (((3 * (uint64_t)x.beta + 2) * (x.L + x.K) + 4 * (uint64_t)x.L) << a.log_n) >= (uint64_t)400 << 16;
    // The digits' words of products whose buffers go round the cache between two uses: see stream_products.
    const bool stream_words = x.fold_ct && stream_products(items, x.L, a.log_n);
    // Twiddles worked out (FpProducts) where one ciphertext's waves are many enough to be bound by what they move: from 3072 on, or with words
    // that pass by the caches; with limbs of both arithmetics up to 11 digits, since a wave works them out once for all of its digits and the waves of
    // integer limbs keep the launch waiting.  One product, us in this kernel read / worked out: 2^16, 24 + 8 limbs 35.2 / 34.7, 20 + 8 30.1 / 28.0, 12 + 3
    // 19.9 / 18.9, 10 + 1 (2816 waves, keys streamed) 30.9 / 30.7, 24 + 2 90.1 / 87.2; 60 / 40 bits 24 + 4 57.3 / 55.9, 16 + 2 (8 digits) 52.2 / 52.5, rotation 50.8 /
    // 50.1, 44 + 4 of 2^14 (11) 39.8 / 39.6, but 24 + 2 of 2^15 (12) 53.4 / 55.3, 24 + 1 100.2 / 101.4, 39 + 1 of 2^14 113.0 / 117.1; whole calls below the line: 832
    // (2^14, 5 + 8 limbs) 31.0 / 31.4, 2816 (2^16, 5 + 6) 44.8 / 45.1.  A batch's waves find them in their
    // CU's cache, read / worked out in this kernel: 4 x 24 + 8 limbs of 2^16 91.3 / 92.6, 16 x 3 + 1 33.6 / 33.8, 8 x 12 + 4 of 2^15 51.7 / 52.2, 60 / 40 bits 8 x 24 + 8
    // 225.9 / 228.8, 4 x 24 + 8 119.1 / 120.4; but with 8192 blocks of FP64, 16 MB of twiddles, they are no loss, 8 x 24 + 8 178.6 / 177.3, and the whole
    // call gains, 691 / 688, 2 x 24 + 8 205.2 / 204.4 (16 x 12 + 4, 4096 blocks, 649 / 652).
    const bool products = backend == NTT_BACKEND_MIXED ? items == 1 && (pairs >= 3072 || stream_keys || stream_words) && x.beta < 12
                          : items == 1                 ? pairs >= 3072 || stream_keys || stream_words
                                                       : pairs >= 8192;
#define HE_INNER_BE(BE, SPLIT, STREAM, PRODUCTS)                                                                                   \
    do {                                                                                                                          \
        if (items == 1 && x.beta <= InnerFew::kDigits)                                                                            \
            hipLaunchKernelGGL((ntt_inner_kernel<BE, SPLIT, STREAM, PRODUCTS, InnerFew>), grid, block, 0, s, HE_HEAD_ARGS(head), few);   \
        else                                                                                                                      \
            hipLaunchKernelGGL((ntt_inner_kernel<BE, SPLIT, STREAM, PRODUCTS, InnerMany>), grid, block, 0, s, HE_HEAD_ARGS(head), many); \
    } while (0)
#define HE_INNER(SPLIT, STREAM, PRODUCTS)                        \
    do {                                                         \
        if (backend == NTT_BACKEND_MIXED)                        \
            HE_INNER_BE(NTT_BACKEND_MIXED, SPLIT, STREAM, PRODUCTS); \
        else if (backend)                                        \
            HE_INNER_BE(NTT_BACKEND_FP, SPLIT, STREAM, PRODUCTS);    \
        else                                                     \
            HE_INNER_BE(NTT_BACKEND_INT, SPLIT, STREAM, false);  \
    } while (0)
#define HE_INNER_ONE(STREAM)            \
    do {                                \
        if (products)                   \
            HE_INNER(1, STREAM, true);  \
        else                            \
            HE_INNER(1, STREAM, false); \
    } while (0)
    if (split == 4)
        HE_INNER(4, 0, false);
    else if (split == 2)
        HE_INNER(2, 0, false);
    else if (stream_keys && stream_words)
        HE_INNER_ONE(3);
    else if (stream_keys)
        HE_INNER_ONE(1);
    else if (stream_words)
        HE_INNER_ONE(2);
    else
        HE_INNER_ONE(0);
#undef HE_INNER_ONE
#undef HE_INNER
#undef HE_INNER_BE
    return hipGetLastError();
}

// Whether a pass over the products of a batch deals a limb's workgroups to all XCDs (limb_block).  A limb's twiddles serve all items:
// dealt out, an XCD keeps its eighth of all of them.  The first pass gains by it once the operands do not fit into the
// L2s, where the launch before has left them otherwise: from 6 * 2^16 words a polynomial on, 10 * 2^16 with limbs of 2^14 and less
// (products of a batch, us together / dealt: 8 x 24 limbs of 2^16 782 / 772, 2 x 3 of 2^16 43.2 / 42.6, 20 x 3 of 2^15 122 / 118, 2 x 3 of
// 2^15 32.4 / 32.7, 8 x 10 of 2^13 62.5 / 61.9; 8 x 3 of 2^14 39.5 / 41.1, 8 x 8 of 2^12 58.7 / 61.6).  The last pass gains a little over the same
// line (8 x 24 + 8 of 2^16 709 / 704, 8 x 12 + 4 of 2^15 182.9 / 180.9, 4 x 6 + 1 of 2^15, 60 / 40 bits, 86.1 / 85.0; 10 x 4 + 1 of 2^14 55.9 / 56.0).
bool spread_products(uint32_t items, uint32_t L, uint32_t log_n) {
    return items > 1 && ((uint64_t)L * items << log_n) >= (uint64_t)(log_n >= 15 ? 6 : 10) << 16;
}

hipError_t launch_tensor_intt_blocks(const NttArgs &args, const TensorFuse &x, uint32_t items, int backend, hipStream_t s) {
    NttArgs a = args;
    a.in = x.ct1;
    if (a.log_n < 9 || a.log_n > 17 || a.jobs || a.map.limbs != x.L || x.L == 0 || items == 0) return hipErrorInvalidValue;
    const uint64_t wgs = ((uint64_t)x.L * items << (a.log_n - 8)) / kBlockWaves;
    if (wgs > most_workgroups(64 * kBlockWaves)) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)wgs), block(64 * kBlockWaves);
    a.spread = spread_products(items, x.L, a.log_n);
    const NttHead h = ntt_head(a, grid.x, x.square ? 1 : 0);
#define HE_TENSOR(BE)                                                                                                             \
    do {                                                                                                                          \
        if (x.last_only)                                                                                                          \
            hipLaunchKernelGGL((tensor_intt_blocks_kernel<BE, true>), grid, block, 0, s, HE_HEAD_ARGS(h), x.ct2, x.d01, x.d2);    \
        else                                                                                                                      \
            hipLaunchKernelGGL((tensor_intt_blocks_kernel<BE, false>), grid, block, 0, s, HE_HEAD_ARGS(h), x.ct2, x.d01, x.d2);   \
    } while (0)
    if (backend == NTT_BACKEND_MIXED)
        HE_TENSOR(NTT_BACKEND_MIXED);
    else if (backend)
        HE_TENSOR(NTT_BACKEND_FP);
    else
        HE_TENSOR(NTT_BACKEND_INT);
#undef HE_TENSOR
    return hipGetLastError();
}

hipError_t launch_product_end(const NttArgs &args, const ProductEnd &x, uint32_t items, int backend, hipStream_t s) {
    NttArgs a = args;
    a.in = x.ct1;
    a.out_poly_stride = 2 * x.L;   // (a job is both polynomials of a limb)
    if (a.log_n < 9 || a.log_n > 17 || a.jobs || a.map.limbs + 1 != x.L || a.map.limbs == 0 || items == 0) return hipErrorInvalidValue;
    const uint64_t wgs = ((uint64_t)a.map.limbs * items << (a.log_n - 8)) / kBlockWaves;
    if (wgs > most_workgroups(64 * kBlockWaves)) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)wgs), block(64 * kBlockWaves);
    a.spread = spread_products(items, x.L, a.log_n);
    const NttHead h = ntt_head(a, grid.x, 0);
    const EndExtra extra{x.cx, x.ct2, x.out, x.p_inv, x.q_last_inv, x.cx_stride};
    // (the factors from half the last-level cache on: smaller ones may be in it for the caller's next product of them)
    const int stream = !stream_products(items, x.L, a.log_n) ? 0 : ((uint64_t)items * x.L << a.log_n) >= (uint64_t)64 << 16 ? 2 : 1;
    // Twiddles worked out (FpProducts): FP64 always; with limbs of both arithmetics, whose integers keep a launch waiting, from 11 limbs of
    // 2^16 words on, when a launch's twiddles are more than its L2s keep for all of its items.  us in this kernel read / worked out, FP64: 8 x 4 + 1
    // limbs of 2^14 8.22 / 7.44, 2 x 8 + 2 of 2^16 13.16 / 12.64, 16 x 3 + 1 26.90 / 27.24, 8 x 24 + 8 147.1 / 141.4; 60 / 40 bits 8 x 4 + 1 of 2^14 9.18 / 9.66, 2 x 8 + 2 of
    // 2^16 14.54 / 14.96, 32 x 6 + 2 of 2^14 34.74 / 35.60, 8 x 8 + 2 of 2^16 45.38 / 45.52, 8 x 12 + 4 68.21 / 68.07, 2 x 16 + 4 27.84 / 26.78, 3 x 24 + 8 of 2^15 29.64 /
    // 28.64, 8 x 24 + 8 of 2^16 147.0 / 141.9.
    const bool products = ((uint64_t)a.map.limbs << a.log_n) >= (uint64_t)11 << 16;
#define HE_END(BE, PRODUCTS)                                                                                       \
    do {                                                                                                           \
        if (stream == 2)                                                                                           \
            hipLaunchKernelGGL((product_end_kernel<BE, 2, PRODUCTS>), grid, block, 0, s, HE_HEAD_ARGS(h), extra);  \
        else if (stream)                                                                                           \
            hipLaunchKernelGGL((product_end_kernel<BE, 1, PRODUCTS>), grid, block, 0, s, HE_HEAD_ARGS(h), extra);  \
        else                                                                                                       \
            hipLaunchKernelGGL((product_end_kernel<BE, 0, PRODUCTS>), grid, block, 0, s, HE_HEAD_ARGS(h), extra);  \
    } while (0)
    if (backend == NTT_BACKEND_MIXED && products)
        HE_END(NTT_BACKEND_MIXED, true);
    else if (backend == NTT_BACKEND_MIXED)
        HE_END(NTT_BACKEND_MIXED, false);
    else if (backend)
        HE_END(NTT_BACKEND_FP, true);
    else
        HE_END(NTT_BACKEND_INT, false);
#undef HE_END
    return hipGetLastError();
}

hipError_t launch_encrypt_blocks(const NttArgs &args, const uint64_t *pk, uint32_t L, uint32_t K, uint32_t size_q, uint32_t items,
                                 int backend, hipStream_t s) {
    NttArgs a = args;
    if (a.log_n < 9 || a.log_n > 17 || items == 0) return hipErrorInvalidValue;
    a.in = pk;
    a.in_poly_stride = items;
    a.map = LimbMap{L + K, 0, L, size_q};
    const dim3 block(192);
    const uint32_t wgs_per_item = (L + K) << (a.log_n - 8), per_launch = most_workgroups(block.x) / wgs_per_item;
    if (per_launch == 0) return hipErrorInvalidValue;
    for (uint32_t first = 0; first < items; first += per_launch) {
        const dim3 grid((items - first < per_launch ? items - first : per_launch) * wgs_per_item);
        a.spread = spread_encryption(a, backend, items, grid.x);
        const NttHead head = ntt_head(a, grid.x, first);
        if (backend == NTT_BACKEND_MIXED)
            hipLaunchKernelGGL(encrypt_blocks_kernel<NTT_BACKEND_MIXED>, grid, block, 0, s, HE_HEAD_ARGS(head), a.pro_itw);
        else if (backend)
            hipLaunchKernelGGL(encrypt_blocks_kernel<NTT_BACKEND_FP>, grid, block, 0, s, HE_HEAD_ARGS(head), a.pro_itw);
        else
            hipLaunchKernelGGL(encrypt_blocks_kernel<NTT_BACKEND_INT>, grid, block, 0, s, HE_HEAD_ARGS(head), a.pro_itw);
        if (hipError_t e = hipGetLastError()) return e;
    }
    return hipSuccess;
}

hipError_t launch_encrypt_products(const NttArgs &args, const uint64_t *pk, uint64_t *wide, uint32_t L, uint32_t K, uint32_t size_q, uint32_t items,
                                   int backend, hipStream_t s) {
    NttArgs a = args;
    if (a.log_n < 9 || a.log_n > 17 || items == 0) return hipErrorInvalidValue;
    a.in = pk;
    a.map = LimbMap{L + K, 0, L, size_q};
    const dim3 block(64 * kBlockWaves);
    const uint32_t wgs_per_item = ((L + 2 * K) << (a.log_n - 8)) / kBlockWaves, per_launch = most_workgroups(block.x) / wgs_per_item;
    if (per_launch == 0) return hipErrorInvalidValue;
    for (uint32_t first = 0; first < items; first += per_launch) {
        const uint32_t now = items - first < per_launch ? items - first : per_launch;
        const dim3 grid(now * wgs_per_item);
        a.spread = spread_encrypt_products(a, backend, items, L + K);
        const NttHead head = ntt_head(a, grid.x, first);
        if (backend == NTT_BACKEND_MIXED)
            hipLaunchKernelGGL(encrypt_products_kernel<NTT_BACKEND_MIXED>, grid, block, 0, s, HE_HEAD_ARGS(head), a.pro_itw, wide);
        else if (backend)
            hipLaunchKernelGGL(encrypt_products_kernel<NTT_BACKEND_FP>, grid, block, 0, s, HE_HEAD_ARGS(head), a.pro_itw, wide);
        else
            hipLaunchKernelGGL(encrypt_products_kernel<NTT_BACKEND_INT>, grid, block, 0, s, HE_HEAD_ARGS(head), a.pro_itw, wide);
        if (hipError_t e = hipGetLastError()) return e;
    }
    return hipSuccess;
}

hipError_t launch_decrypt_blocks(const NttArgs &args, const DecryptArgs &d, uint32_t items, int backend, hipStream_t s) {
    NttArgs a = args;
    if (a.log_n < 9 || a.log_n > 17 || a.jobs || items == 0 || d.size < 2 || d.size > 3) return hipErrorInvalidValue;
    const uint64_t wgs = ((uint64_t)a.map.limbs * items << (a.log_n - 8)) / kBlockWaves;
    if (wgs > most_workgroups(64 * kBlockWaves)) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)wgs), block(64 * kBlockWaves);
    a.in = d.ct;
    const NttHead head = ntt_head(a, grid.x, 0);
    if (backend == NTT_BACKEND_MIXED)
        hipLaunchKernelGGL(decrypt_blocks_kernel<NTT_BACKEND_MIXED>, grid, block, 0, s, HE_HEAD_ARGS(head), d);
    else if (backend)
        hipLaunchKernelGGL(decrypt_blocks_kernel<NTT_BACKEND_FP>, grid, block, 0, s, HE_HEAD_ARGS(head), d);
    else
        hipLaunchKernelGGL(decrypt_blocks_kernel<NTT_BACKEND_INT>, grid, block, 0, s, HE_HEAD_ARGS(head), d);
    return hipGetLastError();
}

}  // namespace he
