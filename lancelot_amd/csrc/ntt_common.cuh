// What the kernels of the transform share: how a job names its limb, the per-limb constants of the two back ends, and the
// prologues that form the input of a forward rows pass.
#pragma once
#include <type_traits>

#include "kernels.h"
#include "modarith.cuh"

namespace he {

namespace {

__host__ __device__ __forceinline__ constexpr uint32_t skew(uint32_t e) { return e + (e >> 4); }

// read-only tables that every lane of a wave reads at one address: through the scalar cache
typedef const double __attribute__((address_space(4))) *ScalarF64;
typedef const uint64_t __attribute__((address_space(4))) *ScalarU64;
__device__ __forceinline__ ScalarF64 scalar(const double *p) { return (ScalarF64)(uintptr_t)p; }
__device__ __forceinline__ ScalarU64 scalar(const uint64_t *p) { return (ScalarU64)(uintptr_t)p; }

// entry idx of a table of (operand, Shoup quotient) pairs
__device__ __forceinline__ Shoup scalar_shoup(const uint64_t *table, size_t idx) { return Shoup{scalar(table)[2 * idx], scalar(table)[2 * idx + 1]}; }

// The arguments of a launch lie in memory that no cache holds yet: the first read of each of their 64-byte lines takes as long as
// one from memory, and the compiler reads a field where it is used, one line after the other in a chain.  A kernel that begins with
// this has asked for all lines at once.
template <int BYTES>
__device__ __forceinline__ void touch_arguments() {
    typedef const uint32_t __attribute__((address_space(4))) *Line;
    const Line p = (Line)__builtin_amdgcn_kernarg_segment_ptr();
    constexpr int LINES = BYTES / 64;
    uint32_t x[LINES];
#pragma unroll
    for (int i = 0; i < LINES; i++) x[i] = p[16 * i];
#pragma unroll
    for (int i = 0; i < LINES; i++) asm volatile("" ::"s"(x[i]));
}

// Workgroup barrier that orders LDS traffic only.  __syncthreads() also waits for every global load and
// store of the wave, which would serialise a prefetch issued before it with the butterflies after it.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Workgroups are dealt round-robin to the 8 XCDs; give every XCD a contiguous range of logical ids so
// that the tiles of one limb (which share a twiddle table) meet in one L2.
// n: workgroups of the launch
__device__ __forceinline__ uint32_t logical_block(uint32_t n) {
    const uint32_t b = blockIdx.x;
    if (n % 8 == 0) return (b % 8) * (n / 8) + b / 8;
    return b;
}

// The same for a launch of limbs of 2^log_tiles workgroups each, where NttArgs::spread says so: an XCD gets the same eighth of every limb.
__device__ __forceinline__ uint32_t limb_block(uint32_t n, uint32_t log_tiles, uint32_t h0) {
    if (log_tiles < 3 || !(h0 >> 16 & 1)) return logical_block(n);
    const uint32_t b = blockIdx.x, k = b >> 3, log_per = log_tiles - 3;
    return (k >> log_per << log_tiles) | (b & 7) << log_per | (k & ((1u << log_per) - 1));
}

// the pointers into a direction's block (NttArgs::tw)
__device__ __forceinline__ const double *block_fp(const uint64_t *block, uint32_t qp, uint32_t log_n) {
    return reinterpret_cast<const double *>(block + ((size_t)(2 * qp) << log_n));
}

// the fields that came as scalar arguments
__device__ __forceinline__ void set_head(NttArgs &a, HE_HEAD_PARAMS) {
    const uint32_t qp = (h0 >> 24) + 1;
    a.in = h_in;
    a.out = h_out;
    a.tw = h_tables;
    a.fp_mask = h_fp_mask;
    a.log_n = h0 & 31;
    a.size_qp = qp;
    a.tw_fp = block_fp(h_tables, qp, a.log_n);
    a.fp_consts = a.tw_fp + ((size_t)qp << a.log_n);
    a.moduli = reinterpret_cast<const uint64_t *>(a.fp_consts + 4 * qp);
    a.barrett = a.moduli + qp;
    a.map = LimbMap{(h0 >> 6) & 0x3ff, h3 & 0x1ff, (h3 >> 9) & 0x1ff, (h3 >> 18) & 0x1ff};
    a.pro_mode = h3 >> 27;
    a.listed = (h0 >> 5) & 1;
    a.in_poly_stride = a.n_jobs = h1;
    a.out_poly_stride = h2;
    a.digit_limbs = h2 & 0xffff;
    a.digits = h2 >> 16;
    a.batch = a.first_job = h5;
}

__device__ __forceinline__ void set_inverse_block(NttArgs &a, const uint64_t *block) {
    a.pro_itw = block;
    a.pro_itw_fp = block_fp(block, a.size_qp, a.log_n);
}

// A unit of a fused base conversion (BconvRows), worked out from the workgroup's number: looked up, it was a trip to memory before the
// one for the words.
struct BconvUnit {
    uint32_t item, copy_first, n_in, n_out;   // (copy_first: the first of a digit's own limbs)
    const uint64_t *in;
    uint64_t *out;
    size_t mat_off;
    uint32_t mx_off, row_off;
    bool up;
    __device__ __forceinline__ uint32_t limb(uint32_t row) const { return up && row >= copy_first ? row + n_in : row; }
};

// packed: limbs of a ModDown polynomial where its inputs are tiled (BconvRows::tiled), 0: they are part of the sum's L + K
__device__ __forceinline__ BconvUnit bconv_unit(const NttArgs &a, uint32_t units, uint32_t K, uint32_t index, uint32_t packed = 0) {
    const uint32_t L = a.map.split, LK = a.map.limbs;
    BconvUnit u;
    u.up = a.pro_mode;
    u.item = index / units;
    u.copy_first = u.mx_off = u.row_off = 0;
    u.mat_off = 0;
    u.n_in = K;
    u.n_out = L;
    if (u.up) {
        const uint32_t d = index - u.item * units;
        u.copy_first = d * K;
        u.n_in = u.copy_first + K < L ? K : L - u.copy_first;
        u.n_out = LK - u.n_in;
        u.mat_off = (size_t)u.copy_first * (LK - K);
        u.mx_off = d * ((LK - K + 3) / 4);
        u.row_off = d * (LK - K);
        u.in = a.in + (((size_t)u.item * L + u.copy_first) << a.log_n);
        u.out = a.out + ((size_t)index * LK << a.log_n);
    } else {
        u.in = a.in + ((packed ? (size_t)index * packed + (packed - K) : (size_t)index * LK + L) << a.log_n);
        u.out = a.out + ((size_t)index * L << a.log_n);
    }
    return u;
}

struct Job {
    const uint64_t *in;
    uint64_t *out;
    uint32_t table;
    uint32_t poly;
    uint32_t limb;
    const uint64_t *src;   // NTT_PRO_SOURCE_[INTT_]REDUCE (rows pass only): the limb that is reduced into this one
    uint32_t src_table;    // NTT_PRO_SOURCE_INTT_REDUCE: its prime
};

// LOOKUP (blocks pass): entries of the list as it is stored, ordered by their primes
template <bool SRC = false, bool LOOKUP = false>
__device__ __forceinline__ Job decode_job(const NttArgs &a, uint32_t job) {
    Job j;
    const size_t n = (size_t)1 << a.log_n;
    if (LOOKUP && a.listed) {
        // job = item * n_jobs + entry of the list
        const uint32_t item = job / a.n_jobs;
        const LimbJob lj = a.jobs[job - item * a.n_jobs];
        j.in = nullptr;
        j.out = a.out + item * a.item_stride + (size_t)lj.data_limb * n;
        j.table = lj.table;
        j.poly = 0;
        j.limb = 0;
        j.src = nullptr;
        j.src_table = 0;
    } else if (a.listed) {
        // job = item * n_jobs + entry of the list, which is worked out (looked up, the entry was a second trip to memory in front of the
        // words)
        const uint32_t item = job / a.n_jobs, r = job - item * a.n_jobs, per = a.map.limbs - a.digit_limbs;
        uint32_t d = r / per;
        d = d < a.digits ? d : a.digits - 1;
        const uint32_t own0 = d * a.digit_limbs, t0 = r - d * per;
        const uint32_t own = own0 + a.digit_limbs < a.map.split ? a.digit_limbs : a.map.split - own0;
        const uint32_t t = t0 < own0 ? t0 : t0 + own, data_limb = d * a.map.limbs + t;
        const bool sourced = a.pro_mode == NTT_PRO_SOURCE_REDUCE || a.pro_mode == NTT_PRO_SOURCE_INTT_REDUCE;
        j.in = sourced ? nullptr : a.in + (size_t)data_limb * n;
        j.out = a.out + (size_t)data_limb * n;
        j.table = map_table(a.map, t);
        j.poly = 0;
        j.limb = 0;
        j.src_table = sourced ? d : 0;
        j.src = sourced ? a.in + (size_t)d * n : nullptr;
        if (item) {
            if (sourced)
                j.src += item * a.pro_item_stride;
            else
                j.in += item * a.item_stride;
            j.out += item * a.item_stride;
        }
    } else {
        j.poly = job / a.map.limbs;
        j.limb = job % a.map.limbs;
        j.in = a.in ? a.in + ((size_t)j.poly * a.in_poly_stride + j.limb) * n : nullptr;
        j.out = a.out + ((size_t)j.poly * a.out_poly_stride + j.limb) * n;
        j.table = map_table(a.map, j.limb);
        // (rows pass: a prologue that has one source limb for every limb of a polynomial finds it, and its stride, in place of the input)
        j.src = a.in + ((size_t)j.poly * a.in_poly_stride << a.log_n);
        j.src_table = SRC ? a.pro_src_table : 0;
    }
    return j;
}

// Per-limb constants of one back end.
struct IntCtx {
    uint64_t q;
    const uint64_t *tw;
};

struct FpCtx {
    FpMod m;
    const double *tw;
};

__device__ __forceinline__ IntCtx int_ctx(const NttArgs &a, uint32_t table) {
    return IntCtx{scalar(a.moduli)[table], a.tw + ((size_t)table << (a.log_n + 1))};
}

__device__ __forceinline__ FpCtx fp_ctx(const NttArgs &a, uint32_t table) {
    const ScalarF64 c = scalar(a.fp_consts) + 4 * (size_t)table;
    return FpCtx{FpMod{c[0], c[1]}, a.tw_fp + ((size_t)table << a.log_n)};
}

// (N^-1 [* w]) for the last multiplication of the inverse transform, centred
__device__ __forceinline__ double inverse_scale(const NttArgs &a, const Job &job, FpMod m) {
    const ScalarF64 c = scalar(a.fp_consts) + 4 * (size_t)job.table;
    const double ninv = c[2];
    if (a.epi_mode != NTT_EPI_MUL) return ninv;
    return fp_reduce(fp_mulmod(fp_from_u64(scalar(a.w)[2 * job.limb]), ninv, m), m);
}

// coefficient at `at` of encoding `poly`, whose slot vector lies in `values`, rounded (NTT_PRO_ROUND)
__device__ __forceinline__ double rounded_coefficient(const NttArgs &a, const double *values, uint32_t poly, uint32_t log_slots, uint32_t at) {
    const uint32_t half = 1u << (a.log_n - 1), log_gap = a.log_n - 1 - log_slots;
    const uint32_t k = at & (half - 1);
    if (k & ((1u << log_gap) - 1)) return 0.0;
    const double *v = values + ((size_t)poly << (log_slots + 1));
    const uint32_t slot = __brev(k >> log_gap) >> (32 - log_slots);
    return round(v[2 * slot + (at >= half ? 1 : 0)] * a.pro_fix);
}
__device__ __forceinline__ double rounded_coefficient(const NttArgs &a, const Job &job, uint32_t at) {
    return rounded_coefficient(a, reinterpret_cast<const double *>(a.in), job.poly, a.in_poly_stride, at);
}
// ... as a residue
__device__ __forceinline__ uint64_t rounded_residue(double x, uint64_t q, uint64_t r1) {
    const uint64_t r = barrett64((uint64_t)fabs(x), q, r1);
    return x < 0 ? neg_mod(r, q) : r;
}

// s + e modulo q for a residue s and a small e
__device__ __forceinline__ uint64_t add_small(uint64_t s, int e, uint64_t q) {
    int64_t t = (int64_t)s + e;
    t += t < 0 ? (int64_t)q : 0;
    return (uint64_t)(t >= (int64_t)q ? t - (int64_t)q : t);
}

// Input of a forward rows pass (a.pro_mode): word j of the thread from global offset glob(j) of its limb, as exact
// doubles; returns whether they have to be reduced before the first stage (else they are canonical).
// MDR: the launch's mode is NTT_PRO_MODDOWN_RESCALE (a template argument: its operands cost the other modes registers, 90 instead of
// 64 for the mixed rows pass; encryption 69.1 -> 68.6 us, a Krum round of 10 clients 4.30 -> 4.23 ms)
// GIVEN: its two sources are in ts and ds already.
template <bool MDR, bool GIVEN, int W, typename Glob>
__device__ __forceinline__ bool rows_input_fp(double (&v)[W], const NttArgs &a, const Job &job, const FpCtx &c, Glob glob, const uint64_t *ts,
                                              const uint64_t *given_ds) {
    if constexpr (MDR) {
        const uint64_t *tsrc = a.pro_src + ((size_t)job.poly * a.pro_poly_stride << a.log_n);
        const uint64_t *dsrc = a.pro_src2 + ((size_t)job.poly * a.pro2_poly_stride << a.log_n);
        const FpMod ml = fp_ctx(a, a.pro_last).m;
        const double w = fp_from_u64(scalar(a.pro_w)[2 * job.limb]), wlast = fp_from_u64(scalar(a.pro_w)[2 * a.pro_last]);
        const uint64_t qj = scalar(a.moduli)[job.table], rj = scalar(a.barrett)[2 * job.table + 1];
        const uint64_t qlast = scalar(a.moduli)[a.pro_last], rlast = scalar(a.barrett)[2 * a.pro_last + 1];
#pragma unroll
        for (int j = 0; j < W; j++) {
            const uint64_t ds = GIVEN ? given_ds[j] : dsrc[glob(j)], t = GIVEN ? ts[j] : tsrc[glob(j)];
            const uint64_t dl = GIVEN || a.pro_k1 ? barrett64(ds, qlast, rlast) : ds;
            const uint64_t dj = GIVEN || a.pro_k1 ? barrett64(ds, qj, rj) : job.in[glob(j)];
            // coefficient of the dropped limb of the ModDown result, canonical mod q_last
            const double r = fp_canonical(fp_from_u64(t) - fp_mulmod(fp_from_u64(dl), wlast, ml), ml);
            v[j] = fp_mulmod(fp_from_u64(dj), w, c.m) + fp_reduce(r, c.m);
        }
        return true;
    }
    if (a.pro_mode == NTT_PRO_BROADCAST_REDUCE) {
        // one source limb for every limb: it may exceed this limb's prime, so reduce first
        const uint64_t *src = job.src;
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = fp_from_u64(src[glob(j)]);
        return true;
    }
    if (a.pro_mode == NTT_PRO_SOURCE_REDUCE) {
        const uint64_t q = scalar(a.moduli)[job.table], r1 = scalar(a.barrett)[2 * job.table + 1];
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = fp_from_u64(barrett64(job.src[glob(j)], q, r1));
    } else if (a.pro_mode == NTT_PRO_SMALL) {
        const int8_t *src = reinterpret_cast<const int8_t *>(a.in) + ((size_t)job.poly << a.log_n);
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = (double)src[glob(j)];
    } else if (a.pro_mode == NTT_PRO_ROUND) {
        // (an integer below 2^62 in magnitude: the quotient estimate is off by at most 1, the fused multiply-add exact)
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = fp_reduce(rounded_coefficient(a, job, (uint32_t)glob(j)), c.m);
    } else {
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = fp_from_u64(job.in[glob(j)]);
    }
    return false;
}

// The same on the integer back end: residues below q.
template <bool MDR, bool GIVEN, int W, typename Glob>
__device__ __forceinline__ void rows_input_int(uint64_t (&v)[W], const NttArgs &a, const Job &job, uint64_t q, Glob glob, const uint64_t *ts,
                                               const uint64_t *given_ds) {
    if constexpr (MDR) {
        const uint64_t r1 = scalar(a.barrett)[2 * job.table + 1];
        const uint64_t *tsrc = a.pro_src + ((size_t)job.poly * a.pro_poly_stride << a.log_n);
        const uint64_t *dsrc = a.pro_src2 + ((size_t)job.poly * a.pro2_poly_stride << a.log_n);
        const uint64_t ql = scalar(a.moduli)[a.pro_last];
        const Shoup w = scalar_shoup(a.pro_w, job.limb), wlast = scalar_shoup(a.pro_w, a.pro_last);
        const uint64_t rlast = scalar(a.barrett)[2 * a.pro_last + 1];
#pragma unroll
        for (int j = 0; j < W; j++) {
            const uint64_t ds = GIVEN ? given_ds[j] : dsrc[glob(j)], t = GIVEN ? ts[j] : tsrc[glob(j)];
            const uint64_t dl = GIVEN || a.pro_k1 ? barrett64(ds, ql, rlast) : ds;
            const uint64_t dj = GIVEN || a.pro_k1 ? barrett64(ds, q, r1) : job.in[glob(j)];
            const uint64_t r = sub_mod(t, mul_shoup(dl, wlast, ql), ql);
            v[j] = add_mod(mul_shoup(dj, w, q), barrett64(r, q, r1), q);
        }
    } else if (a.pro_mode == NTT_PRO_BROADCAST_REDUCE || a.pro_mode == NTT_PRO_SOURCE_REDUCE) {
        const uint64_t r1 = scalar(a.barrett)[2 * job.table + 1];
        const uint64_t *src = job.src;
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = barrett64(src[glob(j)], q, r1);
    } else if (a.pro_mode == NTT_PRO_SMALL) {
        const int8_t *src = reinterpret_cast<const int8_t *>(a.in) + ((size_t)job.poly << a.log_n);
#pragma unroll
        for (int j = 0; j < W; j++) {
            const int64_t x = src[glob(j)];
            v[j] = (uint64_t)x + (x < 0 ? q : 0);
        }
    } else if (a.pro_mode == NTT_PRO_ROUND) {
        const uint64_t r1 = scalar(a.barrett)[2 * job.table + 1];
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = rounded_residue(rounded_coefficient(a, job, (uint32_t)glob(j)), q, r1);
    } else {
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = job.in[glob(j)];
    }
}

// Input of a forward rows pass in the mode NTT_PRO_SOURCE_SMALL_REDUCE.  x: the rounded coefficients (pro_values)
template <typename Glob>
__device__ __forceinline__ void small_source(uint64_t (&v)[4], double (&x)[4], const NttArgs &a, const Job &job, bool values, Glob glob) {
    const uint64_t q = scalar(a.moduli)[job.table], r1 = scalar(a.barrett)[2 * job.table + 1], p = scalar(a.moduli)[a.pro_src_table];
    const int8_t *small = a.pro_small + ((size_t)job.poly << a.log_n);
    int e[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        v[j] = job.src[glob(j)];
        e[j] = small[glob(j)];
    }
    if (values) {
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = rounded_coefficient(a, a.pro_values, job.poly >> 1, a.pro_log_slots, (uint32_t)glob(j));
    }
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = add_small(barrett64(add_small(v[j], e[j], p), q, r1), -e[j], q);
}

// a of the lanes whose bit BIT is set and b of the lanes where it is not change places: the words' register bit becomes that
// bit of the lane
template <int BIT>
__device__ __forceinline__ void swap_lane_bit(uint32_t &a, uint32_t &b) {
    if constexpr (BIT >= 4) {
        const auto r = BIT == 5 ? __builtin_amdgcn_permlane32_swap(a, b, false, false) : __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = r[0];
        b = r[1];
    } else if constexpr (BIT >= 2) {
        // a row's lanes shifted by 8 or 4; the banks (4 lanes) with the bit take b from below, the others a from above
        constexpr int SHIFT = 1 << BIT, WITH = BIT == 3 ? 0xc : 0xa;
        const uint32_t x = (uint32_t)__builtin_amdgcn_update_dpp((int)a, (int)b, 0x110 + SHIFT, 0xf, WITH, false);
        b = (uint32_t)__builtin_amdgcn_update_dpp((int)b, (int)a, 0x100 + SHIFT, 0xf, 0xf ^ WITH, false);
        a = x;
    } else {
        constexpr int PERM = BIT == 1 ? 0x4e : 0xb1;   // lanes 2 3 0 1, or 1 0 3 2, of every four
        const bool with = (__lane_id() >> BIT) & 1;
        const uint32_t pa = (uint32_t)__builtin_amdgcn_mov_dpp((int)a, PERM, 0xf, 0xf, true);
        const uint32_t pb = (uint32_t)__builtin_amdgcn_mov_dpp((int)b, PERM, 0xf, 0xf, true);
        a = with ? pb : a;
        b = with ? b : pa;
    }
}

template <int BIT>
__device__ __forceinline__ void swap_lane_bit(uint64_t &a, uint64_t &b) {
    uint32_t al = (uint32_t)a, ah = (uint32_t)(a >> 32), bl = (uint32_t)b, bh = (uint32_t)(b >> 32);
    swap_lane_bit<BIT>(al, bl);
    swap_lane_bit<BIT>(ah, bh);
    a = ((uint64_t)ah << 32) | al;
    b = ((uint64_t)bh << 32) | bl;
}

// Two stages (ST = 1: only the first of them) on four words; tw entries: the first stage's twiddle, then the two of the
// second.
struct IntArith {
    using V = uint64_t;
    struct Tw {
        Shoup s[3];
    };
    IntMod m;
    const uint64_t *table;
    static __device__ __forceinline__ V from_word(uint64_t x) { return x; }
    static __device__ __forceinline__ uint64_t to_word(V v) { return v; }
    template <int ST, bool UNIFORM>
    __device__ __forceinline__ Tw load(uint32_t idx) const {
        auto at = [&](size_t i) { return UNIFORM ? scalar_shoup(table, i) : load_shoup(table, i); };
        Tw t;
        t.s[0] = at(idx);
        t.s[1] = t.s[2] = Shoup{0, 0};
        if (ST == 2) {
            t.s[1] = at(2 * (size_t)idx);
            t.s[2] = at(2 * (size_t)idx + 1);
        }
        return t;
    }
    __device__ __forceinline__ Tw load_last(uint32_t scale, uint32_t t) const { return load<2, false>((scale << 6) + t); }
    template <int ST>
    __device__ __forceinline__ void ct(V *v, const Tw &t) const {
        ct_butterfly(v[0], v[2], t.s[0], m);
        ct_butterfly(v[1], v[3], t.s[0], m);
        if (ST == 2) {
            ct_butterfly(v[0], v[1], t.s[1], m);
            ct_butterfly(v[2], v[3], t.s[2], m);
        }
    }
    template <int ST>
    __device__ __forceinline__ void gs(V *v, const Tw &t) const {
        if (ST == 2) {
            gs_butterfly(v[0], v[1], t.s[1], m);
            gs_butterfly(v[2], v[3], t.s[2], m);
        }
        gs_butterfly(v[0], v[2], t.s[0], m);
        gs_butterfly(v[1], v[3], t.s[0], m);
    }
    __device__ __forceinline__ void reduce(V *) const {}
    __device__ __forceinline__ void settle(V *) const {}
};

// Bounds, in units of 2^50 > q: |v| < 8 keeps every value exact.  The twiddles are centred, so a product with a word below b is at most
// 0.5 + 0.1875 b (the quotient's estimate is three roundings off).
// Forward, a stage takes b to 1.1875 b + 0.5: six stages from 1 (canonical words, a conversion's sums up to 1.01) end at 7.7, from 0.5
// (reduced) at 6.2, four from 2.63 at 7.9.  One reduction in a rows pass that leaves at most three stages behind it (2.63), one in the
// middle of the blocks pass (3.63 at its end): see Tile4.
// Inverse, a block of two stages leaves sums of four words at 4 b, sums of two products at 1 + 0.75 b, and 0.5 + 0.75 b and less in the
// others.  Reducing the first two (settle) keeps b below 2 from canonical words on: 1, 1.25, 1.44, 1.58, 1.69, 1.77, 1.83, 1.87, ..., and 4 b
// below 8.
struct FpArith {
    using V = double;
    struct Tw {
        double w[3];
    };
    FpMod m;
    const double *table;
    static __device__ __forceinline__ V from_word(uint64_t x) { return __longlong_as_double((long long)x); }
    static __device__ __forceinline__ uint64_t to_word(V v) { return (uint64_t)__double_as_longlong(v); }
    // UNIFORM: idx is the same in every lane of the wave
    template <int ST, bool UNIFORM>
    __device__ __forceinline__ Tw load(uint32_t idx) const {
        auto at = [&](size_t i) { return UNIFORM ? (double)scalar(table)[i] : table[i]; };
        Tw t;
        t.w[0] = at(idx);
        t.w[1] = t.w[2] = 0.0;
        if (ST == 2) {
            t.w[1] = at(2 * (size_t)idx);
            t.w[2] = at(2 * (size_t)idx + 1);
        }
        return t;
    }
    // the last block of a wave's 256 words (Tile4<8, 8>, `scale` as in load_tw)
    __device__ __forceinline__ Tw load_last(uint32_t scale, uint32_t t) const { return load<2, false>((scale << 6) + t); }
    __device__ __forceinline__ void ct1(V &x, V &y, double w) const {
        const double t = fp_mulmod(y, w, m);
        y = x - t;
        x = x + t;
    }
    __device__ __forceinline__ void gs1(V &x, V &y, double w) const {
        const double d = x - y;
        x = x + y;
        y = fp_mulmod(d, w, m);
    }
    template <int ST>
    __device__ __forceinline__ void ct(V *v, const Tw &t) const {
        ct1(v[0], v[2], t.w[0]);
        ct1(v[1], v[3], t.w[0]);
        if (ST == 2) {
            ct1(v[0], v[1], t.w[1]);
            ct1(v[2], v[3], t.w[2]);
        }
    }
    template <int ST>
    __device__ __forceinline__ void gs(V *v, const Tw &t) const {
        if (ST == 2) {
            gs1(v[0], v[1], t.w[1]);
            gs1(v[2], v[3], t.w[2]);
        }
        gs1(v[0], v[2], t.w[0]);
        gs1(v[1], v[3], t.w[0]);
    }
    __device__ __forceinline__ void reduce(V *v) const {
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = fp_reduce(v[j], m);
    }
    __device__ __forceinline__ void settle(V *v) const {
        v[0] = fp_reduce(v[0], m);
        v[1] = fp_reduce(v[1], m);
    }
    // v s as canonical values for the words that the inverse's last block of ST stages has left: with v[0] (and v[1] after one stage)
    // reduced they are at most 2.4, the products at most 0.95 q
    template <int ST>
    __device__ __forceinline__ void scale(V *v, double s) const {
        v[0] = fp_reduce(v[0], m);
        if (ST == 1) v[1] = fp_reduce(v[1], m);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const double p = fp_mulmod(v[j], s, m);
            v[j] = p < 0.0 ? p + m.q : p;
        }
    }
    template <int ST>
    __device__ __forceinline__ void scale(uint64_t *w, V *v, double s) const {
        scale<ST>(v, s);
#pragma unroll
        for (int j = 0; j < 4; j++) w[j] = fp_to_u64(v[j]);
    }
};

// The same with the twiddles of the last block of a wave's 256 words (Tile4<8, 8>) worked out.  They are three quarters of those of a blocks
// pass and, read from their own places, nearly as many bytes as its words; but entry i of the table is psi to the power of i bit-reversed, so
// for numbers without a common bit entry x + y is entry x times entry y: one of the wave's block times one of the first 128, which all
// blocks of the limb read.  It pays where a kernel is bound by what it moves.  us with the entries read / worked out, n = 2^16: the last
// blocks pass of a product of 12 + 4 limbs 11.0 / 9.5, of 24 + 8 18.4 / 16.9, of eight of those (product_end_kernel) 146 / 140, of a
// rotation 8.8 / 8.0 and 15.5 / 14.1, 2^14, 12 + 4 4.6 / 4.5; the inner product of rotations 17.8 / 16.4 and 35.4 / 33.9.  Not where waves wait for
// each other or for scattered words: inner product with blocks shared by two waves, 2^14, 12 + 4 6.8 / 7.2, encryption, 12 + 4 16.8 / 17.5,
// rotation's first pass 8.7 / 9.2 and 8.8 / 10.5, the first pass of eight products 92 / 94.  (In pairs for the integer butterflies a product and
// its quotient would take as many multiplications as a butterfly and a half.)
// The product of two centred entries is at most 0.6 q.  Inverse: the first block of two stages then leaves at most 1.4 in place of 1.25,
// and the bounds above still rise to 2.  Forward: the last two stages end at 3.8 in place of 3.63; CENTRED keeps 3.63, which the inner
// product's sums need (FpSums).
template <bool CENTRED>
struct FpProducts : FpArith {
    __device__ __forceinline__ Tw load_last(uint32_t scale, uint32_t t) const {
        const double b0 = scalar(table)[(size_t)scale << 6], b1 = scalar(table)[(size_t)scale << 7];
        Tw w{{fp_mulmod(table[t], b0, m), fp_mulmod(table[2 * t], b1, m), fp_mulmod(table[2 * t + 1], b1, m)}};
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (CENTRED) w.w[i] = fp_reduce(w.w[i], m);
        return w;
    }
};

// A tile of 2^B words, 4 per thread, whose stages 0 .. LD-1 pair the tile bits B-1, B-2, ...; block k holds the stages
// 2k and 2k+1.  In block k thread t has the words ((t >> low) << (low + 2)) | (j << low) | (t mod 2^low), low = B - 2k - 2,
// and the twiddle index of its first stage is 2^(2k) + (t >> low).  Between the blocks k and k+1 words move inside groups
// of 2^low threads: inside a wave from low = 6 on.
template <int B, int LD>
struct Tile4 {
    static constexpr int kBlocks = (LD + 1) / 2;
    static_assert(B >= 8 && 2 * kBlocks <= B, "four words of every block lie inside the tile");
    static constexpr int stages(int k) { return LD - 2 * k >= 2 ? 2 : 1; }
    // the forward block before which words are reduced (FpArith): whole limbs and the blocks pass (B = LD), rows passes
    static constexpr int kReduceBefore = B == LD ? (LD <= 10 ? 2 : 3) : LD <= 2 ? kBlocks : LD <= 5 ? 1 : LD <= 7 ? 2 : 3;
    static __device__ __forceinline__ uint32_t word(int k, uint32_t t, int j) {
        const int low = B - 2 * k - 2;
        return ((t >> low) << (low + 2)) | ((uint32_t)j << low) | (t & ((1u << low) - 1));
    }
    static __device__ __forceinline__ uint32_t index(int k, uint32_t t) { return (1u << (2 * k)) + (t >> (B - 2 * k - 2)); }

    template <class A, int K>
    static __device__ __forceinline__ void load_tw(typename A::Tw *tw, const A &ar, uint32_t scale, uint32_t t) {
        // scale: the tile's number within the limb enters the index as its upper bits (blocks pass), 1 for a rows pass
        if constexpr (B == 8 && LD == 8 && K == kBlocks - 1)
            tw[K] = ar.load_last(scale, t);
        else
            tw[K] = ar.template load<stages(K), (B - 2 * K - 2 >= 6)>(((scale - 1) << (2 * K)) + index(K, t));
        if constexpr (K + 1 < kBlocks) load_tw<A, K + 1>(tw, ar, scale, t);
    }
    // From the layout of block KLO to that of block KLO + 1, or back: the register bits and the thread bits low - 1 and low - 2
    // change places.  Inside a wave that is done in registers (8 to 16 instructions for 4 words; through LDS 8 accesses
    // and about 300 cycles before the next butterfly starts).
    static constexpr bool in_wave(int klo) { return B - 2 * klo - 2 <= 6; }
    template <int KLO>
    static __device__ __forceinline__ void swap_words(uint64_t *w) {
        constexpr int LOW = B - 2 * KLO - 2;
        swap_lane_bit<LOW - 1>(w[0], w[2]);
        swap_lane_bit<LOW - 1>(w[1], w[3]);
        swap_lane_bit<LOW - 2>(w[0], w[1]);
        swap_lane_bit<LOW - 2>(w[2], w[3]);
    }
    template <class A, int KLO, bool BACK>
    static __device__ __forceinline__ void exchange(typename A::V *v, uint64_t *lds, uint32_t t) {
        uint64_t w[4];
#pragma unroll
        for (int j = 0; j < 4; j++) w[j] = A::to_word(v[j]);
        if constexpr (in_wave(KLO)) {
            swap_words<KLO>(w);
        } else {
            // (bits low and low + 1 of a thread's first word are clear, and low >= 4: the words' slots lie a constant apart)
            constexpr int FROM = BACK ? KLO + 1 : KLO, TO = BACK ? KLO : KLO + 1;
            static_assert(B - 2 * KLO - 4 >= 4, "skew() adds to the words' distances");
            uint64_t *from = lds + skew(word(FROM, t, 0));
            const uint64_t *to = lds + skew(word(TO, t, 0));
#pragma unroll
            for (int j = 0; j < 4; j++) from[j * skew(1u << (B - 2 * FROM - 2))] = w[j];
            lds_barrier();
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = to[j * skew(1u << (B - 2 * TO - 2))];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = A::from_word(w[j]);
    }
    // (lds: only for exchanges across waves)
    template <class A, int K = 0>
    static __device__ __forceinline__ void forward(typename A::V *v, const typename A::Tw *tw, const A &ar, uint64_t *lds, uint32_t t) {
        ar.template ct<stages(K)>(v, tw[K]);
        if constexpr (K + 1 < kBlocks) {
            exchange<A, K, false>(v, lds, t);
            if constexpr (K + 1 == kReduceBefore) ar.reduce(v);
            forward<A, K + 1>(v, tw, ar, lds, t);
        }
    }
    template <class A, int K = kBlocks - 1>
    static __device__ __forceinline__ void inverse(typename A::V *v, const typename A::Tw *tw, const A &ar, uint64_t *lds, uint32_t t) {
        ar.template gs<stages(K)>(v, tw[K]);
        if constexpr (K > 0) {
            ar.settle(v);
            exchange<A, K - 1, true>(v, lds, t);
            inverse<A, K - 1>(v, tw, ar, lds, t);
        } else if constexpr (B == 8 && LD == 8) {
            ar.settle(v);   // (blocks pass: the rows pass goes on)
        }
    }
};

// Where the words of thread t of a tile of 2^B words lie in a limb between the inverse rows pass and a fused base conversion (a rows
// pass ends, and the conversion begins, with the words t + j 2^(B - 2) of the tile in thread t): words j = 0, 1 from here on, words 2, 3
// from 512 words further on.  Half a tile of 2048 words (a tile of 1024) lies together, so that every access is one of 16 bytes a lane
// over whole lines, and a workgroup's accesses go to all channels of its L2.  (As [row][column] a tile of 2048 words at N = 2^16 is 256
// segments of 64 bytes, 2 KiB apart: a quarter of the channels.)
template <int B, int LD>
__device__ __forceinline__ uint32_t conversion_word(uint32_t tile, uint32_t t) {
    if constexpr (B == 10) {
        return (tile << 10) + 2 * t;
    } else {
        static_assert(B == 11, "tiles of the passes from 2^12 words on");
        constexpr int LOGH = 10 - LD;   // columns of half a tile, log2
        const uint32_t u = ((t >> (LOGH + 1)) << LOGH) | (t & ((1u << LOGH) - 1));
        return (tile << 11) + ((t >> LOGH & 1) << 10) + 2 * u;
    }
}

__device__ __forceinline__ IntArith int_arith(const NttArgs &a, uint32_t table) {
    const IntCtx c = int_ctx(a, table);
    return IntArith{int_mod(c.q), c.tw};
}

__device__ __forceinline__ FpArith fp_arith(const NttArgs &a, uint32_t table) {
    const FpCtx c = fp_ctx(a, table);
    return FpArith{c.m, c.tw};
}


// four consecutive words of a lane, as two 16-byte accesses (the polynomials are only 8-byte aligned for certain)
typedef uint64_t Words2 __attribute__((ext_vector_type(2), aligned(8)));

__device__ __forceinline__ void load4(uint64_t *v, const uint64_t *p) {
    const Words2 a = reinterpret_cast<const Words2 *>(p)[0], b = reinterpret_cast<const Words2 *>(p)[1];
    v[0] = a.x;
    v[1] = a.y;
    v[2] = b.x;
    v[3] = b.y;
}

__device__ __forceinline__ void store4(uint64_t *p, const uint64_t *v) {
    reinterpret_cast<Words2 *>(p)[0] = Words2{v[0], v[1]};
    reinterpret_cast<Words2 *>(p)[1] = Words2{v[2], v[3]};
}

__device__ __forceinline__ void load_tiled(uint64_t *v, const uint64_t *p) {
    const Words2 a = reinterpret_cast<const Words2 *>(p)[0], b = reinterpret_cast<const Words2 *>(p + 512)[0];
    v[0] = a.x;
    v[1] = a.y;
    v[2] = b.x;
    v[3] = b.y;
}

__device__ __forceinline__ void store_tiled(uint64_t *p, const uint64_t *v) {
    reinterpret_cast<Words2 *>(p)[0] = Words2{v[0], v[1]};
    reinterpret_cast<Words2 *>(p + 512)[0] = Words2{v[2], v[3]};
}

// A wave's block of 256 words in memory: a lane's words are not the four neighbours 4 lane .. 4 lane + 3 of the last register block
// (Tile4<8, 8>) but two pairs, 128 words apart, so that a 16-byte access of the wave covers 1 KiB without holes.  Four neighbours took
// two accesses that touched the same sixteen lines one after the other, half of each.  turn_pairs goes from one layout to the other:
// word bit 1 (a register's) and word bit 7 (lane bit 5) change places, four instructions.  Everything between the stages and memory
// (products, epilogues) works on pairs.  Before / after, us: L = 24, K = 8 a product 141.6 / 140.9, eight 782 / 769, a rotation 116.9 / 116.6;
// n = 2^15, 10 of 12 limbs of 60 / 40 bits 63.6 / 62.4; 2 x 24 limbs of 2^16 words back the same 24.4.
__device__ __forceinline__ uint32_t pair_lane(uint32_t lane) { return 4 * (lane & 31) + 2 * (lane >> 5); }
__device__ __forceinline__ constexpr uint32_t pair_word(uint32_t j) { return (j & 1) + (j >> 1) * 128; }

__device__ __forceinline__ void load_pairs(uint64_t *v, const uint64_t *p) {
    const Words2 a = reinterpret_cast<const Words2 *>(p)[0], b = reinterpret_cast<const Words2 *>(p + pair_word(2))[0];
    v[0] = a.x;
    v[1] = a.y;
    v[2] = b.x;
    v[3] = b.y;
}

// the same for words that are read once: they pass by without pushing others out of the caches
__device__ __forceinline__ void stream_pairs(uint64_t *v, const uint64_t *p) {
    const Words2 a = __builtin_nontemporal_load(reinterpret_cast<const Words2 *>(p));
    const Words2 b = __builtin_nontemporal_load(reinterpret_cast<const Words2 *>(p + pair_word(2)));
    v[0] = a.x;
    v[1] = a.y;
    v[2] = b.x;
    v[3] = b.y;
}

template <bool STREAM>
__device__ __forceinline__ void load_pairs_or_stream(uint64_t *v, const uint64_t *p) {
    if constexpr (STREAM)
        stream_pairs(v, p);
    else
        load_pairs(v, p);
}

__device__ __forceinline__ void store_pairs(uint64_t *p, const uint64_t *v) {
    reinterpret_cast<Words2 *>(p)[0] = Words2{v[0], v[1]};
    reinterpret_cast<Words2 *>(p + pair_word(2))[0] = Words2{v[2], v[3]};
}

__device__ __forceinline__ void turn_pairs(uint64_t *v) {
    swap_lane_bit<5>(v[0], v[2]);
    swap_lane_bit<5>(v[1], v[3]);
}

__device__ __forceinline__ void turn_pairs(double *v) {
    uint64_t w[4];
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = (uint64_t)__double_as_longlong(v[j]);
    turn_pairs(w);
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = __longlong_as_double((long long)w[j]);
}

}  // namespace

}  // namespace he
