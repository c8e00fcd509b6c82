// What the kernels of the transform share: how a job names its limb, the per-limb constants of the two back ends, and the
// prologues that form the input of a forward rows pass.
#pragma once
#include "kernels.h"
#include "modarith.cuh"

namespace he {

namespace {

__device__ __forceinline__ uint32_t skew(uint32_t e) { return e + (e >> 4); }

// Workgroup barrier that orders LDS traffic only.  __syncthreads() also waits for every global load and
// store of the wave, which would serialise a prefetch issued before it with the butterflies after it.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Workgroups are dealt round-robin to the 8 XCDs; give every XCD a contiguous range of logical ids so
// that the tiles of one limb (which share a twiddle table) meet in one L2.
__device__ __forceinline__ uint32_t logical_block() {
    uint32_t b = blockIdx.x, n = gridDim.x;
    if (n % 8 == 0) return (b % 8) * (n / 8) + b / 8;
    return b;
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

__device__ __forceinline__ Job decode_job(const NttArgs &a, uint32_t job) {
    Job j;
    const size_t n = (size_t)1 << a.log_n;
    if (a.jobs) {
        // job = item * n_jobs + entry of the list
        const uint32_t item = job / a.n_jobs;
        LimbJob lj = a.jobs[job - item * a.n_jobs];
        j.in = a.in + item * a.item_stride + (size_t)lj.data_limb * n;
        j.out = a.out + item * a.item_stride + (size_t)lj.data_limb * n;
        j.table = lj.table;
        j.poly = 0;
        j.limb = 0;
        const bool sourced = a.pro_mode == NTT_PRO_SOURCE_REDUCE || a.pro_mode == NTT_PRO_SOURCE_INTT_REDUCE;
        j.src_table = sourced ? lj.data_limb / a.pro_lk : 0;
        j.src = sourced ? a.pro_src + item * a.pro_item_stride + (size_t)j.src_table * n : nullptr;
    } else {
        j.poly = job / a.map.limbs;
        j.limb = job % a.map.limbs;
        j.in = a.in ? a.in + ((size_t)j.poly * a.in_poly_stride + j.limb) * n : nullptr;
        j.out = a.out + ((size_t)j.poly * a.out_poly_stride + j.limb) * n;
        j.table = map_table(a.map, j.limb);
        j.src = a.pro_src + ((size_t)j.poly * a.pro_poly_stride << a.log_n);
        j.src_table = a.pro_src_table;
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
    return IntCtx{a.moduli[table], a.tw + ((size_t)table << (a.log_n + 1))};
}

__device__ __forceinline__ FpCtx fp_ctx(const NttArgs &a, uint32_t table) {
    const double *c = a.fp_consts + 4 * (size_t)table;
    return FpCtx{FpMod{c[0], c[1]}, a.tw_fp + ((size_t)table << a.log_n)};
}

// (N^-1 [* w]) as an FP twiddle for the last multiplication of the inverse transform
__device__ __forceinline__ FpTw inverse_scale(const NttArgs &a, const Job &job, FpMod m) {
    const double *c = a.fp_consts + 4 * (size_t)job.table;
    FpTw ninv{c[2], c[3]};
    if (a.epi_mode != NTT_EPI_MUL) return ninv;
    const double w = fp_canonical(fp_mulmod(fp_from_u64(a.w[2 * job.limb]), ninv, m), m);
    return FpTw{w, w * m.qinv};
}

// Input of a forward rows pass (a.pro_mode): word j of the thread from global offset glob(j) of its limb, as exact
// doubles; returns whether they have to be reduced before the first stage (else they are canonical).
template <int W, typename Glob>
__device__ __forceinline__ bool rows_input_fp(double (&v)[W], const NttArgs &a, const Job &job, const FpCtx &c, Glob glob) {
    if (a.pro_mode == NTT_PRO_MODDOWN_RESCALE) {
        const uint64_t *tsrc = a.pro_src + ((size_t)job.poly * a.pro_poly_stride << a.log_n);
        const uint64_t *dsrc = a.pro_src2 + ((size_t)job.poly * a.pro2_poly_stride << a.log_n);
        const FpMod ml = fp_ctx(a, a.pro_last).m;
        const double wd = fp_from_u64(a.pro_w[2 * job.limb]), wl = fp_from_u64(a.pro_w[2 * a.pro_last]);
        const FpTw w{wd, wd * c.m.qinv}, wlast{wl, wl * ml.qinv};
        const uint64_t qj = a.moduli[job.table], rj = a.barrett[2 * job.table + 1];
        const uint64_t qlast = a.moduli[a.pro_last], rlast = a.barrett[2 * a.pro_last + 1];
#pragma unroll
        for (int j = 0; j < W; j++) {
            const uint64_t ds = dsrc[glob(j)];
            const uint64_t dl = a.pro_k1 ? barrett64(ds, qlast, rlast) : ds;
            const uint64_t dj = a.pro_k1 ? barrett64(ds, qj, rj) : job.in[glob(j)];
            // coefficient of the dropped limb of the ModDown result, canonical mod q_last
            const double r = fp_canonical(fp_from_u64(tsrc[glob(j)]) - fp_mulmod(fp_from_u64(dl), wlast, ml), ml);
            v[j] = fp_mulmod(fp_from_u64(dj), w, c.m) + fp_reduce(r, c.m);
        }
        return true;
    }
    if (a.pro_mode == NTT_PRO_BROADCAST_REDUCE) {
        // one source limb for every limb: it may exceed this limb's prime, so reduce first
        const uint64_t *src = a.pro_src + ((size_t)job.poly * a.pro_poly_stride << a.log_n);
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = fp_from_u64(src[glob(j)]);
        return true;
    }
    if (a.pro_mode == NTT_PRO_SOURCE_REDUCE) {
        const uint64_t q = a.moduli[job.table], r1 = a.barrett[2 * job.table + 1];
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = fp_from_u64(barrett64(job.src[glob(j)], q, r1));
    } else {
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = fp_from_u64(job.in[glob(j)]);
    }
    return false;
}

// The same on the integer back end: residues below q.
template <int W, typename Glob>
__device__ __forceinline__ void rows_input_int(uint64_t (&v)[W], const NttArgs &a, const Job &job, uint64_t q, Glob glob) {
    if (a.pro_mode == NTT_PRO_BROADCAST_REDUCE || a.pro_mode == NTT_PRO_SOURCE_REDUCE) {
        const uint64_t r1 = a.barrett[2 * job.table + 1];
        const uint64_t *src = a.pro_mode == NTT_PRO_SOURCE_REDUCE ? job.src : a.pro_src + ((size_t)job.poly * a.pro_poly_stride << a.log_n);
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = barrett64(src[glob(j)], q, r1);
    } else if (a.pro_mode == NTT_PRO_MODDOWN_RESCALE) {
        const uint64_t r1 = a.barrett[2 * job.table + 1];
        const uint64_t *tsrc = a.pro_src + ((size_t)job.poly * a.pro_poly_stride << a.log_n);
        const uint64_t *dsrc = a.pro_src2 + ((size_t)job.poly * a.pro2_poly_stride << a.log_n);
        const uint64_t ql = a.moduli[a.pro_last];
        const Shoup w = load_shoup(a.pro_w, job.limb), wlast = load_shoup(a.pro_w, a.pro_last);
        const uint64_t rlast = a.barrett[2 * a.pro_last + 1];
#pragma unroll
        for (int j = 0; j < W; j++) {
            const uint64_t ds = dsrc[glob(j)];
            const uint64_t dl = a.pro_k1 ? barrett64(ds, ql, rlast) : ds;
            const uint64_t dj = a.pro_k1 ? barrett64(ds, q, r1) : job.in[glob(j)];
            const uint64_t r = sub_mod(tsrc[glob(j)], mul_shoup(dl, wlast, ql), ql);
            v[j] = add_mod(mul_shoup(dj, w, q), barrett64(r, q, r1), q);
        }
    } else {
#pragma unroll
        for (int j = 0; j < W; j++) v[j] = job.in[glob(j)];
    }
}

}  // namespace

}  // namespace he
