// CKKS encoding and decoding on the device: the special FFT over the orbit 5^j mod 2N (HEAAN's fftSpecial /
// fftSpecialInv butterfly network, cahel-main/src/fft.cu:194-453), rounding to integer coefficients
// (src/rns_base.cu:121-156) and the CRT composition of a decrypted plaintext (src/rns_base.cu:325-459).
//
// All floating-point steps are plain IEEE double operations in a fixed order (this file is compiled without
// contraction): a butterfly is u = a + b, t = (a - b) * w with the four-multiplication complex product, so
// the result does not depend on how the butterflies are spread over threads.
//
// Layout: v = `slots` complex values as double2.
#include "kernels.h"
#include "modarith.cuh"
#include "ntt_common.cuh"

namespace he {

namespace {

constexpr int kThreads = 256;

// A value of a vector or a result, which are only 8-byte aligned for certain, as one 16-byte access
typedef double Value2 __attribute__((ext_vector_type(2), aligned(8)));

__device__ __forceinline__ double2 get(const double2 *v) {
    const Value2 x = *reinterpret_cast<const Value2 *>(v);
    return double2{x.x, x.y};
}

__device__ __forceinline__ void put(double2 *v, double2 x) { *reinterpret_cast<Value2 *>(v) = Value2{x.x, x.y}; }

__device__ __forceinline__ double2 cmul(double2 a, double2 w) {
    return double2{a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x};
}

// twiddle of butterfly j < len / 2 in a stage of span len: e^{+-2 pi i (5^j mod 4 len) / (4 len)}; a stage's twiddles lie one
// after the other (looked up as root[group[j]], two dependent loads of which the second gathers, the two passes of one
// encoding of 32,768 values took 3 us longer)
template <bool INVERSE>
__device__ __forceinline__ double2 stage_twiddle(const FftTables &t, uint32_t len, uint32_t j) {
    return (INVERSE ? t.inverse : t.forward)[(len >> 1) + j];
}

// INVERSE (encode): decimation in frequency,  (a, b) -> (a + b, (a - b) w)
// forward (decode): decimation in time,       (a, b) -> (a + b w, a - b w)
template <bool INVERSE>
__device__ __forceinline__ void butterfly(double2 &a, double2 &b, double2 w) {
    if (INVERSE) {
        const double2 u{a.x + b.x, a.y + b.y};
        const double2 d{a.x - b.x, a.y - b.y};
        a = u;
        b = cmul(d, w);
    } else {
        const double2 t = cmul(b, w);
        const double2 u = a;
        a = double2{u.x + t.x, u.y + t.y};
        b = double2{u.x - t.x, u.y - t.y};
    }
}

// Where an encoding starts from: the caller's real and imaginary parts (zero padded from `count` on) instead of the
// scratch vector.  re = nullptr: the scratch vector itself.
struct FftSource {
    const double *re, *im;
    uint32_t count;
    size_t value_stride;          // doubles between the items' values
    unsigned long long *max_bits; // one per item, cleared here for the rounding kernel to accumulate into
};

__device__ __forceinline__ double2 source_value(const FftSource &src, uint32_t item, uint32_t i) {
    if (i >= src.count) return double2{0.0, 0.0};
    const size_t at = item * src.value_stride + i;
    return double2{src.re[at], src.im ? src.im[at] : 0.0};
}

// Where a decoding ends: with `re` the real parts of the first `count` values of every item, or both parts, packed, instead of the
// vector.
struct FftTarget {
    double *re;
    uint32_t count;
    bool both;
};

__device__ __forceinline__ void store_value(const FftTarget &dst, uint32_t item, uint32_t i, double2 v) {
    const size_t at = (size_t)item * dst.count + i;
    if (dst.both)
        put(reinterpret_cast<double2 *>(dst.re) + at, v);
    else
        dst.re[at] = v.x;
}

constexpr uint32_t kSmallSlots = 256;   // below this the small kernel runs

// fewer than 256 slots: every stage inside LDS, one workgroup per item
template <bool INVERSE>
__global__ __launch_bounds__(kThreads) void cfft_lds_kernel(double2 *v, uint32_t tile, FftTables t, uint32_t slots,
                                                            FftSource src, FftTarget dst) {
    __shared__ double2 s[kSmallSlots];
    double2 *g = v + (size_t)blockIdx.y * slots + (size_t)blockIdx.x * tile;
    if (INVERSE && src.re) {
        if (threadIdx.x == 0 && src.max_bits) src.max_bits[blockIdx.y] = 0;
        for (uint32_t i = threadIdx.x; i < tile; i += kThreads) s[i] = source_value(src, blockIdx.y, i);
    } else {
        for (uint32_t i = threadIdx.x; i < tile; i += kThreads) s[i] = get(g + i);
    }
    __syncthreads();
    for (uint32_t k = 2; k <= tile; k <<= 1) {
        const uint32_t len = INVERSE ? (tile << 1) / k : k;   // tile, tile/2, ..., 2  or  2, 4, ..., tile
        const uint32_t lenh = len >> 1;
        for (uint32_t b = threadIdx.x; b < (tile >> 1); b += kThreads) {
            const uint32_t j = b & (lenh - 1), pos = ((b / lenh) * len) + j;
            double2 x = s[pos], y = s[pos + lenh];
            butterfly<INVERSE>(x, y, stage_twiddle<INVERSE>(t, len, j));
            s[pos] = x;
            s[pos + lenh] = y;
        }
        __syncthreads();
    }
    if (!INVERSE && dst.re) {
        for (uint32_t i = threadIdx.x; i < dst.count; i += kThreads) store_value(dst, blockIdx.y, i, s[i]);
    } else {
        for (uint32_t i = threadIdx.x; i < tile; i += kThreads) put(g + i, s[i]);
    }
}

// A transform of 2^s >= 256 values as two passes, like the number-theoretic one: the vector is 2^(s - 10) rows x 1024 columns (x 256
// below 1024 values); the rows pass holds the stages whose span is more than a row (a workgroup owns all rows of a few columns),
// the blocks pass the 10 (8) stages inside one row.  A thread holds 4 values in register blocks of two stages (Tile4's
// layout) and fetches its twiddles together with the values.  Every butterfly has the operands and the twiddle that a launch per
// stage would give it, so the results do not depend on the split.
// Why rows of 1024: the rows pass reads an encoding's values from, and writes a decoding's to, page-locked host memory, in segments as long
// as a tile is wide.  A tile of 1024 values has 32 columns at 32,768 values, 256 bytes a segment; with rows of 256 columns it
// had 8, and 256 KB read in segments of 64 bytes take 15.0 us over PCIe (128 bytes 8.7, 256 bytes and more 7.0; written 7.1, 6.3, 6.0).
// Stage sigma of the inverse direction (the forward runs them backwards) pairs index bit s - 1 - sigma; a value's twiddle
// is chosen by the bits below it.
template <bool INVERSE, int B, int LD>
struct FftTile {
    using T4 = Tile4<B, LD>;
    struct Tw {
        double2 a0, a1, b;   // first stage: pairs (0, 2) and (1, 3); second: pairs (0, 1) and (2, 3)
    };
    template <typename Pos, int K = 0>
    static __device__ __forceinline__ void load_tw(Tw *tw, const FftTables &t, uint32_t log_slots, uint32_t stage0, Pos pos) {
        const uint32_t len = 1u << (log_slots - stage0 - 2 * K), mask = (len >> 1) - 1;
        tw[K].a0 = stage_twiddle<INVERSE>(t, len, pos(K, 0) & mask);
        tw[K].a1 = stage_twiddle<INVERSE>(t, len, pos(K, 1) & mask);
        tw[K].b = T4::stages(K) == 2 ? stage_twiddle<INVERSE>(t, len >> 1, pos(K, 0) & (mask >> 1)) : double2{0.0, 0.0};
        if constexpr (K + 1 < T4::kBlocks) load_tw<Pos, K + 1>(tw, t, log_slots, stage0, pos);
    }
    // from the layout of block FROM to that of its neighbour TO
    template <int FROM, int TO>
    static __device__ __forceinline__ void move(double2 *v, double *re, double *im, uint32_t t) {
        constexpr int KLO = FROM < TO ? FROM : TO;
        if constexpr (T4::in_wave(KLO)) {
            uint64_t x[4], y[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                x[j] = (uint64_t)__double_as_longlong(v[j].x);
                y[j] = (uint64_t)__double_as_longlong(v[j].y);
            }
            T4::template swap_words<KLO>(x);
            T4::template swap_words<KLO>(y);
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = double2{__longlong_as_double((long long)x[j]), __longlong_as_double((long long)y[j])};
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t e = skew(T4::word(FROM, t, j));
                re[e] = v[j].x;
                im[e] = v[j].y;
            }
            lds_barrier();
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t e = skew(T4::word(TO, t, j));
                v[j] = double2{re[e], im[e]};
            }
        }
    }
    // the stages in order (INVERSE), values of block 0 -> values of the last block
    template <int K = 0>
    static __device__ __forceinline__ void down(double2 *v, const Tw *tw, double *re, double *im, uint32_t t) {
        butterfly<INVERSE>(v[0], v[2], tw[K].a0);
        butterfly<INVERSE>(v[1], v[3], tw[K].a1);
        if (T4::stages(K) == 2) {
            butterfly<INVERSE>(v[0], v[1], tw[K].b);
            butterfly<INVERSE>(v[2], v[3], tw[K].b);
        }
        if constexpr (K + 1 < T4::kBlocks) {
            move<K, K + 1>(v, re, im, t);
            down<K + 1>(v, tw, re, im, t);
        }
    }
    // backwards (forward direction), values of the last block -> values of block 0
    template <int K = T4::kBlocks - 1>
    static __device__ __forceinline__ void up(double2 *v, const Tw *tw, double *re, double *im, uint32_t t) {
        if (T4::stages(K) == 2) {
            butterfly<INVERSE>(v[0], v[1], tw[K].b);
            butterfly<INVERSE>(v[2], v[3], tw[K].b);
        }
        butterfly<INVERSE>(v[0], v[2], tw[K].a0);
        butterfly<INVERSE>(v[1], v[3], tw[K].a1);
        if constexpr (K > 0) {
            move<K, K - 1>(v, re, im, t);
            up<K - 1>(v, tw, re, im, t);
        }
    }
};

// blockIdx.x = tile of 2^(B - LD) columns, blockIdx.y = item; LR = log2(columns of the vector)
template <bool INVERSE, int B, int LD, int LR>
__global__ __launch_bounds__(1 << (B - 2)) void cfft_rows_kernel(double2 *v, FftTables t, uint32_t log_slots, FftSource src,
                                                                 FftTarget dst) {
    using F = FftTile<INVERSE, B, LD>;
    using T4 = typename F::T4;
    constexpr int LOGC = B - LD, NB = T4::kBlocks;
    __shared__ double re[(1 << B) + (1 << (B - 4))], im[(1 << B) + (1 << (B - 4))];
    const uint32_t item = blockIdx.y, col0 = blockIdx.x << LOGC, tid = threadIdx.x;
    v += (size_t)item << log_slots;
    auto pos = [&](int k, int j) {
        const uint32_t e = T4::word(k, tid, j);
        return ((e >> LOGC) << LR) + col0 + (e & ((1u << LOGC) - 1));
    };
    double2 x[4];
    typename F::Tw tw[NB];
    if (INVERSE) {
        if (src.re) {
            if (src.max_bits && blockIdx.x == 0 && tid == 0) src.max_bits[item] = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = source_value(src, item, pos(0, j));
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = get(v + pos(0, j));
        }
        F::load_tw(tw, t, log_slots, 0, pos);
        F::down(x, tw, re, im, tid);
#pragma unroll
        for (int j = 0; j < 4; j++) put(v + pos(NB - 1, j), x[j]);
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = get(v + pos(NB - 1, j));
        F::load_tw(tw, t, log_slots, 0, pos);
        F::up(x, tw, re, im, tid);
        if (dst.re) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (pos(0, j) < dst.count) store_value(dst, item, pos(0, j), x[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) put(v + pos(0, j), x[j]);
        }
    }
}

// Blocks of 2^B values: a wave of a workgroup of two (B = 8), or a workgroup (B = 10).  blockIdx.y = item
template <int B>
constexpr uint32_t kFftBlocks = B == 8 ? 2 : 1;   // of a workgroup

template <bool INVERSE, int B>
__global__ __launch_bounds__((1 << (B - 2)) * kFftBlocks<B>) void cfft_blocks_kernel(double2 *v, FftTables t, uint32_t log_slots,
                                                                                    FftSource src, FftTarget dst) {
    using F = FftTile<INVERSE, B, B>;
    using T4 = typename F::T4;
    constexpr int LAST = T4::kBlocks - 1, WORDS = T4::in_wave(0) ? 1 : (1 << B) + (1 << (B - 4));
    __shared__ double re[WORDS], im[WORDS];
    const uint32_t w = threadIdx.x >> (B - 2), tid = threadIdx.x & ((1u << (B - 2)) - 1), item = blockIdx.y;
    const uint32_t blk = blockIdx.x * kFftBlocks<B> + w;
    if (kFftBlocks<B> > 1 && blk >= 1u << (log_slots - B)) return;   // (256 slots: one block)
    v += ((size_t)item << log_slots) + ((size_t)blk << B);
    auto pos = [&](int k, int j) { return T4::word(k, tid, j); };   // (the twiddles depend on the position inside the block)
    double2 x[4];
    typename F::Tw tw[LAST + 1];
    if (INVERSE) {
        if (src.re) {
            // (only when the whole vector is this one block: otherwise the rows pass has run before)
            if (src.max_bits && tid == 0) src.max_bits[item] = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = source_value(src, item, pos(0, j));
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = get(v + pos(0, j));
        }
        F::load_tw(tw, t, log_slots, log_slots - B, pos);
        F::down(x, tw, re, im, tid);
#pragma unroll
        for (int j = 0; j < 4; j++) put(v + pos(LAST, j), x[j]);
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = get(v + pos(LAST, j));
        F::load_tw(tw, t, log_slots, log_slots - B, pos);
        F::up(x, tw, re, im, tid);
        if (dst.re && log_slots == B) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (pos(0, j) < dst.count) store_value(dst, item, pos(0, j), x[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) put(v + pos(0, j), x[j]);
        }
    }
}

// The largest magnitude of an item's coefficients (the bit patterns of non-negative doubles order like the values):
// reduced over the wave, then over the workgroup, one atomic per workgroup.  Atomics on one address are served one
// after the other: one per thread took most of the rounding kernel's time, one per wave still half of it.  Every
// thread of the workgroup calls this.
__device__ __forceinline__ void block_max_to(unsigned long long *dst, unsigned long long m) {
    __shared__ unsigned long long wave_max[kThreads / 64];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        const unsigned long long o = __shfl_xor(m, d);
        m = o > m ? o : m;
    }
    if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < kThreads / 64; w++) m = wave_max[w] > m ? wave_max[w] : m;
        if (m) atomicMax(dst, m);
    }
}

// Where the rounded coefficients go: as residues of the first `limbs` primes to out [items][limbs][N], items out_item_stride words
// apart.
struct RoundSink {
    uint64_t *out;
    const uint64_t *moduli, *barrett;
    uint32_t limbs;
    size_t out_item_stride;
};

// residue of a rounded real coefficient (below 2^63 in magnitude: the caller checks the maximum)
__device__ __forceinline__ uint64_t real_residue(double c, uint64_t q, uint64_t r1) {
    const uint64_t r = barrett64((uint64_t)fabs(c), q, r1);
    return c < 0 ? neg_mod(r, q) : r;
}

// coefficient c of the plaintext: real parts fill the first half, imaginary parts the second, `gap` apart;
// value i comes from position bitrev(i) of the transformed vector
__global__ __launch_bounds__(kThreads) void encode_round_kernel(const double2 *v, uint32_t log_slots, uint32_t gap,
                                                                uint32_t half, double fix, RoundSink sink,
                                                                unsigned long long *max_bits) {
    const uint32_t c = blockIdx.x * kThreads + threadIdx.x;
    v += (size_t)blockIdx.y << log_slots;
    max_bits += blockIdx.y;
    const bool imag = c >= half;
    const uint32_t k = imag ? c - half : c;
    double val = 0.0;
    if (k % gap == 0) {
        const uint32_t i = k / gap;
        const double2 z = get(v + (__brev(i) >> (32 - log_slots)));
        val = round((imag ? z.y : z.x) * fix);
    }
    uint64_t *o = sink.out + blockIdx.y * sink.out_item_stride + c;
    for (uint32_t l = 0; l < sink.limbs; l++) o[(size_t)l * 2 * half] = real_residue(val, sink.moduli[l], sink.barrett[2 * l + 1]);
    block_max_to(max_bits, (unsigned long long)__double_as_longlong(fabs(val)));
}

// The same for full packing (gap = 1, at least 256 slots): the bit reversal as a tiled transpose through LDS, so that
// both the reads of the transformed vector and the writes of the coefficients touch whole cache lines (with one thread
// per coefficient every lane of a wave reads a line of its own).  Slot i = (top 4 bits | middle | low 4 bits); a
// workgroup takes one value of the middle bits: thread (x, y) reads the slot with low bits y and top bits brev4(x),
// which sits at position (brev4(y) | brev(middle) | x) of the vector (consecutive in x), and writes the slot with low
// bits x and top bits brev4(y) (consecutive in x), real part to coefficient i, imaginary part to coefficient N/2 + i.
__global__ __launch_bounds__(kThreads) void encode_round_tiled_kernel(const double2 *v, uint32_t log_slots, uint32_t half,
                                                                      double fix, RoundSink sink, unsigned long long *max_bits) {
    __shared__ double2 tile[16][17];
    const uint32_t x = threadIdx.x & 15, y = threadIdx.x >> 4, mid = blockIdx.x, mid_bits = log_slots - 8;
    v += (size_t)blockIdx.y << log_slots;
    max_bits += blockIdx.y;
    const uint32_t rmid = mid_bits ? __brev(mid) >> (32 - mid_bits) : 0;
    const uint32_t brev4_y = __brev(y) >> 28;
    tile[y][x] = get(v + ((brev4_y << (log_slots - 4)) | (rmid << 4) | x));
    __syncthreads();
    const double2 z = tile[x][y];
    const uint32_t i = (brev4_y << (log_slots - 4)) | (mid << 4) | x;
    const double re = round(z.x * fix), im = round(z.y * fix);
    uint64_t *o = sink.out + blockIdx.y * sink.out_item_stride + i;
    for (uint32_t l = 0; l < sink.limbs; l++) {
        const uint64_t q = sink.moduli[l], r1 = sink.barrett[2 * l + 1];
        o[(size_t)l * 2 * half] = real_residue(re, q, r1);
        o[(size_t)l * 2 * half + half] = real_residue(im, q, r1);
    }
    const double big = fabs(re) > fabs(im) ? fabs(re) : fabs(im);
    block_max_to(max_bits, (unsigned long long)__double_as_longlong(big));
}

constexpr int kMaxComposeLimbs = 64;

// Garner's mixed-radix composition of one coefficient from its residues d[0 .. limbs-1] (overwritten), centred around zero,
// as a double divided by the scale.  LIMBS > 0: the number of limbs at compile time (the digits then stay in registers;
// with a run-time count the array lives in scratch memory), 0: any number up to kMaxComposeLimbs.
template <int LIMBS>
__device__ __forceinline__ double compose(uint64_t *d, uint32_t limbs_rt, double inv_scale, const uint64_t *moduli, const uint64_t *barrett,
                                          const uint64_t *garner_inv, uint32_t garner_stride) {
    const uint32_t limbs = LIMBS ? (uint32_t)LIMBS : limbs_rt;
#pragma unroll
    for (uint32_t i = 0; i < limbs; i++) {
        const uint64_t q = moduli[i], r0 = barrett[2 * i], r1 = barrett[2 * i + 1];
        uint64_t t = d[i];
#pragma unroll
        for (uint32_t j = 0; j < i; j++) {
            const uint64_t dj = barrett64(d[j], q, r1);
            t = mul_mod(sub_mod(t, dj, q), garner_inv[(size_t)i * garner_stride + j], q, r0, r1);
        }
        d[i] = t;
    }
    // negative iff the digits, read from the top, exceed those of (Q - 1) / 2, whose digits are (q_i - 1) / 2
    // (written without early exits so that the loops unroll: `decided` / `carry` play the part of the breaks)
    bool negative = false, decided = false;
#pragma unroll
    for (uint32_t k = 0; k < limbs; k++) {
        const uint32_t i = limbs - 1 - k;
        const uint64_t h = (moduli[i] - 1) >> 1;
        if (!decided && d[i] != h) {
            negative = d[i] > h;
            decided = true;
        }
    }
    if (negative) {
        // Q - v = (Q - 1 - v) + 1: digit-wise complement, then increment
        bool carry = true;
#pragma unroll
        for (uint32_t i = 0; i < limbs; i++) {
            uint64_t x = moduli[i] - 1 - d[i];
            if (carry) {
                x++;
                carry = x >= moduli[i];
                if (carry) x = 0;
            }
            d[i] = x;
        }
    }
    double acc = 0.0;
#pragma unroll
    for (uint32_t k = 0; k < limbs; k++) {
        const uint32_t i = limbs - 1 - k;
        acc = acc * (double)moduli[i] + (double)d[i];
    }
    return (negative ? -acc : acc) * inv_scale;
}

// thread s < slots: real part of value s, else imaginary part of value s - slots; stored at position bitrev.
template <int LIMBS>
__global__ __launch_bounds__(kThreads) void decode_compose_kernel(const uint64_t *res, uint32_t limbs_rt, uint32_t log_n,
                                                                  uint32_t log_slots, uint32_t gap, double inv_scale,
                                                                  const uint64_t *moduli, const uint64_t *barrett,
                                                                  const uint64_t *garner_inv, uint32_t garner_stride,
                                                                  double2 *v) {
    const uint32_t limbs = LIMBS ? (uint32_t)LIMBS : limbs_rt;
    const uint32_t s = blockIdx.x * kThreads + threadIdx.x;
    const uint32_t slots = 1u << log_slots, half = 1u << (log_n - 1);
    if (s >= 2 * slots) return;
    res += ((size_t)blockIdx.y * limbs) << log_n;   // blockIdx.y = item: dense plaintexts, dense slot vectors
    v += (size_t)blockIdx.y * slots;
    const bool imag = s >= slots;
    const uint32_t i0 = imag ? s - slots : s;
    const size_t coeff = (imag ? half : 0) + (size_t)i0 * gap;
    uint64_t d[LIMBS ? LIMBS : kMaxComposeLimbs];
#pragma unroll
    for (uint32_t i = 0; i < limbs; i++) d[i] = res[((size_t)i << log_n) + coeff];
    double *slot = reinterpret_cast<double *>(&v[__brev(i0) >> (32 - log_slots)]);
    slot[imag ? 1 : 0] = compose<LIMBS>(d, limbs, inv_scale, moduli, barrett, garner_inv, garner_stride);
}

// The inverse rows pass of all limbs of a plaintext and the composition in one kernel: a workgroup takes one tile of every limb
// through the pass, a limb to each group of four waves, which leaves rows r, r + R/4 (real parts of two values) and r + R/2, r + 3R/4
// (their imaginary parts) of one column in each thread; the groups exchange their words, and the first two compose one of the two
// values each, which go to neighbouring positions of the slot vector.  Full and sparse packing; blockIdx.y = item.
// Bound by the chain from the words' arrival to the composed value: the launch has one tile for every fourth CU.  One group that took
// limb after limb, 7.2 us for 2 limbs of 2^16 words, now 6.2; a decryption to host values of 4 limbs with 2^12 values 49 -> 43.5 us
// (1.6 us of it the sampling, see flood_rows_kernel).
template <int LD, int LIMBS>
__global__ __launch_bounds__(256 * LIMBS) void decode_rows_compose_kernel(HE_HEAD_PARAMS, double2 *v, const uint64_t *garner_inv,
                                                                          double inv_scale, uint32_t log_slots, uint32_t garner_stride) {
    constexpr int B = 10, LOGC = B - LD;
    using T4 = Tile4<B, LD>;
    constexpr int NB = T4::kBlocks;
    __shared__ uint64_t tiles[LIMBS][(1 << B) + (1 << (B - 4))];
    NttArgs a;
    set_head(a, HE_HEAD_NAMES);
    a.epi_mode = NTT_PLAIN;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6), group = wave >> 2;
    const uint32_t t = ((wave & 3) << 6) | (threadIdx.x & 63);
    const uint32_t col0 = blockIdx.x << LOGC, item = blockIdx.y;
    auto glob = [&](int k, int j) {
        const uint32_t e = T4::word(k, t, j);
        return (size_t)(e >> LOGC) * 256 + col0 + (e & ((1u << LOGC) - 1));
    };
    uint64_t *lds = tiles[group];
    const Job job = decode_job(a, item * LIMBS + group);
    uint64_t x[4];
#pragma unroll
    for (int j = 0; j < 4; j++) x[j] = job.in[glob(NB - 1, j)];
    // (the composition's constants, requested with the words: behind the exchange they were another trip to memory)
    uint64_t moduli[LIMBS], barrett[2 * LIMBS], garner[LIMBS * LIMBS];
#pragma unroll
    for (int i = 0; i < LIMBS; i++) {
        moduli[i] = scalar(a.moduli)[i];
        barrett[2 * i] = scalar(a.barrett)[2 * i];
        barrett[2 * i + 1] = scalar(a.barrett)[2 * i + 1];
#pragma unroll
        for (int j = 0; j < i; j++) garner[i * LIMBS + j] = scalar(garner_inv)[(size_t)i * garner_stride + j];
    }
#pragma unroll
    for (int i = 0; i < LIMBS; i++) {
        asm volatile("" ::"s"(moduli[i]), "s"(barrett[2 * i]), "s"(barrett[2 * i + 1]));
#pragma unroll
        for (int j = 0; j < i; j++) asm volatile("" ::"s"(garner[i * LIMBS + j]));
    }
    if ((a.fp_mask >> job.table) & 1) {
        const FpArith ar = fp_arith(a, job.table);
        FpArith::Tw tw[NB];
        T4::template load_tw<FpArith, 0>(tw, ar, 1, t);
        const double scale = inverse_scale(a, job, ar.m);
        double w[4];
#pragma unroll
        for (int j = 0; j < 4; j++) w[j] = FpArith::from_word(x[j]);
        T4::template inverse<FpArith>(w, tw, ar, lds, t);
        ar.template scale<T4::stages(0)>(x, w, scale);
    } else {
        const IntArith ar = int_arith(a, job.table);
        IntArith::Tw tw[NB];
        T4::template load_tw<IntArith, 0>(tw, ar, 1, t);
        T4::template inverse<IntArith>(x, tw, ar, lds, t);
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = reduce_4q(x[j], ar.m);
    }
    uint64_t d[2][LIMBS];
    if constexpr (LIMBS > 1) {
        lds_barrier();   // (the other waves of the group have read the tile)
#pragma unroll
        for (int j = 0; j < 4; j++) lds[256 * j + t] = x[j];
        lds_barrier();
    }
    const uint32_t log_gap = a.log_n - 1 - log_slots;
    v += (size_t)item << log_slots;
#pragma unroll
    for (int pair = 0; pair < (LIMBS > 1 ? 1 : 2); pair++) {
        const uint32_t j = LIMBS > 1 ? group : pair;
        if (j >= 2) return;
#pragma unroll
        for (int l = 0; l < LIMBS; l++) {
            d[0][l] = LIMBS > 1 ? tiles[l][256 * j + t] : x[pair];
            d[1][l] = LIMBS > 1 ? tiles[l][256 * (j + 2) + t] : x[pair + 2];
        }
        double2 val;
        val.x = compose<LIMBS>(d[0], LIMBS, inv_scale, moduli, barrett, garner, LIMBS);
        val.y = compose<LIMBS>(d[1], LIMBS, inv_scale, moduli, barrett, garner, LIMBS);
        const uint32_t k = (uint32_t)glob(0, (int)j);   // (below N / 2)
        if ((k & ((1u << log_gap) - 1)) == 0) put(v + (__brev(k >> log_gap) >> (32 - log_slots)), val);
    }
}

template <bool INVERSE>
hipError_t run_fft(double2 *v, uint32_t slots, uint32_t items, const FftTables &t, hipStream_t s, FftSource src, FftTarget dst) {
    const uint32_t log_slots = 31 - __builtin_clz(slots);
    if (slots < kSmallSlots) {
        hipLaunchKernelGGL(cfft_lds_kernel<INVERSE>, dim3(1, items), dim3(kThreads), 0, s, v, slots, t, slots, src, dst);
        return hipGetLastError();
    }
    const uint32_t lr = log_slots >= 10 ? 10 : 8, ld = log_slots - lr;
    const FftSource none{nullptr, nullptr, 0, 0, nullptr};
    auto rows = [&]() {
        // tiles of 1024 values (256 of the 512)
#define HE_CASE(LD, B, LR)                                                                                                              \
    case LD:                                                                                                                            \
        hipLaunchKernelGGL((cfft_rows_kernel<INVERSE, B, LD, LR>), dim3((1u << LR) >> (B - LD), items), dim3(1u << (B - 2)), 0, s, v, t, \
                           log_slots, src, dst);                                                                                        \
        break;
        if (lr == 8) {
            switch (ld) {
                HE_CASE(1, 8, 8)
                default: return hipErrorInvalidValue;
            }
        } else {
            switch (ld) {
                HE_CASE(1, 10, 10) HE_CASE(2, 10, 10) HE_CASE(3, 10, 10) HE_CASE(4, 10, 10) HE_CASE(5, 10, 10) HE_CASE(6, 10, 10)
                default: return hipErrorInvalidValue;
            }
        }
#undef HE_CASE
        return hipGetLastError();
    };
    auto blocks = [&]() {
        if (lr == 8)
            hipLaunchKernelGGL((cfft_blocks_kernel<INVERSE, 8>), dim3(1, items), dim3(64 * kFftBlocks<8>), 0, s, v, t, log_slots,
                               ld ? none : src, dst);
        else
            hipLaunchKernelGGL((cfft_blocks_kernel<INVERSE, 10>), dim3(1u << ld, items), dim3(256), 0, s, v, t, log_slots, ld ? none : src, dst);
        return hipGetLastError();
    };
    if (INVERSE && ld)
        if (hipError_t e = rows()) return e;
    if (hipError_t e = blocks()) return e;
    if (!INVERSE && ld) return rows();
    return hipSuccess;
}

// out[item][i] = v[item][i] for i < count: the leading slots of every item, packed
__global__ __launch_bounds__(kThreads) void take_slots_kernel(const double2 *v, uint32_t slots, uint32_t count, double2 *out) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i < count) put(out + (size_t)blockIdx.y * count + i, get(v + (size_t)blockIdx.y * slots + i));
}

}  // namespace

hipError_t launch_ckks_encode(const FftTables &t, const Tables &tab, const double *re, const double *im, uint32_t count,
                              uint32_t slots, double scale, double2 *v, uint64_t *max_bits, uint32_t items, size_t value_stride,
                              uint64_t *out, uint32_t limbs, size_t out_item_stride, hipStream_t s) {
    const uint32_t n = 1u << t.log_n, log_slots = 31 - __builtin_clz(slots);
    if (items == 0 || items > 65535 || !out || limbs == 0) return hipErrorInvalidValue;
    unsigned long long *maxima = reinterpret_cast<unsigned long long *>(max_bits);
    hipError_t e = run_fft<true>(v, slots, items, t, s, FftSource{re, im, count, value_stride, maxima}, FftTarget{nullptr, 0, false});
    if (e != hipSuccess) return e;
    const RoundSink sink{out, tab.moduli, tab.barrett, limbs, out_item_stride};
    if (slots == n / 2 && log_slots >= 8)
        hipLaunchKernelGGL(encode_round_tiled_kernel, dim3(slots / kThreads, items), dim3(kThreads), 0, s, v, log_slots, n / 2,
                           scale / (double)slots, sink, maxima);
    else
        hipLaunchKernelGGL(encode_round_kernel, dim3((n + kThreads - 1) / kThreads, items), dim3(kThreads), 0, s, v, log_slots,
                           (n / 2) / slots, n / 2, scale / (double)slots, sink, maxima);
    return hipGetLastError();
}

// Updates of 32-bit floats cross the bus and the host's copying loop as such, half of the bytes: 10 x 62,006 of them 2.5 MB; widened here
// they take 4 us (5 MB written).
__global__ __launch_bounds__(256) void widen_rows_kernel(const float *in, double *out, size_t length, size_t padded) {
    const size_t i = 2 * ((size_t)blockIdx.x * 256 + threadIdx.x), row = blockIdx.y;
    if (i >= padded) return;
    const float *src = in + row * length;
    double2 v;
    v.x = i < length ? (double)src[i] : 0.0;
    v.y = i + 1 < length ? (double)src[i + 1] : 0.0;
    *reinterpret_cast<double2 *>(out + row * padded + i) = v;
}

hipError_t launch_widen_rows(const float *in, double *out, uint32_t rows, size_t length, size_t padded, hipStream_t s) {
    const size_t blocks = (padded + 511) / 512;
    if (rows == 0 || rows > 65535 || padded == 0 || padded % 2 || length > padded || blocks > most_workgroups(256)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(widen_rows_kernel, dim3((uint32_t)blocks, rows), dim3(256), 0, s, in, out, length, padded);
    return hipGetLastError();
}

hipError_t launch_ckks_fft_inverse(const FftTables &t, const double *re, const double *im, uint32_t count, uint32_t slots,
                                   double2 *v, uint32_t items, size_t value_stride, hipStream_t s) {
    if (items == 0 || items > 65535 || !re) return hipErrorInvalidValue;
    return run_fft<true>(v, slots, items, t, s, FftSource{re, im, count, value_stride, nullptr}, FftTarget{nullptr, 0, false});
}

hipError_t launch_ckks_fft_real(const FftTables &t, uint32_t slots, double2 *v, uint32_t items, double *re, uint32_t count,
                                bool both, hipStream_t s) {
    if (items == 0 || items > 65535 || !re || count == 0 || count > slots) return hipErrorInvalidValue;
    return run_fft<false>(v, slots, items, t, s, FftSource{nullptr, nullptr, 0, 0, nullptr}, FftTarget{re, count, both});
}

hipError_t launch_ckks_compose(const FftTables &t, const Tables &tab, const uint64_t *res, uint32_t limbs,
                               uint32_t slots, double scale, const uint64_t *garner_inv, uint32_t garner_stride,
                               double2 *v, uint32_t items, hipStream_t s) {
    const uint32_t n = 1u << t.log_n, log_slots = 31 - __builtin_clz(slots);
    if (limbs == 0 || limbs > (uint32_t)kMaxComposeLimbs || items == 0 || items > 65535) return hipErrorInvalidValue;
    const dim3 grid((2 * slots + kThreads - 1) / kThreads, items);
#define HE_COMPOSE(L)                                                                                                     \
    hipLaunchKernelGGL(decode_compose_kernel<L>, grid, dim3(kThreads), 0, s, res, limbs, t.log_n, log_slots, (n / 2) / slots, \
                       1.0 / scale, tab.moduli, tab.barrett, garner_inv, garner_stride, v)
    switch (limbs) {
        case 1: HE_COMPOSE(1); break;
        case 2: HE_COMPOSE(2); break;
        case 3: HE_COMPOSE(3); break;
        case 4: HE_COMPOSE(4); break;
        default: HE_COMPOSE(0); break;
    }
#undef HE_COMPOSE
    return hipGetLastError();
}

hipError_t launch_ckks_decode(const FftTables &t, const Tables &tab, const uint64_t *res, uint32_t limbs,
                              uint32_t slots, double scale, const uint64_t *garner_inv, uint32_t garner_stride,
                              double2 *v, uint32_t items, hipStream_t s) {
    if (hipError_t e = launch_ckks_compose(t, tab, res, limbs, slots, scale, garner_inv, garner_stride, v, items, s)) return e;
    return run_fft<false>(v, slots, items, t, s, FftSource{nullptr, nullptr, 0, 0, nullptr}, FftTarget{nullptr, 0, false});
}

hipError_t launch_ckks_decode_real(const FftTables &t, const NttArgs &inv, int backend, uint32_t slots, double scale,
                                   const uint64_t *garner_inv, uint32_t garner_stride, double2 *v, uint32_t items, double *re,
                                   uint32_t count, bool both, hipStream_t s) {
    const uint32_t limbs = inv.map.limbs, log_slots = 31 - __builtin_clz(slots);
    if (inv.log_n < 12 || inv.log_n > 16 || inv.jobs || limbs == 0 || limbs > 4 || items == 0 || items > 65535) return hipErrorInvalidValue;
    NttArgs a = inv;   // (the mask stands for the launch's back end)
    a.fp_mask = backend == NTT_BACKEND_INT ? 0 : (backend == NTT_BACKEND_FP ? ~(uint64_t)0 : inv.fp_mask);
    const dim3 grid(1u << (a.log_n - 10), items);
    const NttHead h = ntt_head(a, 0, 0);
#define HE_LIMBS(LD, L)                                                                                                            \
    hipLaunchKernelGGL((decode_rows_compose_kernel<LD, L>), grid, dim3(256 * L), 0, s, HE_HEAD_ARGS(h), v, garner_inv, 1.0 / scale,    \
                       log_slots, garner_stride)
#define HE_CASE(LD)                         \
    case LD:                                \
        switch (limbs) {                    \
            case 1: HE_LIMBS(LD, 1); break; \
            case 2: HE_LIMBS(LD, 2); break; \
            case 3: HE_LIMBS(LD, 3); break; \
            default: HE_LIMBS(LD, 4);       \
        }                                   \
        break;
    switch (a.log_n - 8) {
        HE_CASE(4) HE_CASE(5) HE_CASE(6) HE_CASE(7) HE_CASE(8)
        default: return hipErrorInvalidValue;
    }
#undef HE_CASE
#undef HE_LIMBS
    if (hipError_t e = hipGetLastError()) return e;
    return launch_ckks_fft_real(t, slots, v, items, re, count, both, s);
}

hipError_t launch_take_slots(const double2 *v, uint32_t slots, uint32_t items, uint32_t count, double2 *out, hipStream_t s) {
    if (count == 0 || count > slots || items == 0 || items > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(take_slots_kernel, dim3((count + kThreads - 1) / kThreads, items), dim3(kThreads), 0, s, v, slots,
                       count, out);
    return hipGetLastError();
}

}  // namespace he
