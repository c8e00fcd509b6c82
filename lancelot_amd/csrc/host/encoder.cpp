// CKKS encoder: slots <-> plaintext polynomial through the canonical embedding restricted to the orbit
// 5^j mod 2N (cahel-main/src/ckks.cu:34-209 encode, :292-465 decode; transform of src/fft.cu; rounding and
// residues of src/rns_base.cu:121-156; CRT composition of src/rns_base.cu:325-459).
//
// Everything runs on the GPU (he_ckks_encode / he_ckks_decode: special FFT of HEAAN's fftSpecial / fftSpecialInv
// butterfly network in FP64, rounding, residues, CRT composition, NTTs); the host moves the slot values in and
// out and keeps the reference's argument checks.  Decoded values agree with the reference up to FP64 operation
// order (bounded by the 2^-20 acceptance tolerance), not bit for bit.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "cahel.h"
#include "staging.h"

using namespace cahel;

namespace {

// how much of a batch's values travels at once: 1 MiB takes the link about 20 us, several times what starting a copy costs
constexpr std::size_t kChunkBytes = std::size_t(1) << 20;

// dst = src, and the sum of the magnitudes
template <class T>
double copy_sum(T *dst, const T *src, std::size_t count) {
    double s = 0.0;
#pragma omp simd reduction(+ : s)
    for (std::size_t i = 0; i < count; i++) {
        dst[i] = src[i];
        s += std::fabs((double)src[i]);
    }
    return s;
}

// No coefficient of an encoding exceeds scale / slots times the sum of the values' magnitudes (the transform's twiddles have
// magnitude 1; the margin covers its rounding).  When that already stays inside the bounds that the largest coefficient has to
// keep, the coefficients need not be looked at: the encoding is enqueued and nothing waits for it.
bool surely_small(double sum, double scale, std::size_t slots, int total_bits) {
    const double bound = 1.001 * (scale / static_cast<double>(slots)) * sum + 1.0;
    if (!(bound < 0x1p61)) return false;   // (also: not a number)
    return static_cast<int>(std::ceil(std::log2(bound))) + 1 < total_bits;
}

void check_largest(double max_coeff, int total_bits) {
    const int max_coeff_bit_count = static_cast<int>(std::ceil(std::log2(std::max(max_coeff, 1.0)))) + 1;
    if (max_coeff_bit_count >= total_bits) throw std::invalid_argument("encoded values are too large");
    if (max_coeff_bit_count > 63)
        throw std::invalid_argument("encoded values are too large: coefficients above 2^62 are not supported");
}

}  // namespace

CAHELGPUCKKSEncoder::CAHELGPUCKKSEncoder(const CAHELGPUContext &context) {
    if (context.scheme() != scheme_type::ckks) throw std::invalid_argument("unsupported scheme");
    slots_ = context.poly_degree() >> 1;
    first_chain_index_ = context.get_first_index();
}

std::size_t CAHELGPUCKKSEncoder::message_slots(std::size_t count) {
    if (sparse_slots_ == 0) {
        // the first message fixes the slot count for the lifetime of the encoder (src/ckks.cu:131-142)
        std::size_t s = 1;
        while (s < count) s <<= 1;
        sparse_slots_ = s;
    } else if (count > sparse_slots_) {
        throw std::invalid_argument("values_size exceeds previous message length");
    }
    if (sparse_slots_ < 2) throw std::invalid_argument("single value encoding is not available");
    return sparse_slots_;
}

std::vector<CAHELGPUCiphertext> CAHELGPUCKKSEncoder::encode_encrypt_many(const CAHELGPUContext &context,
                                                                         const CAHELGPUPublicKey &pk, const double *values,
                                                                         std::size_t items, std::size_t count,
                                                                         std::size_t value_stride, double scale) {
    if (items == 0) return {};
    if (count > slots_ || value_stride < count) throw std::invalid_argument("values_size is too large");
    check_batch(context, pk, items, scale);
    const std::size_t ss = message_slots(count);
    Batch batch = begin_batch(context, pk, items, scale);
    he_stream st = context.stream();

    // values -> device, packed, some messages at a time through page-locked memory (the next ones are copied while the last
    // travel)
    DeviceBuffer staging(items * count);
    double *d_values = reinterpret_cast<double *>(staging.get());
    PinnedRing &ring = PinnedRing::of_thread();
    const std::size_t rows = count ? std::max<std::size_t>(1, kChunkBytes / (count * sizeof(double))) : items;
    bool small = true;
    for (std::size_t first = 0; count && first < items; first += rows) {
        const std::size_t taken = std::min(rows, items - first), bytes = taken * count * sizeof(double);
        double *host = static_cast<double *>(ring.take(bytes));
        for (std::size_t k = 0; k < taken; k++)
            small = surely_small(copy_sum(host + k * count, values + (first + k) * value_stride, count), scale, ss, batch.total_bits) && small;
        const int status = he_memcpy_h2d_async(d_values + first * count, host, bytes, st);
        ring.fence(st);
        check_status(status, "upload");
    }
    return end_batch(context, std::move(batch), d_values, small, count, ss);
}

std::vector<CAHELGPUCiphertext> CAHELGPUCKKSEncoder::encode_encrypt_updates(const CAHELGPUContext &context, const CAHELGPUPublicKey &pk,
                                                                            const std::vector<const float *> &rows, std::size_t length,
                                                                            double scale) {
    if (rows.empty() || length == 0) return {};
    const std::size_t chunks = (length + slots_ - 1) / slots_;
    if (chunks > 8192 || rows.size() > 8192) throw std::invalid_argument("too many messages");
    const std::size_t items = rows.size() * chunks, padded = chunks * slots_;
    check_batch(context, pk, items, scale);
    const std::size_t ss = message_slots(slots_);
    Batch batch = begin_batch(context, pk, items, scale);
    he_stream st = context.stream();
    // the floats as they are, row after row, some messages at a time through page-locked memory; the device widens them
    const std::size_t total = rows.size() * length;
    DeviceBuffer narrow((total + 1) / 2), staging(items * slots_);
    float *d_floats = reinterpret_cast<float *>(narrow.get());
    double *d_values = reinterpret_cast<double *>(staging.get());
    PinnedRing &ring = PinnedRing::of_thread();
    const std::size_t room = std::max(kChunkBytes / sizeof(float), slots_);
    bool small = true;
    float *host = nullptr;
    std::size_t filled = 0, sent = 0;
    auto send = [&] {
        const int status = he_memcpy_h2d_async(d_floats + sent, host, filled * sizeof(float), st);
        ring.fence(st);
        check_status(status, "upload");
        sent += filled;
        filled = 0;
    };
    for (const float *row : rows)
        for (std::size_t at = 0; at < length; at += slots_) {
            const std::size_t taken = std::min(slots_, length - at);
            if (filled + taken > room) send();
            if (filled == 0) host = static_cast<float *>(ring.take(room * sizeof(float)));
            small = surely_small(copy_sum(host + filled, row + at, taken), scale, ss, batch.total_bits) && small;
            filled += taken;
        }
    send();
    check_status(he_widen_rows(d_floats, d_values, (uint32_t)rows.size(), length, padded, st), "he_widen_rows");
    return end_batch(context, std::move(batch), d_values, small, slots_, ss);
}

// what a batch needs of its key, level and scale
void CAHELGPUCKKSEncoder::check_batch(const CAHELGPUContext &context, const CAHELGPUPublicKey &pk, std::size_t items, double scale) const {
    if (items > 8192) throw std::invalid_argument("too many messages");
    if (!pk.gen_flag_) throw std::logic_error("public key has not been generated");
    if (first_chain_index_ == 0 || context.size_p() == 0) throw std::logic_error("batched encryption needs a data level and special primes");
    if (scale <= 0 || (static_cast<int>(std::log2(scale)) + 1 >= context.total_coeff_modulus_bit_count(first_chain_index_)))
        throw std::invalid_argument("scale out of bounds");
}

CAHELGPUCKKSEncoder::Batch CAHELGPUCKKSEncoder::begin_batch(const CAHELGPUContext &context, const CAHELGPUPublicKey &pk, std::size_t items,
                                                            double scale) {
    const uint32_t L = (uint32_t)context.limbs_at(first_chain_index_);
    he_context *h = context.handle();
    Batch batch{items, scale, context.total_coeff_modulus_bit_count(first_chain_index_),
                DeviceBuffer(items * 2 * (std::size_t)L * context.poly_degree()),
                DeviceBuffer(he_encrypt_batch_workspace_words(h, L, (uint32_t)items)), StreamIds(context, 3 * items)};
    check_status(he_encrypt_begin(h, L, (uint32_t)items, pk.pk_.data(), context.prng_key(), batch.ids.first(), batch.ws.get(), context.stream()),
                 "he_encrypt_begin");
    return batch;
}

std::vector<CAHELGPUCiphertext> CAHELGPUCKKSEncoder::end_batch(const CAHELGPUContext &context, Batch batch, const double *d_values, bool small,
                                                               std::size_t count, std::size_t ss) {
    const std::size_t n = context.poly_degree(), chain = first_chain_index_, items = batch.items;
    const uint32_t L = (uint32_t)context.limbs_at(chain);
    const double scale = batch.scale;
    he_context *h = context.handle();
    he_stream st = context.stream();
    // plaintexts, where there are any, straight into polynomial 0 of the ciphertexts
    const std::size_t words = 2 * (std::size_t)L * n;
    DeviceBuffer ws(he_ckks_encode_batch_workspace_words(h, (uint32_t)items));
    if (small) {
        check_status(he_encrypt_end_values(h, L, (uint32_t)items, d_values, (uint32_t)count, (uint32_t)ss, scale, count, batch.cts.get(),
                                           batch.ws.get(), ws.get(), st),
                     "he_encrypt_end_values");
    } else {
        check_status(he_ckks_encode_batch(h, d_values, nullptr, (uint32_t)count, (uint32_t)ss, scale, L, (uint32_t)items, count,
                                          batch.cts.get(), 2 * L, ws.get(), st),
                     "he_ckks_encode_batch");
        std::vector<double> maxima(items);
        check_status(he_memcpy_d2h(maxima.data(), ws.get(), items * sizeof(double), st), "download");
        for (double max_coeff : maxima) {
            const int max_coeff_bit_count = static_cast<int>(std::ceil(std::log2(std::max(max_coeff, 1.0)))) + 1;
            if (max_coeff_bit_count >= batch.total_bits || max_coeff_bit_count > 63)
                throw std::invalid_argument("encoded values are too large");
        }
        check_status(he_encrypt_end(h, L, (uint32_t)items, batch.cts.get(), batch.ws.get(), st), "he_encrypt_end");
    }
    // one ciphertext object per message, each a slice of the batch (no copies)
    std::vector<CAHELGPUCiphertext> out(items);
    auto shared = std::make_shared<DeviceBuffer>(std::move(batch.cts));
    for (std::size_t k = 0; k < items; k++) {
        CAHELGPUCiphertext &ct = out[k];
        ct.adopt(DeviceBuffer::slice(shared, k * words, words));
        ct.size_ = 2;
        ct.coeff_modulus_size_ = L;
        ct.poly_modulus_degree_ = n;
        ct.chain_index_ = chain;
        ct.parms_id_ = context.parms_id_at(chain);
        ct.scale_ = scale;
        ct.is_ntt_form_ = true;
        ct.is_asymmetric_ = true;
    }
    batch.ids.keep();
    return out;
}

void CAHELGPUCKKSEncoder::encode_complex(const CAHELGPUContext &context, const double *re, const double *im,
                                         std::size_t count, std::size_t chain_index, double scale,
                                         CAHELGPUPlaintext &destination) {
    const std::size_t n = context.poly_degree();
    if (count > slots_) throw std::invalid_argument("values_size is too large");
    const int total_bits = context.total_coeff_modulus_bit_count(chain_index);
    if (scale <= 0 || (static_cast<int>(std::log2(scale)) + 1 >= total_bits))
        throw std::invalid_argument("scale out of bounds");
    const std::size_t ss = message_slots(count);
    const uint32_t limbs = (uint32_t)context.limbs_at(chain_index);
    // (a block of another lane goes back there: an encoding's block belongs to the lane that writes it)
    if (destination.data_.get() && destination.data_.lane() != current_lane()) destination.data_.release();
    destination.resize(limbs, n);
    he_context *h = context.handle();
    he_stream st = context.stream();
    DeviceBuffer ws(he_ckks_encode_batch_workspace_words(h, 1));
    // the values, real parts then imaginary parts, in page-locked memory that the first kernel reads where it is
    PinnedRing &ring = PinnedRing::of_thread();
    double *host_re = static_cast<double *>(ring.take(2 * ss * sizeof(double))), *host_im = im ? host_re + ss : nullptr;
    double sum = copy_sum(host_re, re, count);
    if (im) sum += copy_sum(host_im, im, count);
    if (surely_small(sum, scale, ss, total_bits)) {
        const int status = he_ckks_encode_bounded(h, host_re, host_im, (uint32_t)count, (uint32_t)ss, scale, limbs, 1, count,
                                                  destination.data_.get(), limbs, ws.get(), st);
        ring.fence(st);
        destination.encoding_enqueued();
        check_status(status, "he_ckks_encode_bounded");
    } else {
        const int status = he_ckks_encode(h, host_re, host_im, (uint32_t)count, (uint32_t)ss, scale, limbs, destination.data_.get(),
                                          ws.get(), st);
        ring.fence(st);
        check_status(status, "he_ckks_encode");
        double max_coeff = 0.0;
        check_status(he_memcpy_d2h(&max_coeff, ws.get(), sizeof(double), st), "download");
        check_largest(max_coeff, total_bits);
    }
    destination.chain_index() = chain_index;
    destination.scale() = scale;
    destination.parms_id() = context.parms_id_at(chain_index);
    destination.is_ntt_form_ = true;
}

void CAHELGPUCKKSEncoder::encode(const CAHELGPUContext &context, const std::vector<double> &values,
                                 std::size_t chain_index, double scale, CAHELGPUPlaintext &destination) {
    encode_complex(context, values.data(), nullptr, values.size(), chain_index, scale, destination);
}

// the first `count` complex values of the decoding, interleaved (re, im), into v
void CAHELGPUCKKSEncoder::decode_values(const CAHELGPUContext &context, const CAHELGPUPlaintext &plain,
                                        std::size_t count, std::vector<double> &v) {
    const std::size_t ss = decode_count(context, plain, 0);   // (once: it may change on another thread)
    if (count == 0 || count > ss) count = ss;
    const uint32_t limbs = (uint32_t)plain.coeff_modulus_size();

    he_context *h = context.handle();
    DeviceBuffer ws(he_ckks_workspace_words(h, limbs));
    DeviceBuffer out(2 * ss);
    check_status(he_ckks_decode(h, plain.lane_data(), limbs, (uint32_t)ss, plain.scale(),
                                reinterpret_cast<double *>(out.get()), ws.get(), context.stream()),
                 "he_ckks_decode");
    v.resize(2 * count);
    check_status(he_memcpy_d2h(v.data(), out.get(), v.size() * sizeof(double), context.stream()), "download");
}

void CAHELGPUCKKSEncoder::decode_complex(const CAHELGPUContext &context, const CAHELGPUPlaintext &plain,
                                         std::vector<double> &re, std::vector<double> &im) {
    std::vector<double> v;
    decode_values(context, plain, 0, v);
    const std::size_t ss = v.size() / 2;
    re.resize(ss);
    im.resize(ss);
    for (std::size_t i = 0; i < ss; i++) {
        re[i] = v[2 * i];
        im[i] = v[2 * i + 1];
    }
}

std::size_t CAHELGPUCKKSEncoder::decode_count(const CAHELGPUContext &context, const CAHELGPUPlaintext &plain, std::size_t count) {
    if (!plain.is_ntt_form()) throw std::invalid_argument("plain is not in NTT form");
    if (plain.coeff_modulus_size() == 0 || !plain.data_.get()) throw std::invalid_argument("plain is empty");
    const int total_bits = context.total_coeff_modulus_bit_count(plain.chain_index());
    if (plain.scale() <= 0 || (static_cast<int>(std::log2(plain.scale())) >= total_bits))
        throw std::invalid_argument("scale out of bounds");
    if (sparse_slots_ == 0) sparse_slots_ = slots_;   // as the reference: decoding first fixes the full slot count
    return count == 0 || count > sparse_slots_ ? sparse_slots_ : count;
}

// the real parts of the first `count` values (decode_count's answer) to `destination`; the last kernel writes them to
// page-locked memory
void CAHELGPUCKKSEncoder::decode_real(const CAHELGPUContext &context, const CAHELGPUPlaintext &plain, std::size_t count,
                                      double *destination) {
    he_context *h = context.handle();
    const uint32_t limbs = (uint32_t)plain.coeff_modulus_size(), slots = (uint32_t)sparse_slots_;   // (once: it may change on another thread)
    DeviceBuffer ws(he_ckks_decode_real_workspace_words(h, limbs, slots));
    PinnedRing &ring = PinnedRing::of_thread();
    double *host = static_cast<double *>(ring.take(count * sizeof(double)));
    const int status = he_ckks_decode_real(h, plain.lane_data(), limbs, slots, plain.scale(), host, (uint32_t)count, ws.get(), context.stream());
    if (status != HE_OK) ring.fence(context.stream());   // (what was launched before the failure may still write the block)
    check_status(status, "he_ckks_decode_real");
    check_status(he_stream_synchronize(context.stream()), "synchronisation failed");
    std::memcpy(destination, host, count * sizeof(double));
}

void CAHELGPUCKKSEncoder::decode_prefix(const CAHELGPUContext &context, const CAHELGPUPlaintext &plain,
                                        std::size_t count, std::vector<double> &destination) {
    count = decode_count(context, plain, count);
    destination.resize(count);
    decode_real(context, plain, count, destination.data());
}

void CAHELGPUCKKSEncoder::decode(const CAHELGPUContext &context, const CAHELGPUPlaintext &plain,
                                 std::vector<double> &destination) {
    decode_prefix(context, plain, 0, destination);
}
