// Host-memory stand-in for the C-ABI entry points that the host layer's table construction, record parsing and
// containers call (he_malloc .. he_context_destroy, and he_keyswitch for a deferred relinearisation), so that those
// CPU code paths can run under AddressSanitizer and UndefinedBehaviorSanitizer without a GPU.  Test infrastructure: "device" memory is malloc'ed host memory, copies
// are memcpy, a context is an opaque token.  Nothing here computes.  Streams are queues: an asynchronous copy reads its source, an encoding
// writes its plaintext, when the stream is next waited for, as late as a device may.
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <vector>

#include "cahel_hip.h"

struct he_context {
    uint32_t log_n, size_q, size_p;
};

// the call that fails from now on, or nullptr
const char *mock_failing = nullptr;
// whether he_ckks_decode_real succeeds; what happens during each he_decrypt_flood and each
// question for a decoding's workspace (another thread's doing)
bool mock_decodes = false;
std::function<void()> mock_meanwhile;

namespace {

std::map<he_stream, std::vector<std::function<void()>>> queues;

bool fails(const char *call) { return mock_failing && !std::strcmp(mock_failing, call); }

void run(he_stream stream) {
    for (auto &work : queues[stream]) work();
    queues[stream].clear();
}

}  // namespace

extern "C" {

const char *he_error_string(int status) { return status == 0 ? "success" : "mock device error"; }

int he_malloc(void **dev_ptr, size_t bytes) {
    if (!dev_ptr) return HE_E_INVALID_ARGUMENT;
    if (fails("he_malloc")) return HE_E_OUT_OF_MEMORY;
    *dev_ptr = bytes ? std::malloc(bytes) : nullptr;
    return (bytes && !*dev_ptr) ? HE_E_OUT_OF_MEMORY : HE_OK;
}

int he_free(void *dev_ptr) {   // (waits for the device, as hipFree does)
    for (auto &q : queues) run(q.first);
    std::free(dev_ptr);
    return HE_OK;
}

int he_memcpy_h2d(void *dst, const void *src, size_t bytes, he_stream stream) {
    run(stream);
    if (bytes) std::memcpy(dst, src, bytes);
    return HE_OK;
}

int he_memcpy_d2h(void *dst, const void *src, size_t bytes, he_stream stream) {
    run(stream);
    if (bytes) std::memcpy(dst, src, bytes);
    return HE_OK;
}

int he_memcpy_d2d(void *dst, const void *src, size_t bytes, he_stream stream) {
    run(stream);
    if (bytes) std::memmove(dst, src, bytes);
    return HE_OK;
}

int he_stream_create(he_stream *stream) {
    if (!stream) return HE_E_INVALID_ARGUMENT;
    static char tokens[64];
    static int used = 0;
    *stream = &tokens[used++ % 64];
    return HE_OK;
}

int he_stream_synchronize(he_stream stream) {
    run(stream);
    return HE_OK;
}

int he_host_malloc(void **host_ptr, size_t bytes) { return he_malloc(host_ptr, bytes); }
int he_host_free(void *host_ptr) { return he_free(host_ptr); }
int he_memcpy_h2d_async(void *dst, const void *src, size_t bytes, he_stream stream) {
    if (fails("he_memcpy_h2d_async")) return HE_E_UNSUPPORTED;
    queues[stream].push_back([=] { std::memcpy(dst, src, bytes); });
    return HE_OK;
}

// an event knows the stream it was recorded on
int he_event_create(he_event *event) {
    *event = new he_stream(nullptr);
    return HE_OK;
}
int he_event_destroy(he_event event) {
    delete static_cast<he_stream *>(event);
    return HE_OK;
}
int he_event_record(he_event event, he_stream stream) {
    *static_cast<he_stream *>(event) = stream;
    return HE_OK;
}
int he_event_synchronize(he_event event) {
    run(*static_cast<he_stream *>(event));
    return HE_OK;
}

int he_context_create(const he_context_desc *d, he_context **out) {
    if (!d || !out || !d->moduli || !d->barrett || !d->psi || !d->ipsi_div2) return HE_E_INVALID_ARGUMENT;
    if (d->log_n < 9 || d->log_n > 16) return HE_E_UNSUPPORTED;
    // touch every table the real library would upload, so that a short array shows up as a sanitizer report
    const size_t n = (size_t)1 << d->log_n, qp = (size_t)d->size_q + d->size_p;
    volatile uint64_t sink = 0;
    for (size_t i = 0; i < qp; i++) sink += d->moduli[i] + d->barrett[2 * i + 1];
    sink += d->psi[2 * qp * n - 1] + d->ipsi_div2[2 * qp * n - 1];
    if (d->size_p)
        sink += d->p_mod_q[2 * d->size_q - 1] + d->pinv_mod_q[2 * d->size_q - 1] + d->phat_inv_mod_p[2 * d->size_p - 1] +
                d->phat_mod_q[(size_t)d->size_q * d->size_p - 1];
    (void)sink;
    *out = new he_context{d->log_n, d->size_q, d->size_p};
    return HE_OK;
}

int he_context_set_level(he_context *ctx, const he_level_desc *d) {
    if (!ctx || !d || d->L == 0 || d->L > ctx->size_q) return HE_E_INVALID_ARGUMENT;
    volatile uint64_t sink = 0;
    if (d->L > 1) sink += d->qlast_inv[2 * (d->L - 1) - 1];
    if (ctx->size_p) {
        sink += d->part_hat_inv[2 * d->L - 1];
        const uint32_t K = ctx->size_p, beta = d->beta;
        for (uint32_t g = 0; g < beta; g++) {
            const uint32_t start = g * K, size = start + K <= d->L ? K : d->L - start, n_out = d->L + K - size;
            sink += d->digit_mats[d->digit_mat_off[g] + (size_t)n_out * size - 1];
        }
    }
    (void)sink;
    return HE_OK;
}

int he_context_destroy(he_context *ctx) {
    delete ctx;
    return HE_OK;
}

// "Encodes" later: the bits of value i as word i of every limb, zeros behind them.
int he_ckks_encode_bounded(const he_context *ctx, const double *re, const double *im, uint32_t count, uint32_t, double, uint32_t limbs,
                           uint32_t items, size_t value_stride, uint64_t *out, uint32_t out_poly_stride, uint64_t *ws, he_stream stream) {
    if (!ctx || !re || im || !out || !ws || items == 0) return HE_E_INVALID_ARGUMENT;
    if (fails("he_ckks_encode_bounded")) return HE_E_UNSUPPORTED;
    const size_t n = (size_t)1 << ctx->log_n;
    queues[stream].push_back([=] {
        for (uint32_t k = 0; k < items; k++)
            for (uint32_t l = 0; l < limbs; l++) {
                uint64_t *limb = out + ((size_t)k * out_poly_stride + l) * n;
                std::memset(limb, 0, n * sizeof(uint64_t));
                std::memcpy(limb, re + k * value_stride, count * sizeof(double));
            }
    });
    return HE_OK;
}

// The same, and the largest |value| times the scale in place of the largest coefficient
int he_ckks_encode_batch(const he_context *ctx, const double *re, const double *im, uint32_t count, uint32_t slots, double scale, uint32_t limbs,
                         uint32_t items, size_t value_stride, uint64_t *out, uint32_t out_poly_stride, uint64_t *ws, he_stream stream) {
    if (fails("he_ckks_encode_batch")) return HE_E_UNSUPPORTED;
    if (int rc = he_ckks_encode_bounded(ctx, re, im, count, slots, scale, limbs, items, value_stride, out, out_poly_stride, ws, stream)) return rc;
    queues[stream].push_back([=] {
        for (uint32_t k = 0; k < items; k++) {
            double largest = 0.0;
            for (uint32_t i = 0; i < count; i++) largest = std::fmax(largest, std::fabs(re[k * value_stride + i]) * scale);
            std::memcpy(ws + k, &largest, sizeof(double));
        }
    });
    return HE_OK;
}

int he_encrypt_end(const he_context *ctx, uint32_t L, uint32_t items, uint64_t *cts, uint64_t *ws, he_stream stream);
int he_encrypt_end_values(const he_context *ctx, uint32_t L, uint32_t items, const double *re, uint32_t count, uint32_t slots, double scale,
                          size_t value_stride, uint64_t *cts, uint64_t *ws, uint64_t *encode_ws, he_stream stream) {
    if (int rc = he_ckks_encode_bounded(ctx, re, nullptr, count, slots, scale, L, items, value_stride, cts, 2 * L, encode_ws, stream)) return rc;
    return he_encrypt_end(ctx, L, items, cts, ws, stream);
}

int he_widen_rows(const float *in, double *out, uint32_t rows, size_t length, size_t padded, he_stream stream) {
    queues[stream].push_back([=] {
        for (uint32_t r = 0; r < rows; r++)
            for (size_t i = 0; i < padded; i++) out[r * padded + i] = i < length ? (double)in[r * length + i] : 0.0;
    });
    return HE_OK;
}

size_t he_ckks_encode_batch_workspace_words(const he_context *, uint32_t items) { return 8 * (size_t)items; }

// "Encrypts" in two calls: what item k draws from, its first stream id, goes to the workspace, and from there into every word of polynomial 1.
size_t he_encrypt_batch_workspace_words(const he_context *, uint32_t, uint32_t items) { return items; }
int he_encrypt_begin(const he_context *ctx, uint32_t L, uint32_t items, const uint64_t *pk, const uint32_t *key, uint64_t stream_id, uint64_t *ws,
                     he_stream stream) {
    if (!ctx || L == 0 || items == 0 || !pk || !key || !ws) return HE_E_INVALID_ARGUMENT;
    queues[stream].push_back([=] {
        for (uint32_t k = 0; k < items; k++) ws[k] = stream_id + 3 * k;
    });
    return fails("he_encrypt_begin") ? HE_E_UNSUPPORTED : HE_OK;
}
int he_encrypt_end(const he_context *ctx, uint32_t L, uint32_t items, uint64_t *cts, uint64_t *ws, he_stream stream) {
    if (!ctx || L == 0 || items == 0 || !cts || !ws) return HE_E_INVALID_ARGUMENT;
    if (fails("he_encrypt_end")) return HE_E_UNSUPPORTED;
    const size_t poly = (size_t)L << ctx->log_n;
    queues[stream].push_back([=] {
        for (uint32_t k = 0; k < items; k++)
            for (size_t i = 0; i < poly; i++) cts[(2 * (size_t)k + 1) * poly + i] = ws[k];
    });
    return HE_OK;
}

// (what encoder.cpp refers to besides)
int he_ckks_encode(const he_context *, const double *, const double *, uint32_t, uint32_t, double, uint32_t, uint64_t *, uint64_t *,
                   he_stream) { return HE_E_UNSUPPORTED; }
int he_encrypt_batch(const he_context *, uint32_t, uint32_t, const uint64_t *, const uint32_t *, uint64_t, uint64_t *, uint64_t *,
                     he_stream) { return HE_E_UNSUPPORTED; }
size_t he_ckks_workspace_words(const he_context *, uint32_t) { return 0; }
int he_ckks_decode(const he_context *, const uint64_t *, uint32_t, uint32_t, double, double *, uint64_t *, he_stream) {
    return HE_E_UNSUPPORTED;
}
// a workspace is for as many slots as were asked for last
static uint32_t decode_workspace_slots = 0;
size_t he_ckks_decode_real_workspace_words(const he_context *, uint32_t, uint32_t slots) {
    decode_workspace_slots = slots;
    if (mock_meanwhile) mock_meanwhile();
    return 0;
}
// "Decodes" later: the bits of word i as value i.  Unless mock_decodes, fails behind its first launches: what they write comes later all the same.
int he_ckks_decode_real(const he_context *, const uint64_t *plain, uint32_t, uint32_t slots, double, double *out, uint32_t count, uint64_t *,
                        he_stream stream) {
    if (count > slots) return HE_E_INVALID_ARGUMENT;
    if (slots > decode_workspace_slots) std::abort();
    if (mock_decodes) {
        queues[stream].push_back([=] { std::memcpy(out, plain, count * sizeof(double)); });
        return HE_OK;
    }
    queues[stream].push_back([=] { std::memset(out, 0x66, count * sizeof(double)); });
    return HE_E_UNSUPPORTED;
}

// "Decrypts" later: the words of polynomial 0.
int he_decrypt_flood(const he_context *ctx, const uint64_t *ct, uint32_t, uint32_t limbs, const uint64_t *, size_t, const uint32_t *, uint64_t,
                     const uint64_t *, uint32_t, uint64_t *plain, uint64_t *, he_stream stream) {
    queues[stream].push_back([=] { std::memcpy(plain, ct, ((size_t)limbs << ctx->log_n) * sizeof(uint64_t)); });
    if (mock_meanwhile) mock_meanwhile();
    return HE_OK;
}
size_t he_decrypt_decode_real_workspace_words(const he_context *, uint32_t, uint32_t, uint32_t) { return 1; }
// Decryption and decoding of a batch, later: the first `count` words of polynomial 0 of every ciphertext, as (re, im) pairs of equal values
int he_decrypt_decode_flood_batch(const he_context *, const uint64_t *const *d_cts, uint32_t items, uint32_t, const uint64_t *, const uint32_t *,
                                  uint64_t, const uint64_t *, uint32_t, uint32_t, double, uint32_t count, double *out, uint64_t *,
                                  he_stream stream) {
    queues[stream].push_back([=] {
        for (size_t k = 0; k < items; k++)
            for (size_t i = 0; i < 2 * (size_t)count; i++) std::memcpy(out + 2 * k * count + i, d_cts[k] + i / 2, sizeof(double));
    });
    return HE_OK;
}

// (what keys.cpp refers to besides; a secret key is sampled and transformed)
int he_sample(const he_context *ctx, int, const uint32_t *, uint64_t stream_id, uint64_t *out, uint32_t limbs, uint32_t, uint32_t, uint32_t,
              const uint64_t *, uint32_t, he_stream stream) {
    queues[stream].push_back([=] {
        for (size_t i = 0; i < (size_t)limbs << ctx->log_n; i++) out[i] = stream_id;
    });
    return HE_OK;
}
int he_ntt_forward(const he_context *, uint64_t *, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, he_stream) { return HE_OK; }
int he_add(const he_context *, const uint64_t *, const uint64_t *, uint64_t *, uint32_t, uint32_t, uint32_t, he_stream) { return HE_E_UNSUPPORTED; }
int he_multiply(const he_context *, const uint64_t *, const uint64_t *, uint64_t *, uint32_t, uint32_t, uint32_t, he_stream) {
    return HE_E_UNSUPPORTED;
}
int he_multiply_add(const he_context *, const uint64_t *, const uint64_t *, const uint64_t *, uint64_t *, uint32_t, uint32_t, uint32_t, int,
                    he_stream) { return HE_E_UNSUPPORTED; }
int he_add_p_multiple(const he_context *, const uint64_t *, const uint64_t *, uint64_t *, uint32_t, uint32_t, he_stream) { return HE_E_UNSUPPORTED; }
int he_galois_ntt(const he_context *, const uint64_t *, uint64_t *, uint32_t, uint32_t, he_stream) { return HE_E_UNSUPPORTED; }
int he_encrypt(const he_context *, uint32_t, const uint64_t *, const uint64_t *, const uint32_t *, uint64_t, uint64_t *, uint64_t *, he_stream) {
    return HE_E_UNSUPPORTED;
}
int he_decrypt_decode_real_batch(const he_context *, const uint64_t *const *, uint32_t, uint32_t, const uint64_t *, const uint32_t *, uint64_t,
                                 const uint64_t *, uint32_t, uint32_t, double, uint32_t, double *, uint64_t *, he_stream) { return HE_E_UNSUPPORTED; }

size_t he_keyswitch_workspace_words(const he_context *ctx, uint32_t L) { return ctx ? (size_t)L << ctx->log_n : 0; }

// Touches what the real call reads and writes (every word of c, of the beta key digits and of ct, and the
// workspace), so that a stale pointer shows up as a sanitizer report; marks ct so that the caller can tell it ran.
int he_keyswitch(const he_context *ctx, uint32_t L, const uint64_t *c, const uint64_t *const *evk, uint64_t *ct,
                 uint32_t, uint64_t *workspace, he_stream) {
    if (!ctx || !c || !evk || !ct || !workspace || L == 0 || L > ctx->size_q || ctx->size_p == 0) return HE_E_INVALID_ARGUMENT;
    const size_t n = (size_t)1 << ctx->log_n, qp = (size_t)ctx->size_q + ctx->size_p;
    const uint32_t beta = (L + ctx->size_p - 1) / ctx->size_p;
    uint64_t sum = 0;
    for (size_t i = 0; i < (size_t)L * n; i++) sum += c[i];
    for (uint32_t d = 0; d < beta; d++)
        for (size_t i = 0; i < 2 * qp * n; i += 97) sum += evk[d][i];
    for (size_t i = 0; i < (size_t)L * n; i++) workspace[i] = sum;
    for (size_t i = 0; i < 2 * (size_t)L * n; i++) ct[i] += 1;
    return HE_OK;
}

}  // extern "C"
