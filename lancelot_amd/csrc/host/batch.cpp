// Batched evaluation for callers that hold many small independent ciphertexts (Lancelot's have three or four limbs:
// one of them neither fills the GPU nor amortises a kernel launch).  Not in the reference, which evaluates one
// ciphertext per call; every item goes through the same arithmetic as the single-ciphertext functions, so its limbs
// equal theirs.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <stdexcept>

#include "cahel.h"
#include "staging.h"

using cahel::check_status;
using cahel::DeviceBuffer;

// a table of device pointers, uploaded through page-locked memory without waiting
static DeviceBuffer upload_table(const std::vector<const uint64_t *> &table, he_stream st) {
    const std::size_t bytes = table.size() * sizeof(uint64_t);
    DeviceBuffer d_table(table.size());
    if (bytes > cahel::PinnedRing::kMaxBytes) {
        check_status(he_memcpy_h2d(d_table.get(), table.data(), bytes, st), "upload");
        return d_table;
    }
    cahel::PinnedRing &ring = cahel::PinnedRing::of_thread();
    void *host = ring.take(bytes);
    std::memcpy(host, table.data(), bytes);
    const int status = he_memcpy_h2d_async(d_table.get(), host, bytes, st);
    ring.fence(st);
    check_status(status, "upload");
    return d_table;
}

// ciphertext objects that are the consecutive slices of a batch (no copies), like `like` but for their size, limbs and scale
static std::vector<CAHELGPUCiphertext> slices(DeviceBuffer batch, std::size_t items, std::size_t size, const CAHELGPUCiphertext &like,
                                              double scale) {
    std::vector<CAHELGPUCiphertext> out(items);
    const std::size_t limbs = like.coeff_modulus_size(), n = like.poly_modulus_degree(), words = size * limbs * n;
    auto shared = std::make_shared<DeviceBuffer>(std::move(batch));
    for (std::size_t k = 0; k < items; k++) {
        CAHELGPUCiphertext &ct = out[k];
        ct.adopt(DeviceBuffer::slice(shared, k * words, words));
        ct.size_ = size;
        ct.coeff_modulus_size_ = limbs;
        ct.poly_modulus_degree_ = n;
        ct.chain_index_ = like.chain_index();
        ct.parms_id_ = like.parms_id();
        ct.scale_ = scale;
        ct.is_ntt_form_ = true;
        ct.is_asymmetric_ = like.is_asymmetric_;
    }
    return out;
}

constexpr std::size_t kRowsPerCall = 16384;   // what he_sum_ciphertexts and he_multiply_sum take at once

// The sum of every row of ciphertexts (add_inplace term by term), all rows in one launch (up to kRowsPerCall).
std::vector<CAHELGPUCiphertext> sum_ciphertexts(const CAHELGPUContext &context,
                                                const std::vector<std::vector<const CAHELGPUCiphertext *>> &rows) {
    if (rows.empty()) return {};
    if (rows[0].empty() || !rows[0][0]) throw std::invalid_argument("no ciphertexts");
    const CAHELGPUCiphertext &first = *rows[0][0];
    std::vector<const uint64_t *> table;
    for (const auto &row : rows) {
        if (row.size() != rows[0].size()) throw std::invalid_argument("rows differ in their number of ciphertexts");
        for (const CAHELGPUCiphertext *ct : row) {
            if (!ct || !ct->is_ntt_form()) throw std::invalid_argument("encrypted is not valid");
            if (ct->parms_id() != first.parms_id() || ct->chain_index() != first.chain_index() || ct->size() != first.size())
                throw std::invalid_argument("encrypted parameter mismatch");
            if (ct->scale() != first.scale()) throw std::invalid_argument("scale mismatch");
            table.push_back(ct->data());
        }
    }
    he_stream st = context.stream();
    const uint32_t size = (uint32_t)first.size(), L = (uint32_t)first.coeff_modulus_size(), count = (uint32_t)rows[0].size();
    const std::size_t items = rows.size(), words = (std::size_t)size * L * context.poly_degree();
    const DeviceBuffer d_table = upload_table(table, st);
    DeviceBuffer out(items * words);
    for (std::size_t k = 0; k < items; k += kRowsPerCall)
        check_status(he_sum_ciphertexts(context.handle(), L, size, (uint32_t)std::min(kRowsPerCall, items - k), count,
                                        reinterpret_cast<const uint64_t *const *>(d_table.get()) + k * count, out.get() + k * words, st),
                     "he_sum_ciphertexts");
    return slices(std::move(out), items, size, first, first.scale());
}

// For every row of ciphertexts the sum of its products with `factors` (multiply, add_inplace term by term; size 3, not
// relinearised), all rows in one launch (up to kRowsPerCall).
std::vector<CAHELGPUCiphertext> multiply_sum(const CAHELGPUContext &context,
                                             const std::vector<std::vector<const CAHELGPUCiphertext *>> &rows,
                                             const std::vector<const CAHELGPUCiphertext *> &factors) {
    if (context.scheme() != cahel::scheme_type::ckks) throw std::logic_error("unsupported scheme");
    if (rows.empty()) return {};
    if (rows[0].empty() || !rows[0][0] || factors.empty() || !factors[0]) throw std::invalid_argument("no ciphertexts");
    const CAHELGPUCiphertext &first = *rows[0][0];
    auto check = [&](const CAHELGPUCiphertext *ct, double scale) {
        if (!ct || ct->size() != 2 || !ct->is_ntt_form()) throw std::invalid_argument("encrypted is not valid");
        if (ct->parms_id() != first.parms_id() || ct->chain_index() != first.chain_index())
            throw std::invalid_argument("encrypted parameter mismatch");
        if (ct->scale() != scale) throw std::invalid_argument("scale mismatch");
    };
    for (const CAHELGPUCiphertext *f : factors) check(f, first.scale());
    std::vector<const uint64_t *> table;
    for (const auto &row : rows) {
        if (row.size() != factors.size()) throw std::invalid_argument("rows differ in their number of ciphertexts");
        for (std::size_t k = 0; k < row.size(); k++) {
            check(row[k], first.scale());
            table.push_back(row[k]->data());
            table.push_back(factors[k]->data());
        }
    }
    // (multiply's condition on the product)
    const double scale = first.scale() * factors[0]->scale();
    if (scale <= 0 || static_cast<int>(std::log2(scale)) >= context.total_coeff_modulus_bit_count(first.chain_index()))
        throw std::invalid_argument("scale out of bounds");
    he_stream st = context.stream();
    const uint32_t L = (uint32_t)first.coeff_modulus_size(), count = (uint32_t)factors.size();
    const std::size_t items = rows.size(), words = 3 * (std::size_t)L * context.poly_degree();
    const DeviceBuffer d_table = upload_table(table, st);
    DeviceBuffer out(items * words);
    for (std::size_t k = 0; k < items; k += kRowsPerCall)
        check_status(he_multiply_sum(context.handle(), L, (uint32_t)std::min(kRowsPerCall, items - k), count,
                                     reinterpret_cast<const uint64_t *const *>(d_table.get()) + k * 2 * count, out.get() + k * words, st),
                     "he_multiply_sum");
    return slices(std::move(out), items, 3, first, scale);
}

namespace {

using Clients = std::vector<std::vector<const CAHELGPUCiphertext *>>;

// What the distances of `clients` and the key switches after them need; throws what the calls one by one would.
void check_clients(const CAHELGPUContext &context, const Clients &clients, const CAHELGPURelinKey &rlk, const CAHELGPUGaloisKey &glk) {
    if (context.scheme() != cahel::scheme_type::ckks) throw std::logic_error("unsupported scheme");
    if (clients.empty() || clients[0].empty()) throw std::invalid_argument("no ciphertexts");
    const CAHELGPUCiphertext &first = *clients[0][0];
    const std::size_t chunks = clients[0].size();
    for (const auto &client : clients) {
        if (client.size() != chunks) throw std::invalid_argument("clients differ in their number of chunks");
        for (const CAHELGPUCiphertext *ct : client) {
            if (!ct || ct->size() != 2 || !ct->is_ntt_form()) throw std::invalid_argument("encrypted is not valid");
            if (ct->parms_id() != first.parms_id() || ct->chain_index() != first.chain_index())
                throw std::invalid_argument("encrypted parameter mismatch");
            if (ct->scale() != first.scale()) throw std::invalid_argument("scale mismatch");
        }
    }
    if (rlk.parms_id() != context.key_parms_id() || glk.parms_id() != context.key_parms_id())
        throw std::invalid_argument("keys are not valid for encryption parameters");
    if (!context.using_keyswitching()) throw std::logic_error("keyswitching is not supported by the context");
    const std::size_t chain = first.chain_index();
    if (chain == 0) throw std::invalid_argument("key switching needs a data-level ciphertext");
    if (chain == context.max_chain_index()) throw std::invalid_argument("end of modulus switching chain reached");
}

// the chunks of both clients of a pair, side by side
void push_pair(std::vector<const uint64_t *> &table, const Clients &clients, const std::pair<std::size_t, std::size_t> &pr) {
    for (std::size_t c = 0; c < clients[0].size(); c++) {
        table.push_back(clients[pr.second][c]->data());
        table.push_back(clients[pr.first][c]->data());
    }
}

// Squared distances (d01 [items][2][L][N], d2 [items][L][N], like products of `first` with itself) relinearised and rescaled, then for
// every round acc += sum over the round's steps of rot(acc, step) (hoisted).  scale > 0 overrides the scale after the rescale
// (the reference's set_scale).  drop_levels > 0 switches the rescaled ciphertexts down by that many further limbs without
// scaling (mod_switch_to_next) before the slot sum, whose key switches then run over fewer limbs.
std::vector<CAHELGPUCiphertext> sum_of_slots(const CAHELGPUContext &context, const CAHELGPUCiphertext &first, const DeviceBuffer &d01,
                                             const DeviceBuffer &d2, uint32_t items, const CAHELGPURelinKey &rlk,
                                             const CAHELGPUGaloisKey &glk, const std::vector<std::vector<int>> &rounds, double scale,
                                             std::size_t drop_levels) {
    he_context *h = context.handle();
    he_stream st = context.stream();
    const std::size_t n = context.poly_degree(), K = context.size_p(), chain = first.chain_index();
    const uint32_t L = (uint32_t)first.coeff_modulus_size();

    // (1) relinearise + rescale
    auto rl = rlk.key_ptrs();
    if (rl.size() < (L + K - 1) / K) throw std::invalid_argument("key_poly_num != 2");
    DeviceBuffer ws(he_keyswitch_batch_workspace_words(h, L, items));
    DeviceBuffer acc((std::size_t)items * 2 * (L - 1) * n);
    check_status(he_keyswitch_rescale_batch(h, L, items, d2.get(), L, rl.data(), d01.get(), acc.get(), 0, ws.get(), st),
                 "he_keyswitch_rescale_batch");
    double out_scale = first.scale() * first.scale() / static_cast<double>(context.key_modulus()[L - 1].value());
    if (scale > 0) out_scale = scale;

    // (2) optional: drop limbs without scaling, the leading limbs of every polynomial move to a denser batch
    uint32_t L1 = L - 1;
    std::size_t out_chain = chain + 1;
    if (drop_levels) {
        if (drop_levels >= L1) throw std::invalid_argument("end of modulus switching chain reached");
        const uint32_t L2 = L1 - (uint32_t)drop_levels;
        DeviceBuffer dense((std::size_t)items * 2 * L2 * n);
        check_status(he_memcpy2d_d2d(dense.get(), (std::size_t)L2 * n * sizeof(uint64_t), acc.get(),
                                     (std::size_t)L1 * n * sizeof(uint64_t), (std::size_t)L2 * n * sizeof(uint64_t),
                                     (std::size_t)items * 2, st),
                     "he_memcpy2d_d2d");
        acc = std::move(dense);
        L1 = L2;
        out_chain += drop_levels;
    }

    // (3) the slot sum, one hoisted round at a time: acc += sum_s rot(acc, s)
    const std::size_t beta = (L1 + K - 1) / K;
    DeviceBuffer next(rounds.empty() ? 0 : (std::size_t)items * 2 * L1 * n);
    for (const auto &steps : rounds) {
        if (steps.empty()) throw std::invalid_argument("steps cannot be empty");
        std::vector<const uint64_t *> ptrs;
        std::vector<uint32_t> elts;
        for (int s : steps) {
            const long idx = context.find_galois_elt(context.get_elt_from_step(s));
            if (idx < 0 || (std::size_t)idx >= glk.relin_keys_.size())
                throw std::logic_error("Galois key not present in hoisting");
            auto key = glk.relin_keys_[(std::size_t)idx].key_ptrs();
            if (key.size() < beta) throw std::invalid_argument("key_poly_num must be 2 in hoisting");
            ptrs.insert(ptrs.end(), key.begin(), key.begin() + beta);
            elts.push_back(context.galois_elts()[(std::size_t)idx]);
        }
        check_status(he_hoisted_rotations_batch(h, L1, items, acc.get(), ptrs.data(), elts.data(), (uint32_t)elts.size(), 1,
                                                next.get(), ws.get(), st),
                     "he_hoisted_rotations_batch");
        std::swap(acc, next);
    }

    // (4) one ciphertext object per item, each a slice of the batch (no copies)
    std::vector<CAHELGPUCiphertext> out(items);
    const std::size_t words = 2 * (std::size_t)L1 * n;
    auto shared = std::make_shared<DeviceBuffer>(std::move(acc));
    for (uint32_t k = 0; k < items; k++) {
        CAHELGPUCiphertext &ct = out[k];
        ct.adopt(DeviceBuffer::slice(shared, k * words, words));
        ct.size_ = 2;
        ct.coeff_modulus_size_ = L1;
        ct.poly_modulus_degree_ = n;
        ct.chain_index_ = out_chain;
        ct.parms_id_ = context.parms_id_at(out_chain);
        ct.scale_ = out_scale;
        ct.is_ntt_form_ = true;
        ct.is_asymmetric_ = first.is_asymmetric_;
    }
    return out;
}

std::vector<CAHELGPUCiphertext> square_distances(const CAHELGPUContext &context, const Clients &clients,
                                                 const std::vector<std::pair<std::size_t, std::size_t>> &pairs,
                                                 const CAHELGPURelinKey &rlk, const CAHELGPUGaloisKey &glk,
                                                 const std::vector<std::vector<int>> &rounds, double scale, std::size_t drop_levels,
                                                 bool packed) {
    if (context.scheme() != cahel::scheme_type::ckks) throw std::logic_error("unsupported scheme");
    if (clients.empty() || clients[0].empty()) throw std::invalid_argument("no ciphertexts");
    if (pairs.empty()) return {};
    if (pairs.size() > 16384) throw std::invalid_argument("too many pairs");
    check_clients(context, clients, rlk, glk);
    for (const auto &pr : pairs)
        if (pr.first >= clients.size() || pr.second >= clients.size()) throw std::invalid_argument("pair out of range");
    const CAHELGPUCiphertext &first = *clients[0][0];
    const std::size_t n = context.poly_degree(), chunks = clients[0].size(), items = packed ? (pairs.size() + 1) / 2 : pairs.size();
    const uint32_t L = (uint32_t)first.coeff_modulus_size();
    he_stream st = context.stream();
    std::vector<const uint64_t *> table;
    table.reserve(2 * chunks * (pairs.size() + 1));
    for (const auto &pr : pairs) push_pair(table, clients, pr);
    if (packed && pairs.size() % 2) table.insert(table.end(), 2 * chunks, nullptr);
    const DeviceBuffer d_table = upload_table(table, st);
    DeviceBuffer d01(items * 2 * L * n), d2(items * L * n);
    check_status((packed ? he_pair_square_sum_packed : he_pair_square_sum)(context.handle(), L, (uint32_t)items, (uint32_t)chunks,
                                                                           reinterpret_cast<const uint64_t *const *>(d_table.get()),
                                                                           d01.get(), d2.get(), st),
                 "he_pair_square_sum");
    return sum_of_slots(context, first, d01, d2, (uint32_t)items, rlk, glk, rounds, scale, drop_levels);
}

}  // namespace

// For every (i, j) of `pairs`: the sum over chunks of (clients[j][c] - clients[i][c])^2 and its slot sum, as
// GPU_compute_pair_distance does per pair (lancelot-main-GPU/utils/byzantine_fl.py:173-321) -- here with one
// launch per stage for all pairs.
std::vector<CAHELGPUCiphertext> pair_square_distances(
    const CAHELGPUContext &context, const std::vector<std::vector<const CAHELGPUCiphertext *>> &clients,
    const std::vector<std::pair<std::size_t, std::size_t>> &pairs, const CAHELGPURelinKey &rlk,
    const CAHELGPUGaloisKey &glk, const std::vector<std::vector<int>> &rounds, double scale, std::size_t drop_levels) {
    return square_distances(context, clients, pairs, rlk, glk, rounds, scale, drop_levels, false);
}

// The same, two pairs per ciphertext: item k holds pair 2 k in the real and pair 2 k + 1 in the imaginary parts of its slots
// (the messages' slots are real), half the key switches.
std::vector<CAHELGPUCiphertext> packed_pair_distances(
    const CAHELGPUContext &context, const std::vector<std::vector<const CAHELGPUCiphertext *>> &clients,
    const std::vector<std::pair<std::size_t, std::size_t>> &pairs, const CAHELGPURelinKey &rlk,
    const CAHELGPUGaloisKey &glk, const std::vector<std::vector<int>> &rounds, double scale, std::size_t drop_levels) {
    return square_distances(context, clients, pairs, rlk, glk, rounds, scale, drop_levels, true);
}

// Every client's sum of squared distances to all others (its score), client 2 k in the real and client 2 k + 1 in the imaginary parts
// of item k: relinearisation, rescale and slot sum are linear, so the scores go through them instead of all pairs.
std::vector<CAHELGPUCiphertext> packed_distance_scores(
    const CAHELGPUContext &context, const std::vector<std::vector<const CAHELGPUCiphertext *>> &clients, const CAHELGPURelinKey &rlk,
    const CAHELGPUGaloisKey &glk, const std::vector<std::vector<int>> &rounds, double scale, std::size_t drop_levels) {
    check_clients(context, clients, rlk, glk);
    if (clients.size() > 32768) throw std::invalid_argument("too many clients");
    const CAHELGPUCiphertext &first = *clients[0][0];
    const std::size_t n = context.poly_degree(), items = (clients.size() + 1) / 2;
    const uint32_t L = (uint32_t)first.coeff_modulus_size(), chunks = (uint32_t)clients[0].size();
    he_stream st = context.stream();
    std::vector<const uint64_t *> table;
    for (const auto &client : clients)
        for (const CAHELGPUCiphertext *ct : client) table.push_back(ct->data());
    const DeviceBuffer d_table = upload_table(table, st);
    DeviceBuffer d01(items * 2 * L * n), d2(items * L * n);
    {
        DeviceBuffer ws(he_row_square_sums_workspace_words(context.handle(), L, chunks));
        check_status(he_row_square_sums_packed(context.handle(), L, (uint32_t)clients.size(), chunks,
                                               reinterpret_cast<const uint64_t *const *>(d_table.get()), d01.get(), d2.get(), ws.get(), st),
                     "he_row_square_sums_packed");
    }
    return sum_of_slots(context, first, d01, d2, (uint32_t)items, rlk, glk, rounds, scale, drop_levels);
}
