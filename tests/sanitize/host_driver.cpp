// Runs the CPU-only parts of the host layer (number theory, BLAKE2b, table construction, record save / load, what waits for an
// encoding) under
// AddressSanitizer + UndefinedBehaviorSanitizer, against the host-memory mock of the device ABI (mock_device.cpp).
// Ends with a bounded, seeded loop that feeds damaged and random records to every load() entry: a parser may refuse
// a record (any std::exception), it may not crash or touch memory it does not own.  Exit code 0 = clean.
#include <cstdio>
#include <cstring>
#include <functional>
#include <random>
#include <sstream>
#include <stdexcept>
#include <string>
#include <vector>

#include "cahel.h"
#include "staging.h"

using namespace cahel;

extern const char *mock_failing;   // mock_device.cpp
extern bool mock_decodes;
extern std::function<void()> mock_meanwhile;

#define REQUIRE(cond)                                                        \
    do {                                                                     \
        if (!(cond)) {                                                       \
            std::fprintf(stderr, "REQUIRE failed: %s (line %d)\n", #cond, __LINE__); \
            return 1;                                                        \
        }                                                                    \
    } while (0)

template <typename T>
static std::string saved(const T &obj) {
    std::ostringstream os(std::ios::binary);
    obj.save(os);
    return os.str();
}

template <typename F>
static bool refuses(F &&f) {
    try {
        f();
    } catch (const std::exception &) {
        return true;
    }
    return false;
}

int main(int argc, char **argv) {
    const long rounds = argc > 1 ? std::atol(argv[1]) : 20000;

    // ---- number theory known answers (cahel-main/unittest/util/numth.cu, the reference's own vectors) ----
    uint64_t root = 0;
    REQUIRE(try_minimal_primitive_root(2, 11, root) && root == 10);
    REQUIRE(try_minimal_primitive_root(4, 29, root) && root == 12);
    REQUIRE(try_minimal_primitive_root(8, 1234565441ull, root) && root == 249725733ull);
    const auto primes = get_primes(8192, 44, 3);
    REQUIRE(primes.size() == 3 && primes[0] == 0xfffffffc001ull && primes[1] == 0xffffff6c001ull &&
            primes[2] == 0xfffffebc001ull);
    const auto digits = naf(-7);  // -8 + 1
    REQUIRE(!digits.empty());
    long sum = 0;
    for (int d : digits) sum += d;
    REQUIRE(sum == -7);
    // RFC 7693 appendix A: BLAKE2b-512("abc") starts ba 80 a5 3f
    unsigned char digest[64];
    blake2b(digest, 64, "abc", 3);
    REQUIRE(digest[0] == 0xba && digest[1] == 0x80 && digest[2] == 0xa5 && digest[3] == 0x3f && digest[63] == 0x23);

    // ---- context: every table of every level is built on the host and handed to the (mock) device ----
    const std::size_t n = 1024;
    EncryptionParameters parms(scheme_type::ckks);
    parms.set_poly_modulus_degree(n);
    parms.set_coeff_modulus(CoeffModulus::Create(n, {40, 30, 30, 30, 30, 30, 40, 40}));
    parms.set_special_modulus_size(2);   // six data limbs, three digits of two
    parms.set_galois_elts(get_elts_from_steps({1, -1, 0, 5}, n));
    CAHELGPUContext context(parms, true, sec_level_type::none);
    REQUIRE(context.size_q() == 6 && context.size_p() == 2);
    REQUIRE(context.limbs_at(1) == context.size_q());
    REQUIRE(context.parms_id_at(0) != context.parms_id_at(1));

    // ---- parameters record ----
    const std::string prec = saved(parms);
    {
        EncryptionParameters back;
        std::istringstream is(prec, std::ios::binary);
        back.load(is);
        REQUIRE(back.poly_modulus_degree() == n && back.coeff_modulus().size() == parms.coeff_modulus().size());
        REQUIRE(back.coeff_modulus()[3].value() == parms.coeff_modulus()[3].value());
    }

    // ---- plaintext and ciphertext records over the mock's host memory ----
    CAHELGPUPlaintext plain(context);
    plain.resize(context.limbs_at(1), n);
    plain.chain_index() = 1;
    plain.parms_id() = context.parms_id_at(1);
    plain.scale() = 1099511627776.0;
    for (std::size_t i = 0; i < context.limbs_at(1) * n; i++) plain.data()[i] = i * 2654435761u;
    CAHELGPUCiphertext cipher(context);
    cipher.resize(context, 2, 3);
    cipher.scale() = 1048576.0;
    for (std::size_t i = 0; i < 3 * context.limbs_at(2) * n; i++) cipher.data()[i] = i * 40503u + 7;
    const std::string ptrec = saved(plain), ctrec = saved(cipher);
    {
        CAHELGPUPlaintext back(context);
        std::istringstream is(ptrec, std::ios::binary);
        back.load(context, is);
        REQUIRE(back.chain_index() == 1 && back.scale() == plain.scale());
        REQUIRE(std::memcmp(back.data(), plain.data(), context.limbs_at(1) * n * 8) == 0);
        CAHELGPUCiphertext cback(context);
        std::istringstream cs(ctrec, std::ios::binary);
        cback.load(context, cs);
        REQUIRE(cback.size() == 3 && cback.chain_index() == 2 && cback.coeff_modulus_size() == context.limbs_at(2));
        REQUIRE(std::memcmp(cback.data(), cipher.data(), 3 * context.limbs_at(2) * n * 8) == 0);
        // copy / shrink / grow of a ciphertext keep the leading words and stay inside their block
        CAHELGPUCiphertext copy = cback;
        copy.resize(2, copy.coeff_modulus_size(), n);
        CAHELGPUCiphertext copy2 = copy;
        REQUIRE(copy2.size() == 2 && std::memcmp(copy2.data(), cipher.data(), 2 * context.limbs_at(2) * n * 8) == 0);
        copy.resize(3, copy.coeff_modulus_size(), n);
        REQUIRE(std::memcmp(copy.data(), cipher.data(), 2 * context.limbs_at(2) * n * 8) == 0);
    }
    // ---- device blocks: slices, shared owners, and a key switch that is deferred past its key's lifetime ----
    {
        auto parent = std::make_shared<DeviceBuffer>(4 * n);
        for (std::size_t i = 0; i < 4 * n; i++) parent->get()[i] = i;
        DeviceBuffer s1 = DeviceBuffer::slice(parent, n, n), s2 = DeviceBuffer::slice(parent, 3 * n, n);
        parent.reset();                       // the slices keep the block
        REQUIRE(s1.get()[0] == n && s2.get()[n - 1] == 4 * n - 1);
        REQUIRE(refuses([&] { DeviceBuffer::slice(s1.owner(), 4 * n, 1); }));
        DeviceBuffer own(n);
        for (std::size_t i = 0; i < n; i++) own.get()[i] = 7 * i;
        s1 = own;                             // copy-assign into a slice of the same size: the words land in the parent's block
        REQUIRE(s1.get()[5] == 35 && s1.owner());
        DeviceBuffer big(2 * n);
        for (std::size_t i = 0; i < 2 * n; i++) big.get()[i] = i + 1;
        s1.assign(big, 2 * n);                // larger than the slice: it takes a block of its own
        REQUIRE(s1.words() == 2 * n && !s1.owner() && s1.get()[2 * n - 1] == 2 * n);
        { DeviceBuffer last = std::move(s2); }   // the last slice to go frees the parent's block
        // a ciphertext whose block is a slice: growing it past the slice moves it to a block of its own
        auto batch = std::make_shared<DeviceBuffer>(4 * context.limbs_at(2) * n);
        for (std::size_t i = 0; i < batch->words(); i++) batch->get()[i] = 3 * i;
        CAHELGPUCiphertext part(context);
        part.adopt(DeviceBuffer::slice(batch, 2 * context.limbs_at(2) * n, 2 * context.limbs_at(2) * n));
        part.size_ = 2;
        part.coeff_modulus_size_ = context.limbs_at(2);
        part.poly_modulus_degree_ = n;
        batch.reset();
        const uint64_t first = part.data()[0];
        part.resize(3, part.coeff_modulus_size(), n);
        REQUIRE(part.data()[0] == first && !part.data_.owner());
        // make_shared keeps the words in place; owners outlive the object that made them
        DeviceBuffer key(2 * context.size_qp() * n);
        for (std::size_t i = 0; i < key.words(); i++) key.get()[i] = i ^ 0x55;
        const uint64_t *where = key.get();
        key.make_shared();
        REQUIRE(key.get() == where && key.owner() && key.owner().use_count() == 1);
        // a relinearisation deferred on `three` (as relinearize_inplace leaves it) while its key object goes away
        const std::size_t L2 = context.limbs_at(2);
        CAHELGPUCiphertext three(context);
        three.resize(context, 2, 3);
        for (std::size_t i = 0; i < 3 * L2 * n; i++) three.data()[i] = i;
        auto pending = std::make_shared<PendingKeySwitch>();
        pending->handle = context.handle();
        pending->limbs = (uint32_t)L2;
        std::vector<DeviceBuffer> digits((L2 + context.size_p() - 1) / context.size_p());
        for (auto &d : digits) {
            d.allocate(2 * context.size_qp() * n);
            std::memset(d.get(), 1, d.words() * 8);
            d.make_shared();
            pending->key_ptrs.push_back(d.get());
            pending->key_owners.push_back(d.owner());
        }
        three.size_ = 2;
        three.pending_ = pending;
        pending.reset();
        digits.clear();                       // the key is gone; the owners in the pending switch keep its blocks
        DeviceBuffer::trim_pool();
        REQUIRE(three.has_pending_key_switch() && three.size() == 2);
        CAHELGPUCiphertext after = three;     // a copy runs the switch on the source first
        REQUIRE(!three.has_pending_key_switch() && !after.has_pending_key_switch());
        REQUIRE(three.data()[0] == 1 && after.data()[1] == 2 && after.size() == 2);   // the mock adds one to (c0, c1)
        three.pending_ = std::make_shared<PendingKeySwitch>();   // overwritten as a whole: nothing runs
        three.adopt(DeviceBuffer(2 * L2 * n));
        REQUIRE(!three.has_pending_key_switch());
    }

    // ---- encodings that nothing has waited for: used at once on other lanes, through data(), copied, written again ----
    {
        CAHELGPUCKKSEncoder encoder(context);
        std::vector<double> values(n / 2), others(n / 2);
        for (std::size_t i = 0; i < n / 2; i++) {
            values[i] = 1.0 + 0.001 * (double)i;
            others[i] = -values[i];
        }
        const std::size_t L1 = context.limbs_at(1), bytes = n / 2 * sizeof(double);
        auto holds = [&](const uint64_t *words, const std::vector<double> &v) {
            for (std::size_t l = 0; l < L1; l++)
                if (std::memcmp(words + l * n, v.data(), bytes) != 0) return false;
            return true;
        };
        auto stale = [&](CAHELGPUPlaintext &p) {   // what the block holds before the encoding runs
            set_lane(0);
            p.resize(L1, n);
            std::memset(p.data_.get(), 0x77, p.data_.words() * 8);
        };
        CAHELGPUPlaintext p(context);
        stale(p);
        encoder.encode(context, values, 1099511627776.0, p);
        REQUIRE(!holds(p.data_.get(), values));        // (the mock's device has not run it)
        (void)p.lane_data();
        REQUIRE(!holds(p.data_.get(), values));        // on its own lane nobody waits
        set_lane(2);
        REQUIRE(holds(p.lane_data(), values));         // another lane
        stale(p);
        encoder.encode(context, values, 1099511627776.0, p);
        REQUIRE(holds(p.data(), values));              // data(): any stream
        stale(p);
        encoder.encode(context, values, 1099511627776.0, p);
        CAHELGPUPlaintext moved = std::move(p);
        set_lane(1);
        CAHELGPUPlaintext copy = moved;                // a copy made on another lane
        REQUIRE(holds(copy.data(), values));
        CAHELGPUPlaintext record(context);
        stale(moved);
        encoder.encode(context, values, 1099511627776.0, moved);
        set_lane(3);
        const std::string bytes_of = saved(moved);     // a record written on another lane
        std::istringstream is(bytes_of, std::ios::binary);
        record.load(context, is);
        REQUIRE(holds(record.data(), values));
        stale(moved);
        encoder.encode(context, values, 1099511627776.0, moved);
        const uint64_t *block = moved.data_.get();
        set_lane(4);
        encoder.encode(context, others, 1099511627776.0, moved);   // encoded again on another lane: in a block of that lane
        REQUIRE(moved.data_.get() != block && moved.data_.lane() == 4);
        set_lane(0);
        REQUIRE(holds(moved.lane_data(), others));
        stale(p);
        encoder.encode(context, others, 1099511627776.0, p);
        set_lane(5);
        p = copy;                                      // assigned to while its encoding runs: what is assigned stays
        synchronize_lanes();
        REQUIRE(holds(p.data_.get(), values));
        set_lane(0);
        // a decoding that fails behind its first launches: their writes come before the staging block is handed out again
        PinnedRing &ring = PinnedRing::of_thread();
        for (int i = 0; i < PinnedRing::kBlocks; i++) (void)ring.take(bytes);   // (nothing is left of the encodings above)
        REQUIRE(refuses([&] { encoder.decode_real(context, p, n / 2, others.data()); }));
        std::vector<double *> blocks;
        for (int i = 0; i < PinnedRing::kBlocks; i++) {
            blocks.push_back(static_cast<double *>(ring.take(bytes)));
            std::memcpy(blocks.back(), values.data(), bytes);
        }
        synchronize_lanes();
        for (double *b : blocks) REQUIRE(std::memcmp(b, values.data(), bytes) == 0);
    }

    // ---- batches: the random part is on its way before the messages are looked at.  One that fails behind it, wherever that is, leaves
    // the next one the stream ids that it would have drawn from without it. ----
    {
        set_lane(0);
        CAHELGPUCKKSEncoder encoder(context);
        CAHELGPUPublicKey pk(context);
        pk.pk_.resize(context, 0, 2);
        pk.gen_flag_ = true;
        const std::size_t L1 = context.limbs_at(1), items = 3, count = n / 2;
        std::vector<double> values(items * count, 0.5), huge(items * count, 1e30);
        std::vector<float> floats(items * count, 0.5f);
        const std::vector<const float *> rows{floats.data(), floats.data() + count, floats.data() + 2 * count};
        const double scale = 1099511627776.0;
        const uint64_t first = context.next_stream(0);
        auto refused = [&](const char *call, const std::vector<double> &v) {
            DeviceBuffer::trim_pool();
            { DeviceBuffer cts(items * 2 * L1 * n), ws(items); }   // (in the pool: what he_malloc is asked for is the staging between the two calls)
            mock_failing = call;
            const bool threw = refuses([&] { encoder.encode_encrypt_many(context, pk, v.data(), items, count, count, scale); });
            mock_failing = nullptr;
            return threw && context.next_stream(0) == first;
        };
        REQUIRE(refused("", huge));
        REQUIRE(refused("he_encrypt_begin", values));
        REQUIRE(refused("he_memcpy_h2d_async", values));
        REQUIRE(refused("he_ckks_encode_bounded", values));
        REQUIRE(refused("he_ckks_encode_batch", huge));
        REQUIRE(refused("he_encrypt_end", values));
        REQUIRE(refused("he_malloc", values));
        mock_failing = "he_memcpy_h2d_async";
        REQUIRE(refuses([&] { encoder.encode_encrypt_updates(context, pk, rows, count, scale); }) && context.next_stream(0) == first);
        mock_failing = nullptr;
        auto cts = encoder.encode_encrypt_many(context, pk, values.data(), items, count, count, scale);
        REQUIRE(cts.size() == items && context.next_stream(0) == first + 3 * items);
        synchronize_lanes();
        for (std::size_t k = 0; k < items; k++)
            REQUIRE(cts[k].data()[0] == cts[0].data()[0] && cts[k].data()[L1 * n] == first + 3 * k && cts[k].data()[2 * L1 * n - 1] == first + 3 * k);
        // floats: rows that end inside, at and right behind a message, and more than all staging blocks hold (the fifth one is the first
        // again, which its copy has to have left)
        const std::size_t one_block = (std::size_t(1) << 20) / sizeof(float);
        for (const std::size_t length : {std::size_t(1), count - 1, count, count + 1, 3 * count + 77, one_block + 5, 2 * one_block - 1}) {
            const std::size_t chunks = (length + count - 1) / count, clients = length > count ? 3 : 2;
            std::vector<std::vector<float>> updates(clients);
            std::vector<const float *> starts;
            for (std::size_t r = 0; r < clients; r++) {
                for (std::size_t i = 0; i < length; i++) updates[r].push_back(0.25f + 1e-6f * (float)((i * 7 + r) % 1000));
                starts.push_back(updates[r].data());
            }
            auto encrypted = encoder.encode_encrypt_updates(context, pk, starts, length, scale);
            REQUIRE(encrypted.size() == clients * chunks);
            synchronize_lanes();
            for (std::size_t k = 0; k < encrypted.size(); k++)
                for (std::size_t i = 0; i < count; i++) {
                    const std::size_t at = k % chunks * count + i;
                    double got;
                    std::memcpy(&got, encrypted[k].data() + i, sizeof(got));
                    REQUIRE(got == (at < length ? (double)updates[k / chunks][at] : 0.0));
                }
        }
        REQUIRE(encoder.encode_encrypt_updates(context, pk, {}, 5, scale).empty());
    }

    // ---- decryptions that are enqueued before the values in front are waited for: the values of every ciphertext in their place, in an array
    // of the slot count that the encoder had at the start, whatever becomes of that meanwhile ----
    {
        set_lane(0);
        CAHELGPUCKKSEncoder encoder(context);
        CAHELGPUSecretKey secret(parms);
        secret.gen_secretkey(context);
        const std::size_t L2 = context.limbs_at(2), few = n / 8;
        auto value = [](std::size_t k, std::size_t i) { return 1.0 + (double)k + 1e-6 * (double)i; };
        std::vector<CAHELGPUCiphertext> cts;
        std::vector<const CAHELGPUCiphertext *> ptrs;
        for (std::size_t k = 0; k < 7; k++) {
            cts.emplace_back(context);
            cts.back().resize(context, 2, 2);
            cts.back().scale() = 1048576.0;
            cts.back().is_ntt_form() = true;
            for (std::size_t i = 0; i < L2 * n; i++) {
                const double v = value(k, i);
                std::memcpy(cts.back().data() + i, &v, sizeof(v));
            }
        }
        for (const auto &ct : cts) ptrs.push_back(&ct);
        CAHELGPUPlaintext message(context);
        encoder.encode(context, std::vector<double>(few, 0.5), 1048576.0, message);   // fixes the slot count
        mock_decodes = true;
        auto decoded = [&](std::size_t slots) {
            std::vector<double> out(cts.size() * slots);
            secret.decrypt_decode_each(context, encoder, ptrs, slots, out.data());
            for (std::size_t k = 0; k < cts.size(); k++)
                for (std::size_t i = 0; i < slots; i++)
                    if (out[k * slots + i] != value(k, i)) return false;
            return true;
        };
        REQUIRE(encoder.decoded_slots() == few && decoded(few));
        {   // what is to be enqueued behind them comes once, in front of the last values
            std::vector<double> out(cts.size() * few, 0.0);
            int times = 0;
            bool early = false;
            secret.decrypt_decode_each(context, encoder, ptrs, few, out.data(), [&] {
                times++;
                early = out[(cts.size() - 1) * few] == 0.0;
            });
            REQUIRE(times == 1 && early && out.back() == value(cts.size() - 1, few - 1));
            secret.decrypt_decode_each(context, encoder, {}, few, nullptr, [&] { times++; });
            REQUIRE(times == 2);
            REQUIRE(refuses([&] { secret.decrypt_decode_each(context, encoder, ptrs, few, out.data(), [] { throw std::runtime_error("behind"); }); }));
        }
        {   // a decoding by itself: its workspace is for the slots that it decodes
            CAHELGPUPlaintext p(context);
            secret.decrypt(context, cts[1], p);
            std::vector<double> out(few);
            mock_meanwhile = [&] {
                encoder.reset_sparse_slots();
                CAHELGPUPlaintext q(context);
                encoder.encode(context, std::vector<double>(2 * few, 0.5), 1048576.0, q);
            };
            encoder.decode_real(context, p, few, out.data());
            REQUIRE(out[0] == value(1, 0) && out[few - 1] == value(1, few - 1) && encoder.decoded_slots() == 2 * few);
            mock_meanwhile = nullptr;
            encoder.reset_sparse_slots();
            encoder.encode(context, std::vector<double>(few, 0.5), 1048576.0, message);
        }
        int calls = 0;
        mock_meanwhile = [&] {
            if (++calls == 3) encoder.reset_sparse_slots();
        };
        REQUIRE(decoded(few) && encoder.decoded_slots() == n / 2);   // (a decoding fixes the full count)
        calls = 0;
        mock_meanwhile = [&] {
            if (++calls == 2) {
                encoder.reset_sparse_slots();
                CAHELGPUPlaintext p(context);
                encoder.encode(context, std::vector<double>(few, 0.5), 1048576.0, p);
            }
        };
        REQUIRE(decoded(n / 2) && encoder.decoded_slots() == few);
        mock_meanwhile = nullptr;
        mock_decodes = false;

        // a batch whose caller enqueues more work, staging blocks of its own with it, before the values are waited for, or fails there
        const std::size_t items = cts.size(), count = 5;
        std::vector<double> pairs(2 * items * count);
        PinnedRing &ring = PinnedRing::of_thread();
        secret.decrypt_decode_many(context, ptrs, few, count, pairs.data(), true, [&] {
            for (int i = 0; i < 2 * PinnedRing::kBlocks + 1; i++) {
                std::memset(ring.take(2 * items * count * sizeof(double)), 0x55, 2 * items * count * sizeof(double));
                ring.fence(current_stream());
            }
        });
        for (std::size_t i = 0; i < pairs.size(); i++) REQUIRE(pairs[i] == value(i / (2 * count), i / 2 % count));
        REQUIRE(refuses([&] { secret.decrypt_decode_many(context, ptrs, few, count, pairs.data(), true, [] { throw std::runtime_error("meanwhile"); }); }));
        secret.decrypt_decode_many(context, {}, few, count, pairs.data(), true, [&] { pairs[0] = -1.0; });
        REQUIRE(pairs[0] == -1.0);
    }

    // ---- blocks of the page-locked ring that are held: never handed out meanwhile, afterwards only when their work is done ----
    {
        set_lane(0);
        const he_stream stream = current_stream();
        const std::vector<double> written(16, 3.5);
        const std::size_t bytes = written.size() * sizeof(double);
        PinnedRing ring;
        auto started = [&] {   // a block that work on the stream will write
            void *block = ring.take(bytes);
            std::memset(block, 0, bytes);
            check_status(he_memcpy_h2d_async(block, written.data(), bytes, stream), "copy");
            return block;
        };
        auto handed_out = [&](const void *block, int times) {
            bool met = false;
            for (int i = 0; i < times; i++) met = ring.take(bytes) == block || met;
            return met;
        };
        auto done = [&](const void *block) { return std::memcmp(block, written.data(), bytes) == 0; };
        for (int turn = 0; turn < PinnedRing::kBlocks; turn++) {   // (the held blocks lie at every place of the ring)
            void *one = started();
            {
                PinnedRing::Held held(ring, stream);
                REQUIRE(!handed_out(one, 2 * PinnedRing::kBlocks) && !done(one));
                void *two = started();
                REQUIRE(two != one);
                PinnedRing::Held first(ring, stream);
                PinnedRing::Held second = std::move(first);
                REQUIRE(!handed_out(one, 2 * PinnedRing::kBlocks) && !handed_out(two, 2 * PinnedRing::kBlocks) && !done(two));
                second.wait();
                REQUIRE(done(two) && !handed_out(two, 2 * PinnedRing::kBlocks));
            }
            REQUIRE(done(one) && handed_out(one, PinnedRing::kBlocks));
            void *thrown = nullptr;
            REQUIRE(refuses([&] {
                thrown = started();
                PinnedRing::Held held(ring, stream);
                throw std::runtime_error("while a block is held");
            }));
            REQUIRE(!done(thrown));   // (nobody has waited)
            while (ring.take(bytes) != thrown) REQUIRE(!done(thrown));
            REQUIRE(done(thrown));    // its event was waited for before it was handed out
            (void)ring.take(bytes);
        }
    }

    // a record of another level, a truncated one and one with a wrong degree are refused
    REQUIRE(refuses([&] {
        std::string bad = ctrec.substr(0, ctrec.size() / 2);
        std::istringstream is(bad, std::ios::binary);
        CAHELGPUCiphertext c(context);
        c.load(context, is);
    }));

    // ---- bounded fuzz: damaged copies of the valid records and pure noise into every loader ----
    std::mt19937_64 rng(20250117);
    long refused = 0, accepted = 0;
    const std::string *seeds[3] = {&prec, &ptrec, &ctrec};
    for (long it = 0; it < rounds; it++) {
        std::string rec;
        const int kind = (int)(rng() % 4);
        if (kind == 3) {
            rec.resize(rng() % 200);
            for (auto &ch : rec) ch = (char)rng();
        } else {
            rec = *seeds[kind];
            // headers sit in the first bytes: damage mostly there, sometimes anywhere, sometimes truncate
            const int hits = 1 + (int)(rng() % 4);
            for (int h = 0; h < hits; h++) {
                const std::size_t span = (rng() & 3) ? std::min<std::size_t>(rec.size(), 96) : rec.size();
                rec[rng() % span] = (char)rng();
            }
            if ((rng() & 7) == 0) rec.resize(rng() % rec.size());
        }
        const int target = (int)(rng() % 6);
        const bool bad = refuses([&] {
            std::istringstream is(rec, std::ios::binary);
            switch (target) {
                case 0: { EncryptionParameters p; p.load(is); break; }
                case 1: { CAHELGPUPlaintext p(context); p.load(context, is); break; }
                case 2: { CAHELGPUCiphertext c(context); c.load(context, is); break; }
                case 3: { CAHELGPUPublicKey k(context); k.load(context, is); break; }
                case 4: { CAHELGPURelinKey k; k.load(context, is); break; }
                default: { CAHELGPUGaloisKey k(context); k.load(context, is); break; }
            }
        });
        (bad ? refused : accepted)++;
    }
    std::printf("host sanitize driver ok: %ld records refused, %ld accepted\n", refused, accepted);
    return 0;
}
