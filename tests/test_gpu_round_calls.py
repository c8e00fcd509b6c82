"""Calls of an aggregated Krum round that enqueue what follows before they wait: the same words and values as the calls one by one, which draw
the same randomness in the same order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SCALE = 2.0 ** 40


def state_of(seed, log_n):
    from lancelot_amd import krum
    return krum.gpu_init(krum.KrumConfig(log_n=log_n, seed=seed, sec_level="none"))


def encrypted(state, items, slots):
    values = np.random.default_rng(items).uniform(-1, 1, (items, slots))
    return values, state.encoder.encode_encrypt_many(state.context, state.pk, values, SCALE)


# (15: the values of one message are more than a block of the page-locked ring starts with; 9 messages go round the ring twice)
@pytest.mark.parametrize("log_n,items", [(13, 1), (13, 2), (13, 9), (15, 3)])
@pytest.mark.parametrize("size", [2, 3])
def test_decrypt_and_decode_one_after_the_other(log_n, items, size):
    a, b = state_of(5, log_n), state_of(5, log_n)
    out = []
    for state in (a, b):
        values, cts = encrypted(state, items, state.slots)
        if size == 3:
            cts = state.cahel.multiply_sum(state.context, [[ct] for ct in cts], cts[:1])
            assert all(ct.size() == 3 for ct in cts)
        if state is a:
            got = state.sk.decrypt_decode_each(state.context, state.encoder, cts)
            assert got.shape == (items * state.slots,)
            out.append(got.reshape(items, -1))
        else:
            out.append(np.stack([state.encoder.decode_array(state.context, state.sk.decrypt(state.context, ct)) for ct in cts]))
    assert (out[0] == out[1]).all()
    assert np.abs(out[0] - (values if size == 2 else values * values[0])).max() < 1e-3
    assert a.sk.decrypt_decode_each(a.context, a.encoder, []).size == 0


@pytest.mark.parametrize("length", [100, 1025])
def test_each_decoded_with_the_slot_count_of_the_encoder(length):
    """An encoder whose first message has fixed fewer slots than the ring has."""
    state = state_of(8, 13)
    values = np.random.default_rng(length).uniform(-1, 1, (3, length))
    cts = state.encoder.encode_encrypt_many(state.context, state.pk, values, SCALE)
    slots = 1 << (length - 1).bit_length()
    got = state.sk.decrypt_decode_each(state.context, state.encoder, cts)
    assert got.shape == (3 * slots,)
    got = got.reshape(3, slots)
    assert np.abs(got[:, :length] - values).max() < 1e-4 and np.abs(got[:, length:]).max() < 1e-4
    state.encoder.reset_sparse_slots()
    assert state.sk.decrypt_decode_each(state.context, state.encoder, cts[:1]).shape == (state.slots,)


@pytest.mark.parametrize("log_n,items,messages", [(13, 1, 2), (13, 5, 1), (15, 2, 17)])   # 17: five blocks of messages in a ring of four
def test_values_and_encryptions_at_once(log_n, items, messages):
    a, b = state_of(6, log_n), state_of(6, log_n)
    constants = np.zeros((messages, a.slots))
    constants[-1] = 1.0
    _, cts = encrypted(a, items, a.slots)
    got, got_cts = a.sk.decrypt_decode_complex_and_encrypt_many(a.context, cts, a.slots, 3, a.encoder, a.pk, constants, SCALE)
    _, cts = encrypted(b, items, b.slots)
    want = b.sk.decrypt_decode_complex_many(b.context, cts, b.slots, 3)
    want_cts = b.encoder.encode_encrypt_many(b.context, b.pk, constants, SCALE)
    assert (got == want).all() and len(got_cts) == messages
    assert all((x.to_numpy() == y.to_numpy()).all() for x, y in zip(got_cts, want_cts))
    # messages that are refused leave the ring as it was, and nothing held
    before = a.context
    with pytest.raises(ValueError):
        a.sk.decrypt_decode_complex_and_encrypt_many(a.context, got_cts[:1], a.slots, 1, a.encoder, a.pk, np.full((1, a.slots), 1e30), SCALE)
    for _ in range(5):
        assert a.sk.decrypt_decode_complex_many(before, got_cts[:1], a.slots, 1).shape == (1, 1)


@pytest.mark.parametrize("aggregate", [False, True])
def test_phases_of_a_round_add_up(aggregate):
    from lancelot_amd import krum
    state = state_of(7, 13)
    rng = np.random.default_rng(1)
    updates = [rng.normal(0, 0.01, 5000).astype(np.float32) for _ in range(4)]
    for _ in range(2):
        timings = (krum.gpu_krum_aggregate if aggregate else krum.gpu_krum)(updates, state=state)[2]
    phases = ["encode", "evaluate", "mask", "mask_multiply"] if aggregate else ["encode", "evaluate", "decrypt"]
    assert all(timings[k] > 0 for k in phases) and not state.marks
    assert timings["encode"] + timings["evaluate"] < timings["total"]


@pytest.mark.parametrize("aggregate", [False, True])
def test_no_time_of_a_round_is_in_two_phases(aggregate):
    """At 2^16 the mask's constants take the device some 50 us, which are the mask's and not the masked sum's as well.  15 us: by what the device
    reaches the last mark behind the clock that ends the round."""
    from lancelot_amd import krum
    state = state_of(9, 16)
    rng = np.random.default_rng(2)
    updates = [rng.normal(0, 0.01, 40000).astype(np.float32) for _ in range(4)]
    over = []
    for _ in range(9):
        timings = dict((krum.gpu_krum_aggregate if aggregate else krum.gpu_krum)(updates, state=state)[2])
        over.append(sum(timings.values()) - 2 * timings["total"])
    assert np.median(over[2:]) < 15e-6, (over, timings)
