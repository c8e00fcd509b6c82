"""Updates of 32-bit floats, split, padded and widened on the device, against the host's splitting: the same ciphertexts word for word."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LOG_N = 13
SLOTS = 1 << (LOG_N - 1)


def _states():
    from lancelot_amd import krum
    return krum, [krum.gpu_init(krum.KrumConfig(log_n=LOG_N, seed=5)) for _ in range(2)]


@pytest.mark.parametrize("length", [1, SLOTS - 1, SLOTS, SLOTS + 1, 3 * SLOTS + 77])
@pytest.mark.parametrize("clients", [1, 3])
def test_float_updates_equal_split_updates(length, clients):
    krum, (a, b) = _states()
    rng = np.random.default_rng(length)
    updates = [rng.normal(0, 0.01, length).astype(np.float32) for _ in range(clients)]
    got = krum.encrypt_all(a, updates)
    want = krum.encrypt_updates(b, krum.split_updates(updates, b.slots))
    assert [len(row) for row in got] == [len(row) for row in want] == [-(-length // SLOTS)] * clients
    for row, other in zip(got, want):
        for x, y in zip(row, other):
            assert (x.to_numpy() == y.to_numpy()).all()
            assert x.scale() == y.scale() and x.chain_index() == y.chain_index()


def test_float_updates_of_other_forms():
    """More floats than a staging block holds, arrays that are not flat or not contiguous, other types, and what is refused."""
    krum, (a, b) = _states()
    rng = np.random.default_rng(1)
    base = [rng.normal(0, 0.01, (200, 1501)).astype(np.float32) for _ in range(2)]
    forms = [base[0].reshape(-1), np.asfortranarray(base[1])]     # (taken in C order, as the host's splitting takes them)
    got, want = krum.encrypt_all(a, forms), krum.encrypt_updates(b, krum.split_updates(base, b.slots))
    for row, other in zip(got, want):
        assert len(row) == len(other)
        for x, y in list(zip(row, other))[::37] + [(row[-1], other[-1])]:
            assert (x.to_numpy() == y.to_numpy()).all()
    doubles = [u.astype(np.float64) for u in base]
    assert len(krum.encrypt_all(a, doubles)[0]) == len(want[0])
    with pytest.raises(ValueError):
        krum.encrypt_all(a, [np.zeros(3, np.float32), np.zeros(4, np.float32)])
    with pytest.raises(ValueError):                               # (the encoding's own bound)
        krum.encrypt_all(a, [np.full(SLOTS, 1e30, np.float32)])
