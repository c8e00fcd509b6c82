"""Two squared distances per ciphertext (real and imaginary parts of the slots) and row sums formed before the relinearisation:
the size-3 ciphertexts against the oracle's squares word for word, the scores and distances against float64."""
import numpy as np
import pytest

from gpu_util import DeviceArray, make_pair, rand_limbs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


def _monomial(p, L):
    """X^(N/2) in NTT form."""
    x = np.zeros((L, p.n), dtype=np.uint64)
    x[:, p.n // 2] = 1
    return p.ntt_fwd(x)


def _square(p, a, b):
    d = np.stack([p.sub(a[i], b[i]) for i in range(2)])
    return p.tensor(d, d)


def _total(p, terms):
    total = terms[0]
    for t in terms[1:]:
        total = np.stack([p.add(x, y) for x, y in zip(total, t)])
    return total


def _packed(p, sums, L):
    w = _monomial(p, L)
    out = []
    for k in range(0, len(sums), 2):
        item = sums[k]
        if k + 1 < len(sums):
            item = np.stack([p.mul_add(w, y, x) for x, y in zip(item, sums[k + 1])])
        out.append(item)
    return np.stack(out)


@pytest.mark.parametrize("logn,bits,L", [(9, [60, 40, 40, 60], 3), (10, [50, 50, 50], 2), (11, [60, 60, 30, 60], 3)])
@pytest.mark.parametrize("pairs,chunks", [(1, 1), (2, 3), (5, 17), (3, 33)])
def test_pairs_of_square_sums(oracle, capi, logn, bits, L, pairs, chunks):
    """he_pair_square_sum_packed; 17 and 33 terms cross the points where the running sums are reduced."""
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, 1)
    rng = np.random.default_rng(pairs + chunks)
    lib, h = capi.lib(), ctx.he_handle()
    host = [rand_limbs(p, rng, range(L), n_polys=2) for _ in range(5)]
    host[0][:], host[1][:] = 0, np.array([p.moduli[i] - 1 for i in range(L)], dtype=np.uint64)[None, :, None]   # differences of q - 1
    cts = [DeviceArray(capi, host=x) for x in host]
    which = rng.integers(0, 5, (pairs, chunks, 2))
    which[0, 0] = [1, 0]
    table = np.zeros((pairs + pairs % 2, chunks, 2), dtype=np.uint64)
    table[:pairs] = np.array([c.ptr for c in cts], dtype=np.uint64)[which]
    items, dtab = len(table) // 2, DeviceArray(capi, host=table)
    d01, d2 = DeviceArray(capi, shape=(items, 2, L, p.n)), DeviceArray(capi, shape=(items, 1, L, p.n))
    capi.check(lib.he_pair_square_sum_packed(h, L, items, chunks, dtab.ptr, d01.ptr, d2.ptr, None))
    got = np.concatenate([d01.numpy(), d2.numpy()], axis=1)
    sums = [_total(p, [_square(p, host[a], host[b]) for a, b in pair]) for pair in which]
    assert (got == _packed(p, sums, L)).all()
    assert lib.he_pair_square_sum_packed(h, L, 0, chunks, dtab.ptr, d01.ptr, d2.ptr, None) == -1
    assert lib.he_pair_square_sum_packed(h, L, items, 0, dtab.ptr, d01.ptr, d2.ptr, None) == -1


@pytest.mark.parametrize("items,chunks", [(1, 1), (3, 17), (16, 32), (16, 33)])
def test_square_sums_with_one_and_with_two_words_a_thread(oracle, capi, items, chunks):
    """he_pair_square_sum; up to 48 * 2^16 words a side, 512 terms of three limbs of 2^11, a thread takes one word, beyond two."""
    cahel, parms, ctx, p = make_pair(oracle, 11, [60, 60, 30, 60], 1)
    rng = np.random.default_rng(items + chunks)
    lib, h, L = capi.lib(), ctx.he_handle(), 3
    host = [rand_limbs(p, rng, range(L), n_polys=2) for _ in range(3)]
    host[0][:], host[1][:] = 0, np.array([p.moduli[i] - 1 for i in range(L)], dtype=np.uint64)[None, :, None]
    cts = [DeviceArray(capi, host=x) for x in host]
    which = rng.integers(0, 3, (items, chunks, 2))
    which[0, 0] = [1, 0]
    table = DeviceArray(capi, host=np.array([c.ptr for c in cts], dtype=np.uint64)[which])
    d01, d2 = DeviceArray(capi, shape=(items, 2, L, p.n)), DeviceArray(capi, shape=(items, 1, L, p.n))
    capi.check(lib.he_pair_square_sum(h, L, items, chunks, table.ptr, d01.ptr, d2.ptr, None))
    got = np.concatenate([d01.numpy(), d2.numpy()], axis=1)
    squares = {(a, b): _square(p, host[a], host[b]) for a in range(3) for b in range(3)}
    for k in range(items):
        assert (got[k] == _total(p, [squares[tuple(pair)] for pair in which[k]])).all(), k


@pytest.mark.parametrize("logn,bits,L", [(9, [60, 40, 40, 60], 3), (11, [60, 60, 30, 60], 3)])
@pytest.mark.parametrize("clients,chunks", [(1, 1), (2, 1), (3, 2), (5, 4), (17, 1), (2, 17)])
def test_row_sums_of_squares(oracle, capi, logn, bits, L, clients, chunks):
    """he_row_square_sums_packed against the sum of all squared differences of a row."""
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, 1)
    rng = np.random.default_rng(100 * clients + chunks)
    lib, h = capi.lib(), ctx.he_handle()
    host = [[rand_limbs(p, rng, range(L), n_polys=2) for _ in range(chunks)] for _ in range(clients)]
    host[0][0][:] = np.array([p.moduli[i] - 1 for i in range(L)], dtype=np.uint64)[None, :, None]
    cts = [[DeviceArray(capi, host=x) for x in row] for row in host]
    table = DeviceArray(capi, host=np.array([[c.ptr for c in row] for row in cts], dtype=np.uint64))
    items = (clients + 1) // 2
    d01, d2 = DeviceArray(capi, shape=(items, 2, L, p.n)), DeviceArray(capi, shape=(items, 1, L, p.n))
    ws = DeviceArray(capi, shape=(lib.he_row_square_sums_workspace_words(h, L, chunks),))
    capi.check(lib.he_row_square_sums_packed(h, L, clients, chunks, table.ptr, d01.ptr, d2.ptr, ws.ptr, None))
    got = np.concatenate([d01.numpy(), d2.numpy()], axis=1)
    sums = [_total(p, [_square(p, host[i][c], host[j][c]) for j in range(clients) for c in range(chunks)]) for i in range(clients)]
    assert (got == _packed(p, sums, L)).all()
    assert lib.he_row_square_sums_packed(h, L, clients, 0, table.ptr, d01.ptr, d2.ptr, ws.ptr, None) == -1


@pytest.mark.parametrize("clients,drop", [(2, 0), (3, 0), (4, 1), (5, 0)])
def test_packed_results_decode_to_the_distances(oracle, clients, drop):
    """packed_pair_distances and packed_distance_scores through decrypt_decode_complex_many: the float64 distances and their row sums
    within the budget of the encrypted round (set_scale after the rescale, noise of the key switches)."""
    from lancelot_amd import krum
    rng = np.random.default_rng(clients)
    updates = [rng.normal(0, 0.01, 5000).astype(np.float32) for _ in range(clients)]
    updates[-1] = updates[-1] * 5
    state = krum.gpu_init(krum.KrumConfig(log_n=13, modulus_bits=(60, 40, 40, 60), seed=5, sum_drop_levels=drop))
    c, ctx, cfg = state.cahel, state.context, state.config
    cts = krum.encrypt_updates(state, krum.split_updates(updates, state.slots))
    pairs = [(i, j) for i in range(clients) for j in range(i + 1, clients)]
    rounds = krum.rotate_sum_plan(12, cfg)
    want = krum.plain_distance_matrix(updates)

    def unpacked(packed, count):
        z = state.sk.decrypt_decode_complex_many(ctx, packed, state.slots, 3)
        assert z.shape == ((count + 1) // 2, 3) and z.dtype == np.complex128
        assert np.abs(z - z[:, :1]).max() < 1e-4 * np.abs(z).max()          # every slot holds the sum
        return np.stack([z[:, 0].real, z[:, 0].imag], axis=1).reshape(-1)[:count]

    dist = unpacked(c.packed_pair_distances(ctx, cts, pairs, state.rlk, state.glk, rounds, cfg.scale, drop), len(pairs))
    assert np.allclose(dist, [want[i, j] for i, j in pairs], rtol=2e-5)
    scores = unpacked(c.packed_distance_scores(ctx, cts, state.rlk, state.glk, rounds, cfg.scale, drop), clients)
    assert np.allclose(scores, want.sum(axis=0), rtol=2e-5)
    assert c.packed_pair_distances(ctx, cts, [], state.rlk, state.glk, rounds) == []
    with pytest.raises(ValueError, match="pair out of range"):
        c.packed_pair_distances(ctx, cts, [(0, clients)], state.rlk, state.glk, rounds)
    with pytest.raises(ValueError, match="no ciphertexts"):
        c.packed_distance_scores(ctx, [], state.rlk, state.glk, rounds)
